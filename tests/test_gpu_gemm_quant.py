"""GPU parity: linear (fp32 / bf16), W8A16 GEMM and teeny-quant on the GPU."""
import numpy as np
import pytest

import teenygrad_amd as tg
from conftest import load_golden
from gpu_util import check_bf16, check_f32, stream_workspace
from quant_cases import KNOWN
from teenygrad_amd import _lib, kernels as K
from teenygrad_amd.dtypes import from_bf16, to_bf16

pytestmark = pytest.mark.gpu


def rb(a):
    return from_bf16(to_bf16(a))


@pytest.mark.parametrize("with_bias", [False, True])
def test_linear_f32_fixture(dev, orc, with_bias):
    x = load_golden("linear/input.bin").reshape(64, 64)
    w = load_golden("linear/weight.bin").reshape(48, 64)
    b = load_golden("linear/bias.bin")
    want = load_golden(f"linear/expected_{'with' if with_bias else 'no'}_bias.bin").reshape(64, 48)
    got = K.linear(dev.upload(x), dev.upload(w), dev.upload(b) if with_bias else None).to_host()
    np.testing.assert_allclose(got, want, rtol=0.02, atol=0.1)  # test_linear.rs:48-54
    check_f32(got, orc.linear(x, w, b if with_bias else None), "linear f32")


SMALL_GRID = [  # (M, N, K, K slices): 64 x 64 tiles with ragged edges, unsplit and in four slices of ragged K
    (65, 65, 64, 1), (130, 72, 272, 1), (1000, 520, 1040, 1), (100, 200, 2048, 4), (257, 130, 2064, 4),
    (70, 1000, 4112, 4), (1023, 1024, 4096, 1), (1100, 1000, 4624, 4),
    # K shared by two and four groups of waves (runs of k-tiles past K), on 64 x 64, 128 x 64 and 128 x 128 tiles
    (300, 520, 976, 1), (500, 600, 2064, 1), (450, 500, 2032, 1), (1100, 1000, 1104, 1), (2100, 1000, 1040, 1),
    # few rows whose narrow output and deep K stay on the tiles
    (64, 130, 4656, 4)]


@pytest.mark.parametrize("m,n,k,slices", SMALL_GRID)
@pytest.mark.parametrize("weights", ["int8", "bf16"])
def test_small_grids(dev, m, n, k, slices, weights):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    x = rb(rng.standard_normal((m, k), dtype=np.float32)).reshape(m, k)
    bias = rb(rng.standard_normal(n, dtype=np.float32))
    xb = dev.upload(to_bf16(x), tg.bf16)
    need = K.linear_workspace_size(m, n, k, tg.i8 if weights == "int8" else tg.bf16)
    if dev.info()["compute_units"] == 256:
        assert need == (slices * m * n * 4 if slices > 1 else 0), need
    if weights == "int8":
        q = rng.integers(-128, 128, (n, k)).astype(np.int8)
        scale = rng.uniform(0.005, 0.02, n).astype(np.float32)
        w, args = q.astype(np.float64) * scale[:, None], (dev.upload(q), dev.upload(scale), dev.upload(bias))
        fn = K.w8a16_linear
    else:
        w = rb(rng.standard_normal((n, k), dtype=np.float32)).reshape(n, k).astype(np.float64)
        args, fn = (dev.upload(to_bf16(w.astype(np.float32)), tg.bf16), dev.upload(to_bf16(bias), tg.bf16)), K.linear
    ref = x.astype(np.float64) @ w.T + bias
    # k fp32 sums, each within 2^-24 of at most sum |x| |w|, and the bf16 result
    bound = (k + 8) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + np.abs(bias)) + 2.0 ** -8 * np.abs(ref)
    for ws in {need, 0}:
        print(f"[small grid] M={m} N={n} K={k} {weights} workspace={ws}", flush=True)
        with stream_workspace(dev, ws):
            got = fn(xb, *args).to_host()
        err = np.abs(from_bf16(got).astype(np.float64).reshape(m, n) - ref)
        assert np.all(err <= bound), f"{np.max(err - bound)} beyond the bound"


SKINNY = [  # (M, N, K): row blocks of 16, column tails, K tails of 16 .. 64, fewer chunks than waves
    (1, 16, 16), (1, 1, 64), (7, 100, 528), (15, 33, 4096), (16, 48, 80), (17, 65, 1008), (32, 31, 2080), (33, 47, 1040),
    (64, 130, 2032), (2, 11008, 64),
    # two and four blocks of 16 columns per workgroup, the last one ragged (bf16 past 32 rows has no four)
    (19, 5130, 528), (31, 10250, 208), (40, 5130, 1040), (64, 10250, 144)]


@pytest.mark.parametrize("m,n,k", SKINNY)
@pytest.mark.parametrize("weights", ["int8", "bf16"])
def test_few_rows(dev, m, n, k, weights):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    x = rb(rng.standard_normal((m, k), dtype=np.float32)).reshape(m, k)
    bias = rb(rng.standard_normal(n, dtype=np.float32))
    xb = dev.upload(to_bf16(x), tg.bf16)
    print(f"[few rows] M={m} N={n} K={k} {weights}", flush=True)
    if weights == "int8":
        q = rng.integers(-128, 128, (n, k)).astype(np.int8)
        scale = rng.uniform(0.005, 0.02, n).astype(np.float32)
        w = q.astype(np.float64) * scale[:, None]
        got = K.w8a16_linear(xb, dev.upload(q), dev.upload(scale), dev.upload(bias)).to_host()
    else:
        w = rb(rng.standard_normal((n, k), dtype=np.float32)).reshape(n, k).astype(np.float64)
        got = K.linear(xb, dev.upload(to_bf16(w.astype(np.float32)), tg.bf16), dev.upload(to_bf16(bias), tg.bf16)).to_host()
    ref = x.astype(np.float64) @ w.T + bias
    # k fp32 sums, each within 2^-24 of at most sum |x| |w|, and the bf16 result
    bound = (k + 3) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + np.abs(bias)) + 2.0 ** -8 * np.abs(ref)
    err = np.abs(from_bf16(got).astype(np.float64).reshape(m, n) - ref)
    assert np.all(err <= bound), f"{np.max(err - bound)} beyond the bound"


@pytest.mark.parametrize("m,n,k", [
    # ragged K in rows padded to 16 bytes: K shared by two and four groups of waves on 64 x 64 tiles (with runs of
    # k-tiles past K), by two on 128 x 64 and 128 x 128 tiles
    (300, 130, 1001), (70, 200, 2051), (70, 72, 1985), (1100, 1000, 1101), (2100, 1000, 1039)])
def test_small_grids_padded_rows(dev, m, n, k):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    x, w = (rb(rng.standard_normal((r, k), dtype=np.float32)).reshape(r, k) for r in (m, n))
    ld = -(-k // 8) * 8
    pad = lambda a: np.pad(a, ((0, 0), (0, ld - k)), constant_values=np.nan)  # noqa: E731 (not to be read)
    xb, wb = (dev.upload(to_bf16(pad(a)), tg.bf16) for a in (x, w))
    y = tg.Buffer(tg.bf16, (m, n))
    print(f"[small grid] M={m} N={n} K={k} rows of {ld}", flush=True)
    tg.check(_lib.lib.teeny_linear_forward(xb.ptr, wb.ptr, None, y.ptr, m, n, k, ld, 1, ld, 1, n, 1, tg.bf16.code, None))
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    # k fp32 sums, each within 2^-24 of at most sum |x| |w|, and the bf16 result
    bound = (k + 8) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T) + 2.0 ** -8 * np.abs(ref)
    err = np.abs(from_bf16(y.to_host()).astype(np.float64).reshape(m, n) - ref)
    assert np.all(err <= bound), f"{np.max(err - bound)} beyond the bound"


def test_few_rows_widest(dev):
    # 2^27 columns: 2^32 threads at 512 for every 16 columns, past what a launch takes
    n, k, at = 2 ** 27, 16, [0, 1, 2 ** 26 - 1, 2 ** 26, 2 ** 27 - 9, 2 ** 27 - 1]
    x, q, scale = np.full((1, k), 0.5, np.float32), tg.Buffer(tg.i8, (n, k)), tg.Buffer(tg.f32, (n,))
    xb = dev.upload(to_bf16(x), tg.bf16)
    tg.check(_lib.lib.teeny_hip_memset(q.ptr, 1, q.nbytes, None))
    tg.check(_lib.lib.teeny_hip_memset(scale.ptr, 0, scale.nbytes, None))
    vals = np.arange(1, len(at) + 1, dtype=np.float32)
    for i, v in zip(at, vals):
        tg.check(_lib.lib.teeny_hip_memcpy_h2d(scale.ptr + 4 * i, np.float32([v]).ctypes.data, 4, None))
    print(f"[few rows] M=1 N={n} K={k} int8", flush=True)
    got = K.w8a16_linear(xb, q, scale).to_host().reshape(-1)
    np.testing.assert_array_equal(from_bf16(got[at]), 8 * vals)  # 16 times 0.5, times the scale
    assert np.count_nonzero(got) == len(at)


@pytest.mark.parametrize("k", [2 ** 30 + 48, 2 ** 31 - 64, 2 ** 31 - 16])
@pytest.mark.parametrize("weights", ["int8", "bf16"])
def test_few_rows_longest_k(dev, k, weights):
    # offsets past 2^31 bytes in bf16; ends of chunks and of groups of them past 2^31 products
    at = [0, 63, 2 ** 28 - 1, 2 ** 29, 2 ** 30 - 1, 2 ** 30, k - 33, k - 32, k - 16, k - 1]
    vals = np.arange(1, len(at) + 1, dtype=np.float32)
    x, y = tg.Buffer(tg.bf16, (1, k)), tg.Buffer(tg.bf16, (1, 1))
    w = tg.Buffer(tg.i8 if weights == "int8" else tg.bf16, (1, k))
    for buf in (x, w):
        tg.check(_lib.lib.teeny_hip_memset(buf.ptr, 0, buf.nbytes, None))
        for j, v in zip(at, vals):
            v = np.int8([v]) if buf.dtype == tg.i8 else to_bf16(np.float32([v]))
            tg.check(_lib.lib.teeny_hip_memcpy_h2d(buf.ptr + j * v.itemsize, v.ctypes.data, v.itemsize, None))
    print(f"[few rows] M=1 N=1 K={k} {weights}", flush=True)
    if weights == "int8":
        K.w8a16_linear(x, w, dev.upload(np.float32([0.5])), y=y)
    else:
        K.linear(x, w, y=y)
    ref = float(np.sum(vals * vals)) * (0.5 if weights == "int8" else 1.0)
    assert from_bf16(y.to_host()).reshape(-1)[0] == from_bf16(to_bf16(np.float32([ref])))[0]


F32_GEMM = [  # (M, N, K): tile edges, ragged vectors, k tails, splits, fewer than a 16-byte load spans
    (1, 5, 4), (3, 3, 3), (31, 65, 29), (33, 64, 31), (64, 64, 32), (65, 63, 33), (129, 127, 97), (4, 4, 161),
    (5, 1000, 700), (200, 72, 3001), (2300, 2200, 40)]


@pytest.mark.parametrize("m,n,k", F32_GEMM)
@pytest.mark.parametrize("xt,wt", [(False, False), (True, False), (False, True), (True, True)])
def test_linear_f32_strides(dev, m, n, k, xt, wt):
    # x and w along k or along their rows, rows padded by 3 (NaN between them), y transposed as well
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    x = rng.standard_normal((m, k), dtype=np.float32)
    w = rng.standard_normal((n, k), dtype=np.float32)
    b = rng.standard_normal(n, dtype=np.float32)

    def pad(a):
        out = np.full((a.shape[0], a.shape[1] + 3), np.nan, np.float32)
        out[:, :a.shape[1]] = a
        return out

    xb, wb = dev.upload(pad(x.T if xt else x)), dev.upload(pad(w.T if wt else w))
    bb = dev.upload(b)
    sx, sw = ((1, m + 3) if xt else (k + 3, 1)), ((1, n + 3) if wt else (k + 3, 1))
    ref = x.astype(np.float64) @ w.astype(np.float64).T + b
    # k fp32 products and sums: each within 2^-24 of a partial sum no larger than sum |x| |w| (+ |b|)
    bound = (k + 2) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + np.abs(b))
    for ws in (K.linear_workspace_size(m, n, k, tg.f32), 0):
        for yt in (False, True):
            print(f"[linear f32] M={m} N={n} K={k} xt={xt} wt={wt} yt={yt} workspace={ws}", flush=True)
            y = dev.upload(np.full((n, m) if yt else (m, n), np.nan, np.float32))
            with stream_workspace(dev, ws):
                tg.check(_lib.lib.teeny_linear_forward(xb.ptr, wb.ptr, bb.ptr, y.ptr, m, n, k, *sx, *sw,
                                                       *((1, m) if yt else (n, 1)), tg.f32.code, None))
                got = y.to_host()
            err = np.abs((got.T if yt else got).astype(np.float64) - ref)
            assert np.all(err <= bound), f"{np.max(err - bound)} beyond the bound"


@pytest.mark.parametrize("k", [2 ** 31 - 1, 2 ** 31 - 31, 2 ** 31 - 32, 2 ** 31 - 33])
def test_linear_f32_longest_k(dev, k):
    # the last chunk and the last of 512 slices end at, or would end past, the
    # largest 32-bit count; strides of 0 along k: every product is x[m] w[n]
    m = n = 4
    x, w, b = np.arange(1, 5, dtype=np.float32), np.float32([0.5, -1, 2, 4]), np.float32([1, 2, 3, 4])
    y = tg.Buffer(tg.f32, (m, n))
    xb, wb, bb = dev.upload(x), dev.upload(w), dev.upload(b)
    need = K.linear_workspace_size(m, n, k, tg.f32)
    assert need > 0
    print(f"[linear f32] K={k} workspace={need}", flush=True)
    with stream_workspace(dev, need):
        tg.check(_lib.lib.teeny_linear_forward(xb.ptr, wb.ptr, bb.ptr, y.ptr, m, n, k, 1, 0, 1, 0, n, 1,
                                               tg.f32.code, None))
        got = y.to_host().astype(np.float64)
    # four waves share a slice's 2^22 k's: their sums of 2^20 small multiples of 0.5 are exact, and
    # adding the 512 slices rounds by at most 512 * 2^-24 = 2^-15; a slice left out would show as 2^-9
    ref = float(k) * np.outer(x, w).astype(np.float64) + b
    assert np.all(np.abs(got - ref) <= 2.0 ** -12 * np.abs(ref)), got / ref


def with_scratch(dev, scratch, need, fn):
    """Runs fn() with no stream workspace, or with one of ``need`` bytes."""
    if scratch == "workspace":
        if need == 0:
            pytest.skip("no scratch plan at this shape: same path as scratch=none")
        with stream_workspace(dev, need):
            return fn()
    return fn()


@pytest.mark.parametrize("m,n,k", [(128, 128, 64), (200, 300, 136), (64, 48, 64), (33, 17, 70), (256, 512, 1000),
                                   (64, 256, 4096), (96, 200, 3100)])
@pytest.mark.parametrize("scratch", ["none", "workspace"])
def test_linear_bf16(dev, orc, m, n, k, scratch):
    # (64, 256, 4096) splits along K given a workspace; (33, 17, 70) and
    # (96, 200, 3100) have K % 8 != 0 and take the generic kernel
    rng = np.random.default_rng(m + n + k)
    x = rb(rng.standard_normal((m, k), dtype=np.float32))
    w = rb((rng.standard_normal((n, k), dtype=np.float32) / np.sqrt(k)).astype(np.float32))
    b = rb(rng.normal(0, 0.5, n).astype(np.float32))
    need = K.linear_workspace_size(m, n, k, tg.bf16)
    if dev.info()["compute_units"] == 256:
        assert (need > 0) == ((m, n, k) == (64, 256, 4096)), need
    got = with_scratch(dev, scratch, need, lambda: K.linear(
        dev.upload(to_bf16(x), tg.bf16), dev.upload(to_bf16(w), tg.bf16), dev.upload(to_bf16(b), tg.bf16)).to_host())
    check_bf16(got, orc.linear(x, w, b), "linear bf16")


@pytest.mark.parametrize("m,n,k", [(16421, 64, 128), (16384, 128, 256), (20000, 256, 64)])
def test_linear_bf16_stream(dev, orc, m, n, k):
    # M >= 16384 with K, N in {64, 128, 256}: the streaming kernel (B staged
    # once per workgroup, 32-row blocks per wave; 16421 and 20000 end in a
    # partial block)
    rng = np.random.default_rng(m + n + k)
    x = rb(rng.standard_normal((m, k), dtype=np.float32))
    w = rb((rng.standard_normal((n, k), dtype=np.float32) / np.sqrt(k)).astype(np.float32))
    b = rb(rng.normal(0, 0.5, n).astype(np.float32))
    assert K.linear_workspace_size(m, n, k, tg.bf16) == 0
    got = K.linear(dev.upload(to_bf16(x), tg.bf16), dev.upload(to_bf16(w), tg.bf16),
                   dev.upload(to_bf16(b), tg.bf16)).to_host()
    check_bf16(got, orc.linear(x, w, b), "linear bf16 stream")


@pytest.mark.parametrize("pad,offset", [(8, 0), (4, 0), (0, 8), (8, 16)])
def test_linear_bf16_stream_padded_rows(dev, orc, pad, offset):
    # the reference's LinearForward passes output_row_stride as stride_ym
    # (linear.rs:297-311), which may be padded; M = 16421 with K = 128, N = 64 is
    # a streaming shape.  Row pitch N + pad and y offset by `offset` bytes: the
    # streaming kernel takes 16-byte aligned rows (pad 8, offset 0 or 16), the
    # tiled kernels the rest; padding columns and the bytes before y stay untouched
    m, n, k = 16421, 64, 128
    print(f"[linear stream padded] ldy={n + pad} offset={offset}", flush=True)
    rng = np.random.default_rng(pad + offset)
    x = rb(rng.standard_normal((m, k), dtype=np.float32))
    w = rb((rng.standard_normal((n, k), dtype=np.float32) / np.sqrt(k)).astype(np.float32))
    xb, wb = dev.upload(to_bf16(x), tg.bf16), dev.upload(to_bf16(w), tg.bf16)
    ldy = n + pad
    sentinel = np.uint16(0x7FC1)  # a NaN pattern no result has
    ybuf = dev.upload(np.full(offset // 2 + m * ldy, sentinel, np.uint16), tg.bf16)
    tg.check(_lib.lib.teeny_linear_forward(xb.ptr, wb.ptr, None, ybuf.ptr + offset, m, n, k, k, 1, k, 1,
                                           ldy, 1, _lib.BF16, None))
    host = ybuf.to_host()
    assert np.all(host[:offset // 2] == sentinel)
    y = host[offset // 2:].reshape(m, ldy)
    assert np.all(y[:, n:] == sentinel)
    rows = np.concatenate([np.arange(0, 64), np.arange(0, m, 97), np.arange(m - 64, m)])
    check_bf16(y[rows, :n], orc.linear(x[rows], w), f"ldy={ldy} offset={offset}")


def tile_rows(m, tile, rng):
    """One row inside every `tile`-row block of [0, m), plus the first and last 64 rows."""
    starts = np.arange(0, m, tile, dtype=np.int64)
    pick = starts + (rng.random(starts.size) * np.minimum(tile, m - starts)).astype(np.int64)
    return np.unique(np.concatenate([np.arange(64), pick, np.arange(m - 64, m)]))


@pytest.mark.parametrize("m,n,k,pad", [(50000, 512, 128, 0), (50000, 512, 256, 8), (131072, 128, 384, 0),
                                       (40000, 1024, 512, 16), (12544, 1024, 256, 0), (12544, 512, 1024, 0),
                                       (20000, 384, 768, 8)])
def test_linear_bf16_persistent(dev, orc, m, n, k, pad):
    # >= 1.5 tiles of 128 x 128 per CU and 128 <= K <= 512 (<= 1024 for
    # N <= 1024): the persistent LDS-DMA kernel (one DMA ring per workgroup
    # across its tiles; 50000, 40000 and 20000 end in a partial row tile,
    # K = 128 is shorter than the ring; 12544 x 512 x 1024 and 20000 x 384
    # x 768 run 1.5-1.8 tiles per CU, some workgroups one tile).
    # Output rows padded to N + pad: the padding columns stay untouched.
    # One row of every 128-row tile (each workgroup's every tile) vs the oracle.
    print(f"[linear persistent] m={m} n={n} k={k} ldy={n + pad}", flush=True)
    rng = np.random.default_rng(m + n + k)
    x = rb(rng.standard_normal((m, k), dtype=np.float32))
    w = rb((rng.standard_normal((n, k), dtype=np.float32) / np.sqrt(k)).astype(np.float32))
    b = rb(rng.normal(0, 0.5, n).astype(np.float32))
    assert K.linear_workspace_size(m, n, k, tg.bf16) == 0
    xb, wb, bb = dev.upload(to_bf16(x), tg.bf16), dev.upload(to_bf16(w), tg.bf16), dev.upload(to_bf16(b), tg.bf16)
    ldy = n + pad
    sentinel = np.uint16(0x7FC1)
    ybuf = dev.upload(np.full(m * ldy, sentinel, np.uint16), tg.bf16)
    tg.check(_lib.lib.teeny_linear_forward(xb.ptr, wb.ptr, bb.ptr, ybuf.ptr, m, n, k, k, 1, k, 1, ldy, 1,
                                           _lib.BF16, None))
    y = ybuf.to_host().reshape(m, ldy)
    assert np.all(y[:, n:] == sentinel)
    assert np.all(np.isfinite(from_bf16(y[:, :n])))
    rows = tile_rows(m, 128, rng)
    check_bf16(y[rows, :n], orc.linear(x[rows], w, b), f"{rows.size} sampled rows")


def test_linear_bf16_large_tile(dev, orc):
    # 4096 x 512 x 4096: 256 x 256 tiles fill the chip -> large-tile kernel;
    # rows 0..31 and the last 32 rows against the oracle
    m, k, n = 4096, 512, 4096
    rng = np.random.default_rng(4096)
    x = rb(rng.standard_normal((m, k), dtype=np.float32))
    w = rb(rng.normal(0, 0.05, (n, k)).astype(np.float32))
    y = K.linear(dev.upload(to_bf16(x), tg.bf16), dev.upload(to_bf16(w), tg.bf16)).to_host()
    for lo, hi in ((0, 32), (m - 32, m)):
        check_bf16(y[lo:hi], orc.linear(x[lo:hi], w), f"rows {lo}..{hi}")


def test_linear_bf16_strided_generic(dev, orc):
    # x given as a transposed view (stride_xk = M): the generic kernel path
    rng = np.random.default_rng(3)
    m, n, k = 40, 24, 56
    xt = rb(rng.standard_normal((k, m), dtype=np.float32))  # x = xt^T
    w = rb((rng.standard_normal((n, k), dtype=np.float32) / 8).astype(np.float32))
    xb, wb = dev.upload(to_bf16(xt), tg.bf16), dev.upload(to_bf16(w), tg.bf16)
    y = tg.Buffer(tg.bf16, (m, n))
    tg.check(_lib.lib.teeny_linear_forward(xb.ptr, wb.ptr, None, y.ptr, m, n, k, 1, m, k, 1, n, 1,
                                           _lib.BF16, None))
    check_bf16(y.to_host(), orc.linear(np.ascontiguousarray(xt.T), w), "strided linear")


def quantized_weight(orc, rng, n, k):
    wf = rng.normal(0, 0.02, (n, k)).astype(np.float32)
    q, s, _, _ = orc.quantize_affine(wf, [n, k], "channel", 0)
    return q.reshape(n, k), s


@pytest.mark.parametrize("m,n,k,act", [(100, 200, 256, None), (256, 384, 512, "silu"),
                                       (64, 64, 4096, "gelu"), (37, 70, 40, "relu"), (5, 9, 48, None),
                                       (600, 96, 128, "relu"), (530, 200, 64, None)])
@pytest.mark.parametrize("scratch", ["none", "workspace"])
def test_w8a16_small(dev, orc, m, n, k, act, scratch):
    # (37, 70, 40) and (5, 9, 48): K % 16 != 0 -> generic kernel; others MFMA;
    # given a workspace, (64, 64, 4096) splits along K
    rng = np.random.default_rng(m * n + k)
    x = rb(rng.standard_normal((m, k), dtype=np.float32))
    q, s = quantized_weight(orc, rng, n, k)
    bias = rng.normal(0, 0.1, n).astype(np.float32)
    need = K.linear_workspace_size(m, n, k, tg.i8)
    if dev.info()["compute_units"] == 256:
        assert (need > 0) == ((m, n, k) == (64, 64, 4096)), need
    got = with_scratch(dev, scratch, need, lambda: K.w8a16_linear(
        dev.upload(to_bf16(x), tg.bf16), dev.upload(q), dev.upload(s), dev.upload(bias), act=act).to_host())
    ref = orc.w8a16_linear(x, q, s, bias)
    if act is not None:
        ref = getattr(orc, act)(ref)
    check_bf16(got, ref, "w8a16")


_CONFIG_REF = {}


@pytest.mark.parametrize("scratch", ["none", "workspace"])
@pytest.mark.parametrize("k,n", [(4096, 11008), (11008, 4096)])
def test_w8a16_config(dev, orc, k, n, scratch):
    # M = 4096 tokens; weights N(0, 0.02) quantised per output channel on the GPU
    # (bit-exact with the oracle); the whole [M, N] output against the oracle
    m = 4096
    rng = np.random.default_rng(0x7EE70005 + k)
    x = rb(rng.standard_normal((m, k), dtype=np.float32))
    wf = rng.normal(0, 0.02, (n, k)).astype(np.float32)
    print(f"[w8a16 config] M={m} K={k} N={n} scratch={scratch}", flush=True)
    qg, sg, zg, _ = K.quantize_affine(dev.upload(wf), [n, k], "channel", 0)
    q, s, z, _ = orc.quantize_affine(wf, [n, k], "channel", 0)
    np.testing.assert_array_equal(qg.to_host().reshape(-1), q)
    np.testing.assert_array_equal(sg.to_host(), s)
    # the 256 x 256 LDS-DMA kernel converts the int8 weights in registers
    # ahead of each MFMA: no scratch, and an attached workspace changes nothing
    need = K.linear_workspace_size(m, n, k, tg.i8)
    assert need == 0, need
    need = 1 << 20
    y = with_scratch(dev, scratch, need, lambda: K.w8a16_linear(dev.upload(to_bf16(x), tg.bf16), qg, sg).to_host())
    if (k, n) not in _CONFIG_REF:  # one oracle run per shape, shared by both scratch modes
        _CONFIG_REF.clear()
        wdeq = orc.dequantize_affine(q, s, None, [n, k], "channel", 0)
        _CONFIG_REF[(k, n)] = orc.linear(x, wdeq)
    ref = _CONFIG_REF[(k, n)]
    for lo in range(0, m, 1024):
        check_bf16(y[lo:lo + 1024], ref[lo:lo + 1024], f"rows {lo}..{lo + 1023}")


# ── teeny-quant on the GPU: bit-exact with the oracle ──────────────────────


@pytest.mark.parametrize("case", KNOWN, ids=[c[0] for c in KNOWN])
def test_quant_known_answers(dev, case):
    name, data, shape, gran, axis, gs, sym, bits, want_q, want_s, want_z = case
    q, s, z, g = K.quantize_affine(dev.upload(np.array(data, np.float32)), shape, gran, axis, gs,
                                   sym, bits, want_groups=True)
    np.testing.assert_array_equal(q.to_host().reshape(-1), np.array(want_q, np.int8))
    np.testing.assert_array_equal(s.to_host(), np.array(want_s, np.float32))
    np.testing.assert_array_equal(z.to_host(), np.array(want_z, np.int32))


RANDOM = [((64, 96), "channel", 0, 1, True, 8), ((64, 96), "channel", 1, 1, True, 8),
          ((64, 96), "tensor", 0, 1, False, 8), ((8, 5, 33), "group", 2, 8, True, 8),
          ((8, 5, 33), "group", 1, 2, False, 4), ((8, 5, 33), "group", 0, 3, True, 4),
          ((256, 3, 3, 256), "channel", 0, 1, True, 8), ((3000, 17), "channel", 0, 1, False, 8),
          # contiguous groups split over several workgroups (rows of 40000 and a
          # 100003-element tensor), groups of 7 and 5 (quads straddling two
          # groups), and groups of 3 (the per-element kernel)
          ((5, 40000), "channel", 0, 1, True, 8), ((100003,), "tensor", 0, 1, False, 8),
          ((33, 7), "channel", 0, 1, True, 8), ((9, 5), "channel", 0, 1, False, 4), ((6, 3), "channel", 0, 1, True, 8)]


@pytest.mark.parametrize("shape,gran,axis,gs,sym,bits", RANDOM)
def test_quant_vs_oracle(dev, orc, shape, gran, axis, gs, sym, bits):
    x = np.random.default_rng(len(shape) + axis).normal(0, 0.02, shape).astype(np.float32)
    x.reshape(-1)[::5] *= 3.0
    q, s, z, g = K.quantize_affine(dev.upload(x), shape, gran, axis, gs, sym, bits, want_groups=True)
    oq, os_, oz, og = orc.quantize_affine(x, shape, gran, axis, gs, sym, bits)
    np.testing.assert_array_equal(g.to_host(), og)
    np.testing.assert_array_equal(s.to_host(), os_)
    np.testing.assert_array_equal(z.to_host(), oz)
    np.testing.assert_array_equal(q.to_host().reshape(-1), oq)
    d = K.dequantize_affine(q, s, z, shape, gran, axis, gs).to_host()
    np.testing.assert_array_equal(d.reshape(-1), orc.dequantize_affine(oq, os_, oz, shape, gran, axis, gs).reshape(-1))


def test_quant_empty_groups(dev):
    # shape [0, 4], per-channel over axis 1: 4 groups, no elements -> scale 1, zp = qmin (asym)
    ng = K.quant_num_groups([0, 4], "channel", 1)
    assert ng == 4
    x = tg.Buffer(tg.f32, (0,))
    q, s, z, _ = K.quantize_affine(x, [0, 4], "channel", 1, symmetric=False)
    np.testing.assert_array_equal(s.to_host(), np.ones(4, np.float32))
    np.testing.assert_array_equal(z.to_host(), np.full(4, -128, np.int32))
