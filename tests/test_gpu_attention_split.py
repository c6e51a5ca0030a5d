"""bf16 attention with few queries per K/V head (the keys shared out over waves
and, given a workspace, over workgroups) against the CPU oracle."""
import numpy as np
import pytest

import teenygrad_amd as tg
from gpu_util import check_bf16, stream_workspace
from teenygrad_amd import kernels as K
from teenygrad_amd.dtypes import from_bf16, to_bf16

pytestmark = pytest.mark.gpu

CASES = [  # batch, q_heads, kv_heads, nq, nk, d: rows of a column block, tile and range edges
    (1, 1, 1, 1, 1, 128), (2, 2, 1, 1, 31, 64), (1, 8, 2, 1, 129, 128), (3, 4, 4, 2, 512, 64),
    (1, 32, 4, 5, 1000, 128), (2, 8, 1, 4, 257, 64), (1, 3, 1, 32, 700, 128), (1, 2, 2, 31, 2049, 64),
    (2, 16, 2, 1, 3001, 128), (1, 1, 1, 32, 33, 128),
    # both sides of the plan's lines on a full chip (256 CUs): blocks as many as heads, 5 to 8 heads (400, 800 of
    # them), 7 to 8; one tile of keys per wave
    (36, 16, 2, 32, 70, 128), (20, 32, 4, 20, 70, 128), (40, 32, 4, 20, 70, 128), (10, 64, 8, 28, 70, 64),
    (80, 8, 2, 32, 40, 64), (65, 4, 4, 17, 64, 128), (65, 4, 4, 17, 65, 128), (1, 4, 2, 33, 128, 128),
    (1, 4, 2, 33, 129, 128), (1, 8, 1, 1, 128, 128),
    (32, 8, 1, 32, 200, 128), (31, 8, 1, 32, 200, 128), (32, 4, 2, 64, 140, 128)]


@pytest.mark.parametrize("b,hq,hkv,nq,nk,d", CASES)
@pytest.mark.parametrize("scale", [None, -0.1, 0.0])
def test_few_queries(dev, orc, b, hq, hkv, nq, nk, d, scale):
    rng = np.random.default_rng(nq + 3 * nk + d)
    q, k, v = (from_bf16(to_bf16(rng.standard_normal((n, m, d), dtype=np.float32)))
               for n, m in ((b * hq, nq), (b * hkv, nk), (b * hkv, nk)))
    scale = 1 / np.sqrt(d) if scale is None else scale
    oo, ol = orc.flash_attention(q, *(np.repeat(a, hq // hkv, axis=0) for a in (k, v)), scale)
    bufs = [dev.upload(to_bf16(a), tg.bf16) for a in (q, k, v)]
    for ws in (K.attention_workspace_size(b, hq, hkv, nq, nk, d), 0):
        print(f"[attn split] b={b} hq={hq} hkv={hkv} nq={nq} nk={nk} d={d} scale={scale} workspace={ws}", flush=True)
        lse = tg.Buffer(tg.f32, (b * hq, nq))
        with stream_workspace(dev, ws):
            o = K.attention(*bufs, hq, hkv, scale, lse=lse).to_host()
        check_bf16(o, oo, "o")
        assert np.max(np.abs(lse.to_host() - ol)) < 1e-3


@pytest.mark.parametrize("b,hq,hkv,nq,nk,d", [
    # rows of one and of several heads in a block, ranges past the last query, keys that no query sees
    (1, 4, 2, 20, 300, 128), (2, 2, 2, 33, 33, 64), (1, 6, 1, 50, 70, 64), (1, 1, 1, 1500, 1400, 128),
    (1, 2, 2, 700, 1100, 64), (3, 4, 1, 129, 129, 128)])
def test_causal(dev, orc, b, hq, hkv, nq, nk, d):
    rng = np.random.default_rng(nq + 3 * nk + d)
    q, k, v = (from_bf16(to_bf16(rng.standard_normal((n, m, d), dtype=np.float32)))
               for n, m in ((b * hq, nq), (b * hkv, nk), (b * hkv, nk)))
    oo, ol = orc.flash_attention(q, *(np.repeat(a, hq // hkv, axis=0) for a in (k, v)), 1 / np.sqrt(d), True)
    bufs = [dev.upload(to_bf16(a), tg.bf16) for a in (q, k, v)]
    for ws in (K.attention_workspace_size(b, hq, hkv, nq, nk, d, True), 0):
        print(f"[attn split] causal b={b} hq={hq} hkv={hkv} nq={nq} nk={nk} d={d} workspace={ws}", flush=True)
        lse = tg.Buffer(tg.f32, (b * hq, nq))
        with stream_workspace(dev, ws):
            o = K.attention(*bufs, hq, hkv, causal=True, lse=lse).to_host()
        check_bf16(o, oo, "o")
        assert np.max(np.abs(lse.to_host() - ol)) < 1e-3


def test_rows_past_the_keys(dev, orc):
    # the head after this one holds no numbers: its rows are read only as padding
    q, k, v = (from_bf16(to_bf16(np.random.default_rng(1).standard_normal((2, n, 128), dtype=np.float32)))
               for n in (1, 300, 300))
    k[1], v[1] = np.nan, np.inf
    oo, _ = orc.flash_attention(q[:1], k[:1], v[:1])
    with stream_workspace(dev, K.attention_workspace_size(2, 1, 1, 1, 300, 128)):
        o = K.flash_attention(*(dev.upload(to_bf16(a), tg.bf16) for a in (q, k, v))).to_host()
    check_bf16(o[:1], oo, "o")
    assert np.isnan(from_bf16(o[1])).all()


@pytest.mark.parametrize("b,hq,hkv,n,cut,d", [
    # `cut`: the first row that holds no numbers, at a 64-key tile's edge; the rows before it see no key from there on
    (1, 2, 1, 200, 128, 128), (1, 8, 2, 100, 64, 64), (2, 6, 2, 77, 64, 64), (1, 4, 1, 333, 256, 128)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_causal_rows_without_numbers(dev, orc, b, hq, hkv, n, cut, d, bad):
    # a padded batch: early queries of every head of a group, the ones that
    # follow another head's last query in a column block among them
    rng = np.random.default_rng(n + d)
    q, k, v = (from_bf16(to_bf16(rng.standard_normal((m, n, d), dtype=np.float32))) for m in (b * hq, b * hkv, b * hkv))
    oo, ol = orc.flash_attention(q, *(np.repeat(a, hq // hkv, axis=0) for a in (k, v)), 1 / np.sqrt(d), True)
    k[:, cut:], v[:, cut:] = bad, bad
    bufs = [dev.upload(to_bf16(a), tg.bf16) for a in (q, k, v)]
    for ws in (K.attention_workspace_size(b, hq, hkv, n, n, d, True), 0):
        print(f"[attn split] masked b={b} hq={hq} hkv={hkv} n={n} cut={cut} d={d} bad={bad} workspace={ws}", flush=True)
        lse = tg.Buffer(tg.f32, (b * hq, n))
        with stream_workspace(dev, ws):
            o = K.attention(*bufs, hq, hkv, causal=True, lse=lse).to_host()
        check_bf16(o[:, :cut], oo[:, :cut], "o")
        assert np.max(np.abs(lse.to_host()[:, :cut] - ol[:, :cut])) < 1e-3


@pytest.mark.parametrize("b,hq,hkv,nq,nk,d", [
    (1, 8, 2, 64, 4096, 128), (1, 1, 1, 5, 16384, 64), (2, 8, 8, 100, 2048, 64), (1, 2, 1, 128, 1100, 128), (1, 4, 2, 700, 3000, 64)])
def test_causal_keys_past_the_queries(dev, orc, b, hq, hkv, nq, nk, d):
    # keys that no query sees take no part: no numbers there, and no share of the plan
    assert K.attention_workspace_size(b, hq, hkv, nq, nk, d, True) == K.attention_workspace_size(b, hq, hkv, nq, nq, d, True)
    rng = np.random.default_rng(nq + nk)
    q, k, v = (from_bf16(to_bf16(rng.standard_normal((m, n, d), dtype=np.float32)))
               for m, n in ((b * hq, nq), (b * hkv, nk), (b * hkv, nk)))
    oo, ol = orc.flash_attention(q, *(np.repeat(a[:, :nq], hq // hkv, axis=0) for a in (k, v)), 1 / np.sqrt(d), True)
    cut = -(-nq // 64) * 64  # the edge of the last queries' own tile
    k[:, cut:], v[:, cut:] = np.nan, np.nan
    bufs = [dev.upload(to_bf16(a), tg.bf16) for a in (q, k, v)]
    for ws in {K.attention_workspace_size(b, hq, hkv, nq, nk, d, True), 0}:
        print(f"[attn split] causal b={b} hq={hq} hkv={hkv} nq={nq} nk={nk} d={d} workspace={ws}", flush=True)
        lse = tg.Buffer(tg.f32, (b * hq, nq))
        with stream_workspace(dev, ws):
            o = K.attention(*bufs, hq, hkv, causal=True, lse=lse).to_host()
        check_bf16(o, oo, "o")
        assert np.max(np.abs(lse.to_host() - ol)) < 1e-3
