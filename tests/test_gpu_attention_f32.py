"""Attention with fp32 products on the fp32 matrix cores, forward and backward,
against the CPU oracle and 64-bit results: tile and share edges, both launch
shapes, grouped heads, bf16 operands, and masked rows that hold no numbers."""
import math

import numpy as np
import pytest

import teenygrad_amd as tg
from gpu_util import check_bf16, check_f32, stream_workspace
from teenygrad_amd import kernels as K
from teenygrad_amd.dtypes import from_bf16, to_bf16

pytestmark = pytest.mark.gpu


def reference(q, k, v, do, causal, group):
    """(o, lse, dq, dk, dv) in float64."""
    q, k, v, do = (a.astype(np.float64) for a in (q, k, v, do))
    kr, vr = np.repeat(k, group, 0), np.repeat(v, group, 0)
    nq, nk, d = q.shape[1], k.shape[1], q.shape[2]
    s = q @ kr.transpose(0, 2, 1) / math.sqrt(d)
    if causal:
        s = np.where(np.arange(nk)[None, :] <= np.arange(nq)[:, None], s, -np.inf)
    m = s.max(-1, keepdims=True)
    e = np.exp(s - m)
    lse = (m + np.log(e.sum(-1, keepdims=True)))[..., 0]
    p = e / e.sum(-1, keepdims=True)
    o = p @ vr
    ds = p * (do @ vr.transpose(0, 2, 1) - (do * o).sum(-1, keepdims=True)) / math.sqrt(d)
    sum_group = lambda a: a.reshape(k.shape[0], group, nk, d).sum(1)  # noqa: E731
    return o, lse, ds @ kr, sum_group(ds.transpose(0, 2, 1) @ q), sum_group(p.transpose(0, 2, 1) @ do)


CASES = [  # bh, nq, nk, d, causal, group
    (1, 1, 3, 16, False, 1), (2, 31, 33, 16, True, 1), (3, 32, 32, 32, True, 1), (2, 33, 65, 64, False, 1),
    # four waves sharing 1, 3, 4, 5 and 9 tiles (a single key would leave gradients of exactly zero to compare with)
    (1, 40, 31, 64, False, 1), (1, 97, 96, 128, False, 1), (2, 128, 128, 128, True, 1), (1, 150, 129, 32, True, 1),
    (2, 260, 270, 64, True, 1),
    # causal with keys that no query sees, and queries past the last key
    (2, 40, 140, 64, True, 1), (2, 140, 40, 128, True, 1),
    (6, 70, 50, 64, True, 3), (8, 40, 100, 32, False, 4),
    # eight waves sharing 12, 13 and 20 tiles
    (1, 390, 384, 16, True, 1), (2, 400, 410, 64, False, 1), (2, 630, 640, 32, True, 2),
    # enough blocks for a wave each, and blocks that do not fill a workgroup
    (2100, 20, 30, 16, True, 1), (1100, 40, 40, 16, False, 1), (700, 90, 70, 32, True, 1), (1024, 50, 33, 64, True, 2)]


@pytest.mark.parametrize("bh,nq,nk,d,causal,group", CASES)
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_forward_backward(dev, dtype, bh, nq, nk, d, causal, group):
    bf = dtype == "bf16"
    if bf and d > 32:
        pytest.skip("bf16 at head_dim 64 and 128 runs the bf16 MFMA kernels")
    rng = np.random.default_rng(bh + 7 * nq + 13 * nk + d)
    make = lambda n, m: rng.standard_normal((n, m, d), dtype=np.float32)  # noqa: E731
    q, k, v, do = make(bh, nq), make(bh // group, nk), make(bh // group, nk), make(bh, nq)
    if bf:
        q, k, v, do = (from_bf16(to_bf16(a)) for a in (q, k, v, do))
    up = (lambda a: dev.upload(to_bf16(a), tg.bf16)) if bf else dev.upload  # noqa: E731
    qb, kb, vb, gb = (up(a) for a in (q, k, v, do))
    lse = tg.Buffer(tg.f32, (bh, nq))
    print(f"[attn f32] {dtype} bh={bh} nq={nq} nk={nk} d={d} causal={causal} group={group}", flush=True)
    ob = K.attention(qb, kb, vb, group, 1, causal=causal, lse=lse)
    ref = reference(q, k, v, do, causal, group)
    for ws in (0, K.attention_backward_workspace_size(bh // group, group, nq)):
        with stream_workspace(dev, ws):
            dq, dk, dv = K.attention_backward(qb, kb, vb, ob, gb, lse, group, 1, causal=causal)
            got = [b.to_host() for b in (ob, lse, dq, dk, dv)]
        for name, g, r in zip(("o", "lse", "dq", "dk", "dv"), got, ref):
            if bf and name != "lse":
                # each gradient is a sum over at most 140 rounded o . do, next to the bf16 bound
                check_bf16(g, r, name)
            else:
                check_f32(g, r, name)


LEAST = [  # bh, nq, nk, d, causal, group: both sides of the lines between these kernels and the per-row ones (256 CUs)
    (32, 16, 64, 128, False, 1), (33, 16, 64, 128, True, 1), (2, 16, 65, 64, False, 1), (128, 16, 16, 32, True, 1),
    (512, 1, 128, 64, False, 1), (512, 1, 129, 64, False, 1), (1024, 1, 256, 16, False, 2), (520, 2, 64, 32, False, 4),
    (520, 2, 65, 32, False, 4), (512, 4, 32, 128, False, 1), (512, 16, 9, 128, False, 2), (2048, 2, 70, 16, False, 1),
    (2048, 2, 70, 64, False, 8), (2048, 4, 70, 128, True, 8), (2047, 3, 17, 64, False, 1), (4, 8, 256, 64, False, 1),
    (4, 8, 257, 64, False, 1), (16, 16, 16, 32, True, 1), (512, 16, 2, 16, False, 1)]


@pytest.mark.parametrize("bh,nq,nk,d,causal,group", LEAST)
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_least_work(dev, dtype, bh, nq, nk, d, causal, group):
    test_forward_backward(dev, dtype, bh, nq, nk, d, causal, group)


@pytest.mark.parametrize("bh,nk", [(2048, 130), (8, 140)])  # the per-row kernel, and this file's
def test_first_keys_without_weight(dev, bh, nk):
    # the first keys' scores are all -inf: they weigh nothing, the others as if alone
    rng = np.random.default_rng(nk)
    q, k, v = (rng.standard_normal((bh, n, 16), dtype=np.float32) for n in (1, nk, nk))
    q[..., 0] = 1.0
    o, lse, *_ = reference(q, k[:, 70:], v[:, 70:], q, False, 1)
    k[:, :70, 0] = -np.inf
    print(f"[attn f32] scores of -inf bh={bh} nk={nk}", flush=True)
    lb = tg.Buffer(tg.f32, (bh, 1))
    ob = K.flash_attention(*(dev.upload(x) for x in (q, k, v)), lse=lb)
    check_f32(ob.to_host(), o, "o")
    check_f32(lb.to_host(), lse, "lse")


@pytest.mark.parametrize("d", [16, 64, 128])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_masked_rows_without_numbers(dev, d, bad):
    # rows from `cut` on hold no numbers (a padded batch): the queries before
    # it see none of them, in the block that the cut divides as well
    bh, n, cut = 2, 80, 45
    rng = np.random.default_rng(d)
    a = [rng.standard_normal((bh, n, d), dtype=np.float32) for _ in range(4)]
    q, k, v, do = a
    o, lse, dq, _, _ = reference(*(x[:, :cut] for x in a), True, 1)
    k[:, cut:], v[:, cut:] = bad, bad
    print(f"[attn f32 masked] d={d} bad={bad}", flush=True)
    lb = tg.Buffer(tg.f32, (bh, n))
    bufs = [dev.upload(x) for x in (q, k, v)]
    ob = K.flash_attention(*bufs, causal=True, lse=lb)
    check_f32(ob.to_host()[:, :cut], o, "o")
    check_f32(lb.to_host()[:, :cut], lse, "lse")
    check_f32(K.flash_attention_backward_dq(*bufs, ob, dev.upload(do), lb, causal=True).to_host()[:, :cut], dq, "dq")

    # queries before `cut` hold none: the keys from there on are seen by none of them
    q, k, v, do = (rng.standard_normal((bh, n, d), dtype=np.float32) for _ in range(4))
    o, lse, _, dk, dv = reference(q, k, v, do, True, 1)
    s = np.where(np.arange(n)[None, :] <= np.arange(n)[:, None], q.astype(np.float64) @ k.transpose(0, 2, 1) / math.sqrt(d),
                 -np.inf)[:, cut:]
    p = np.exp(s - lse[:, cut:, None])
    g = do[:, cut:].astype(np.float64)
    ds = p * (g @ v.transpose(0, 2, 1) - (g * o[:, cut:]).sum(-1, keepdims=True)) / math.sqrt(d)
    dk, dv = ds.transpose(0, 2, 1) @ q[:, cut:], p.transpose(0, 2, 1) @ g
    q[:, :cut], do[:, :cut] = bad, bad
    bufs = [dev.upload(x.astype(np.float32)) for x in (q, k, v, o, do, lse)]
    gk, gv = K.flash_attention_backward_dkv(*bufs, causal=True)
    check_f32(gk.to_host()[:, cut:], dk[:, cut:], "dk")
    check_f32(gv.to_host()[:, cut:], dv[:, cut:], "dv")


def test_rows_without_softmax(dev):
    # a row whose scores are all -inf, or hold a NaN or +inf, is NaN in o and lse; the others are not
    rng = np.random.default_rng(3)
    q, k, v = (rng.standard_normal((1, 70, 32), dtype=np.float32) for _ in range(3))
    k[0, :, 0] = 1.0  # q's component 0 shifts a whole row of scores
    q[0, 3, 0], q[0, 40, 0], q[0, 69, 0] = -np.inf, np.nan, np.inf
    lse = tg.Buffer(tg.f32, (1, 70))
    o = K.flash_attention(dev.upload(q), dev.upload(k), dev.upload(v), lse=lse).to_host()
    nan = np.zeros(70, bool)
    nan[[3, 40, 69]] = True
    np.testing.assert_array_equal(np.isnan(lse.to_host()[0]), nan)
    np.testing.assert_array_equal(np.isnan(o[0]).all(-1), nan)
    np.testing.assert_array_equal(np.isnan(o[0]).any(-1), nan)


def test_bf16_dkv_alone(dev, orc):
    # dk/dv of bf16 at head_dim 64 and 128 without a workspace for D_m
    for d in (64, 128):
        rng = np.random.default_rng(d)
        q, k, v, do = (from_bf16(to_bf16(rng.standard_normal((2, 70, d), dtype=np.float32))) for _ in range(4))
        o, l = orc.flash_attention(q, k, v, causal=True)
        o = from_bf16(to_bf16(o))
        _, rk, rv = orc.flash_attention_backward(q, k, v, o, do, l, 1 / math.sqrt(d), True)
        bufs = [dev.upload(to_bf16(a), tg.bf16) for a in (q, k, v, o, do)]
        print(f"[attn bf16 dkv alone] d={d}", flush=True)
        dk, dv = K.flash_attention_backward_dkv(*bufs, dev.upload(l), causal=True)
        check_bf16(dk.to_host(), rk, "dk")
        check_bf16(dv.to_host(), rv, "dv")
