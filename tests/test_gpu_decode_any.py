"""The decode kernel for the caches the tiled one does not take (head sizes that are no 64 / 128 / 256, more than 16 q heads per
kv head, pages below 16 positions, 2-byte aligned bases) against the float64 oracle.

Its only rounding below fp32 is that of Q, and the inputs take that one out: q holds f16 values and the softmax scale is
2^-4 / log2(e), so q * scale * log2(e) rounds back to an f16 value. What is left are fp32 sums: scores of at most 2^5 in the
log2 domain are off by at most 2^5 2^-24 times a few roundings (the sums of a block and of the blocks), and P by ln 2 times
that - about 5e-6 at the very worst, 1e-6 in the 2-norm; P in 16 bits would give 2e-4. The bound is 1e-5."""
import numpy as np
import pytest
import torch

import _inputs as I
import _oracle as O
from _gpu import Pool, dev

pytestmark = pytest.mark.gpu
SCALE = float(np.float32(2.0 ** -4 / 1.4426950408889634))
TOL = 1e-5


def close(out, ref, what):
    rl = float(np.linalg.norm(out.astype(np.float64) - ref) / np.linalg.norm(ref))
    assert np.all(np.isfinite(out)) and rl <= TOL, (what, rl)
    print(f"[parity] {what}: rel_l2={rl:.2e}")


# (type, q heads, kv heads, D, log2 of the page): builds of 8 and of 4 waves, one and more column
# tiles (17 and 20 heads of a group), short pages, the 51- and 27-value-wide odd rows of D = 96 and one kv head
SHAPES = [(O.KV_F16, 6, 1, 96, 4), (O.KV_Q8_0, 24, 4, 96, 8), (O.KV_Q4_0, 4, 1, 96, 4), (O.KV_Q8_0, 3, 1, 96, 0),
          (O.KV_F16, 16, 2, 192, 6), (O.KV_Q8_0, 16, 4, 192, 4), (O.KV_Q4_0, 8, 8, 192, 4),
          (O.KV_F16, 17, 1, 64, 4), (O.KV_Q8_0, 40, 2, 256, 6), (O.KV_Q4_0, 4, 2, 256, 2), (O.KV_F16, 4, 2, 32, 3),
          (O.KV_Q8_0, 4, 2, 160, 4), (O.KV_Q4_0, 2, 1, 224, 4),
          (O.KV_F16, 4, 2, 512, 4), (O.KV_Q8_0, 6, 2, 320, 4), (O.KV_Q4_0, 2, 2, 288, 1)]


@pytest.mark.parametrize("kv_type,Hq,Hkv,D,psh", SHAPES)
def test_any_shape_vs_float64(p1a, kv_type, Hq, Hkv, D, psh):
    unit = 128 if D <= 256 else 64                              # positions of a workgroup's unit: 16 per wave
    lens = [1, 17, unit, unit + 1, 9 * unit + 5]
    pool = Pool(p1a, kv_type, Hq, Hkv, D, psh, lens, seed=D + Hq)
    for s, n in enumerate(lens):
        T = min(n, 3)
        q, _, _, gate = I.qkv(7 * D + s, 1, T, Hq, Hkv, D, f16_inputs=True)
        pos = (n - T + np.arange(T)).astype(np.int32)
        ref = O.attn_rows(pool.host_seq(s), q, pos, Hq, SCALE, gate=gate, f64=True)
        c, dq, dg = pool.dev_seq(s), dev(q), dev(gate)
        out = torch.full((T, Hq, D), float("nan"), device="cuda")
        p1a.attn_decode(dq, c, out, T, n - T, Hq, SCALE, gate=dg)
        close(out.cpu().numpy(), ref, f"type {kv_type} {Hq}/{Hkv}/{D} pages {1 << psh} n {n}")
        one = torch.empty((1, Hq, D), device="cuda")
        for t in range(T):                                      # a row of its own, and by device position: the same bits
            p1a.attn_decode(dq[t:t + 1], c, one, 1, n - T + t, Hq, SCALE, gate=dg[t:t + 1])
            assert torch.equal(one[0], out[t]), (s, t)
            p1a.attn_decode_rows(dq[t:t + 1], c, one, 1, dev(pos[t:t + 1]), Hq, SCALE, gate=dg[t:t + 1])
            assert torch.equal(one[0], out[t]), (s, t)
    # the sequences in one call; an idle slot (position -1) sees no key and disturbs nobody
    S = len(lens)
    q, _, _, _ = I.qkv(9 * D, 1, S, Hq, Hkv, D, f16_inputs=True)
    pos = np.array([lens[0] - 1, -1] + [n - 1 for n in lens[2:]], np.int32)
    rows = pool.devkv.with_rows(dev(np.array([s * pool.maxp for s in range(S)], np.int32)))
    out = torch.zeros((S, Hq, D), device="cuda")
    p1a.attn_decode_rows(dev(q), rows, out, S, dev(pos), Hq, SCALE)
    got = out.cpu().numpy()
    for s in (0, 2, 3, 4):
        close(got[s:s + 1], O.attn_rows(pool.host_seq(s), q[s:s + 1], pos[s:s + 1], Hq, SCALE, f64=True), f"slot {s}")
    assert np.all(np.isnan(got[1]))


@pytest.mark.parametrize("kv_type", [O.KV_F16, O.KV_Q8_0, O.KV_Q4_0])
@pytest.mark.parametrize("D", range(32, 513, 32))
def test_any_head_size(p1a, kv_type, D):
    """a build for each number of 32-dim blocks: a unit's first wave alone, and several units with a ragged end"""
    Hq, Hkv, psh, lens = 3, 1, 2, [5, 400]
    pool = Pool(p1a, kv_type, Hq, Hkv, D, psh, lens, seed=D)
    for s, n in enumerate(lens):
        q, _, _, gate = I.qkv(3 * D + s, 1, 1, Hq, Hkv, D, f16_inputs=True)
        ref = O.attn_rows(pool.host_seq(s), q, np.array([n - 1], np.int32), Hq, SCALE, gate=gate, f64=True)
        out = torch.full((1, Hq, D), float("nan"), device="cuda")
        p1a.attn_decode(dev(q), pool.dev_seq(s), out, 1, n - 1, Hq, SCALE, gate=dev(gate))
        close(out.cpu().numpy(), ref, f"type {kv_type} D {D} n {n}")


@pytest.mark.parametrize("kv_type", [O.KV_F16, O.KV_Q8_0, O.KV_Q4_0])
def test_any_misaligned_contiguous_base(p1a, kv_type):
    """a contiguous cache of D = 256 two bytes off any alignment"""
    Hq, Hkv, D, n = 12, 2, 256, 300
    pool = Pool(p1a, kv_type, Hq, Hkv, D, 4, [n], seed=4)
    h = pool.host_contiguous(0)
    kb, vb = (torch.zeros(x.view(np.uint8).size + 2, dtype=torch.uint8, device="cuda") for x in (h.k, h.v))
    kb[2:] = dev(h.k.view(np.uint8).reshape(-1))
    vb[2:] = dev(h.v.view(np.uint8).reshape(-1))
    c = p1a.KVCache(kv_type, n, Hkv, D, kb.data_ptr() + 2, vb.data_ptr() + 2, keep=(kb, vb))
    q, _, _, _ = I.qkv(5, 1, 2, Hq, Hkv, D, f16_inputs=True)
    out = torch.empty((2, Hq, D), device="cuda")
    p1a.attn_decode(dev(q), c, out, 2, n - 2, Hq, SCALE)
    close(out.cpu().numpy(), O.attn_rows(h, q, np.array([n - 2, n - 1], np.int32), Hq, SCALE, f64=True), f"type {kv_type}")


def test_any_infinite_values_and_low_scores(p1a):
    """f16: an infinite V of a key with a small weight gives an infinite result, not a NaN, and none at all in a row that does
    not see its key; scores 2^40 below the rest neither raise the reference maximum nor leave a NaN"""
    Hq, Hkv, D, n = 4, 1, 96, 200
    pool = Pool(p1a, O.KV_F16, Hq, Hkv, D, 4, [n], seed=6, fill="none")
    q, k, v, _ = I.qkv(8, n, 2, Hq, Hkv, D, f16_inputs=True)
    k[100] = -(40.0 / 2.0 ** -4) * q[0, 0] / float(q[0, 0] @ q[0, 0])
    v[100, 0, 5] = np.inf
    v[n - 1, 0, 7] = -np.inf
    O.kv_append_rows(pool.host_seq(0), k, v, np.arange(n))
    p1a.kv_append(pool.dev_seq(0), dev(k), dev(v), 0, n)
    out = torch.empty((2, Hq, D), device="cuda")
    p1a.attn_decode(dev(q), pool.dev_seq(0), out, 2, n - 2, Hq, SCALE)
    got = out.cpu().numpy()
    assert np.all(got[:, :, 5] == np.inf)
    assert np.all(np.isfinite(got[0, :, 7])) and np.all(got[1, :, 7] == -np.inf)
    keep = [d for d in range(D) if d not in (5, 7)]
    v0 = v.copy()
    v0[~np.isfinite(v0)] = 0.0
    O.kv_append_rows(pool.host_seq(0), k, v0, np.arange(n))
    ref = O.attn_rows(pool.host_seq(0), q, np.array([n - 2, n - 1], np.int32), Hq, SCALE, f64=True)
    close(got[:, :, keep], ref[:, :, keep], "the other dims")


@pytest.mark.parametrize("kv_type", [O.KV_F16, O.KV_Q8_0, O.KV_Q4_0])
@pytest.mark.parametrize("D,low", [(96, 60.0), (192, 43.0), (320, 30.0)])
def test_any_weights_have_the_range_of_fp32(p1a, kv_type, D, low):
    """one key with a small V beside thousands whose V is the largest f16 holds and whose weight is 2^-low of its own: what those
    add is below, at and above an ulp of the result, and weights of any narrower range (f16 pieces end at 2^-24) make it more
    than the result. The scores are twice the 2^5 of TOL, so twice TOL."""
    Hq, Hkv, n = 4, 1, 8190
    pool = Pool(p1a, kv_type, Hq, Hkv, D, 4, [n], seed=D, fill="none")
    q, k, v, _ = I.qkv(D, n, 1, Hq, Hkv, D, f16_inputs=True)
    q[:] = q[0, 0]
    k[:] = -(low / 2.0 ** -4) * q[0, 0] / float(q[0, 0] @ q[0, 0])
    k[4001] = 0.0
    v[:] = 60000.0
    v[4001] = (1.0 + 0.01 * np.arange(D)) * 2.0 ** -10
    O.kv_append_rows(pool.host_seq(0), k, v, np.arange(n))
    p1a.kv_append(pool.dev_seq(0), dev(k), dev(v), 0, n)
    ref = O.attn_rows(pool.host_seq(0), q, np.array([n - 1], np.int32), Hq, SCALE, f64=True)
    out = torch.empty((1, Hq, D), device="cuda")
    p1a.attn_decode(dev(q), pool.dev_seq(0), out, 1, n - 1, Hq, SCALE)
    rl = float(np.linalg.norm(out.cpu().numpy().astype(np.float64) - ref) / np.linalg.norm(ref))
    assert rl <= 2 * TOL, (kv_type, D, low, rl)


def test_any_infinite_value_under_equal_weights(p1a):
    """f16: weights of a single bit (q = 0: every key the same) have nothing left for the lower pieces of a cut; an infinite V
    stays infinite all the same, and the other dims are the mean"""
    Hq, Hkv, D, n = 3, 1, 96, 128
    pool = Pool(p1a, O.KV_F16, Hq, Hkv, D, 4, [n], seed=7, fill="none")
    _, k, v, _ = I.qkv(9, n, 1, Hq, Hkv, D, f16_inputs=True)
    v[50, 0, 3], v[7, 0, 90] = np.inf, -np.inf
    O.kv_append_rows(pool.host_seq(0), k, v, np.arange(n))
    p1a.kv_append(pool.dev_seq(0), dev(k), dev(v), 0, n)
    out = torch.empty((1, Hq, D), device="cuda")
    p1a.attn_decode(dev(np.zeros((1, Hq, D), np.float32)), pool.dev_seq(0), out, 1, n - 1, Hq, SCALE)
    got = out.cpu().numpy()[0]
    assert np.all(got[:, 3] == np.inf) and np.all(got[:, 90] == -np.inf)
    keep = [d for d in range(D) if d not in (3, 90)]
    mean = np.broadcast_to(v[:, 0].astype(np.float64).mean(0)[keep], (Hq, len(keep)))
    close(got[:, keep], mean, "equal weights")
