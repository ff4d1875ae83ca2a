"""attn_prep on the GPU (through the C ABI) vs the oracle: gate, q and the KV bytes (K codes included) must match bit for
bit - both sides keep one operation order and spell out power, cosine and sine in IEEE double operations instead of
calling a math library; then the prepared cache and q drive a decode."""
import numpy as np
import pytest
import torch

import _inputs as I
import _oracle as O
from _gpu import check, dev

pytestmark = pytest.mark.gpu
TYPES = [O.KV_F16, O.KV_Q8_0, O.KV_Q4_0]


def make(seed, T, Hq, Hkv, D):
    g = I.rng(seed)
    qg = I.normal(g, (T, Hq, 2 * D))
    k = I.normal(g, (T, Hkv, D)) * 1.3
    v = I.normal(g, (T, Hkv, D))
    qn = (1.0 + 0.1 * I.normal(g, (D,))).astype(np.float32)
    kn = (1.0 + 0.1 * I.normal(g, (D,))).astype(np.float32)
    return qg, k, v, qn, kn


def ulp_diff(a, b):
    ia = a.view(np.int32).astype(np.int64)
    ib = b.view(np.int32).astype(np.int64)
    ia = np.where(ia < 0, -(ia & 0x7fffffff), ia)
    ib = np.where(ib < 0, -(ib & 0x7fffffff), ib)
    return np.abs(ia - ib)


@pytest.mark.parametrize("kv_type", TYPES)
@pytest.mark.parametrize("Hq,Hkv,D,n_rot", [(24, 4, 256, 64), (4, 1, 64, 64), (8, 2, 128, 32)])
def test_host_position_contiguous(p1a, kv_type, Hq, Hkv, D, n_rot):
    T, p0, n_ctx, base, eps = 7, 9, 32, 1e7, 1e-6
    qg, k, v, qn, kn = make(D + n_rot, T, Hq, Hkv, D)
    pos = (p0 + np.arange(T)).astype(np.int32)
    host = O.HostKV.contiguous(kv_type, n_ctx, Hkv, D)
    q_ref, gate_ref = O.attn_prep(host, qg, k, v, qn, kn, pos, p0, Hq, n_rot, base, eps)
    c = p1a.KVCache.contiguous(kv_type, n_ctx, Hkv, D)
    q = torch.zeros((T, Hq, D), device="cuda")
    gate = torch.zeros((T, Hq * D), device="cuda")
    p1a.attn_prep(dev(qg), dev(k), dev(v), dev(qn), dev(kn), dev(pos), q, gate, c, p0, T, Hq, n_rot, base, eps)
    torch.cuda.synchronize()
    assert np.array_equal(gate.cpu().numpy(), gate_ref)
    assert np.array_equal(q.cpu().numpy().view(np.int32), q_ref.view(np.int32))
    assert np.array_equal(c._keep[1].cpu().numpy(), host.v)
    assert np.array_equal(c._keep[0].cpu().numpy(), host.k)


@pytest.mark.parametrize("kv_type", TYPES)
def test_device_positions_paged_rows_then_decode(p1a, kv_type):
    """rows of four sequences, each at its own position through its own page table (p0 < 0), strided inputs; then the
    prepared q / gate / cache drive attn_decode_rows and must give the oracle's attention"""
    Hq, Hkv, D, n_rot, base, eps, psh = 12, 2, 256, 64, 1e7, 1e-6, 4
    lens = [40, 17, 63, 5]
    T = len(lens)
    max_pages, n_pages = 5, 24
    g = I.rng(77)
    table = g.permutation(n_pages)[: T * max_pages].astype(np.int32)
    rtab = (np.arange(T) * max_pages).astype(np.int32)
    hostp = O.HostKV.paged(kv_type, Hkv, D, psh, n_pages, table, max_pages)
    host = hostp.view(rtab=rtab)
    dtab, drt = dev(table), dev(rtab)
    dc = p1a.KVCache.paged(kv_type, Hkv, D, psh, n_pages, dtab, max_pages).with_rows(drt)
    # history: every sequence gets lens[s] - 1 earlier rows through the plain append (same bytes on both sides)
    for s, n in enumerate(lens):
        if n > 1:
            _, kh, vh, _ = I.qkv(900 + s, n - 1, 1, Hq, Hkv, D)
            O.kv_append_rows(host.view(rtab=np.full(n - 1, s * max_pages, np.int32)), kh, vh, np.arange(n - 1))
            p1a.kv_append(dc.slot(s, max_pages), dev(kh), dev(vh), 0, n - 1)
    qg, k, v, qn, kn = make(5, T, Hq, Hkv, D)
    pos = np.array([n - 1 for n in lens], np.int32)
    # strided inputs: rows carry padding, as slices of a concatenated projection output do
    ldq, ldk, ldv = Hq * 2 * D + 8, Hkv * D + 4, Hkv * D + 12
    def strided(a, ld):
        buf = np.full((T, ld), 7.0, np.float32)
        buf[:, : a[0].size] = a.reshape(T, -1)
        return buf
    q_ref, gate_ref = O.attn_prep(host, qg, k, v, qn, kn, pos, -1, Hq, n_rot, base, eps)
    q = torch.zeros((T, Hq, D), device="cuda")
    gate = torch.zeros((T, Hq * D), device="cuda")
    dpos = dev(pos)
    p1a.attn_prep(dev(strided(qg, ldq)), dev(strided(k, ldk)), dev(strided(v, ldv)), dev(qn), dev(kn), dpos, q, gate, dc, -1, T, Hq,
                  n_rot, base, eps, ldq=ldq, ldk=ldk, ldv=ldv)
    torch.cuda.synchronize()
    assert np.array_equal(gate.cpu().numpy(), gate_ref)
    assert np.array_equal(q.cpu().numpy().view(np.int32), q_ref.view(np.int32))
    assert np.array_equal(dc._keep[0].cpu().numpy(), hostp.pool)          # every byte of the pool: history rows and the prepared ones
    out = torch.zeros((T, Hq, D), device="cuda")
    p1a.attn_decode_rows(q, dc, out, T, dpos, Hq, 1 / 16, gate=gate)
    torch.cuda.synchronize()
    ref = O.attn_rows(host, q_ref, pos, Hq, 1 / 16, gate=gate_ref)
    check(out.cpu().numpy(), ref, f"prep -> decode_rows type {kv_type}")


def test_refusals(p1a):
    c = p1a.KVCache.contiguous(O.KV_Q8_0, 8, 2, 256)
    z = torch.zeros(4 * 2 * 256 * 2, device="cuda")
    pos = torch.zeros(1, dtype=torch.int32, device="cuda")
    with pytest.raises(p1a.P1AError):       # n_rot not a multiple of 8
        p1a.attn_prep(z, z, z, None, None, pos, z, z, c, 0, 1, 4, 12, 1e7, 1e-6)
    with pytest.raises(p1a.P1AError):       # no positions
        p1a.attn_prep(z, z, z, None, None, None, z, z, c, 0, 1, 4, 64, 1e7, 1e-6)
    with pytest.raises(p1a.P1AError):       # row stride shorter than a row
        p1a.attn_prep(z, z, z, None, None, pos, z, z, c, 0, 1, 4, 64, 1e7, 1e-6, ldq=64)
    torch.cuda.synchronize()


def test_ew_quant_sigmoid_and_silu(p1a):
    """gate + a16 emit (src/fast/fused.cu:478-496): y within fp32 rounding of the oracle, the a16 bytes exactly the oracle's
    quantization of the y the GPU wrote; strided a / b; y aliasing a"""
    T, n = 3, 6144
    g = I.rng(41)
    a = I.normal(g, (T, n)) * 2.0
    b = I.normal(g, (T, n))
    a[1, 64:96] = 0.0                                           # an all-zero group
    lda, ldb = n + 8, n + 32
    ap = np.zeros((T, lda), np.float32); ap[:, :n] = a
    bp = np.zeros((T, ldb), np.float32); bp[:, :n] = b
    for op in (1, 0):
        y = torch.zeros((T, n), device="cuda")
        qb = torch.zeros(p1a.a16_bytes(T, n) // 2, dtype=torch.int16, device="cuda")
        p1a.ew_quant(op, dev(ap), dev(bp), y, qb, T, n, lda=lda, ldb=ldb)
        torch.cuda.synchronize()
        yh = y.cpu().numpy()
        if op == 1:
            ref = a.astype(np.float64) / (1.0 + np.exp(-b.astype(np.float64)))
        else:
            ref = a.astype(np.float64) / (1.0 + np.exp(-a.astype(np.float64))) * b.astype(np.float64)
        assert np.max(np.abs(yh - ref)) <= 4e-7 * max(1.0, np.abs(ref).max())
        assert np.array_equal(qb.cpu().numpy().view(np.uint16), O.a16_quant(yh)), op
    # in place: y aliases a (dense rows)
    ya = dev(a)
    qb = torch.zeros(p1a.a16_bytes(T, n) // 2, dtype=torch.int16, device="cuda")
    p1a.ew_quant(1, ya, dev(b), ya, qb, T, n)
    torch.cuda.synchronize()
    assert np.array_equal(qb.cpu().numpy().view(np.uint16), O.a16_quant(ya.cpu().numpy()))
    with pytest.raises(p1a.P1AError):
        p1a.ew_quant(1, ya, dev(b), ya, qb, T, n - 4)          # n % 32 != 0
    torch.cuda.synchronize()


@pytest.mark.parametrize("kv_type", [O.KV_Q8_0, O.KV_F16])
def test_decode_emits_a16(p1a, kv_type):
    """the decode call with a qbuf: same output bits as without, and qbuf = a16(gated output)"""
    from _gpu import Pool
    Hq, Hkv, D, psh = 24, 4, 256, 6
    lens = [300, 77]
    pool = Pool(p1a, kv_type, Hq, Hkv, D, psh, lens, seed=13)
    T = 3
    q, _, _, gate = I.qkv(61, 1, T, Hq, Hkv, D)
    pos = np.array([299, 76, 150], np.int32)
    rt = np.array([0, pool.maxp, 0], np.int32)
    c = pool.devkv.with_rows(dev(rt))
    o1 = torch.zeros((T, Hq, D), device="cuda"); o2 = torch.zeros((T, Hq, D), device="cuda")
    qb = torch.zeros(p1a.a16_bytes(T, Hq * D) // 2, dtype=torch.int16, device="cuda")
    dq, dg, dp = dev(q), dev(gate), dev(pos)
    p1a.attn_decode_rows(dq, c, o1, T, dp, Hq, 1 / 16, gate=dg)
    p1a.attn_decode_rows(dq, c, o2, T, dp, Hq, 1 / 16, gate=dg, qbuf=qb)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2)
    assert np.array_equal(qb.cpu().numpy().view(np.uint16), O.a16_quant(o2.cpu().numpy().reshape(T, Hq * D)))


@pytest.mark.parametrize("kv_type", TYPES)
def test_mrope_positions(p1a, kv_type):
    """interleaved M-RoPE (src/fast/mrope.cuh): image rows with their own t / h / w, the same bars as the plain rotation;
    and text rows (t = h = w = p) give the plain call's bits."""
    Hq, Hkv, D, n_rot, T, n_ctx, base, eps = 24, 4, 256, 64, 9, 64, 1e7, 1e-6
    qg, k, v, qn, kn = make(77, T, Hq, Hkv, D)
    pos = (20 + np.arange(T)).astype(np.int32)                            # cache rows
    P = 1000                                                               # a 3 x 3 image placed at P: t = P, h = P + i / 3, w = P + i % 3
    mp = np.zeros((3, T + 3), np.int32)                                   # (a stride larger than T)
    mp[0, :T], mp[1, :T], mp[2, :T] = P, P + np.arange(T) // 3, P + np.arange(T) % 3
    host = O.HostKV.contiguous(kv_type, n_ctx, Hkv, D)
    q_ref, gate_ref = O.attn_prep(host, qg, k, v, qn, kn, pos, -1, Hq, n_rot, base, eps, mrope=(mp, (11, 11, 10), 32))
    c = p1a.KVCache.contiguous(kv_type, n_ctx, Hkv, D)
    q = torch.zeros((T, Hq, D), device="cuda")
    gate = torch.zeros((T, Hq * D), device="cuda")
    p1a.attn_prep(dev(qg), dev(k), dev(v), dev(qn), dev(kn), dev(pos), q, gate, c, -1, T, Hq, n_rot, base, eps,
                  mrope=(dev(mp), T + 3, (11, 11, 10), 32))
    torch.cuda.synchronize()
    assert np.array_equal(gate.cpu().numpy(), gate_ref)
    assert np.array_equal(q.cpu().numpy().view(np.int32), q_ref.view(np.int32))
    assert np.array_equal(c._keep[1].cpu().numpy(), host.v)
    assert np.array_equal(c._keep[0].cpu().numpy(), host.k)
    # text rows
    c1, c2 = p1a.KVCache.contiguous(kv_type, n_ctx, Hkv, D), p1a.KVCache.contiguous(kv_type, n_ctx, Hkv, D)
    q1, q2 = torch.zeros_like(q), torch.zeros_like(q)
    p1a.attn_prep(dev(qg), dev(k), dev(v), dev(qn), dev(kn), dev(pos), q1, gate, c1, -1, T, Hq, n_rot, base, eps)
    p1a.attn_prep(dev(qg), dev(k), dev(v), dev(qn), dev(kn), dev(pos), q2, gate, c2, -1, T, Hq, n_rot, base, eps,
                  mrope=(dev(np.stack([pos, pos, pos])), T, (11, 11, 10), 32))
    torch.cuda.synchronize()
    assert torch.equal(q1, q2) and torch.equal(c1._keep[0], c2._keep[0]) and torch.equal(c1._keep[1], c2._keep[1])
    with pytest.raises(p1a.P1AError, match="M-RoPE"):
        p1a.attn_prep(dev(qg), dev(k), dev(v), dev(qn), dev(kn), dev(pos), q2, gate, c2, -1, T, Hq, n_rot, base, eps,
                      mrope=(dev(mp), T + 3, (11, 11, 10), 0))


@pytest.mark.parametrize("kv_type", TYPES)
@pytest.mark.parametrize("Hq,Hkv,D,n_rot,by_pos", [(24, 4, 256, 64, False), (2, 1, 256, 256, True), (5, 1, 192, 184, False), (32, 8, 128, 128, True),
                                                   (4, 2, 96, 96, False), (6, 3, 64, 0, True), (7, 1, 32, 8, False)])
def test_calls_of_many_tokens(p1a, kv_type, Hq, Hkv, D, n_rot, by_pos):
    """a call large enough for the workgroup-per-token kernel (64, 32, 16 and 8 lanes to a head, dead lanes at D = 192 and 96):
    the oracle's bits, and those of the same rows in calls of one token (one wave per head), strided inputs, no norm weight
    where n_rot is 0"""
    base, eps = 1e6, 1e-6
    T = 16384 // (Hq + 2 * Hkv) + 1
    p0, n_ctx = 11, T + 16
    qg, k, v, qn, kn = make(D + n_rot + Hq, T, Hq, Hkv, D)
    if n_rot == 0:
        qn = kn = None
    pos = (p0 + np.arange(T)).astype(np.int32)
    if by_pos:
        pos = pos[I.rng(5).permutation(T)].copy()
    host = O.HostKV.contiguous(kv_type, n_ctx, Hkv, D)
    q_ref, gate_ref = O.attn_prep(host, qg, k, v, qn, kn, pos, -1 if by_pos else p0, Hq, n_rot, base, eps)
    c = p1a.KVCache.contiguous(kv_type, n_ctx, Hkv, D)
    c1 = p1a.KVCache.contiguous(kv_type, n_ctx, Hkv, D)
    ldq, ldk, ldv = Hq * 2 * D + 8, Hkv * D + 4, Hkv * D + 12

    def strided(a, ld):
        buf = np.full((T, ld), 7.0, np.float32)
        buf[:, : a[0].size] = a.reshape(T, -1)
        return dev(buf)
    dqg, dk, dv, dpos = strided(qg, ldq), strided(k, ldk), strided(v, ldv), dev(pos)
    dqn, dkn = (None if x is None else dev(x) for x in (qn, kn))
    q, gate = torch.zeros((T, Hq, D), device="cuda"), torch.zeros((T, Hq * D), device="cuda")
    p1a.attn_prep(dqg, dk, dv, dqn, dkn, dpos, q, gate, c, -1 if by_pos else p0, T, Hq, n_rot, base, eps, ldq=ldq, ldk=ldk, ldv=ldv)
    assert np.array_equal(gate.cpu().numpy(), gate_ref)
    assert np.array_equal(q.cpu().numpy().view(np.int32), q_ref.view(np.int32))
    assert np.array_equal(c._keep[0].cpu().numpy(), host.k)
    assert np.array_equal(c._keep[1].cpu().numpy(), host.v)
    for t in (0, T // 2, T - 1):
        q1, g1 = torch.zeros((1, Hq, D), device="cuda"), torch.zeros((1, Hq * D), device="cuda")
        p1a.attn_prep(dqg[t:], dk[t:], dv[t:], dqn, dkn, dpos[t:], q1, g1, c1, -1 if by_pos else p0 + t, 1, Hq, n_rot, base, eps, ldq=ldq, ldk=ldk, ldv=ldv)
        assert torch.equal(q1[0], q[t]) and torch.equal(g1[0], gate[t])


@pytest.mark.parametrize("Hq,D,n_rot", [(24, 256, 64), (8, 128, 128)])
def test_mrope_in_a_call_of_many_tokens(p1a, Hq, D, n_rot):
    """interleaved M-RoPE positions through the workgroup-per-token kernel: the bits of one-token calls"""
    Hkv, sect = 2, (11, 11, 10)
    T = 16384 // (Hq + 2 * Hkv) + 3
    g = I.rng(9)
    qg, k, v, qn, kn = make(3, T, Hq, Hkv, D)
    mr = dev(np.ascontiguousarray(g.integers(0, 5000, (3, T)).astype(np.int32)))
    pos = dev(np.arange(T, dtype=np.int32))
    dqg, dk, dv, dqn, dkn = (dev(x) for x in (qg, k, v, qn, kn))
    out = []
    for step in (T, 1):
        c = p1a.KVCache.contiguous(O.KV_Q8_0, T, Hkv, D)
        q, gate = torch.zeros((T, Hq, D), device="cuda"), torch.zeros((T, Hq * D), device="cuda")
        for a in (range(0, T, step) if step == T else (0, 1, T - 2, T - 1)):
            n = min(step, T - a)
            p1a.attn_prep(dqg[a:], dk[a:], dv[a:], dqn, dkn, pos[a:], q[a:a + n], gate[a:a + n], c, a, n, Hq, n_rot, 1e6, 1e-6,
                          mrope=(mr[:, a:a + n].contiguous(), n, sect, 32))
        out.append((q, gate, c._keep[0].reshape(T, -1), c._keep[1].reshape(T, -1)))
    for x, y in zip(*out):
        for t in (0, 1, T - 2, T - 1):
            assert torch.equal(x[t], y[t]), t


@pytest.mark.parametrize("kv_type,Hq,Hkv,D,n_rot", [(O.KV_Q8_0, 24, 4, 256, 64), (O.KV_F16, 32, 8, 128, 128), (O.KV_Q4_0, 40, 2, 192, 64)])
def test_call_past_the_caches(p1a, kv_type, Hq, Hkv, D, n_rot):
    """from 80 MB of q | gate rows on they are read past the caches: the bits of the same rows in two calls of half as many tokens"""
    T = -(-(80 << 20) // (Hq * D * 8))
    T += T & 1
    g = torch.Generator(device="cuda").manual_seed(D)
    qg, k, v = (torch.randn((T, n), generator=g, device="cuda") for n in (Hq * 2 * D, Hkv * D, Hkv * D))
    qn, kn = (1 + 0.1 * torch.randn(D, generator=g, device="cuda") for _ in range(2))
    pos, outs = torch.arange(T, dtype=torch.int32, device="cuda"), []
    for step in (T, T // 2):
        c = p1a.KVCache.contiguous(kv_type, T, Hkv, D)
        q, gate = torch.zeros((T, Hq, D), device="cuda"), torch.zeros((T, Hq * D), device="cuda")
        for a in range(0, T, step):
            b = a + step
            p1a.attn_prep(qg[a:b], k[a:b], v[a:b], qn, kn, pos[a:b], q[a:b], gate[a:b], c, a, step, Hq, n_rot, 1e6, 1e-6)
        outs.append((q, gate, *c._keep))
    for x, y in zip(*outs):
        assert torch.equal(x, y)
    assert torch.equal(outs[0][1].view(T, Hq, D), qg.view(T, Hq, 2 * D)[:, :, D:])
