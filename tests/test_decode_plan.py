"""The grid of a decode call, on the CPU: whatever the call, there is one, and it visits every split stream of every sequence's row
groups and kv heads exactly once."""
import random

import pytest

from _plan import plan

F16, Q4_0, Q8_0 = 1, 2, 8


def visits(p, Hkv, T):
    """how often each (stream number or (row group, stream), kv head, row group of the sequence) is taken, as dec_mfma_k counts
    blockIdx: with a list, number q of the streams there could be, else the stream itself"""
    seen = {}
    groups = -(-T // p["RG"])
    inner, nseq = Hkv * p["GPS"], -(-groups // p["GPS"])
    if not p["list"]:
        assert (p["x"], p["y"]) == (p["nsplit"] * Hkv, groups)
        return None
    assert p["y"] == 1 and p["x"] % (8 * inner) == 0
    step = (p["x"] >> 3) // inner * 8
    for i in range(p["x"]):
        j = i >> 3
        jq, q = j // inner, j // inner * 8 + (i & 7)
        while q < nseq * p["nsplit"]:
            key = (q, j - jq * inner)
            seen[key] = seen.get(key, 0) + 1
            if not p["loop"]:
                break
            q += step
    return seen, {(q, r) for q in range(nseq * p["nsplit"]) for r in range(inner)}


# rows of a sequence that no group of two to four divides, and many kv heads: more (kv head, row group) pairs than two for every unit
MANY = [(F16, 32, 32, 128, 512, 17, 17), (F16, 32, 32, 128, 513, 17, 17), (F16, 64, 64, 128, 256, 22, 11), (F16, 40, 40, 64, 300, 13, 13), (Q8_0, 32, 32, 256, 512, 31, 31),
        (Q4_0, 128, 128, 256, 100, 10, 5), (F16, 16, 16, 256, 100, 29, 29), (Q8_0, 128, 64, 128, 64, 22, 11)]


@pytest.mark.parametrize("kv_type,Hq,Hkv,D,n_ctx,T,rows", MANY)
def test_many_heads_and_row_groups(kv_type, Hq, Hkv, D, n_ctx, T, rows):
    for cus in (256, 304, 64):
        p = plan(kv_type, Hq, Hkv, D, n_ctx, T, rows, cus=cus)
        assert p["x"] > 0 and p["y"] > 0, (cus, p)
        if p["list"] and cus == 256:
            seen, all_ = visits(p, Hkv, T)
            assert set(seen) == all_ and set(seen.values()) == {1}, cus


def test_drawn_calls():
    rng = random.Random(5)
    kinds = set()
    for _ in range(700):
        kv_type, D = rng.choice([F16, Q4_0, Q8_0]), rng.choice([64, 128, 256])
        Hkv, gqa = rng.choice([1, 2, 3, 4, 5, 8, 16, 24, 32, 40, 64, 128]), rng.choice([1, 1, 2, 3, 4, 6, 8, 16])
        T, cus = rng.randint(1, 32), rng.choice([256, 256, 304, 80])
        rows, n_ctx = rng.randint(1, T + 3), int(2 ** rng.uniform(0, 18))
        p = plan(kv_type, Hkv * gqa, Hkv, D, n_ctx, T, rows, cus=cus, nsplit=rng.choice([0, 0, 0, 1, 24, 1024]))
        assert p["mfma"] and 0 < p["x"] * 64 * p["NW"] < 1 << 32 and 0 < p["y"] < 65536, p
        assert p["RG"] == 1 or rows % p["RG"] == 0               # (a group never holds rows of two sequences)
        if p["list"] and p["x"] * p["GPS"] < 3000:
            seen, all_ = visits(p, Hkv, T)
            assert set(seen) == all_ and set(seen.values()) == {1}, p
            kinds.add((p["sb"], p["loop"], p["NT"]))
    assert len(kinds) >= 5, kinds                              # (two to a unit and one, one stream and several, one column tile and two)


def direct_items(p, Hkv):
    """(row group, kv head, XCD) of each workgroup of a direct call, as dec_mfma_k takes them from blockIdx (workgroup i is on XCD i mod 8)"""
    sh = p["deal_sh"]
    return [(((i >> sh) // Hkv << sh) + (i & ((1 << sh) - 1)), (i >> sh) % Hkv, i & 7) for i in range(p["x"])]


@pytest.mark.parametrize("kv_type,Hq,Hkv,D,T,rows", [(F16, 4, 1, 64, 1, 1), (Q8_0, 24, 4, 256, 32, 4), (F16, 24, 4, 256, 31, 1), (Q8_0, 32, 8, 128, 32, 1), (F16, 12, 6, 128, 9, 3), (Q4_0, 16, 2, 256, 2, 1)])
def test_calls_of_one_unit(kv_type, Hq, Hkv, D, T, rows):
    """a workgroup for every (row group, kv head) where the host knows that no row sees more than a unit - from the positions before n_ctx -, each taken once,
    the heads of a group on one XCD; everything else has the grids above"""
    unit = 128 if kv_type == F16 and D == 256 else 256
    for n_ctx, host_n, direct in ((unit, 0, 1), (unit + 1, 0, 0), (0, 0, 0), (1 << 17, unit, 1), (1, unit + 1, 0)):
        p = plan(kv_type, Hq, Hkv, D, n_ctx, T, rows, pos_rows=host_n == 0, host_n=host_n)
        assert p["direct"] == direct, (n_ctx, host_n)
        assert not plan(kv_type, Hq, Hkv, D, n_ctx, T, rows, pos_rows=host_n == 0, host_n=host_n, partials=True)["direct"]
        if not direct:
            continue
        groups = -(-T // p["RG"])
        taken = direct_items(p, Hkv)
        live = [(g, h) for g, h, _ in taken if g * p["RG"] < T]
        assert p["y"] == 1 and sorted(live) == [(g, h) for g in range(groups) for h in range(Hkv)]
        assert all(len({x for g, _, x in taken if g == k}) == 1 for k in range(groups))
    assert not plan(Q4_0, 24, 4, 256, 256, 8, 4)["direct"]     # (two column tiles of q4_0: no registers for it)
    assert not plan(F16, 32, 32, 64, 256, 9, 1)["direct"]      # (more workgroups than compute units)


@pytest.mark.parametrize("kv_type,D", [(F16, 64), (F16, 128), (F16, 256), (Q8_0, 128), (Q8_0, 256), (Q4_0, 256)])
def test_calls_of_one_unit_fit_every_xcd(kv_type, D):
    """no XCD gets more live workgroups than its compute units, whatever the number of heads: all kv heads of a row group are on one
    XCD only where they fit so"""
    rng, seen = random.Random(6), {0: 0, 3: 0}
    calls = [(Hkv, 1, T, 1, 256) for Hkv, T in ((32, 1), (33, 1), (40, 1), (64, 1), (128, 1), (24, 8), (24, 9), (16, 16), (15, 17), (8, 32), (10, 24), (10, 25))]
    for _ in range(400):
        calls.append((rng.randint(1, 130), rng.choice([1, 2, 4, 6]), rng.randint(1, 32), rng.choice([1, 2, 3, 4]), rng.choice([256, 256, 304, 80])))
    for Hkv, gqa, T, rows, cus in calls:
        p = plan(kv_type, Hkv * gqa, Hkv, D, 100, T, rows, cus=cus)
        if not p["direct"]:
            continue
        live = [(g, h, x) for g, h, x in direct_items(p, Hkv) if g * p["RG"] < T]
        assert sorted(i[:2] for i in live) == [(g, h) for g in range(-(-T // p["RG"])) for h in range(Hkv)], (Hkv, gqa, T, rows, cus, p)
        assert max(sum(x == k for _, _, x in live) for k in range(8)) <= cus // 8, (Hkv, gqa, T, rows, cus, p)
        seen[p["deal_sh"]] += 1
    assert min(seen.values()) > 10, seen


@pytest.mark.parametrize("kv_type", [F16, Q8_0, Q4_0])
def test_positions_the_host_knows_count_before_n_ctx(kv_type):
    """the grid of a call whose positions the host gives does not depend on how wide its page table is"""
    rng, kinds = random.Random(7), set()
    for _ in range(200):
        D, Hkv, T, host_n = rng.choice([64, 128, 128, 256]), rng.choice([1, 2, 4, 8, 16]), rng.randint(1, 32), int(2 ** rng.uniform(5, 17))
        for partials in (False, True):
            grids = [plan(kv_type, 4 * Hkv, Hkv, D, n_ctx, T, T, pos_rows=False, host_n=max(host_n, T), partials=partials) for n_ctx in (0, 100, host_n, 1024, 1 << 17)]
            assert all(g == grids[0] for g in grids), (D, Hkv, T, host_n, partials)
        kinds.add((grids[0]["sb"], D))
    assert (1, 128) in kinds and (0, 128) in kinds
