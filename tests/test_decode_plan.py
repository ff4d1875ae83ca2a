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
