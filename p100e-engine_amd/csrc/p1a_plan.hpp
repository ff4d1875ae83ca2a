// The decode launch plan: which kernel a shape takes, how its keys are split and how large its grid is. Host arithmetic only, on the
// descriptor and the call's numbers.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include "p1a_attn.h"

namespace p1a {

// ---- launch plan: which kernel a shape takes, and how the keys are split ----
// The MFMA kernel needs 16-byte aligned head rows (f16: D in {64, 128, 256}; q8_0 / q4_0: D == 256), 16-byte aligned
// bases and strides, pages of >= 16 positions and GQA <= 16; q8_0 / q4_0 at D = 64 or 128 (head rows of whole dwords)
// take its staged build, which fetches 4 bytes per lane and only needs 4-byte alignment. Everything else takes the
// kernel of p1a_decode_any.hip.
struct dec_plan {
    bool mfma;
    int GQA, NW, NT, RG;
    int nsplit;    // split streams: partials per output row
};

inline bool mfma_ok(const p1a_kv & c, int GQA) {
    if (GQA < 1 || GQA > 16) return false;
    if (c.D != 64 && c.D != 128 && c.D != 256) return false;
    const bool staged = c.type != P1A_KV_F16 && c.D != 256;   // q8_0 / q4_0 head rows are whole 16-byte chunks only at D = 256
    const uintptr_t al = staged ? 3 : 15;
    if (((uintptr_t) c.k | (uintptr_t) c.v) & al) return false;
    if (c.pt && ((c.pstride & al) || c.psh < 4)) return false;
    return true;
}

inline dec_plan make_plan(const p1a_kv & c, int Hq, int rows_per_group, int nsplit_req, int cus) {
    dec_plan p;
    p.GQA = Hq / c.Hkv;
    p.mfma = mfma_ok(c, p.GQA);
    if (!p.mfma) {
        p.NW = 4; p.NT = 1;
        p.RG = rows_per_group < 1 ? 1 : rows_per_group;   // no sharing here: the group only selects the page table
        // one workgroup per CU, and not more than 4 partials for every 2 CUs per q head
        int n = nsplit_req;
        if (n <= 0) {
            const int most = 4 * (2 * cus / Hq < 1 ? 1 : (2 * cus / Hq > 1024 ? 1024 : 2 * cus / Hq));
            n = cus / c.Hkv < most ? cus / c.Hkv : most;
        }
        n = n < 1 ? 1 : (nsplit_req > 1024 ? 1024 : n);
        p.nsplit = n >= 8 ? n & ~7 : n;
        return p;
    }
    const int cap = 32 / p.GQA < 4 ? 32 / p.GQA : 4;
    p.RG = rows_per_group < 1 ? 1 : (rows_per_group > cap ? cap : rows_per_group);
    // One kv head per workgroup: its waves fold into ONE partial, which keeps the split traffic at a few percent of the KV
    // bytes; the heads of a split stream are placed on one XCD so shared cache lines meet in its L2.
    const bool big_tiles = c.type == P1A_KV_F16 && c.D == 256;   // 34 KB of LDS per wave
    p.NW = big_tiles ? 4 : 8;
    const int HG = c.Hkv;
    // (one workgroup per CU for every variant: the four-wave one keeps 128 KB of f16 tiles in LDS; measured for f16 at
    // 32 K: 64 streams 27.2 us, 128 streams - two rounds of workgroups - 30.2 us)
    int n = nsplit_req > 0 ? nsplit_req : cus / HG;
    if (n >= 8) n &= ~7;
    p.nsplit = n < 1 ? 1 : (n > 1024 ? 1024 : n);
    return p;
}

inline void finish_plan(dec_plan & p) { p.NT = p.RG * p.GQA <= 16 ? 1 : 2; }

// The grid of the MFMA kernel: a workgroup for every (split stream, kv head) and row group, or - `list` - for every kv head and row
// group of the streams that hold keys, counted through on the device: x = 8 * Hkv * GPS * nq, nq eights of streams (`loop`: a workgroup
// takes the streams q, q + 8 nq, ...)
struct decode_grid {
    bool sb, list, loop, direct;   // two workgroups to a compute unit; kinds of dec_mfma_k
    int RPS, GPS;          // rows and row groups of a sequence
    int deal_sh;           // direct: log2 of the row groups that are dealt to the XCDs at a time
    unsigned x, y;
};

inline decode_grid plan_grid(const dec_plan & pl, uint32_t type, int D, int Hkv, int n_ctx, int T, int rows_per_seq, bool pos_rows, int cus_,
                             long long host_n, bool partials) {
    decode_grid r;
    const int cus = cus_ > 0 ? cus_ : 256, groups = (T + pl.RG - 1) / pl.RG;
    const bool staged = type != P1A_KV_F16 && D != 256;
    r.RPS = rows_per_seq < T ? rows_per_seq : T;
    r.GPS = rows_per_seq > pl.RG ? rows_per_seq / pl.RG : 1;
    if (r.GPS > groups) r.GPS = groups;
    const int nseq = (groups + r.GPS - 1) / r.GPS, inner = Hkv * r.GPS;
    // One unit at most, as far as the host knows - from the positions (host_n of them; 0: they are in device memory)
    // or from what a page-table row holds: the workgroup of a (row group, kv head) writes the results, and there is no merge behind
    // it (`partials`: they are what the call is for). Steps of two layers, prep included, with merge_k and so: q8_0, 24 / 4 heads of 256,
    // one sequence of 250 keys 34.4 and 29.6 us, 32 of them 42.8 and 33.4; f16, 32 / 8 of 128 30.6 and 26.0, 32 of them 40.2 and 33.4;
    // 8 x 4 rows of 250 (24 / 4) 48.1 and 42.0; plain calls of 100 keys 28.4 and 26.5. (Positions in device memory behind table rows of a
    // server's context limit go by merge_k: 32 of 256, q8_0, 32 / 8 of 128 32.5 with rows of 256 positions, 40 with 512, 42.5 with 32768.)
    // A workgroup has its compute unit to itself. All kv heads of a row group go to one XCD, eights of groups at a time, where no XCD gets more of them than it
    // has units so; else workgroups go to the XCDs in turn. Rows of 250 keys, heads of 256 (q8_0), with merge_k, by groups and in turn: one row of 40 heads
    // 33.8, 44.7, 28.7, of 128 36.8, 77.9, 32.5, 9 rows of 24 heads 47.9, 47.3, 35.5; but 8 rows of 24 38.8, 32.8, 34.6, 16 of 8 heads of
    // 128 37.2, 30.2, 31.8 (cache lines that two heads share; f16 level).
    // Not from two units on: whoever folds last would have to merge, and its stores, counter and loads past the L2s cost what merge_k does
    // (500 keys 34.6 and 35.3, 2000 35.1 and 36.2, 8000 37 and 48).
    r.sb = r.list = r.loop = false;
    r.deal_sh = 0;
    const long long sees = host_n ? host_n : n_ctx;
    r.direct = !partials && sees > 0 && sees <= 32 * pl.NW && (long long) groups * Hkv <= cus && !(pl.NT == 2 && type == P1A_KV_Q4_0 && !staged);
    if (r.direct) {
        r.deal_sh = (groups + 7) / 8 * Hkv <= cus / 8 ? 3 : 0;
        r.x = (unsigned) (((groups + (1 << r.deal_sh) - 1) >> r.deal_sh << r.deal_sh) * Hkv);
        r.y = 1;
        return r;
    }
    // A call of at least two workgroups per CU whose row groups fit one column tile takes the single-buffered variant, two
    // workgroups to a CU (same partials, bit for bit; measured at 24 / 4 heads, D = 256: 8 q8_0 slots of 1 K ... 27 K 56 ->
    // 47 us, 4 x 64 K q4_0 single rows 92 -> 73 us, 16 x 2 rows q4_0 at 16 K 143 -> 115 us, 32 slots of 2 ... 5 K 104 -> 71 us).
    // Staged tiles, D = 128: so too where more workgroups than compute units can have keys - by the positions, or by what a page-table row holds (two layers with
    // prep, one to a unit and two: q8_0, 32 / 8 heads, 16 sequences of 2000 ... 8000 keys 161 and 112 us, 4 of 8000 ... 32000 120 and 101; q4_0, 24 / 4, 8 x 2
    // rows of 8000 ... 32000 136 and 108, 32 sequences of 1000 53 and 45; but 8 x 2 rows of 1000 36.7 and 38.3). Not at D = 64, whose conversions
    // are half as long (q8_0, 16 / 4, 32 of 2000 ... 8000 79 and 85; q4_0, 8 / 8, 2 of 32000 54.4 and 53.5).
    // One sequence's rows have a workgroup for every stream there could be, and from eight for every unit on half of the empty ones' time is worth it, whatever the
    // keys (q8_0, 32 rows of 1000 keys, 32 / 8 heads 68.8 and 62.2, 16 / 4 56.2 and 50.7; with four for every unit, 16 rows, 16 / 4 41.0 and 45.9, 32 / 8
    // 45.9 and 46.9, 8 / 8 44.1 and 41.7; with two, 8 rows of 32 / 8, 37.7 and 44.7).
    const long long all = (long long) pl.nsplit * Hkv * groups;
    const bool two = !staged || (D == 128 && ((sees + 32 * pl.NW - 1) / (32 * pl.NW) * groups * Hkv > cus || (!pos_rows && all >= 8LL * cus)));
    r.sb = pl.NT == 1 && two && all >= 2LL * cus;
    // The list (see dec_mfma_k) costs a workgroup some 0.2 us before its first request. Where two workgroups share a compute unit that hides,
    // and every call of several row groups takes it. Several sequences (110 calls of 2 ... 32 drawn over 4 ... 131072 keys, D = 256 and f16):
    // 0.98 - 1.6 times as fast, 1.1 in the mean. One sequence of 5 ... 32 rows (200 calls over 200, 3000 and 20000 keys, six head shapes):
    // 0.84 - 1.6, 1.1 in the mean - the row groups of a stream are side by side on an XCD, which long sequences gain from (f16, 32 / 8 of 128, 13 rows
    // of 20000 keys 150 -> 98 us, 8 rows 33 -> 26; 200 keys 14.1 -> 11.9); what loses most are row counts that only groups of one
    // divide (q4_0, 16 / 16 of 256, 31 rows of 3000 keys 143 -> 166, f16, 16 / 4 of 64, 20000 keys 80 -> 95). Where one has a unit to itself (two
    // column tiles, staged tiles that do not go two to a unit) it shows: calls of four row groups and more whose page-table rows - as wide as n_ctx
    // says, whatever the sequences hold - cannot hold the keys that half of the streams begin with (without it, with a workgroup for every
    // stream: 8 x 4 rows of 300 ... 5000 keys, q8_0, 24 / 4 heads of 256, two layers 71.0 and 61.1 us, 16 of 300 ... 5000, 16 / 4 of 64
    // 49.9 and 41.5). With every stream live it costs what it takes: 8 of 18797, q8_0, 24 / 4 of 128, four layers 233 and 235.5.
    const long long once = (long long) pl.nsplit * 32 * pl.NW;   // the keys that every stream holds a unit of
    r.list = pos_rows && groups > 1 && (r.sb || (groups >= 4 && 2LL * n_ctx <= once));
    r.loop = false;
    r.x = (unsigned) (pl.nsplit * Hkv);
    r.y = (unsigned) groups;
    if (!r.list) return r;
    long long nq = ((long long) nseq * pl.nsplit + 7) / 8;   // streams there could be, in eights
    // Where most workgroups would find nothing to do, at 0.5 us for every 1000 of them, fewer walk the list. (Three times each: without the list,
    // with a workgroup for every stream, so; two layers with prep, page-table rows as wide as the sequences.)
    //   Two to a unit: more than 16 for every compute unit, i.e. 32 sequences (q8_0, 24 / 4 heads of 256, 500 keys 66.4, 56.5, 44.2 us, 300 ... 5000
    //   88.1, 83.9, 77.6; f16, 32 / 8 of 128, 1024 76.2, 81.3, 71.2). Fewer would lose more where all streams are live (16 of 20000: 314, 306 with a
    //   workgroup for every stream, 333 with eight for every unit); but four for every unit where page-table rows hold a quarter of that at most
    //   (32 of 1024, f16, 16 / 4 of 64 54.9, 56.4, 39.4 - with 16, behind rows of 32768 positions, 45.2; 24 / 4 of 256, q8_0 73.6, 68.8, 56.6;
    //   where they hold half, f16, 8 / 8 of 256, 2000 keys 212 with 16 and 220 with four).
    //   One to a unit: more than two for every compute unit; at least half of the streams are known to be empty there (8 x 4 rows of 300 ... 5000,
    //   q8_0, 24 / 4 of 256 71.0, 61.1, 54.2; 16 / 4 of 64, 32 of 500 54.3, 45.2, 33.2, 16 of 300 ... 5000 49.9, 41.5, 37.5; 32 / 8 of 128,
    //   16 of 500 57.8, 51.4, 39.1).
    //   Staged tiles, two to a unit: two for every compute unit where page-table rows cannot hold half of it, as in the second kind (q8_0,
    //   32 / 8 of 128, 32 of 500 67.8, 60.0, 46.7).
    // Rows of 32768 positions, a server's limit, take the other route whatever the sequences hold: 71.2 us for the 8 x 4 rows, 49.6 for the 16 of
    // 16 / 4 heads, 52.5 for the last.
    const bool resident = !r.sb || (staged && 2LL * n_ctx <= once);
    const long long most = (resident ? 2LL : 16LL) * cus / (8 * inner);
    const bool can_loop = pl.NT == 2 ? staged || type != P1A_KV_Q4_0 : r.sb || staged;   // (q4_0 with two column tiles has no register left for it)
    r.loop = can_loop && nq > most;
    // (never none: 8 * inner workgroups are more than that where kv heads and row groups are many)
    if (r.loop) nq = std::max(1LL, r.sb && !staged && 4LL * n_ctx <= once ? (most + 3) / 4 : most);
    r.x = (unsigned) (8 * inner * nq);
    r.y = 1;
    return r;
}

}   // namespace p1a
