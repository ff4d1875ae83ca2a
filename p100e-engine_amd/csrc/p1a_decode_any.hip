// Split-K paged-KV decode for the caches dec_mfma_k does not take: any D % 32 == 0 up to 512, any GQA, pages of any length,
// any alignment, f16 / q8_0 / q4_0. Nothing here is narrower than fp32 except Q, which is rounded to f16 once.
//
// Work decomposition
//   grid = (nsplit * kv heads, column tiles of 16 q heads, rows), block = NW waves; a row is never shared with another one,
//   so every key below its position is visible to every column. In unit u (16 NW positions) wave w owns the 16 positions
//   from 16 w on; split stream s owns units s, s + nsplit, ... - a partition that depends on the device and the head shape
//   only, so a row gives the same bits in whichever call it stands. The waves fold into one partial per (workgroup, head).
// Arithmetic: exact operands on the matrix cores. (Plain fp32 vector code, one wave per (stream, q head), re-read and
// re-expanded a row for every head of its group and reduced every key's product over 64 lanes in turn, 1.6 us a key.)
//   S^T = K Q^T, 16 keys x 16 columns at a time. f16 keys and the integer codes of quantized ones are f16 operands as they
//   are; the products are exact in fp32, and a block's scale multiplies its fp32 partial result.
//   O^T = V^T P^T. Quantized: the codes are exact in bf16, and P * scale (fp32) is cut into three bf16 pieces of 8 bits - all
//   24 of its mantissa - so the three products add up to the fp32 one. f16: P carries a factor 2^15. Where every P of a tile
//   that is not zero is at least 1, it is cut into three f16 pieces, 11, 11 and the 2 to 4 bits left: exact (the last bit of
//   such a P is 2^-23, f16 ends at 2^-24) and each above zero, so that an infinite V stays infinite. A tile with a smaller P
//   takes fp32 matrix products, at a fifth of the rate: pieces would end at 2^-39 of the largest weight, where fp32 does not,
//   and thousands of light keys with a large V are more than the result. (24 / 4 heads of 96, 8 sequences x 4 rows of 2500
//   keys: two pieces whatever P is 37.6 us, as it is 40.9; 24 / 4 of 256 in pages of 4 cost the same both ways.)
// Data movement
//   A lane reads what it feeds to the products straight into registers: 8 consecutive values (16 / 8 / 4 bytes) of its key
//   per K block, 2 consecutive dims (4 / 2 bytes; q4_0: one byte, dims c and c + 16) of 4 keys per V block. Only the
//   block scales change lanes, through a small table in LDS. No LDS tile: such head rows are 2-byte aligned, which the
//   LDS-direct loads of dec_mfma_k cannot take.
// Builds: one for each number of 32-dim blocks a head can have. (Heads of other than 96 and 192 dims shared one for up to 8
// blocks and one for up to 16: a branch per block keeps the loads and products of two blocks from being scheduled side by side, and
// the LDS of the largest head keeps a second workgroup off the CU. 8 sequences x 4 rows of 2500 keys in pages of 8, q8_0,
// 32 / 8 heads of 128 141 -> 74 us; 16 / 2 of 320 138 -> 66; 4 / 4 of 32 63 -> 27; 24 / 4 of 256 in pages of 4 121 -> 112.)
// What bounds it: latency. At 24 / 4 heads, D = 96, q8_0 a context of 8190 is one tile per wave: positions, page entry, tile,
// fold, each waiting for the one before. Two layers of it (prep, this kernel and the merge each) took 325 us and take 54, of
// which the launches from Python are most; recorded, a layer of 2000 keys takes 15 us, one of 20000 keys (16 MB) 19 us.
#include "p1a_common.hpp"

namespace p1a {
namespace {

constexpr float NEG_INF = -__builtin_inff();

struct any_params {
    const float * q;
    const char * kc;
    const char * vc;
    float * part_o;
    float * part_ml;
    kv_view pg;
    int p0;
    const int32_t * p0_dev;
    const int32_t * pos_rows;
    int RG, Hq, Hkv, GQA, D;
    float qscale;     // softmax scale * log2(e)
    int nsplit;
    int SQ;           // rows of a sequence (1 << 30: all rows are one sequence's)
    int T, RPS, rps_magic, inner;   // list: rows, those of a sequence (at most T), 65536 / RPS + 1, workgroups of a stream
};

template <typename T> __device__ __forceinline__ T ld(const char * p) {   // (any alignment)
    T x;
    __builtin_memcpy(&x, p, sizeof x);
    return x;
}
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }
__device__ __forceinline__ float asf(uint32_t x) { return __builtin_bit_cast(float, x); }
__device__ __forceinline__ uint32_t asu(float x) { return __builtin_bit_cast(uint32_t, x); }
// the upper halves of two fp32 words (bf16 by truncation) as one operand dword
__device__ __forceinline__ uint32_t bf2(float lo, float hi) { return perm(asu(hi), asu(lo), 0x07060302u); }
// 4 bytes -> 4 f16 values byte - off (0x6400 | n = 1024 + n; off = 1152 for x ^ 0x80, 1032 for a nibble)
__device__ __forceinline__ void codes4(uint32_t x, float off, uint32_t & a, uint32_t & b) {
    const h2 o = {(half_t) off, (half_t) off};
    a = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, perm(0x64646464u, x, 0x04010400u)) - o);
    b = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, perm(0x64646464u, x, 0x04030402u)) - o);
}

// the fp32 value below x > 0 (0 for 0)
__device__ __forceinline__ float below(float x) { return asf(__builtin_elementwise_sub_sat(asu(x), 1u)); }
// two values to f16, towards zero
__device__ __forceinline__ h2 cut2(float x, float y) { return __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(x, y)); }

// LIST: blockIdx.x counts the streams that hold keys (live_streams), the others behind them
template <uint32_t KT, int NB, int NW, bool LIST>
__device__ __forceinline__ void any_body(const any_params & P) {
    constexpr bool F16 = KT == P1A_KV_F16, Q8 = KT == P1A_KV_Q8_0;
    constexpr int OS = NB * 32 + 4;                          // floats per parked column (padded)
    constexpr int PC = 8;                                     // columns parked at a time
    __shared__ __attribute__((aligned(16))) float parked[NW * PC * OS];
    __shared__ __attribute__((aligned(16))) float stab[F16 ? 4 : NW * 2 * NB * 16];   // per wave: K scales [block][key], V scales
    __shared__ float ml[NW][2][16];
    constexpr int D = NB * 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    // the kv heads of one split stream share cache lines: given the same index mod 8 they sit on one XCD, and sequence r of a batch
    // starts on XCD r mod 8 (short ones only fill the first streams; the reasons for that and for the list are p1a_decode.hip's)
    constexpr int U = 16 * NW;
    int split, hk, t, ct, rt = 0;
    const bool has_rt = P.pg.pt && P.pg.rtab;
    if constexpr (LIST) {
        const int i = blockIdx.x, j = i >> 3, jq = j / P.inner, q = jq * 8 + (i & 7);
        int in = j - jq * P.inner, rt_lanes;
        const int rest = in / P.Hkv, nct = (P.GQA + 15) / 16;
        hk = in - rest * P.Hkv;
        const int sub = rest / nct;
        ct = rest - sub * nct;
        const uint32_t u_sum = live_streams<U>(P.pos_rows, P.pg.rtab, P.T, P.RPS, P.rps_magic, P.nsplit, lane, rt_lanes);
        const uint32_t all = (uint32_t) __builtin_amdgcn_readlane((int) u_sum, 31);
        const int q_a = (int) (all & 0xffff);
        if (q >= q_a + (int) (all >> 16)) return;
        const stream_at at = pick_stream(u_sum, q, q_a, lane);
        split = at.split;
        t = at.first + sub;
        if (t >= P.T) return;                                 // (a last sequence of fewer rows)
        if (has_rt) rt = P.T < 8 ? __builtin_amdgcn_readlane(rt_lanes, t / P.RG * P.RG) : sload_i32(P.pg.rtab + t / P.RG * P.RG);
    } else {
        if ((P.nsplit & 7) == 0) {
            const int i = blockIdx.x, j = i >> 3, jq = j / P.Hkv;
            hk = j - jq * P.Hkv;
            split = jq * 8 + ((i - (int) blockIdx.z / P.SQ) & 7);
        } else {
            split = blockIdx.x / P.Hkv;
            hk = blockIdx.x - split * P.Hkv;
        }
        t = blockIdx.z;
        ct = blockIdx.y;
        if (has_rt) rt = sload_i32(P.pg.rtab + (P.pos_rows ? (t / P.RG) * P.RG : 0));
    }
    const int col0 = ct * 16, R = min(16, P.GQA - col0);
    const size_t row0 = (size_t) t * P.Hq + (size_t) hk * P.GQA + col0;   // the output row of column 0
    const int n = (P.pos_rows ? sload_i32(P.pos_rows + t) : (P.p0_dev ? sload_i32(P.p0_dev) : P.p0) + t) + 1;
    const int32_t * ptab = P.pg.pt ? P.pg.pt + rt : nullptr;
    if (split * U >= n) return;                               // no key in this stream (the merge does not look at it)
    const size_t hoff = (size_t) hk * head_bytes(KT, 32) * NB;
    const int SC = Q8 ? 2 : 18;                               // distance of two block scales

    // Q^T operands of column c; the 8 k-slots of lane group g are dims 32 b + 8 g .., for q4_0 the low and the high
    // nibbles of bytes 4 g .. 4 g + 3. Asked for ahead of the first tile, converted behind its requests.
    f4 qa[NB][2];
    {
        const float * qr = P.q + (row0 + min(c, R - 1)) * D;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const float * x = qr + 32 * b + (KT == P1A_KV_Q4_0 ? 4 : 8) * g;
            qa[b][0] = *reinterpret_cast<const f4 *>(x);
            qa[b][1] = *reinterpret_cast<const f4 *>(x + (KT == P1A_KV_Q4_0 ? 16 : 4));
        }
    }
    f4 o[NB][2];
#pragma unroll
    for (int b = 0; b < NB; ++b) o[b][0] = o[b][1] = f4{0.f, 0.f, 0.f, 0.f};
    float m = NEG_INF, l = 0.f;                               // l: over this lane's keys
    float * const tk = stab + (F16 ? 0 : wave * 2 * NB * 16), * const tv = tk + (F16 ? 0 : NB * 16);

    const int last = n - 1;
    // a tile's K operands, V values and block scales, all asked for before any of them is used
    u4 kr[F16 ? NB : 1];
    uint64_t k8[Q8 ? NB : 1];
    uint32_t k4[!F16 && !Q8 ? NB : 1];
    uint32_t vr[NB][4];
    constexpr int NSC = (NB + 3) / 4;
    uint16_t sk[NSC], sv[NSC];
    auto request = [&](int ts) {
        // keys past the last one are read as the last one and weighted with nothing
        size_t ko, vo[4];
        if (!ptab || P.pg.psh >= 4) {                         // (16 positions from a multiple of 16 on: one page)
            size_t base = (size_t) ts * P.pg.rowb;
            if (ptab) base = (size_t) sload_i32(ptab + (ts >> P.pg.psh)) * P.pg.pstride + (size_t) (ts & ((1 << P.pg.psh) - 1)) * P.pg.rowb;
            base += hoff;
            ko = base + (size_t) min(c, last - ts) * P.pg.rowb;
#pragma unroll
            for (int i = 0; i < 4; ++i) vo[i] = base + (size_t) min(4 * g + i, last - ts) * P.pg.rowb;
        } else {
            ko = kv_off_tab(P.pg, ptab, min(ts + c, last)) + hoff;
#pragma unroll
            for (int i = 0; i < 4; ++i) vo[i] = kv_off_tab(P.pg, ptab, min(ts + 4 * g + i, last)) + hoff;
        }
        const char * kp = P.kc + ko;
        if constexpr (!F16) {
#pragma unroll
            for (int x = 0; x < NSC; ++x) {
                const int b = min(4 * x + g, NB - 1);         // (lanes without a block of their own repeat the last one)
                sk[x] = ld<uint16_t>(kp + b * SC);
                sv[x] = ld<uint16_t>(P.vc + ko + b * SC);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (F16) kr[b] = ld<u4>(kp + 64 * b + 16 * g);
            else if constexpr (Q8) k8[b] = ld<uint64_t>(kp + 2 * NB + 32 * b + 8 * g);
            else k4[b] = ld<uint32_t>(kp + 18 * b + 2 + 4 * g);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const char * vp = P.vc + vo[i] + (F16 ? 4 * c : Q8 ? 2 * NB + 2 * c : 2 + c);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (F16) vr[b][i] = ld<uint32_t>(vp + 64 * b);
                else if constexpr (Q8) vr[b][i] = ld<uint16_t>(vp + 32 * b);
                else vr[b][i] = *reinterpret_cast<const uint8_t *>(vp + 18 * b);
            }
        }
    };
    int ts = split * U + wave * 16;
    if (ts < n) request(ts);
    h8 qf[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int e = 0; e < 4; ++e) { qf[b][e] = (half_t) (qa[b][0][e] * P.qscale); qf[b][4 + e] = (half_t) (qa[b][1][e] * P.qscale); }
    }

    while (ts < n) {
        const bool tail = ts + 15 > last;
        if constexpr (!F16) {
#pragma unroll
            for (int x = 0; x < NSC; ++x) {
                const int b = min(4 * x + g, NB - 1);
                tk[b * 16 + c] = (float) __builtin_bit_cast(half_t, sk[x]);
                tv[b * 16 + c] = ts + c > last ? 0.f : (float) __builtin_bit_cast(half_t, sv[x]);
            }
            __builtin_amdgcn_wave_barrier();
        }
        // ---- S^T: this lane holds keys ts + 4 g + i of column c ----
        f4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (F16) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kr[b]), qf[b], s, 0, 0, 0);
            else {
                uint32_t a[4];
                if constexpr (Q8) {
                    codes4((uint32_t) k8[b] ^ 0x80808080u, 1152.f, a[0], a[1]);
                    codes4((uint32_t) (k8[b] >> 32) ^ 0x80808080u, 1152.f, a[2], a[3]);
                } else {
                    codes4(k4[b] & 0x0f0f0f0fu, 1032.f, a[0], a[1]);
                    codes4((k4[b] >> 4) & 0x0f0f0f0fu, 1032.f, a[2], a[3]);
                }
                const u4 av = {a[0], a[1], a[2], a[3]};
                const f4 sb = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, av), qf[b], f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                const f4 d = *reinterpret_cast<const f4 *>(tk + b * 16 + 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) s[i] = fmaf(sb[i], d[i], s[i]);
            }
        }
        // ---- online softmax (log2 domain) ----
        if (tail) {
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] = ts + 4 * g + i <= last ? s[i] : NEG_INF;
        }
        const float mx = max_swap32(max_swap16(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
        const float mnew = fmaxf(m, F16 ? mx - 15.f : mx);    // (f16: P runs up to 2^15, see above)
        if (__any(mnew != m)) {
            const float alpha = m == mnew ? 1.f : __builtin_amdgcn_exp2f(m - mnew);   // (m = -inf: nothing accumulated yet, 0)
            l *= alpha;
#pragma unroll
            for (int b = 0; b < NB; ++b) { o[b][0] *= alpha; o[b][1] *= alpha; }
            m = mnew;
        }
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = m == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(s[i] - m);
        l += (p[0] + p[1]) + (p[2] + p[3]);
        // ---- O^T += V^T P^T ----
        if constexpr (F16) {
            if (tail) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (ts + 4 * g + i > last) {
#pragma unroll
                        for (int b = 0; b < NB; ++b) vr[b][i] = 0;
                    }
            }
            if (__builtin_expect(__any((p[0] < 1.f && p[0] > 0.f) || (p[1] < 1.f && p[1] > 0.f) || (p[2] < 1.f && p[2] > 0.f) || (p[3] < 1.f && p[3] > 0.f)), 0)) {
#pragma unroll
                for (int b = 0; b < NB; ++b) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {             // keys 4 g + i of the four lane groups
                        uint32_t w = vr[b][i];
                        asm volatile("" : "+v"(w));           // (here, one at a time: 512 registers do not hold all of them as fp32)
                        const h2 v = __builtin_bit_cast(h2, w);
                        o[b][0] = __builtin_amdgcn_mfma_f32_16x16x4f32((float) v[0], p[i], o[b][0], 0, 0, 0);
                        o[b][1] = __builtin_amdgcn_mfma_f32_16x16x4f32((float) v[1], p[i], o[b][1], 0, 0, 0);
                    }
                }
            } else {
                h4 pc[3];                                     // the largest f16 value below what is left, twice, and the rest
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    float r0 = p[i], r1 = p[i + 1];
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const h2 h = k < 2 ? cut2(below(r0), below(r1)) : cut2(r0, r1);
                        pc[k][i] = h[0];
                        pc[k][i + 1] = h[1];
                        r0 -= (float) h[0];
                        r1 -= (float) h[1];
                    }
                }
#pragma unroll
                for (int b = 0; b < NB; ++b) {
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        const uint32_t sel = x ? 0x07060302u : 0x05040100u;
                        const i2 a = {(int) perm(vr[b][1], vr[b][0], sel), (int) perm(vr[b][3], vr[b][2], sel)};
#pragma unroll
                        for (int k = 2; k >= 0; --k) o[b][x] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, a), pc[k], o[b][x], 0, 0, 0);
                    }
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const f4 d = *reinterpret_cast<const f4 *>(tv + b * 16 + 4 * g);
                float w0[4], w1[4], w2[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    w0[i] = p[i] * d[i];
                    const float r1 = w0[i] - asf(asu(w0[i]) & 0xffff0000u);
                    w1[i] = r1 == r1 ? r1 : 0.f;              // (an infinite scale: its upper piece says it all)
                    w2[i] = w1[i] - asf(asu(w1[i]) & 0xffff0000u);
                }
                const i2 p0 = {(int) bf2(w0[0], w0[1]), (int) bf2(w0[2], w0[3])}, p1 = {(int) bf2(w1[0], w1[1]), (int) bf2(w1[2], w1[3])};
                const i2 p2 = {(int) bf2(w2[0], w2[1]), (int) bf2(w2[2], w2[3])};
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = Q8 ? (float) (int8_t) (vr[b][i] >> (8 * x)) : (float) ((int) ((vr[b][i] >> (4 * x)) & 15) - 8);
                    const i2 a = {(int) bf2(v[0], v[1]), (int) bf2(v[2], v[3])};
                    o[b][x] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, a), __builtin_bit_cast(s4, p2), o[b][x], 0, 0, 0);
                    o[b][x] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, a), __builtin_bit_cast(s4, p1), o[b][x], 0, 0, 0);
                    o[b][x] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, a), __builtin_bit_cast(s4, p0), o[b][x], 0, 0, 0);
                }
            }
            __builtin_amdgcn_wave_barrier();                  // (the next tile's scales go where these were read)
        }
        ts += P.nsplit * U;
        if (ts < n) request(ts);
    }
    // ---- fold the waves, in wave order, 8 columns at a time ----
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (g == 0) { ml[wave][0][c] = m; ml[wave][1][c] = l; }
    for (int h0 = 0; h0 < R; h0 += PC) {
        const int he = min(h0 + PC, R);
        if (h0) __syncthreads();
        if (c >= h0 && c < he) {
            float * dst = parked + (wave * PC + c - h0) * OS;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (KT == P1A_KV_Q4_0) {            // row r of tile x: dim 32 b + 16 x + r
                    *reinterpret_cast<f4 *>(dst + 32 * b + 4 * g) = o[b][0];
                    *reinterpret_cast<f4 *>(dst + 32 * b + 16 + 4 * g) = o[b][1];
                } else {                                      // row r of tile x: dim 32 b + 2 r + x
                    *reinterpret_cast<f4 *>(dst + 32 * b + 8 * g) = f4{o[b][0][0], o[b][1][0], o[b][0][1], o[b][1][1]};
                    *reinterpret_cast<f4 *>(dst + 32 * b + 8 * g + 4) = f4{o[b][0][2], o[b][1][2], o[b][0][3], o[b][1][3]};
                }
            }
        }
        __syncthreads();
        const int D4 = D / 4;
        for (int i = threadIdx.x; i < (he - h0) * D4; i += NW * 64) {
            const int cc = i / D4, d4 = i - cc * D4, col = h0 + cc;
            f4 aw[NW];
            float mw[NW];
            float M = NEG_INF, lt = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                aw[w] = *reinterpret_cast<const f4 *>(parked + (w * PC + cc) * OS + 4 * d4);
                mw[w] = ml[w][0][col];
                M = fmaxf(M, mw[w]);
            }
            f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const float f = mw[w] == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(mw[w] - M);
                lt += ml[w][1][col] * f;
                acc += aw[w] * f;
            }
            const size_t row = row0 + col;
            if (M != NEG_INF) *reinterpret_cast<f4 *>(P.part_o + (row * P.nsplit + split) * D + 4 * d4) = acc;
            if (d4 == 0) {
                float * pm = P.part_ml + (row * P.nsplit + split) * 2;
                pm[0] = M;
                pm[1] = lt;
            }
        }
    }
}

template <uint32_t KT, int NB, int NW>
__global__ void __launch_bounds__(NW * 64) dec_any_k(const any_params P) { any_body<KT, NB, NW, false>(P); }
template <uint32_t KT, int NB, int NW>
__global__ void __launch_bounds__(NW * 64) dec_list_any_k(const any_params P) { any_body<KT, NB, NW, true>(P); }

template <uint32_t KT, int NB> void launch_nb(const any_params & P, bool list, dim3 grid, hipStream_t s) {
    constexpr int NW = NB <= 8 ? 8 : 4;
    if constexpr (NB <= 8) { if (list) { dec_list_any_k<KT, NB, NW><<<grid, NW * 64, 0, s>>>(P); return; } }
    dec_any_k<KT, NB, NW><<<grid, NW * 64, 0, s>>>(P);
}
template <uint32_t KT> void launch_kt(const any_params & P, bool list, dim3 grid, hipStream_t s) {
    switch (P.D / 32) {
#define P1A_ANY(NB_) case NB_: launch_nb<KT, NB_>(P, list, grid, s); break
        P1A_ANY(1); P1A_ANY(2); P1A_ANY(3); P1A_ANY(4); P1A_ANY(5); P1A_ANY(6); P1A_ANY(7); P1A_ANY(8);
        P1A_ANY(9); P1A_ANY(10); P1A_ANY(11); P1A_ANY(12); P1A_ANY(13); P1A_ANY(14); P1A_ANY(15); P1A_ANY(16);
#undef P1A_ANY
    }
}

}   // namespace

int decode_any_unit(int D) { return D <= 256 ? 128 : 64; }

int launch_decode_any(const p1a_kv & c, const decode_args & a, int rows_per_group, int nsplit, hipStream_t s) {
    any_params P;
    P.q = a.q; P.kc = (const char *) c.k; P.vc = (const char *) c.v;
    P.part_o = a.part_o; P.part_ml = a.part_ml; P.pg = view_of(c);
    P.p0 = a.p0; P.p0_dev = a.p0_dev; P.pos_rows = a.pos_rows; P.RG = rows_per_group;
    P.Hq = a.Hq; P.Hkv = c.Hkv; P.GQA = a.Hq / c.Hkv; P.D = c.D; P.qscale = a.scale * 1.4426950408889634f; P.nsplit = nsplit;
    P.SQ = a.rows_per_seq;
    P.T = a.T;
    P.RPS = a.rows_per_seq < a.T ? a.rows_per_seq : a.T;
    P.rps_magic = 65536 / P.RPS + 1;
    const int nct = (P.GQA + 15) / 16, nseq = (a.T + P.RPS - 1) / P.RPS;
    P.inner = c.Hkv * nct * P.RPS;
    // Four to 16 rows of several sequences: calls drawn over 4 ... 7600 keys are 0.95 - 1.27 times as fast, 1.1 in the mean (4 of 616, q8_0,
    // 16 / 4 heads of 96, four layers 65.6 -> 57.9 us, 8 of 211 ... 3391, 4 / 1 of 192 86.7 -> 68.4). With 32 rows a grid of 8192 workgroups is mostly
    // empty and each reads all positions before it knows (f16, 24 / 4 of 192, 8 x 4 rows of 11 ... 188 keys 37 us, 48 with the list); with two
    // there is little to spread (16 / 2 of 96, 15 ... 246 keys 19.8 and 21.9).
    // Larger heads, a compute unit to a workgroup, only while few heads keep most streams empty (q8_0, 16 rows of 1000 keys, two layers: 16 / 2 of 192 1.25
    // times as fast, 24 / 4 1.02, 32 / 8 0.98; f16 1.14, 0.94, 0.88, with 8 rows 1.22, 1.02, 0.94).
    const bool list = a.pos_rows && nseq > 1 && a.T >= 4 && a.T <= 16 && (c.D <= 128 || (c.D <= 256 && c.Hkv * a.T <= 32));
    const dim3 grid = list ? dim3((unsigned) (((long long) nseq * nsplit + 7) / 8 * 8 * P.inner)) : dim3(nsplit * c.Hkv, nct, a.T);
    if (c.type == P1A_KV_F16) launch_kt<P1A_KV_F16>(P, list, grid, s);
    else if (c.type == P1A_KV_Q8_0) launch_kt<P1A_KV_Q8_0>(P, list, grid, s);
    else launch_kt<P1A_KV_Q4_0>(P, list, grid, s);
    return launched();
}

}   // namespace p1a
