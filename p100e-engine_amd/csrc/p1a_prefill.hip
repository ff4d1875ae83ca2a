// Chunked causal prefill attention over a paged f16 / q8_0 / q4_0 KV cache for gfx950 (MI355X).
//
// One workgroup (4 waves) owns 128 consecutive query ROWS of one kv head (64 or 32 in a call of few) - row r is token r / GQA
// under q head r % GQA of the group; wave w owns 32 (16, 8) of them as the N = 32 columns of v_mfma_f32_32x32x16_f16 tiles.
// (Rows, not the tokens of one q head: a chunk of few tokens fills its blocks - 77 tokens under 6 heads are 4 blocks, not
// 6 - and a block spans 128 / GQA tokens, so fewer of the keys it walks are behind the diagonal for most of its rows. 24 / 4
// heads of 256, q8_0: 77 tokens behind 16000 88.7 -> 79.7 us for the whole call; a full chunk, 4096 behind 28672, the same.)
// Keys are walked in tiles of 64, kept in LDS as f16 (two K and two V tiles). f16 rows in pages of 16 positions or more are
// moved from global memory straight into LDS (global_load_lds_dwordx4); everything else is fetched into registers with
// 16-byte loads, dequantized and stored to the same LDS places.
//   S^T = K Q^T : A = K rows straight from LDS (ds_read_b128), B = Q^T held in registers for the whole kernel (pre-multiplied
//                 by scale * log2 e, rounded to f16). A lane then holds 16 keys of ONE query row, so the row maximum
//                 needs no cross-lane work beyond one half-wave swap.
//   O^T = V^T P^T : A = V^T read with the transposing ds_read_b64_tr_b16, B = P^T straight from the S^T registers.
// Two builds of that, chosen by where the registers and the LDS reads end (pf_solo):
//   pairs (D = 256, and whatever is staged through registers): one wave per SIMD with 512 registers. Two waves share their
//                 64 rows for O^T, each accumulating half the dims of both, so a V^T fragment feeds two MFMAs; the partner's
//                 P^T comes through LDS.
//   solo (D = 64 / 128, tiles straight into LDS): a wave accumulates all dims of its own rows in 256 registers, and a CU
//                 holds two workgroups.
// The loop is software-pipelined so that every iteration holds two independent instruction streams side by side: the
// MFMAs of S^T for tile j+1 next to exp2 / f16 conversion of tile j, then the MFMAs of O^T for tile j next to masking and
// the row maximum of tile j+1 (and the dequantization of the tiles that come after). With one or two waves per SIMD little
// else hides one pipe behind the other.
// fp32 accumulation; the softmax denominator is a packed dot product of the rounded P with ones, so that it sums the same
// rounded P that multiplies V. The reference maximum of a row moves lazily (only when the row maximum has grown
// by more than 2^RESCALE_STEP), so the accumulators are rescaled a handful of times per row. Keys above a row's
// diagonal are masked; the sigmoid output gate is applied in the epilogue.
// Workgroup order: up to GQA consecutive row blocks of one kv head (with key splits all of them) get consecutive dispatch slots
// on the same XCD, so they stream the same K/V tiles through one L2.
#include "p1a_common.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace p1a {
size_t prefill_stage_bytes(int n, int Hkv, int D);
namespace {

constexpr int BM = 128;   // query rows per workgroup
constexpr int BN = 64;    // keys per tile
constexpr int NTHR = 256;
constexpr float NEG_INF = -__builtin_inff();

template <int D> struct pf_cfg {
    static constexpr int NKS = D / 16;         // k-steps of S^T (16 dims each)
    static constexpr int NDT = D / 32;         // 32-dim tiles of O^T
};

// Where the f16 tiles sit in LDS: in blocks of 1 KB - RPB = 2, 4 or 8 rows of 512, 256 or 128 bytes - and padding. A block is
// exactly what one global_load_lds_dwordx4 moves (64 lanes x 16 bytes to consecutive LDS); its rows are keys of one 16-key
// group, so one page base serves it: group q of the tile has the NJ = 16 / RPB blocks NJ q .. , key k of it sits in block
// NJ q + k % NJ, slot k / NJ. Tiles staged through registers use the same places. The padding (K 16 bytes, V 64) puts
// the rows that are read together into disjoint banks: 16 consecutive rows of an S^T operand are 16 blocks 4 banks apart
// (D = 64: 8 blocks, and two slots 32 banks apart), the four rows of a transposing V read 4 blocks 16 banks apart. So row
// c of half u of S^T is block c % NB (NB = 64 / RPB blocks; D = 256: + 16 u), slot (c / NB) + u (32 / NB) - which key that is
// follows - and the rows of O^T's operand follow from the order of the S^T values. Every read address is (per-lane base)
// + (compile-time offset).
template <int D> struct pf_lay {
    static constexpr int RB = 2 * D;                            // bytes of a row
    static constexpr int RPB = 1024 / RB, NJ = 16 / RPB, NB = BN / RPB;
    static constexpr int KB = 1024 + 16, VB = 1024 + 64;        // block strides
    static constexpr int KT_B = NB * KB, VT_B = NB * VB;
    static constexpr int STAGE_B = KT_B + VT_B;
    static __device__ __forceinline__ int key_off(int key, int bstride) { return (NJ * (key >> 4) + key % NJ) * bstride + (key & 15) / NJ * RB; }
    // row r (0 .. 31) of half u: its block and slot
    static constexpr __host__ __device__ int block(int u, int r) { return D == 256 ? 16 * u + (r & 15) : r % NB; }
    static constexpr __host__ __device__ int slot(int u, int r) { return D == 256 ? r >> 4 : r / NB + u * (32 / NB); }
    // S^T operand rows: lane base of row c, offset of half u
    static __device__ __forceinline__ int k_lane(int c) { return block(0, c) * KB + slot(0, c) * RB; }
    static constexpr int k_half(int u) { return block(u, 0) * KB + slot(u, 0) * RB; }
    // which key of the tile value i of half u of a lane's S^T column is: key_of(u, i) + KG g (row 8 (i / 4) + 4 g + i % 4)
    static constexpr __host__ __device__ int key_at(int u, int r) { return 16 * (block(u, r) / NJ) + block(u, r) % NJ + NJ * slot(u, r); }
    static constexpr int key_of(int u, int i) { return key_at(u, 8 * (i >> 2) + (i & 3)); }
    static constexpr int KG = key_at(0, 4) - key_at(0, 0);
    // V^T operand of k-step ps (half ps / 2 of the tile): rows 16 (ps % 2) + 4 g + kk (lane part: 4 g + kk), and the same + 8
    static __device__ __forceinline__ int v_lane(int r) { return r * VB; }
    static constexpr int v_lo(int ps) { return block(ps >> 1, 16 * (ps & 1)) * VB + slot(ps >> 1, 16 * (ps & 1)) * RB; }
    static constexpr int v_hi(int ps) { return block(ps >> 1, 16 * (ps & 1) + 8) * VB + slot(ps >> 1, 16 * (ps & 1) + 8) * RB; }
};


struct pf_params {
    const float * q;
    float * out;
    const float * gate;
    const char * kc;
    const char * vc;
    kv_view pg;
    int T, p0, Hq, Hkv, GQA;
    int n_rows;   // positions the cache holds (contiguous caches: rows that may be read)
    float qscale;
    int R;        // query rows of a kv head: T * GQA
    uint32_t gqa_magic;   // floor(2^32 / GQA) (2^32 - 1 for GQA = 1)
    int rpw;      // rows of a wave: 32, or 16 or 8 (a call of few blocks)
    int nblk;     // row blocks (4 rpw rows) of a kv head
    int nbg;      // groups of row blocks
    int bpg;      // blocks of a group
    int turn_a, turn_b;   // slots of an XCD taken in reverse order
    int run;      // key splits: consecutive workgroups of an XCD (0: groups in turn)
    // key splits: with nks > 1 workgroup (block, kv head, ks) walks its share of the block's tiles and leaves an unnormalised
    // partial (O relative to m, and (m, l)) per row in part_o [T*Hq][nks][D] / part_ml [T*Hq][nks][2] for the merge; out is part_o
    // then, and gate null
    int nks;
    float * part_o;
    float * part_ml;
};

__device__ __forceinline__ uint32_t perm_b(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }

// 4 int8 codes -> 4 halves (code * d), packed
struct pair32 { uint32_t lo, hi; };
__device__ __forceinline__ pair32 deq8x4(uint32_t w, h2 dd) {
    const uint32_t x = w ^ 0x80808080u;
    const h2 off = {(half_t) 1152, (half_t) 1152};
    const h2 a = __builtin_bit_cast(h2, perm_b(0x64646464u, x, 0x04010400u));
    const h2 b = __builtin_bit_cast(h2, perm_b(0x64646464u, x, 0x04030402u));
    return pair32{__builtin_bit_cast(uint32_t, (a - off) * dd), __builtin_bit_cast(uint32_t, (b - off) * dd)};
}
// 4 nibbles (in the low nibbles of the 4 bytes of w) -> 4 halves ((n - 8) * d)
__device__ __forceinline__ pair32 deq4x4(uint32_t w, h2 dd) {
    const h2 off = {(half_t) 1032, (half_t) 1032};
    const h2 a = __builtin_bit_cast(h2, perm_b(0x64646464u, w, 0x04010400u));
    const h2 b = __builtin_bit_cast(h2, perm_b(0x64646464u, w, 0x04030402u));
    return pair32{__builtin_bit_cast(uint32_t, (a - off) * dd), __builtin_bit_cast(uint32_t, (b - off) * dd)};
}

// sigmoid(g) through the hardware exponential and reciprocal (each within an ulp or two; exact at g = 0): the library's
// full-range expf and IEEE division are some twenty instructions per value, 128 values per lane
__device__ __forceinline__ float sigmoid(float g) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g)); }

constexpr float RESCALE_STEP = 8.0f;   // log2 units: the reference maximum of a row only moves in steps larger than this

// ---- per-type staging: raw tile of one kv head -> registers -> f16 rows in LDS ----
// Every thread owns a fixed set of items (key, chunk) of the tile: item x of thread tid is i = x * NTHR + tid,
// key = i / CPK, chunk = i % CPK. `raw` keeps what was loaded for them. A load names its address as
// gb[x] + vo[x][n]: gb = cache base + the base of the item's 16-key group (wave-uniform whenever 16 * CPK is a multiple
// of the wave size, so it sits in scalar registers), vo = the loop-invariant 32-bit offset of the item inside its group
// (row in the group * row bytes + offs()[n]); the loads then need no address arithmetic at all.
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef uint32_t __attribute__((may_alias)) u32a;   // the parked scale blocks are written as dwords and read as halves
typedef uint16_t __attribute__((may_alias)) u16a;
typedef const __attribute__((address_space(1))) char * gptr;      // global memory, so the loads are global_load (vmcnt only)
#define P1A_GLOAD(T, p) (*(const __attribute__((address_space(1))) T *) (p))
template <uint32_t KT, int D> struct stager;
// Which (key, chunk) of the 64-key tile item x of thread tid is. Wave-major whenever the chunks of a key divide a wave
// evenly: wave w owns keys 16 w .. 16 w + 15 - exactly one 16-key group, so one page base serves all its loads - and
// item x covers KPW = 64 / CPK of them. (Otherwise: items dealt out thread by thread over the whole tile.)
template <int CPK> struct item_map {
    static constexpr bool WAVE_MAJOR = CPK % 4 == 0 && CPK <= 64;
    static constexpr int KPW = WAVE_MAJOR ? 64 / CPK : 1;
    static __device__ __forceinline__ int key(int x, int tid) { return WAVE_MAJOR ? 16 * (tid >> 6) + x * KPW + (tid & 63) / CPK : (x * NTHR + tid) / CPK; }
    static __device__ __forceinline__ int cc(int x, int tid) { return WAVE_MAJOR ? (tid & 63) % CPK : (x * NTHR + tid) % CPK; }
};

template <int D> struct stager<P1A_KV_Q8_0, D> {
    static constexpr int CPK = D / 16;                    // 16-code chunks per key
    static constexpr int NPT = BN * CPK / NTHR;           // items per thread
    static constexpr int NOFF = 1;                        // codes
    // Sub-dword loads cost twice the issue time of a 16-byte one, so an item does not fetch its own f16 scale: each wave
    // fetches the scale blocks (D/32 scales) of the 16 keys its items belong to with ONE load per tile, parks them in a
    // small LDS area of its own and every lane picks its scales up from there.
    static constexpr bool SCALES_VIA_LDS = true;
    static constexpr int SB = (D / 32) * 2;               // bytes of scales per key head
    static_assert(BN * CPK % NTHR == 0, "tile must split evenly over the threads");
    struct raw { u4 w[NPT]; uint32_t d[NPT]; };           // d: one zero-extended f16 scale per item
    static __device__ __forceinline__ void offs(uint32_t * o, int cc) { o[0] = (D / 32) * 2 + cc * 16; }
    static __device__ __forceinline__ void load_item(raw & r, gptr gb, const uint32_t * vo, int x, int) {
        r.w[x] = P1A_GLOAD(u4, gb + vo[0]);
    }
    static constexpr int PARTS = 2;                       // 16-byte LDS stores per item
    static __device__ __forceinline__ void store_part(const raw & r, char * tile, int stride, int tid, int x, int part) {
        const int key = item_map<CPK>::key(x, tid), cc = item_map<CPK>::cc(x, tid);
        const uint32_t d16 = r.d[x];
        const h2 dd = __builtin_bit_cast(h2, d16 | (d16 << 16));
        const pair32 x0 = deq8x4(r.w[x][2 * part], dd), x1 = deq8x4(r.w[x][2 * part + 1], dd);
        *reinterpret_cast<u4 *>(tile + pf_lay<D>::key_off(key, stride) + cc * 32 + part * 16) = u4{x0.lo, x0.hi, x1.lo, x1.hi};
    }
};

template <int D> struct stager<P1A_KV_F16, D> {
    static constexpr int CPK = D / 8;                     // 16-byte chunks (8 halves) per key
    static constexpr int NPT = BN * CPK / NTHR;
    static constexpr int NOFF = 1;
    static constexpr bool SCALES_VIA_LDS = false;
    static constexpr int SB = 4;
    static_assert(BN * CPK % NTHR == 0, "tile must split evenly over the threads");
    struct raw { u4 w[NPT]; };
    static __device__ __forceinline__ void offs(uint32_t * o, int cc) { o[0] = cc * 16; }
    static __device__ __forceinline__ void load_item(raw & r, gptr gb, const uint32_t * vo, int x, int) {
        r.w[x] = P1A_GLOAD(u4, gb + vo[0]);
    }
    static constexpr int PARTS = 1;
    static __device__ __forceinline__ void store_part(const raw & r, char * tile, int stride, int tid, int x, int) {
        const int key = item_map<CPK>::key(x, tid), cc = item_map<CPK>::cc(x, tid);
        *reinterpret_cast<u4 *>(tile + pf_lay<D>::key_off(key, stride) + cc * 16) = r.w[x];
    }
};

template <int D> struct stager<P1A_KV_Q4_0, D> {
    static constexpr int CPK = D / 32;                    // 18-byte blocks per key: one block (32 values) per item
    static constexpr int NPT = (BN * CPK + NTHR - 1) / NTHR;
    static constexpr int NOFF = 1;
    static constexpr bool SCALES_VIA_LDS = false;
    static constexpr int SB = 4;
    struct raw { uint16_t h[NPT][9]; };
    static __device__ __forceinline__ void offs(uint32_t * o, int cc) { o[0] = cc * 18; }
    static __device__ __forceinline__ void load_item(raw & r, gptr gb, const uint32_t * vo, int x, int tid) {
        const int key = item_map<CPK>::key(x, tid);
        if (BN * CPK % NTHR == 0 || key < BN) {
            const gptr blk = gb + vo[0];   // 2-byte aligned
#pragma unroll
            for (int k = 0; k < 9; ++k) r.h[x][k] = P1A_GLOAD(uint16_t, blk + 2 * k);
        }
    }
    static constexpr int PARTS = 4;                       // part 0, 1: values 0..15 (low nibbles), part 2, 3: values 16..31
    static __device__ __forceinline__ void store_part(const raw & r, char * tile, int stride, int tid, int x, int part) {
        const int key = item_map<CPK>::key(x, tid), b = item_map<CPK>::cc(x, tid);
        if (!(BN * CPK % NTHR == 0 || key < BN)) return;
        const uint32_t d16 = r.h[x][0];
        const h2 dd = __builtin_bit_cast(h2, d16 | (d16 << 16));
        // byte j of the block: low nibble = value j, high nibble = value j + 16; this part covers bytes 8 (part & 1) .. + 7
        pair32 q[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int kb = 2 * (part & 1) + k;
            const uint32_t w = (uint32_t) r.h[x][1 + 2 * kb] | ((uint32_t) r.h[x][2 + 2 * kb] << 16);   // bytes 4 kb .. 4 kb + 3
            q[k] = deq4x4((part & 2 ? w >> 4 : w) & 0x0f0f0f0fu, dd);
        }
        *reinterpret_cast<u4 *>(tile + pf_lay<D>::key_off(key, stride) + b * 64 + part * 16) = u4{q[0].lo, q[0].hi, q[1].lo, q[1].hi};
    }
};

// whole-tile store (prologue): every part of every item
template <class S> __device__ __forceinline__ void store_tile(const typename S::raw & r, char * tile, int stride, int tid) {
#pragma unroll
    for (int x = 0; x < S::NPT; ++x)
#pragma unroll
        for (int part = 0; part < S::PARTS; ++part) S::store_part(r, tile, stride, tid, x, part);
}

// GROUPED: pages hold at least 16 positions (or the cache is contiguous), so a 16-key group has one base
__device__ __forceinline__ uint32_t lds_addr(const char * p) { return (uint32_t) (size_t) (const __attribute__((address_space(3))) char *) p; }
// 64 lanes x 16 bytes, global (scalar base + 32-bit lane offset) -> LDS at `lds` + a constant + 16 * lane, no registers in between
__device__ __forceinline__ void dma16_at(const char * sbase, uint32_t voff, uint32_t lds, int at) {
    asm volatile("s_add_u32 m0, %2, %3\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(voff), "s"(sbase), "s"(lds), "i"(at) : "memory", "m0", "scc");
}

// D <= 128: a wave keeps all the dims of its own 32 rows (the V^T reads are few enough), so no P^T changes hands, no barrier
// stands between the two products, and a workgroup fits twice on a CU: 68 KB of LDS, 256 registers. One workgroup's
// set-up, epilogue and tile latency then run beside the other's products - at D = 128 a tile's products take about as long
// as a tile takes to arrive. Measured with f16, 32 / 8 heads of 128 (registers -> LDS as pairs, LDS-direct as pairs, LDS-direct
// solo): 4096 tokens behind 12000 1227, 1029, 868 us (1.09 PFLOP/s); the first 2003 tokens 71, 59, 53 us; D = 64, 16 / 2 heads,
// 4096 behind 12000: 318, 319 (pairs), 275 us.
constexpr bool pf_solo(int D, bool dma) { return dma && D <= 128; }

template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

template <uint32_t KT, int D, bool GROUPED, bool DMA>
__global__ void __launch_bounds__(NTHR, pf_solo(D, DMA) ? 2 : 1) prefill_k(const pf_params P) {
    static_assert(!DMA || (KT == P1A_KV_F16 && GROUPED), "the LDS-direct loads move f16 rows, a 16-key group at a time");
    constexpr bool PAIR = !pf_solo(D, DMA);
    using C = pf_cfg<D>;
    using L = pf_lay<D>;
    using S = stager<KT, D>;
    extern __shared__ __attribute__((aligned(16))) char lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;
    // blockIdx.x -> (group of row blocks, kv head, block of the group): the blocks of a group share an XCD. Groups are dealt to
    // the XCDs in turn; with key splits a unit is (key split, kv head) with all of its row blocks, and an XCD may take a run of
    // `run` consecutive workgroups instead of whole units
    const int id = blockIdx.x, xcd = id & 7;
    int slot = id >> 3;
    if constexpr (!PAIR) { if (slot >= P.turn_a && slot < P.turn_b) slot = P.turn_a + P.turn_b - 1 - slot; }
    const int lin = P.run ? xcd * P.run + slot : ((slot / P.bpg) * 8 + xcd) * P.bpg + slot % P.bpg;
    const int vunit = lin / P.bpg, hh = lin - vunit * P.bpg;
    const int nunits = P.nbg * P.Hkv;
    if (vunit >= nunits * P.nks) return;
    const int ksp = vunit / nunits, unit = vunit - ksp * nunits;
    // longest blocks (most keys) first
    const int rb = (P.nbg - 1 - unit / P.Hkv) * P.bpg + hh, hk = unit % P.Hkv;
    if (rb >= P.nblk) return;                                 // (the last group need not be full)

    const int row0 = rb * 4 * P.rpw;                          // first row of the block
    const int wrow0 = row0 + P.rpw * wave;                    // first row of this wave
    const int wrows = min(P.rpw, P.R - wrow0);                // how many it has (<= 0: none)
    const int my_row = wrow0 + c;                             // this lane's query row
    const bool live = c < wrows;
    // row -> token (the multiplication is at most one short)
    auto tok_of = [&](int r) {
        const int t = (int) __umulhi((uint32_t) r, P.gqa_magic);
        return r - t * P.GQA >= P.GQA ? t + 1 : t;
    };
    const int my_tok = tok_of(min(my_row, P.R - 1));
    const int my_pos = P.p0 + my_tok;
    const int wave_vis = __builtin_amdgcn_readfirstlane(my_pos);  // every row of this wave sees the positions up to here
    const int pmax = P.p0 + tok_of(min(P.R, row0 + 4 * P.rpw) - 1);   // last position any row of the block sees
    // a row -> its index among the T * Hq rows of q, out, gate and the partials
    auto row_index = [&](int r) { const int t = tok_of(r); return (size_t) t * P.Hq + (size_t) hk * P.GQA + (r - t * P.GQA); };
    const int ntiles_all = pmax / BN + 1;                         // tiles the block sees
    // this workgroup's share of them: tiles tile_a .. tile_a + ntiles - 1
    int tile_a = 0, ntiles = ntiles_all;
    if (P.nks > 1) {
        const int tps = (ntiles_all + P.nks - 1) / P.nks;
        tile_a = ksp * tps;
        ntiles = min(tps, ntiles_all - tile_a);
        if (ntiles <= 0) {   // nothing left for this split: an empty partial (the merge skips it)
            if (g == 0 && live) {
                float * ml = P.part_ml + (row_index(my_row) * P.nks + ksp) * 2;
                ml[0] = NEG_INF;
                ml[1] = 0.f;
            }
            return;
        }
    }

    const int32_t * ptab = P.pg.pt ? (P.pg.rtab ? P.pg.pt + P.pg.rtab[0] : P.pg.pt) : nullptr;
    const size_t hb = KT == P1A_KV_F16 ? (size_t) D * 2 : KT == P1A_KV_Q8_0 ? (size_t) (D / 32) * 34 : (size_t) (D / 32) * 18;
    const size_t head_off = (size_t) hk * hb;

    // ---- Q^T operands (B: k = 16 dims per step, n = query row): lane (row c, half g) holds dims 16 ks + 8 g .. + 7 ----
    h8 qf[C::NKS];
    // fp32 rows of q, out, gate and the partials are moved whole, 16 bytes per lane in memory order: RPI rows of LPF lanes per
    // instruction, NRI instructions for 32 rows (a lane's own operands are 32 bytes of each of 32 rows per instruction: four
    // times the cache lines; 300 tokens, 24 / 4 heads of 256: 25.1 -> 24.8 us, with short blocks 17.6)
    constexpr int LPF = D / 4, RPI = 64 / LPF, NRI = 32 / RPI, N8 = 8 / RPI;   // (N8: instructions of 8 rows)
    const int wlast = wrows > 0 ? wrows - 1 : P.R - 1 - wrow0;   // the row that stands in for those past the wave's last
    auto row_at = [&](int i) { return i * RPI + lane / LPF; };   // the row of the wave that this lane moves in instruction i
    // the wave's Q rows -> f16 row images at `img` (rows padded by 16 bytes) -> operands. All loads first, then the conversions.
    auto load_q = [&](char * img, auto && between) {
        constexpr int QRS = 2 * D + 16;
        float4 a[NRI];
        auto fetch = [&](int i) { a[i] = *reinterpret_cast<const float4 *>(P.q + row_index(wrow0 + min(row_at(i), wlast)) * D + 4 * (lane % LPF)); };
#pragma unroll
        for (int i = 0; i < N8; ++i) fetch(i);
#pragma unroll
        for (int i = N8; i < NRI; ++i) a[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (P.rpw > 8) {
#pragma unroll
            for (int i = N8; i < NRI; ++i) fetch(i);
        }
        between();
        const float s = P.qscale;
#pragma unroll
        for (int i = 0; i < NRI; ++i)
            *reinterpret_cast<h4 *>(img + (i * RPI + lane / LPF) * QRS + (lane % LPF) * 8) = h4{(half_t) (a[i].x * s), (half_t) (a[i].y * s), (half_t) (a[i].z * s), (half_t) (a[i].w * s)};
#pragma unroll
        for (int ks = 0; ks < C::NKS; ++ks) {
            qf[ks] = *reinterpret_cast<const h8 *>(img + c * QRS + ks * 32 + g * 16);
            // Q stays in accumulation registers for the whole kernel: the matrix instructions read them in place, and
            // the vector registers are left to the tiles in flight
            if constexpr (PAIR) asm volatile("" : "+a"(qf[ks]));
        }
    };
    // where the images go before the tiles need the room: with LDS-direct tiles, whose K is on its way by then, two waves' into
    // each V stage (D = 64: the padded rows have an area behind the stages)
    char * const q_img = !DMA ? lds + wave * 32 * (2 * D + 16) : D == 64 ? lds + 2 * L::STAGE_B + wave * 32 * (2 * D + 16) : lds + (wave >> 1) * L::STAGE_B + L::KT_B + (wave & 1) * 32 * (2 * D + 16);
    if constexpr (!DMA) {
        load_q(q_img, [] {});
        __syncthreads();                                      // (the tiles that follow go over the images)
    }

    // Waves pair up for O^T: the pair (w, w ^ 1) shares its 64 query rows, each wave accumulating HALF the dims
    // (tiles HD * (w & 1) ..) for ALL 64 rows: a V^T fragment read from LDS then feeds two MFMAs (own rows, partner's
    // rows) instead of one, which halves the transposing reads - the slowest LDS traffic of the kernel. The price is
    // that P^T (and the rare rescale factors) of the partner come through LDS, behind one more barrier per tile.
    constexpr int NR = PAIR ? 2 : 1;                          // row blocks a wave accumulates
    constexpr int HD = C::NDT / NR;                           // dim tiles per wave
    static_assert(C::NDT % NR == 0, "the dims split over a pair of waves");
    const int dh = PAIR ? wave & 1 : 0;                       // which half of the dims
    f16x o[NR][HD];                                            // [0]: own rows, [1]: the partner's rows
    // softmax denominator of the own rows: this lane's share, per key half of a tile - the sum of the ROUNDED P values
    // (a packed dot product with ones, fp32 accumulation: v_dot2 keeps f16 denormals), so that it matches what
    // multiplies V. 16 vector instructions in the shadow of the S^T products instead of four more matrix instructions
    // per tile (-1.3 % of the call). Kept per (key half, lane half) and added up once, in a fixed order, at the end.
    float lp[2] = {0.f, 0.f};
    // The reference maximum of the own row (-inf: no visible key yet) rides in the S^T products as the value they accumulate
    // on: they deliver S - m, and exp2 takes them as they are.
    float m_run = NEG_INF;
    f16x neg_m;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        neg_m[i] = 0.f;
#pragma unroll
        for (int dt = 0; dt < HD; ++dt)
#pragma unroll
            for (int r = 0; r < NR; ++r) o[r][dt][i] = 0.f;
    }
    asm volatile("" : "+v"(neg_m));                          // (16 registers of one value: not to be rebuilt at every use)
    // exchange areas behind the tile stages: P^T of every wave (BN / 16 k-steps x 64 lanes x 16 bytes), then one float
    // per query row (rescale factor during the loop, denominator at the end)
    char * const xbase = lds + 2 * L::STAGE_B + (S::SCALES_VIA_LDS ? 2 * 4 * 16 * S::SB : 0);
    constexpr int PX_B = (BN / 16) * 64 * 16;
    char * const px_own = xbase + wave * PX_B, * const px_par = xbase + (wave ^ 1) * PX_B;
    float * const ax_own = reinterpret_cast<float *>(xbase + 4 * PX_B) + wave * 32;
    float * const ax_par = reinterpret_cast<float *>(xbase + 4 * PX_B) + (wave ^ 1) * 32;
    const h2 one2 = {(half_t) 1, (half_t) 1};

    // ---- addressing of the raw tile ----
    // A tile is four groups of 16 keys, one per wave. With pages of >= 16 positions (or a contiguous cache) a group lies
    // in one page, so its base is a scalar: one page-table entry per wave and tile, fetched with a hand-issued scalar
    // load (s_load_dword does not share the in-order vector-memory counter with the tile loads in flight) well before the
    // base is formed. Inside the group an item sits at a loop-invariant offset; only the tile that holds pmax clamps the
    // rows past it (they would otherwise read rows nobody has written); that tile's offsets are prepared once, up front.
    constexpr bool grouped = GROUPED;
    const int pmask = (1 << P.pg.psh) - 1;
    const int last_tile = ntiles_all - 1;                     // the tile that holds pmax
    using IM = item_map<S::CPK>;
    uint32_t voff[S::NPT][S::NOFF], voff_last[S::NPT][S::NOFF];
    int grp[S::NPT];                                             // (wave-major: all equal to the wave number)
#pragma unroll
    for (int x = 0; x < S::NPT; ++x) {
        const int key = min(IM::key(x, tid), BN - 1), cc = IM::cc(x, tid);
        grp[x] = key >> 4;
        uint32_t co[S::NOFF];
        S::offs(co, cc);
        const int room = pmax - (last_tile * BN + 16 * grp[x]);         // keys of the group before pmax (< 0: none)
        const int kl = min(key & 15, max(room, 0));
#pragma unroll
        for (int n = 0; n < S::NOFF; ++n) {
            voff[x][n] = (uint32_t) (key & 15) * (uint32_t) P.pg.rowb + co[n];
            voff_last[x][n] = (uint32_t) kl * (uint32_t) P.pg.rowb + co[n];
        }
    }
    // FAST: the wave's 16 keys of a tile lie in one page (or the cache is contiguous): one table entry, one scalar base;
    // otherwise every item and scale block has an entry of its own, asked for a step ahead of the tile too (AHEAD). (Looked up where
    // the loads are made, a tile took a round trip to L2 per row: the entry of the next row stood behind the load of this one.
    // Pages of 8, 1000 tokens behind 2000: f16, 24 / 4 heads of 256 312 -> 135 us, 32 / 8 of 128 162 -> 84; q8_0 of 256 252
    // -> 140; q4_0 of 128, one item a thread, 99 -> 81.) The build whose items are not dealt out wave by wave - q4_0 at D = 64, half an
    // item a thread - has no such chain, and it is faster looking up on the spot (4096 tokens behind 4096, 16 / 2 heads 216 us, 234 ahead).
    constexpr bool FAST = GROUPED && IM::WAVE_MAJOR, AHEAD = !FAST && IM::WAVE_MAJOR;
    struct gpages { int pg; int it[AHEAD ? S::NPT : 1], sb; };
    struct gbases { size_t go; gpages p; };
    // a group past the last position takes the base of the last one that holds a position: the LDS-direct loads then
    // fetch that group's 16 rows (all inside its page) instead of clamping row by row
    const int gclamp = DMA ? (pmax & ~15) : pmax;
    auto group_pages = [&](int tile) {
        gpages r;
        r.pg = 0;
        if constexpr (!FAST) {
            if (AHEAD && ptab) {
#pragma unroll
                for (int x = 0; x < S::NPT; ++x) r.it[AHEAD ? x : 0] = ptab[min(tile * BN + IM::key(x, tid), pmax) >> P.pg.psh];
                if constexpr (S::SCALES_VIA_LDS) r.sb = ptab[min(tile * BN + 16 * wave + (lane & 15), pmax) >> P.pg.psh];
            }
        } else if (ptab) {
            // (a load from the constant address space at a wave-uniform address is an s_load_dword whose wait the compiler
            // places itself, before the first use; the table does not change while the kernel runs)
            const int32_t * e = ptab + (__builtin_amdgcn_readfirstlane(min(tile * BN + 16 * wave, gclamp)) >> P.pg.psh);
            const size_t eu = (size_t) e;
            const uint32_t elo = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) eu);
            const uint32_t ehi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (eu >> 32));
            r.pg = *reinterpret_cast<const __attribute__((address_space(4))) int32_t *>(((size_t) ehi << 32) | elo);
        }
        return r;
    };
    auto group_bases = [&](int tile, gpages & gp) {
        gbases r;
        if constexpr (!FAST) { r.go = 0; r.p = gp; return r; }
        const int p = __builtin_amdgcn_readfirstlane(min(tile * BN + 16 * wave, gclamp));
        r.go = (ptab ? (size_t) gp.pg * P.pg.pstride + (size_t) (p & pmask) * P.pg.rowb : (size_t) p * P.pg.rowb) + head_off;
        return r;
    };
    // the head row of one position, whose page is known
    auto row_off = [&](int pos, int page) { return (ptab ? (size_t) page * P.pg.pstride + (size_t) (pos & pmask) * P.pg.rowb : (size_t) pos * P.pg.rowb) + head_off; };
    // where item x of `tile` starts: base (scalar registers when GROUPED) + 32-bit offsets
    struct iaddr { gptr base; uint32_t vo[S::NOFF]; };
    auto item_addr = [&](const char * cache, int tile, const gbases & gb, int x) {
        iaddr r;
        if constexpr (FAST) {
            r.base = (gptr) cache + gb.go;
            const bool is_last = tile == last_tile;
#pragma unroll
            for (int n = 0; n < S::NOFF; ++n) r.vo[n] = is_last ? voff_last[x][n] : voff[x][n];
        } else {   // pages shorter than a group (or items not dealt out wave by wave)
            const int key = min(IM::key(x, tid), BN - 1), pos = min(tile * BN + key, pmax);
            r.base = (gptr) cache + (AHEAD ? row_off(pos, gb.p.it[AHEAD ? x : 0]) : kv_off_tab(P.pg, ptab, pos) + head_off);
#pragma unroll
            for (int n = 0; n < S::NOFF; ++n) r.vo[n] = voff[x][n] - (uint32_t) (key & 15) * (uint32_t) P.pg.rowb;
        }
        return r;
    };
    auto load_tile = [&](typename S::raw & r, const char * cache, int tile, const gbases & gb) {
#pragma unroll
        for (int x = 0; x < S::NPT; ++x) {
            const iaddr ia = item_addr(cache, tile, gb, x);
            S::load_item(r, ia.base, ia.vo, x, tid);
        }
    };

    // ---- scale blocks (types that keep their scales apart from the codes) ----
    // Lane l of a wave (l mod 16) fetches the block of the l-th of the wave's 16 keys; all four quarters of the wave fetch
    // and park the same 16 blocks, which saves masking lanes off.
    constexpr bool SVL = S::SCALES_VIA_LDS;
    static_assert(!SVL || IM::WAVE_MAJOR, "parked scale blocks are per wave");
    constexpr int KPW = IM::KPW;
    struct sblk { uint32_t w[S::SB / 4]; };
    const int l16 = lane & 15;
    const int lkey = 16 * wave + l16;
    const uint32_t sb_full = (uint32_t) l16 * (uint32_t) P.pg.rowb;
    const uint32_t sb_last = (uint32_t) min(l16, max(pmax - (last_tile * BN + 16 * wave), 0)) * (uint32_t) P.pg.rowb;
    char * const ksc = lds + 2 * L::STAGE_B + wave * 16 * S::SB;           // this wave's parking area: K blocks
    char * const vsc = ksc + 4 * 16 * S::SB;                               // ... V blocks
    auto load_sblk = [&](const char * cache, int tile, const gbases & gb) {
        sblk r;
        size_t off;
        if constexpr (FAST) {
            off = gb.go + (tile == last_tile ? sb_last : sb_full);
        } else {
            off = row_off(min(tile * BN + lkey, pmax), gb.p.sb);
        }
        const gptr p_ = (gptr) cache + off;
        if constexpr (S::SB == 16) { const u4 t = P1A_GLOAD(u4, p_); r.w[0] = t[0]; r.w[1] = t[1]; r.w[2] = t[2]; r.w[3] = t[3]; }
        else if constexpr (S::SB == 8) { const u2v t = P1A_GLOAD(u2v, p_); r.w[0] = t[0]; r.w[1] = t[1]; }
        else r.w[0] = P1A_GLOAD(uint32_t, p_);
        return r;
    };
    auto park_sblk = [&](char * area, const sblk & b) {
#pragma unroll
        for (int j = 0; j < S::SB / 4; ++j) reinterpret_cast<u32a *>(area + l16 * S::SB)[j] = b.w[j];
    };
    auto pick_scales = [&](typename S::raw & r, const char * area) {
        if constexpr (SVL) {
#pragma unroll
            for (int x = 0; x < S::NPT; ++x)
                r.d[x] = *reinterpret_cast<const u16a *>(area + (x * KPW + lane / S::CPK) * S::SB + ((lane % S::CPK) >> 1) * 2);
        }
    };
    // prologue helper: a whole raw tile, scales included
    auto fetch_tile = [&](typename S::raw & r, const char * cache, char * area, int tile, const gbases & gb) {
        load_tile(r, cache, tile, gb);
        if constexpr (SVL) {
            const sblk b = load_sblk(cache, tile, gb);
            park_sblk(area, b);
            pick_scales(r, area);
        }
    };

    // Every workgroup walks its tiles in ascending order: those that share a kv head then ask for a tile within a step of
    // one another and find it in L2. (Each used to start at a tile of its own, to keep them off one L2 channel; the tiles then
    // came from the Infinity Cache: 4096 tokens behind 28672 2815 -> 2740 us without, 77 behind 16000 73.5 -> 69.6.)
    // Steps past the last one (the pipeline looks up to four tiles ahead) wrap around; nothing uses them.
    const int tile_z = tile_a + ntiles - 1;
    auto tile_after = [&](int tile) { return tile == tile_z ? tile_a : tile + 1; };
    const int tile0 = tile_a, tile1 = tile_after(tile0), tile2 = tile_after(tile1);

    // S^T of one tile: 32-key halves u = 0, 1
    auto qk = [&](const char * kt, f16x (&s)[2]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[u][i] = 0.f;
            const char * krow = kt + L::k_lane(c) + L::k_half(u) + g * 16;
#pragma unroll
            for (int ks = 0; ks < C::NKS; ++ks) {
                const h8 a = *reinterpret_cast<const h8 *>(krow + ks * 32);
                s[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[ks], s[u], 0, 0, 0);
            }
        }
    };

    // ---- LDS-direct tile loads (DMA): wave w moves the NJ blocks of its 16-key group; instruction j takes the keys j, j + NJ,
    // ... of the group (16 bytes of a row per lane): the group's base and a loop-invariant lane offset per
    // instruction - registers that spare the loop two 64-bit scalar additions a load. Rows past the last position are fetched as they are (the group lies
    // inside one page, or inside the cache when it is contiguous - the host checks): as K they only make scores that the
    // mask replaces; as V they are overwritten with zeros in LDS once the tile has landed (P = 0 times anything finite).
    constexpr int NJ = L::NJ, LPR = 64 / L::RPB;              // loads per tile and wave; lanes per row
    uint32_t dma_vo[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) dma_vo[j] = (uint32_t) (NJ * (lane / LPR) + j) * (uint32_t) P.pg.rowb + (uint32_t) (lane % LPR) * 16u;
    const uint32_t k_dst = lds_addr(lds) + NJ * wave * L::KB, v_dst = lds_addr(lds) + L::KT_B + NJ * wave * L::VB;   // this wave's blocks of stage 0
    auto dma_k = [&](const gbases & gb, int stage, int j) { dma16_at(P.kc + gb.go, dma_vo[j], k_dst, stage * L::STAGE_B + j * L::KB); };
    auto dma_v = [&](const gbases & gb, int stage, int j) { dma16_at(P.vc + gb.go, dma_vo[j], v_dst, stage * L::STAGE_B + j * L::VB); };
    auto zero_v_tail = [&](int tile, char * vtile) {
        if (tile != last_tile) return;
        const int room = pmax - (last_tile * BN + 16 * wave);             // the wave's last key that exists (< 0: none)
        for (int kg = max(room + 1, 0); kg < 16; ++kg)
            if (lane * 8 < L::RB) *reinterpret_cast<u2v *>(vtile + L::key_off(16 * wave + kg, L::VB) + lane * 8) = u2v{0u, 0u};
    };

    // ---- prologue: K(0), V(0), K(1) in LDS; (staged through registers: V(1) and K(2) on their way); S^T(0) ----
    typename S::raw rk, rv;
    sblk sk, sv;                                           // scale blocks that belong to rk, rv
    // group bases of the V tile and (DMA) the K tile that the next step fetches, table entry of the K tile of the one after
    gbases gb_v, gb_k;
    gpages gp_ahead;
    if constexpr (DMA) {
        gpages g0 = group_pages(tile0), g1 = group_pages(tile1), g2 = group_pages(tile2);
        const gbases b0 = group_bases(tile0, g0);
        gb_v = group_bases(tile1, g1);
        load_q(q_img, [&] {
#pragma unroll
            for (int j = 0; j < NJ; ++j) dma_k(b0, 0, j);
#pragma unroll
            for (int j = 0; j < NJ; ++j) dma_k(gb_v, 1, j);
        });
        gb_k = group_bases(tile2, g2);
        gp_ahead = group_pages(tile_after(tile2));
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int j = 0; j < NJ; ++j) dma_v(b0, 0, j);         // (over the Q images, which every wave is done with)
    } else {
        gpages g0 = group_pages(tile0), g1 = group_pages(tile1), g2 = group_pages(tile2);
        const gbases b0 = group_bases(tile0, g0), b1 = group_bases(tile1, g1);
        gb_v = group_bases(tile2, g2);
        fetch_tile(rk, P.kc, ksc, tile0, b0);
        fetch_tile(rv, P.vc, vsc, tile0, b0);
        store_tile<S>(rk, lds, L::KB, tid);
        store_tile<S>(rv, lds + L::KT_B, L::VB, tid);
        fetch_tile(rk, P.kc, ksc, tile1, b1);
        store_tile<S>(rk, lds + L::STAGE_B, L::KB, tid);
        load_tile(rv, P.vc, tile1, b1);
        load_tile(rk, P.kc, tile2, gb_v);
        if constexpr (SVL) { sv = load_sblk(P.vc, tile1, b1); sk = load_sblk(P.kc, tile2, gb_v); }
    }
    if constexpr (!DMA) __syncthreads();
    // S^T of two tiles: that of the tile in hand and that of the next, taking turns. (DMA: a step is written out twice, so that
    // neither the values nor the LDS addresses of the two stages have to be moved about. A step is then 64 matrix and 346
    // other instructions instead of 461 - one wave per SIMD issues one in four clocks - and its maximum and denominator
    // sums sit beside matrix instructions instead of behind the last one: 3060 -> 2860 us for 4096 tokens behind 28672.)
    f16x s_a[2], s_b[2];
    qk(lds, s_a);
    // Masking and the row maximum of a tile are done one step ahead of its softmax (in the shadow of the O^T products of
    // the tile before it): value i of half u of a lane's S^T column is key k0 + key_of(u, i) + KG g of the lane's own row.
    auto mask_max = [&](f16x (&sv_)[2], int k0_, int idx, float m) {
        const int su = idx >> 4, i = idx & 15;
        sv_[su][i] = L::key_of(su, i) <= my_pos - k0_ - L::KG * g ? sv_[su][i] : NEG_INF;
        return fmaxf(m, sv_[su][i]);
    };
    // both lane halves of a row -> the row's maximum
    auto row_max = [&](float m) { return max_swap32(m); };
    float mloc = NEG_INF;
#pragma unroll
    for (int idx = 0; idx < 32; ++idx) mloc = mask_max(s_a, tile0 * BN, idx, mloc);
    mloc = row_max(mloc);
    // (the first step overwrites K(0) while it runs; every wave has to be done reading it)
    if constexpr (DMA) {
        if constexpr (!PAIR) {                                // (pairs wait for V(0) at their first exchange)
            wait_vm<0>();
            zero_v_tail(tile0, lds + L::KT_B);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }

    int tile_c = tile0, tile_n = tile1, tile_nn = tile2;      // the tiles of this step, the next and the one after
    auto step = [&](auto par, f16x (&s)[2], f16x (&s_next)[2]) {   // s: S^T of this step's tile, masked; mloc: its row maximum
        const int ST = par;
        char * const st_cur = lds + ST * L::STAGE_B;                   // holds K(it) (done with) and V(it)
        char * const st_nxt = lds + (1 - ST) * L::STAGE_B;             // holds K(it+1); V(it-1) is done with
        const int k0n = tile_n * BN;
        gpages gp_k;
        if constexpr (!DMA) gp_k = group_pages(tile_after(tile_nn));   // entries for the K fetch at the end of this step

        // Lazy reference maximum: m_run follows the row maximum (mloc, relative to it) only when that has grown by more than
        // RESCALE_STEP, so P stays below 2^RESCALE_STEP (well inside f16) and the accumulators are rescaled a handful of times
        // per row instead of at every tile. A row that has seen no visible key yet just adopts its first maximum (mloc = -inf
        // never moves anything; the exponentials of such a row are 0).
        const bool fresh = m_run == NEG_INF;
        const bool move = mloc > (fresh ? NEG_INF : RESCALE_STEP);
        float alpha = 1.0f;
        if (__builtin_expect(__any(move), 0)) {
            const float shift = move ? mloc : 0.0f;
            if (move) {
                alpha = fresh ? 1.0f : __builtin_amdgcn_exp2f(-shift);   // (fresh: nothing accumulated)
                m_run = (fresh ? 0.0f : m_run) + shift;
            }
            lp[0] *= alpha;
            lp[1] *= alpha;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                neg_m[i] = m_run == NEG_INF ? 0.0f : -m_run;
                s[0][i] -= shift;
                s[1][i] -= shift;
#pragma unroll
                for (int dt = 0; dt < HD; ++dt) o[0][dt][i] *= alpha;
            }
            asm volatile("" : "+v"(neg_m));
        }
        // ---- stream 1: S^T(it+1) on the matrix pipe; stream 2: P^T(it) = exp2(S^T(it) - m) on the vector pipe ----
        // Written step by step, one MFMA per step, with a scheduling fence after each: the LDS read of the K fragment
        // PF_K steps ahead, the MFMA, and a slice of the softmax that fits in the MFMA's shadow.
        h8 pb[BN / 16];
        constexpr int NQK = 2 * C::NKS, VPS = 32 / NQK, PF_K = 4;
        static_assert(32 % NQK == 0 && (VPS == 1 || VPS % 2 == 0), "softmax slices must tile the 32 values of a lane");
        const char * krow = st_nxt + L::k_lane(c) + g * 16;
        auto kfrag = [&](int k) { return *reinterpret_cast<const h8 *>(krow + L::k_half(k / C::NKS) + (k % C::NKS) * 32); };
        h8 fr[NQK];
#pragma unroll
        for (int k = 0; k < PF_K; ++k) fr[k] = kfrag(k);
#pragma unroll
        for (int k = 0; k < NQK; ++k) {
            if (k + PF_K < NQK) fr[k + PF_K] = kfrag(k + PF_K);
            if constexpr (DMA) {   // one tile load every other step: K(it+2) first (it is needed first), then V(it+1)
                if (k % 2 == 0) {
                    const int j = k / 2;
                    if (j < NJ) dma_k(gb_k, ST, j);                    // over K(it)
                    else if (j < 2 * NJ) dma_v(gb_v, 1 - ST, j - NJ);  // over V(it-1)
                }
            }
            const int u = k / C::NKS;
            s_next[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[k], qf[k % C::NKS], k % C::NKS ? s_next[u] : neg_m, 0, 0, 0);
            if constexpr (SVL) {   // the scales of the raw tiles fetched one step ago: through LDS to the lanes that use them
                if (k == NQK - 4) { park_sblk(ksc, sk); park_sblk(vsc, sv); }
                if (k == NQK - 2) { pick_scales(rk, ksc); pick_scales(rv, vsc); }
            }
#pragma unroll
            for (int v = 0; v < VPS; ++v) {
                const int idx = k * VPS + v, su = idx >> 4, i = idx & 15;
                s[su][i] = __builtin_amdgcn_exp2f(s[su][i]);
                if (idx & 1) {   // packed conversion (round to nearest even), two values per instruction
                    const h2 pr = __builtin_convertvector(f2v{s[su][i - 1], s[su][i]}, h2);
                    lp[su] = __builtin_amdgcn_fdot2(pr, one2, lp[su], false);
                    asm volatile("" : "+v"(lp[su]));   // (here, in the shadow of this product, not at the end of the step)
                    pb[idx >> 3][(idx & 7) - 1] = pr[0];
                    pb[idx >> 3][idx & 7] = pr[1];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- O^T += V^T(it) P^T: set-up. V(it) has been in LDS since the last barrier, so its first fragments are asked
        // for ahead of the exchange: their latency hides behind it ----
        // Slot e of lane half g in k-step ps is row 16 (ps % 2) + 4 g + e (e < 4) of half ps / 2, or row + 8 for e - 4
        const int i16 = lane & 15, blk = lane >> 4;        // 16-lane block: dims 16 (blk & 1) .., lane half blk >> 1 == g
        const int kk = i16 >> 2, jq = i16 & 3;
        const char * vbase = st_cur + L::KT_B + L::v_lane(4 * g + kk) + (16 * (blk & 1) + 4 * jq) * 2 + dh * HD * 64;
        // per k-step: HD fragments of V^T, each multiplied with the own and the partner's P^T, then the denominator
        constexpr int NFR = (BN / 16) * HD, PF_V = 3;
        constexpr int NP = 2 * S::NPT * S::PARTS;                             // store parts: K items, then V items
        struct vfrag { s4 lo, hi; };
        auto vread = [&](int f) {
            const char * p0_ = vbase + (f % HD) * 64;
            return vfrag{__builtin_amdgcn_ds_read_tr16_b64_v4i16((s4 __attribute__((address_space(3))) *) (p0_ + L::v_lo(f / HD))),
                         __builtin_amdgcn_ds_read_tr16_b64_v4i16((s4 __attribute__((address_space(3))) *) (p0_ + L::v_hi(f / HD)))};
        };
        vfrag vf[NFR];
        if constexpr (!PAIR || !DMA) {
#pragma unroll
            for (int f = 0; f < PF_V && f < NFR; ++f) vf[f] = vread(f);
        }
        if constexpr (PAIR) {
            // ---- hand P^T and the rescale factor of the own rows to the partner ----
#pragma unroll
            for (int ps = 0; ps < BN / 16; ++ps) *reinterpret_cast<h8 *>(px_own + (ps * 64 + lane) * 16) = pb[ps];
            ax_own[c] = alpha;                                    // (both lane halves: the same value)
            // (the V(it) loads of the previous step are older than this step's 2 NJ: they have landed when those are left)
            if constexpr (DMA) {
                wait_vm<2 * NJ>();
                zero_v_tail(tile_c, st_cur + L::KT_B);
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        // ---- stream 1: O^T += V^T(it) P^T on the matrix pipe; stream 2: masking and row maximum of S^T(it+1) (and K(it+2),
        // V(it+1) -> f16 tiles in LDS when they are staged through registers) ----
        {
            if constexpr (PAIR && DMA) {
#pragma unroll
                for (int f = 0; f < PF_V && f < NFR; ++f) vf[f] = vread(f);
            }
            float alpha_p = 1.0f;
            h8 pp[BN / 16];
            if constexpr (PAIR) {
                alpha_p = ax_par[c];                                              // (needed before the partner's first product)
                pp[0] = *reinterpret_cast<const h8 *>(px_par + lane * 16);
            }
            constexpr int MPS = 32 / NFR;                                          // next tile's values masked per step
            static_assert(32 % NFR == 0, "mask slices must tile the 32 values of a lane");
            mloc = NEG_INF;
#pragma unroll
            for (int f = 0; f < NFR; ++f) {
                if (f + PF_V < NFR) vf[f + PF_V] = vread(f + PF_V);
                const int ps = f / HD, dt = f % HD;
                if (PAIR && dt == 0 && ps + 1 < BN / 16) pp[ps + 1] = *reinterpret_cast<const h8 *>(px_par + ((ps + 1) * 64 + lane) * 16);
                const h4 l4 = __builtin_bit_cast(h4, vf[f].lo), h4_ = __builtin_bit_cast(h4, vf[f].hi);
                const h8 a = {l4[0], l4[1], l4[2], l4[3], h4_[0], h4_[1], h4_[2], h4_[3]};
                o[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb[ps], o[0][dt], 0, 0, 0);
                if constexpr (PAIR) {
                    if (f == 0 && __builtin_expect(__any(alpha_p != 1.0f), 0)) {   // the partner's rows moved their reference maximum
#pragma unroll
                        for (int i = 0; i < 16; ++i)
#pragma unroll
                            for (int d2 = 0; d2 < HD; ++d2) o[1][d2][i] *= alpha_p;
                    }
                    o[1][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pp[ps], o[1][dt], 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < MPS; ++v) mloc = fmaxf(mloc, s_next[(f * MPS + v) >> 4][(f * MPS + v) & 15]);
                asm volatile("" : "+v"(mloc));
                if constexpr (DMA) {   // where the next step's tiles come from
                    if (f == 1) { gb_v = gb_k; gb_k = group_bases(tile_after(tile_nn), gp_ahead); }
                    if (f == 2) gp_ahead = group_pages(tile_after(tile_after(tile_nn)));
                }
#pragma unroll
                for (int pt = DMA ? NP : f * NP / NFR; pt < (f + 1) * NP / NFR; ++pt) {
                    const int item = pt / S::PARTS, part = pt % S::PARTS;
                    if (item < S::NPT) S::store_part(rk, st_cur, L::KB, tid, item, part);                          // K(it+2) over K(it)
                    else               S::store_part(rv, st_nxt + L::KT_B, L::VB, tid, item - S::NPT, part);       // V(it+1) over V(it-1)
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // A tile that every row of the wave sees whole - all but the last few of a block - is not masked: the 64 compares
            // and selects run for the others only, out of line (with S - m straight from the products 257 -> 127 vector
            // instructions a tile, 4096 tokens behind 28672 3182 -> 3060 us)
            if (__builtin_expect(k0n + BN - 1 > wave_vis, 0)) {
                mloc = NEG_INF;
#pragma unroll
                for (int idx = 0; idx < 32; ++idx) mloc = mask_max(s_next, k0n, idx, mloc);
            }
        }

        mloc = row_max(mloc);
        // ---- raw loads of K(it+3), V(it+2): one whole step to arrive. Issued back to back: a vector memory instruction
        // holds the wave for as long as the CU's address path needs for it, wherever it is placed ----
        if constexpr (DMA) {
            if constexpr (PAIR) wait_vm<NJ>();                      // K(it+2) has landed; V(it+1) has until the next exchange
            else {
                wait_vm<0>();
                zero_v_tail(tile_n, st_nxt + L::KT_B);
            }
        } else {
            const int tile_3 = tile_after(tile_nn);
            const gbases gb_3 = group_bases(tile_3, gp_k);
            load_tile(rk, P.kc, tile_3, gb_3);
            load_tile(rv, P.vc, tile_nn, gb_v);
            if constexpr (SVL) { sk = load_sblk(P.kc, tile_3, gb_3); sv = load_sblk(P.vc, tile_nn, gb_v); }
            gb_v = gb_3;
        }
        tile_c = tile_n;
        tile_n = tile_nn;
        tile_nn = tile_after(tile_nn);
        // LDS stores retired, then the barrier (without the global-memory fence of __syncthreads())
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    if constexpr (DMA) {
        for (int it = 0;;) {
            step(std::integral_constant<int, 0>{}, s_a, s_b);
            if (++it == ntiles) break;
            step(std::integral_constant<int, 1>{}, s_b, s_a);
            if (++it == ntiles) break;
        }
    } else {   // (staged through registers there are none left for two copies)
        for (int it = 0; it < ntiles; ++it) {
            step(it & 1, s_a, s_b);
            s_a[0] = s_b[0];
            s_a[1] = s_b[1];
        }
    }

    // ---- epilogue: the pair swaps denominators, then each wave normalises, gates and stores its half of the dims of
    // all 64 rows. Lane (row c, half g) holds dims 32 dt + 8 (i / 4) + 4 g + (i % 4) of tile dt ----
    const float l_own = (lp[0] + __shfl_xor(lp[0], 32)) + (lp[1] + __shfl_xor(lp[1], 32));
    if constexpr (PAIR) { if (g == 0) ax_own[c] = l_own; }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (also: no tile load is left in flight)
    const float l_par = PAIR ? ax_par[c] : 0.f;
    const bool part = P.nks > 1;   // one of several key splits: the unnormalised partial of every row, for the merge
    if (part && g == 0 && live) {
        float * ml = P.part_ml + (row_index(my_row) * P.nks + ksp) * 2;
        ml[0] = m_run;
        ml[1] = l_own;
    }
    // Full blocks, two workgroups on a CU: each lane stores the 16 bytes it holds of its row, which the other workgroup's products
    // cover. Against the way below: 2003 tokens, 16 / 2 heads of 64 28.5 -> 27.2 us, 8 / 8 of 128 35.2 -> 34.2; 32 / 8 of 128
    // 54.1 -> 53.7; 24 / 4 of 128, 4096 tokens 116.9 -> 118.4, the one of thirty calls that loses more than the runs differ. (Short
    // blocks are alone on their CU: 40 tokens behind 100 9.7 us below, 11.2 this way.)
    if (!PAIR && P.rpw == 32) {
        const float inv = part ? 1.0f : 1.0f / l_own;
        const size_t rr = row_index(min(my_row, P.R - 1));
        f4 gt[HD][4];
        if (P.gate)
#pragma unroll
            for (int dt = 0; dt < HD; ++dt)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) gt[dt][q4] = *reinterpret_cast<const f4 *>(P.gate + rr * D + 32 * dt + 8 * q4 + 4 * g);
        if (live) {
            float * orow = P.out + (part ? rr * P.nks + ksp : rr) * D;
#pragma unroll
            for (int dt = 0; dt < HD; ++dt)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    f4 v = {o[0][dt][4 * q4] * inv, o[0][dt][4 * q4 + 1] * inv, o[0][dt][4 * q4 + 2] * inv, o[0][dt][4 * q4 + 3] * inv};
                    if (P.gate)
#pragma unroll
                        for (int x = 0; x < 4; ++x) v[x] *= sigmoid(gt[dt][q4][x]);
                    *reinterpret_cast<f4 *>(orow + 32 * dt + 8 * q4 + 4 * g) = v;
                }
        }
        return;
    }
    // through LDS, where a row is put together (4 D bytes and 16 of padding; the tiles are done with), to whole rows in memory
    constexpr int ORS = 4 * D + 16;
    const int d4 = 4 * (lane % LPF);
    // f16 caches and copies: all of the wave's gate rows are asked for before the first result is put down: eight at a time, each batch
    // behind the stores of the one before, a round trip to memory stood in front of every quarter of the rows (prep and prefill of the first
    // 512 tokens, f16, 24 / 4 heads of 256 37.8 -> 36.1 us, pages of 4 47.1 -> 45.8; 32 / 8 of 128 31.1 -> 30.3). Not where tiles are converted
    // inside: with that many more registers asked for behind it the compiler arranges their key loop otherwise, and slower, gate or none
    // (150 tokens behind 17112, 8 / 8 heads of 256, q4_0 69.2 us, 71.9 so; 77 behind 17000, 24 / 4 71.0 and 73.3; q8_0 71.9 and 72.4).
    constexpr bool GATES_AHEAD = KT == P1A_KV_F16;
    f4 gt[GATES_AHEAD ? NRI : N8];
    auto fetch_gate = [&](int i) { gt[GATES_AHEAD ? i : i % N8] = *reinterpret_cast<const f4 *>(P.gate + row_index(wrow0 + min(row_at(i), wlast)) * D + d4); };
    if (GATES_AHEAD && P.gate) {
#pragma unroll
        for (int i = 0; i < N8; ++i) fetch_gate(i);
        if (wrows > 8) {
#pragma unroll
            for (int i = N8; i < 2 * N8; ++i) fetch_gate(i);
        }
        if (wrows > 16) {
#pragma unroll
            for (int i = 2 * N8; i < NRI; ++i) fetch_gate(i);
        }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const float inv = part ? 1.0f : 1.0f / (r ? l_par : l_own);
        char * const orow = lds + (32 * (r ? wave ^ 1 : wave) + c) * ORS + dh * HD * 128 + 16 * g;
#pragma unroll
        for (int dt = 0; dt < HD; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                *reinterpret_cast<f4 *>(orow + 128 * dt + 32 * q4) = f4{o[r][dt][4 * q4] * inv, o[r][dt][4 * q4 + 1] * inv, o[r][dt][4 * q4 + 2] * inv, o[r][dt][4 * q4 + 3] * inv};
    }
    const char * const img = lds + (32 * wave + lane / LPF) * ORS + (lane % LPF) * 16;
#pragma unroll
    for (int i0 = 0; i0 < NRI; i0 += N8) {
        f4 v[N8];
        if (!GATES_AHEAD && P.gate) {
#pragma unroll
            for (int i = 0; i < N8; ++i) fetch_gate(i0 + i);
        }
        if (PAIR && i0 == 0) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int i = 0; i < N8; ++i) v[i] = *reinterpret_cast<const f4 *>(img + (i0 + i) * RPI * ORS);
        if (P.gate) {
#pragma unroll
            for (int i = 0; i < N8; ++i)
#pragma unroll
                for (int x = 0; x < 4; ++x) v[i][x] *= sigmoid(gt[GATES_AHEAD ? i0 + i : i][x]);
        }
        // (f16 tiles, D = 256: results, which nothing here reads again, go past the caches: 600 tokens behind 300, 24 / 4 heads, f16 53.9 -> 51.1 us, 2000, 32 / 8, q8_0
        // 157 -> 151. What reads them next gives most of it back: the first 4096 of 24 / 4, f16, alone 252 -> 239, with a cast to f16 behind the call 271.8
        // and 272.5, with that and a product of 5120 columns 525.8 and 524.8; seven calls of 600 ... 4096 tokens alone 1.02 times as fast in the
        // mean, with the cast 0.996 (0.988 - 1.009), with both 1.004 (0.997 - 1.018).
        // Not partials, which the merge reads at once: q4_0, 77 behind 16000 71.6 -> 73.2.)
        if constexpr (DMA && PAIR) {
            f4 * po[N8];
#pragma unroll
            for (int i = 0; i < N8; ++i) {
                const size_t row = row_index(wrow0 + row_at(i0 + i));
                po[i] = reinterpret_cast<f4 *>(P.out + (part ? row * P.nks + ksp : row) * D + d4);
            }
            if (!part) {
#pragma unroll
                for (int i = 0; i < N8; ++i) if (row_at(i0 + i) < wrows) __builtin_nontemporal_store(v[i], po[i]);
            } else {
#pragma unroll
                for (int i = 0; i < N8; ++i) if (row_at(i0 + i) < wrows) *po[i] = v[i];
                asm volatile("");                             // (or the two would be merged into one, through the caches)
            }
        } else {
#pragma unroll
            for (int i = 0; i < N8; ++i) {
                const size_t row = row_index(wrow0 + row_at(i0 + i));
                if (row_at(i0 + i) < wrows) *reinterpret_cast<f4 *>(P.out + (part ? row * P.nks + ksp : row) * D + d4) = v[i];
            }
        }
        if ((i0 + N8) * RPI >= wrows) break;
    }
}

template <uint32_t KT, int D, bool GROUPED, bool DMA = false>
int launch_pf_g(const pf_params & P, hipStream_t s) {
    using L = pf_lay<D>;
    constexpr int lds = 2 * L::STAGE_B + (stager<KT, D>::SCALES_VIA_LDS ? 2 * 4 * 16 * stager<KT, D>::SB : 0) +
                    (pf_solo(D, DMA) ? (D == 64 ? BM * (2 * D + 16) : 0) : 4 * (BN / 16) * 64 * 16 + 4 * 32 * 4);
    static_assert(BM * (4 * D + 16) <= lds, "the output rows fit where the tiles (and P^T) were");
    // (the attribute belongs to the function on ONE device: remembered per device, set again on another)
    static std::atomic<uint32_t> attr_set{0};
    int dev = 0;
    (void) hipGetDevice(&dev);
    const uint32_t bit = 1u << (dev & 31);
    if (!(attr_set.load(std::memory_order_acquire) & bit)) {
        if (hipFuncSetAttribute((const void *) prefill_k<KT, D, GROUPED, DMA>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) {
            (void) hipGetLastError();
            set_error("p1a_attn_prefill: cannot reserve %d bytes of LDS", lds);
            return P1A_E_LAUNCH;
        }
        attr_set.fetch_or(bit, std::memory_order_release);
    }
    const int units = P.nbg * P.Hkv * P.nks;
    const int slots = P.run ? P.run : ((units + 7) / 8) * P.bpg;
    pf_params Q = P;
    Q.turn_a = Q.turn_b = 0;
    // Two workgroups to a compute unit, which an XCD deals them to in turn: the unit of slot s also gets slot s + per. Longest blocks first
    // would give it two long ones (63 blocks of 1 ... 32 tiles: 32 + 16 ... 17 + 1 tiles); the second round is taken in reverse
    // (33 each). First 2003 tokens, 32 / 8 heads of 128, f16, prep included 85.0 -> 81.2 us, 24 / 4 of 64 37.1 -> 34.5. What fits
    // one round is as it was; calls of more than two have their second one reversed too and are level (70 drawn prefills 0.98 - 1.10).
    if (pf_solo(D, DMA) && P.nks == 1) {
        const int per = std::max(cu_count() / 8, 1);          // compute units of an XCD
        if (slots > per) { Q.turn_a = per; Q.turn_b = std::min(2 * per, slots); }
    }
    prefill_k<KT, D, GROUPED, DMA><<<slots * 8, NTHR, lds, s>>>(Q);
    return launched();
}
template <uint32_t KT, int D>
int launch_pf(const pf_params & P, hipStream_t s) {
    const bool grouped = !P.pg.pt || P.pg.psh >= 4;
    if constexpr (KT == P1A_KV_F16) {
        // (rows of whole 16-byte units at 16-byte aligned addresses: what a 16-byte load per lane needs)
        // and whole 16-key groups that can be read: always inside a page; inside a contiguous cache when it holds them
        const bool groups_ok = P.pg.pt || ((P.p0 + P.T - 1) | 15) < P.n_rows;
        if (grouped && groups_ok && P.pg.rowb % 16 == 0 && P.pg.rowb * 16 < (1ull << 32)) return launch_pf_g<KT, D, true, true>(P, s);
    }
    return grouped ? launch_pf_g<KT, D, true>(P, s) : launch_pf_g<KT, D, false>(P, s);
}

}   // namespace

namespace {
// Staging pass of the scratch variant: positions 0 .. n-1 of one sequence of a q8_0 / q4_0 cache -> contiguous f16 rows
// [n][Hkv][D] (K, then V). Same conversion as the in-kernel stagers (code * f16 scale, rounded once to f16), so the
// attention kernel sees the very tiles it would have built itself. One thread per 16 codes (q8_0), per quarter of a block (q4_0: a
// thread per block had 18 two-byte loads one behind the other and stores of 16 bytes 64 apart; 4012 positions of 4 heads of 256 9.2 -> 6.4 us).
template <uint32_t KT>
__global__ void __launch_bounds__(256) dq_k(const char * kc, const char * vc, kv_view pg, int n, int Hkv, int D, char * ko, char * vo) {
    const int32_t * ptab = pg.pt ? (pg.rtab ? pg.pt + pg.rtab[0] : pg.pt) : nullptr;
    const int per = KT == P1A_KV_Q8_0 ? 16 : 8;                // values per item
    const int ipr = Hkv * D / per;                             // items per position
    int row, it;
    if ((ipr & (ipr - 1)) == 0) {
        const long long idx = (long long) blockIdx.x * 256 + threadIdx.x;
        row = (int) (idx >> __builtin_ctz(ipr));
        it = (int) idx & (ipr - 1);
    } else {   // (a 64-bit division: 0.3 us of the 6.6 that 4012 positions would take)
        const long long idx = (long long) blockIdx.x * 256 + threadIdx.x;
        row = (int) (idx / ipr);
        it = (int) (idx - (long long) row * ipr);
    }
    if (row >= n) return;
    const size_t off = kv_off_tab(pg, ptab, row);
    const int iph = D / per, h = it >> __builtin_ctz(iph), cc = it & (iph - 1);   // (D is 64, 128 or 256)
    const size_t orow = ((size_t) row * Hkv + h) * D * 2;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        const char * src = (which ? vc : kc) + off;
        char * dst = (which ? vo : ko) + orow;
        if constexpr (KT == P1A_KV_Q8_0) {
            const char * head = src + (size_t) h * (D / 32) * 34;
            const u4 w = *reinterpret_cast<const u4 *>(head + (D / 32) * 2 + cc * 16);
            const uint32_t d16 = *reinterpret_cast<const uint16_t *>(head + (cc >> 1) * 2);
            const h2 dd = __builtin_bit_cast(h2, d16 | (d16 << 16));
            const pair32 x0 = deq8x4(w[0], dd), x1 = deq8x4(w[1], dd), x2 = deq8x4(w[2], dd), x3 = deq8x4(w[3], dd);
            u4 * o = reinterpret_cast<u4 *>(dst + cc * 32);
            o[0] = u4{x0.lo, x0.hi, x1.lo, x1.hi};
            o[1] = u4{x2.lo, x2.hi, x3.lo, x3.hi};
        } else {
            const uint16_t * blk = reinterpret_cast<const uint16_t *>(src + ((size_t) h * (D / 32) + (cc >> 2)) * 18);
            const uint32_t d16 = blk[0];
            const h2 dd = __builtin_bit_cast(h2, d16 | (d16 << 16));
            // quarter 0, 1: the low nibbles of bytes 0 .. 7, 8 .. 15 (values 0 .. 15), 2, 3: the high ones
            const uint16_t * b = blk + 1 + 4 * (cc & 1);
            const int sh = cc & 2 ? 4 : 0;
            const uint32_t w0 = (uint32_t) b[0] | ((uint32_t) b[1] << 16), w1 = (uint32_t) b[2] | ((uint32_t) b[3] << 16);
            const pair32 x0 = deq4x4((w0 >> sh) & 0x0f0f0f0fu, dd), x1 = deq4x4((w1 >> sh) & 0x0f0f0f0fu, dd);
            *reinterpret_cast<u4 *>(dst + cc * 16) = u4{x0.lo, x0.hi, x1.lo, x1.hi};
        }
    }
}
}   // namespace

// Key splits of a call: a chunk of few row blocks over a long context would leave most of the device idle (one
// workgroup per block and kv head, each walking every tile), so the tiles of a block are dealt to nks workgroups and the
// partials merged. Chosen from the shape and the device alone (never from what scratch the caller brought: the result
// bits depend on the split): the count that minimises, in units of a tile step, rounds of workgroups x (tiles per
// workgroup + 6 for its set-up and partial stores) + the merge (its launch, 2, and its read of the partials, 1 per 6900
// rows and split); a split is at least 8 tiles; 1 unless that saves 15 %. (The figures are D = 256's, a workgroup to a CU; at
// D <= 128, where the kernel on f16 tiles has two, they have not been taken.)
// `units` are the row blocks the call really has, the last of each kv head full or not: planned for the blocks its rows could
// fill, 12 / 12 heads, 1357 tokens behind 20453 - 132 of them, not 128 - got two splits and a second round of workgroups for
// eight of 264: q8_0 of 256 658 us, five 488; f16 of 128 256 and 206.
static int plan_splits(long units, int T, int p0, int Hq, int cus) {
    const long nt = (p0 + T - 1) / BN + 1;
    if (cus < 1) cus = 1;
    auto cost = [&](long k) {
        const long c = ((units * k + cus - 1) / cus) * ((nt + k - 1) / k + 6);
        return k > 1 ? c + 2 + (long) T * Hq * k / 6900 : c;
    };
    long best = 1, cbest = cost(1);
    for (long k = 2; k <= 64 && nt / k >= 8; ++k)
        if (cost(k) < cbest) { best = k; cbest = cost(k); }
    return cbest * 100 <= cost(1) * 85 ? (int) best : 1;
}
int prefill_key_splits(int T, int p0, int Hq, int Hkv, int cus) {
    return plan_splits(((long) T * (Hq / Hkv) + BM - 1) / BM * Hkv, T, p0, Hq, cus);
}
// the most any Hkv makes of it
static int most_key_splits(int T, int p0, int Hq, int cus) {
    int most = 1;
    for (int h = 1; h <= Hq / h; ++h)
        if (Hq % h == 0) most = std::max({most, prefill_key_splits(T, p0, Hq, h, cus), prefill_key_splits(T, p0, Hq, Hq / h, cus)});
    return most;
}
// Rows of a block: 128, halved (down to 32) while the call would still leave half of the device without a workgroup. A
// workgroup's set-up and epilogue are bound by its own CU's memory path (some 20 bytes a clock: 128 rows of q, gate and out
// take 11 us), its key loop takes the same time however many of its rows are live. 85 tokens behind 126, 24 / 4 heads of 256:
// 22.8 -> 15.4 us (20.8 when a block was 128 tokens of one head), the first 69 tokens of 4 / 1 heads 22.4 -> 15.4.
static int block_rows(int R, int Hkv, int nks, int cus) {
    int b = BM;
    while (b > 32 && 2L * ((R + b - 1) / b) * Hkv * nks <= cus) b /= 2;
    return b;
}
// A quantized cache is converted inside the kernel, without a copy, where few row blocks would share the copy: one block
// makes every tile exactly once either way. A copy costs its bytes (about 0.5 us per million values of K and V each), the
// conversion in the kernel some 1.5 us per tile of a workgroup (q8_0 a little more: two loads a key), and those are few only
// while the splits spread them. Copy / inside, us:
//   D = 256, q8_0: level at 3 to 4 million values a block for up to four blocks (24 / 4 heads, 4 M: one block 36 / 36, three 52 / 48,
//   four 66 / 65; 2.5 M: 35 / 37, 43 / 44, 50 / 50; 8 M: 44 / 41, 78 / 71, 107 / 103), behind with five (4 M: 86 / 90) and six (109 / 118).
//   q4_0: level at 2 to 2.5 M (2.5 M: one 36 / 38, two 44 / 42, four 54 / 50; 8 M: 48 / 42, 60 / 49, 117 / 101); five and six gain little
//   (4 M: 92 / 89, 116 / 116).
//   D <= 128, where the kernel on a copy has two workgroups to a CU: one block from 2.5 M on (32 / 8 of 128 q8_0 26 / 25 and, at 5 M,
//   30 / 27; q4_0 28 / 24 and 34 / 26). Two to four would gain too at 128 (12 M for four: 53 / 51 and 58 / 49), not at 64 (55 / 72).
static bool convert_inside(const p1a_kv & c, int R, int n) {
    const int blocks = (R + BM - 1) / BM;
    if (c.pt && c.psh < 4) return false;                      // (a page lookup per key: measured nowhere as good)
    return blocks <= (c.D == 256 ? 4 : 1) && (long long) n * c.Hkv * c.D >= (c.type == P1A_KV_Q8_0 ? 4000000LL : 2500000LL) * blocks;
}
size_t prefill_part_bytes_o(int T, int Hq, int D, int nks) { return nks > 1 ? (size_t) T * Hq * nks * D * 4 : 0; }
size_t prefill_part_bytes_ml(int T, int Hq, int nks) { return nks > 1 ? (((size_t) T * Hq * nks * 2 * 4) + 255) & ~(size_t) 255 : 0; }
void prefill_part_need(int T, int p0, int Hq, int Hkv, int D, size_t & bytes_o, size_t & bytes_ml) {
    const int nks = prefill_key_splits(T, p0, Hq, Hkv, cu_count());
    bytes_o = prefill_part_bytes_o(T, Hq, D, nks);
    bytes_ml = prefill_part_bytes_ml(T, Hq, nks);
}

// bytes of the f16 staging copy of the first n positions (K and V)
// (rows rounded up to whole 16-key groups: the attention kernel fetches whole groups)
size_t prefill_stage_bytes(int n, int Hkv, int D) { return 2 * (size_t) ((n + 15) & ~15) * Hkv * D * 2; }

int launch_prefill(const p1a_kv & c, const float * q, float * out, const float * gate, int T, int p0, int Hq,
                   float scale, void * scratch, size_t scratch_bytes, hipStream_t s) {
    if (c.D != 64 && c.D != 128 && c.D != 256) { set_error("p1a_attn_prefill: unsupported head size D=%d", c.D); return P1A_E_SHAPE; }
    if ((((uintptr_t) c.k | (uintptr_t) c.v) & 15) || (c.pt && (c.pstride & 15))) { set_error("p1a_attn_prefill: cache base / page stride must be 16-byte aligned"); return P1A_E_SHAPE; }
    pf_params P;
    P.q = q; P.out = out; P.gate = gate; P.kc = (const char *) c.k; P.vc = (const char *) c.v; P.pg = view_of(c);
    P.T = T; P.p0 = p0; P.Hq = Hq; P.Hkv = c.Hkv; P.GQA = Hq / c.Hkv;
    P.n_rows = c.n_ctx;
    P.qscale = scale * 1.4426950408889634f;
    P.R = T * P.GQA;
    P.gqa_magic = (uint32_t) ((P.GQA == 1 ? (1ull << 32) - 1 : (1ull << 32) / (unsigned) P.GQA));
    P.nks = 1; P.part_o = nullptr; P.part_ml = nullptr;
    // the caller's scratch: first the f16 staging copy of a quantized cache (when it fits), then the split partials (when
    // they fit behind it); partials that do not fit go to the library's own per-stream buffers
    const int n = p0 + T;
    const bool aligned = scratch && !((uintptr_t) scratch & 255);
    const bool want_copy = c.type != P1A_KV_F16 && !convert_inside(c, P.R, n);
    const bool stage_caller = want_copy && aligned && scratch_bytes >= prefill_stage_bytes(n, c.Hkv, c.D);
    const size_t used = stage_caller ? (prefill_stage_bytes(n, c.Hkv, c.D) + 255) & ~(size_t) 255 : 0;
    // no room in the caller's scratch (the reference's attn_prefill brings none): the library's own staging copy, if it has one
    void * stage_own = nullptr;
    if (want_copy && !stage_caller) stage_own = stage_scratch(s, prefill_stage_bytes(n, c.Hkv, c.D));
    const bool stage = stage_caller || stage_own;
    const int nks = prefill_key_splits(T, p0, Hq, c.Hkv, cu_count());
    if (nks > 1) {
        const size_t bo = prefill_part_bytes_o(T, Hq, c.D, nks), bm = prefill_part_bytes_ml(T, Hq, nks);
        if (aligned && scratch_bytes >= used + bm + bo) {
            P.part_ml = reinterpret_cast<float *>((char *) scratch + used);
            P.part_o = reinterpret_cast<float *>((char *) scratch + used + bm);
        } else if (!split_scratch(s, bo, bm, P.part_o, P.part_ml)) return P1A_E_SCRATCH;   // (the split count fixes the result bits: never fewer splits for want of room)
    }
    P.nks = nks;
    if (nks > 1) { P.out = P.part_o; P.gate = nullptr; }
    P.rpw = block_rows(P.R, c.Hkv, nks, cu_count()) / 4;
    P.nblk = (P.R + 4 * P.rpw - 1) / (4 * P.rpw);
    // Groups of at most GQA blocks, as even as can be: a group's missing blocks are workgroups that find nothing to do, but
    // each takes a compute unit's LDS before it can say so, and the blocks behind it wait. A key-split call is planned to fill
    // the device in so many rounds, and a unit too many on one XCD (three blocks a unit, 84 units: 33 workgroups on an XCD of
    // 32 compute units) is a round more: the XCDs take equal runs of workgroups where whole units in turn would not be
    // equal. q8_0, 64 tokens behind 16000 (24 / 4 heads of 256) 83 -> 63 us, 17 behind 16000 (32 / 8) 132 -> 72, 85 behind 16000
    // (16 / 2) 79 -> 54. (Runs everywhere: 39 -> 43 us for 8 / 8 heads, 32 behind 5000, whose units in turn are equal.)
    P.nbg = nks > 1 ? 1 : (P.nblk + P.GQA - 1) / P.GQA;
    P.bpg = (P.nblk + P.nbg - 1) / P.nbg;
    const int units = P.nbg * c.Hkv * nks, even = (units * P.bpg + 7) / 8;
    P.run = nks > 1 && (units + 7) / 8 * P.bpg > even ? even : 0;
    auto finish = [&](int rc) {
        if (rc != P1A_OK || P.nks == 1) return rc;
        return launch_merge(P.part_o, P.part_ml, out, gate, P.nks, c.D, Hq, T, s);
    };
#define PF(KT_) finish(c.D == 256 ? launch_pf<KT_, 256>(P, s) : c.D == 128 ? launch_pf<KT_, 128>(P, s) : launch_pf<KT_, 64>(P, s))
    if (c.type == P1A_KV_F16) return PF(P1A_KV_F16);
    // A quantized cache with room for a copy: convert the visible positions to f16 once (tens of microseconds, the
    // copy stays in the Infinity Cache) and run the f16 kernel on it - every workgroup then skips the dequantization it
    // would otherwise repeat per 128 query rows. Same tiles, same products, same bits as the direct kernel.
    if (stage) {
        const int n16 = (n + 15) & ~15;
        char * ko = (char *) (stage_caller ? scratch : stage_own), * vo = ko + (size_t) n16 * c.Hkv * c.D * 2;
        const long long items = (long long) n * (c.Hkv * c.D / (c.type == P1A_KV_Q8_0 ? 16 : 8));
        const unsigned blocks = (unsigned) ((items + 255) / 256);
        if (c.type == P1A_KV_Q8_0) dq_k<P1A_KV_Q8_0><<<blocks, 256, 0, s>>>(P.kc, P.vc, P.pg, n, c.Hkv, c.D, ko, vo);
        else dq_k<P1A_KV_Q4_0><<<blocks, 256, 0, s>>>(P.kc, P.vc, P.pg, n, c.Hkv, c.D, ko, vo);
        if (launched() != P1A_OK) return P1A_E_LAUNCH;
        P.kc = ko; P.vc = vo;
        P.pg.pt = nullptr; P.pg.rtab = nullptr; P.pg.psh = 0; P.pg.pstride = 0;
        P.pg.rowb = (size_t) c.Hkv * c.D * 2;
        P.n_rows = n16;
        return PF(P1A_KV_F16);
    }
    if (c.type == P1A_KV_Q8_0) return PF(P1A_KV_Q8_0);
    return PF(P1A_KV_Q4_0);
#undef PF
}

}   // namespace p1a


extern "C" size_t p1a_attn_prefill_scratch_bytes(int T, int p0, int Hq, int Hkv, int D) {
    if (T < 1 || p0 < 0 || Hkv < 1 || D < 1) return 0;
    // optional: with this much scratch a quantized cache is converted to f16 once per call instead of once per
    // workgroup, and the partials of a key-split call (few token blocks over a long context) live in it; with less (or
    // none) the kernel converts on the fly and the partials go to the library's own per-stream buffers
    const int nks = Hq < 1 ? 1 : Hq % Hkv ? p1a::most_key_splits(T, p0, Hq, p1a::cu_count()) : p1a::prefill_key_splits(T, p0, Hq, Hkv, p1a::cu_count());
    return ((p1a::prefill_stage_bytes(p0 + T, Hkv, D) + 255) & ~(size_t) 255) + p1a::prefill_part_bytes_ml(T, Hq, nks) +
           p1a::prefill_part_bytes_o(T, Hq, D, nks);
}

extern "C" int p1a_attn_prefill_key_splits(int T, int p0, int Hq) {
    if (T < 1 || p0 < 0 || Hq < 1) return 1;
    return p1a::most_key_splits(T, p0, Hq, p1a::cu_count());
}

extern "C" int p1a_attn_prefill_call_splits(int T, int p0, int Hq, int Hkv) {
    if (T < 1 || p0 < 0 || Hkv < 1 || Hq < Hkv || Hq % Hkv) return 1;
    return p1a::prefill_key_splits(T, p0, Hq, Hkv, p1a::cu_count());
}
