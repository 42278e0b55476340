// kvm_fa_prefill.hip -- flash attention for long query chunks (chunked prefill,
// long MTP verify) on the matrix cores.
//
// The op is ggml_flash_attn_ext as build_attn calls it
// (patches/0002-attn-qk-capture-hook.patch:225, kq_scale at :256), causal over
// the window plus the chunk's own cells: a cell is visible to a query token iff
// it is live (pos >= 0) and its original position is <= the token's
// (patches/0003-kv-cache-skip-hole-purge.patch:78-90).  For a quantised cache
// and a multi-token query, ggml's GPU backends convert K and V to f16 and run
// an f16 matrix-core kernel; this file does the same with CDNA4 MFMA.
//
// One workgroup of 8 waves per CU; a row is (token, query head of the group), so the
// query heads of a kv head share every K/V tile.  A wave has 32 rows: the 32x32x16
// MFMA reads half the LDS bytes per flop of 16 rows a wave.  A unit is 256 rows of a
// kv head (k_pf_attn: eight such waves) or 128 (k_pf_attn_split: four, and four that
// bring the tiles).  The units' keys are dealt to the workgroups in equal shares, or
// whole units over few tiles (pf_shares); k_pf_combine merges the units that several
// workgroups share.
// S^T = K Q^T and O^T += V^T P^T.  Key order: score row i of a 32-key sub tile is
// key i with bits 2 and 3 swapped (the lane that supplies K row i reads that key),
// so that the accumulator holds for each lane the 8 consecutive keys that the P V
// operand wants and P needs no cross-lane exchange.  Online softmax in the log2
// domain with a lazy running maximum (rescale only when a row max grows by more
// than 2^8).  Tiles no row of the unit can see are left out of its list; tiles
// every row sees in full skip the mask.
// Where the tiles come from (SRC):
//   PF_F16    an f16 window's tiles, which are the MFMA operands already, copied
//             global -> LDS, double buffered;
//   PF_STAGED the same from a workspace into which k_pf_stage converted the
//             quantised window: one conversion for all row tiles (256-row units);
//   PF_QUANT  the quantised tiles, converted by the attention's own waves (128-row
//             units).
// f16 tiles: K as kvm_kh_idx; V units of 8 keys of a dim (as kvm_vh_idx), in LDS
// and in the workspace in the order [32-key half][16-dim tile][8-key group][dim].
// What bounds it: large chunks, the matrix cores at the clock that the power limit
// leaves (2,048 tokens x 34,816 cells, 16 rows a wave and this: 1.02 -> 1.10 PFLOP/s on
// one card, where a large f16 matrix product reaches 1.33; the matrix cores are busy 0.66
// of the cycles, the LDS 0.33); small ones, the attention waves' chain, the latencies of
// the start and the piece traffic (37 tokens x 32,768 cells: 152 -> 53 us; 700 x 8,192 on
// an f16 cache of 2 heads x 128: 49 -> 44).
#include "kvm_internal.h"

#include <algorithm>
#include <type_traits>

#define KVM_PF_LAZY 8.0f         // log2 growth of a row max tolerated before a rescale
#define KVM_PF_LIST 8192u        // tiles of a segment: the keys of a unit are listed at most this many tiles at a time

// Nothing moves over it, the MFMA that wrote x included: the operand loads stay
// where the ring issues them (a scheduling barrier alone keeps the loads, but the
// MFMAs, which nothing orders, sink below all of them and every operand is live).
#define PF_PIN(x)                                    \
    do {                                             \
        asm volatile("" : "+v"(x) : : "memory");     \
        __builtin_amdgcn_sched_barrier(0);           \
    } while (0)

enum { PF_STAGED, PF_F16, PF_QUANT };

typedef __attribute__((address_space(3))) void *kvm_lds_ptr;
typedef float kvm_f32x16 __attribute__((ext_vector_type(16)));
typedef float kvm_f32x2 __attribute__((ext_vector_type(2)));

extern "C" int kvm_fa_prefill_chunked(kvm_state *st, const kvm_window *w, const void *q, int q_type,
                                      const int32_t *q_pos, uint32_t n_tokens, uint32_t n_head,
                                      float scale, float *out);

// ---------------------------------------------------------------------------
// Quantised tile -> f16 operands.  A byte under 0x64 is the f16 number 1024 +
// byte, so four values take two v_perm and two packed subtractions (exact); the
// packed product with the f16 scale rounds once, as (f16)((float)q * d) does.
// ---------------------------------------------------------------------------
__device__ __forceinline__ kvm_f16x2 pf_bits2(uint32_t u) {
    kvm_f16x2 v;
    __builtin_memcpy(&v, &u, 4);
    return v;
}
__device__ __forceinline__ void pf_pairs(uint32_t bytes, kvm_f16x2 &a, kvm_f16x2 &b) {
    a = pf_bits2(__builtin_amdgcn_perm(0x64646464u, bytes, 0x04010400u));
    b = pf_bits2(__builtin_amdgcn_perm(0x64646464u, bytes, 0x04030402u));
}
// 8 int8 quants times one scale
__device__ __forceinline__ kvm_f16x8 pf_q8(uint32_t w0, uint32_t w1, uint32_t dbits) {
    const kvm_f16x2 off = {(_Float16)1152.0f, (_Float16)1152.0f}, d = pf_bits2(dbits * 0x10001u);
    kvm_f16x2 r[4];
    pf_pairs(w0 ^ 0x80808080u, r[0], r[1]);
    pf_pairs(w1 ^ 0x80808080u, r[2], r[3]);
    kvm_f16x8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r[i] = (r[i] - off) * d;
        o[2 * i] = r[i][0];
        o[2 * i + 1] = r[i][1];
    }
    return o;
}
// the 8 q4_0 nibbles of a V word (kvm_vq_nib_shift) times their keys' scales
__device__ __forceinline__ kvm_f16x8 pf_q4(uint32_t w, kvm_u32x4 scales) {
    const kvm_f16x2 off = {(_Float16)1032.0f, (_Float16)1032.0f};
    kvm_f16x2 r[4];
    pf_pairs(w & 0x0f0f0f0fu, r[0], r[1]);
    pf_pairs((w >> 4) & 0x0f0f0f0fu, r[2], r[3]);
    kvm_f16x8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r[i] = (r[i] - off) * pf_bits2(scales[i]);
        o[2 * i] = r[i][0];
        o[2 * i + 1] = r[i][1];
    }
    return o;
}

// x, from which the compiler cannot tell that a value formed of it does not
// change in a loop: hoisted, lane addresses take the registers that the
// accumulators need.
__device__ __forceinline__ uint32_t opaque(int x) {
    asm volatile("" : "+v"(x));
    return (uint32_t)x;
}

// A tile without a live cell is in no unit's list, so it is left as it is: the first
// chunks over a large window convert what they wrote, not the window (1,024 tokens
// in 34,816 cells of 8 heads x 128: 70.7 us for the call with all of it, 42.1 so).
// The look at the cells is a round trip more; a grid that the chip holds at once
// (SKIP false) has nothing to win by it (512 tokens in 8,192 cells: 32.0 and 34.3).
struct pf_stage_args {
    const uint8_t *k, *v;        // window K / V tiles (q8_0 / q4_0)
    const int32_t *cell_pos;
    uint8_t *kh, *vh;            // f16 operand tiles [H][n_tiles][64 * D]
    uint32_t n_tiles;
};

template <int D, bool SKIP>
__global__ void __launch_bounds__(256) k_pf_stage(pf_stage_args a) {
    constexpr int NB = D / 32;
    const uint32_t t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const uint64_t tile = (uint64_t)h * a.n_tiles + t;
    if (SKIP && __builtin_amdgcn_ballot_w64(a.cell_pos[64ull * t + (tid & 63u)] >= 0) == 0) return;     // (every wave reads all of them)
    uint8_t *kh = a.kh + tile * 128 * D, *vh = a.vh + tile * 128 * D;
    // K unit = the 16 quant bytes of (sub s, block pair p, lane 16g+m): key
    // 16s+m, blocks 2p and 2p+1, dims 8g..8g+7 of each
    const uint8_t *kt = a.k + tile * kvm_ktile_bytes(KVM_TYPE_Q8_0, D);
#pragma unroll
    for (uint32_t u = tid; u < 4u * (NB / 2) * 64u; u += 256) {
        const uint32_t ln = u & 63u, sp = u >> 6, s = sp / (NB / 2), p = sp % (NB / 2), m = ln & 15u;
        const kvm_u32x4 qw = *(const kvm_u32x4 *)(kt + (u << 4));
        const uint32_t d0 = *(const uint16_t *)(kt + kvm_kd_off(D, 16 * s + m, 2 * p));
        const uint32_t d1 = *(const uint16_t *)(kt + kvm_kd_off(D, 16 * s + m, 2 * p + 1));
        *(kvm_f16x8 *)(kh + ((s * NB + 2 * p) * 64 + ln) * 16) = pf_q8(qw[0], qw[1], d0);
        *(kvm_f16x8 *)(kh + ((s * NB + 2 * p + 1) * 64 + ln) * 16) = pf_q8(qw[2], qw[3], d1);
    }
    // V unit = the two words (32-key halves) of (dim tile dt, group g, dim m)
    const uint8_t *vt = a.v + tile * kvm_vtile_bytes(KVM_TYPE_Q4_0, D);
#pragma unroll
    for (uint32_t u = tid; u < 4u * D; u += 256) {
        const kvm_u32x2 vw = *(const kvm_u32x2 *)(vt + 8 * u);
        const uint8_t *sc = vt + D * 32u + ((u >> 7) * 128u + ((u >> 4) & 3u) * 16u);
#pragma unroll
        for (uint32_t ks = 0; ks < 2; ++ks)
            *(kvm_f16x8 *)(vh + ks * 64u * D + 16 * u) = pf_q4(vw[ks], *(const kvm_u32x4 *)(sc + 64 * ks));
    }
}

// The keys of U units (unit u: segment u % n_seg of row tile (u / n_seg) %
// n_row_tiles of kv head u / n_seg / n_row_tiles), each counted as P, are dealt
// to P workgroups in order: workgroup p has [p U, (p + 1) U) of U P.  The part of
// a unit that a workgroup has is a piece; the pieces of a row tile and kv head that
// has more than one (every one, if there are several segments) go to slots.  With
// one segment only a workgroup's first and last unit can be cut: slots 2 p and
// 2 p + 1.  With several, from one piece to the next the workgroup, the unit or both
// go on by one, so p + u is another number for each.  (p + u for one segment as well,
// which leaves no slot out: 26.6 us where these take 26.0, 200 tokens in an empty
// f16 window of 4 heads x 256.)
__host__ __device__ inline uint32_t pf_slot(uint32_t U, uint32_t P, uint32_t n_seg, uint32_t p, uint32_t u,
                                            uint32_t u_first) {
    return n_seg == 1 ? 2 * p + (u != u_first) : p + u;
}
__host__ inline uint64_t pf_slots(uint32_t U, uint32_t P, uint32_t n_seg) {
    if (n_seg == 1 && U % P == 0) return 0;               // every unit whole
    return n_seg == 1 ? 2ull * P : (uint64_t)P + U - 1;
}

struct pf_args {
    const uint8_t *k, *v;        // f16 operand tiles, f16 window tiles or quantised window tiles
    const int32_t *cell_pos;
    const void *q;
    const int32_t *q_pos;
    float *out;                  // [token][n_head][D] fp32
    float *ws_o;                 // pieces [slot][32-row group][dim / 4 of a lane half][lane][4]
    float *ws_ml;                // [slot][row][2]: scaled max, sum
    uint32_t U, P;               // U P < 2^32
    uint32_t n_tiles, n_seg, H, G, n_head, n_rows, n_row_tiles;
    float c;                     // kq_scale * log2(e)
    int q_bf16;
    int longest;                 // whole units, more than the CUs: pf_longest
};

// The row tile of a unit.  With more units than workgroups a workgroup has several
// after each other, and in a chunk that attends to itself the later rows see more
// tiles: first and last row tiles take turns, so that shares have like numbers of
// tiles.  32 heads on 8 x 128, 8,192 tokens (1,024 units, 4 a workgroup): 812 us in row
// order, 551 here; 24 on 4 x 256, 8,192 over 16,384 cells (768 units): 2,414 and 2,117.
__device__ __forceinline__ uint32_t pf_row_tile(const pf_args &a, uint32_t i) {
    return a.U > a.P ? (i & 1u ? a.n_row_tiles - 1 - (i >> 1) : i >> 1) : i;
}

// The unit of the i-th workgroup where each has a whole one and they outnumber the
// CUs: the last row tiles, which see the most, first, so that what is left at the
// end is short; the heads of a row tile next to each other, so that an XCD (every
// eighth workgroup) keeps to few of them.
__device__ __forceinline__ uint32_t pf_longest(const pf_args &a, uint32_t i) {
    return i % a.H * a.n_row_tiles + a.n_row_tiles - 1 - i / a.H;
}

// Q rows of a unit into LDS, coalesced (as operand loads, 32 rows of 32 bytes an
// instruction, they took 4 us): unit c of 16 bytes of row r at slot c ^ r, so that a
// column's reads use every bank; Q_UC units of each row a pass.  Rows past the last
// are row 0's: their results are never stored.
template <int D, int ROWS, uint32_t Q_UC, bool BF16>
__device__ __forceinline__ void pf_copy_q(const pf_args &a, uint32_t rt_i, uint32_t h, int pass, uint32_t lds, int w, int l) {
    constexpr uint32_t Q_UNITS = D * (BF16 ? 2 : 4) / 16;
    constexpr int N = ROWS * Q_UC / 64 / 8;               // 1 KB copies of a wave
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t x = opaque((w * N + i) * 64 + l), r = x / Q_UC, c = (x ^ r) % Q_UC;
        const uint32_t rr = rt_i * ROWS + r < a.n_rows ? rt_i * ROWS + r : 0u, t = rr / a.G;
        const uint8_t *src = (const uint8_t *)a.q + (((uint64_t)t * a.n_head + h * a.G + (rr - t * a.G)) * Q_UNITS + pass * Q_UC + c) * 16;
        uint32_t m0_saved;
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                     : "=&s"(m0_saved) : "v"(src), "s"(lds + (w * N + i) * 1024u) : "memory");
    }
}

// The start of a unit's piece: the lane's visibility limit, and the piece's tiles in
// fr.list: the segment's tiles that some row of the workgroup can see, in order, and
// of these the share [f_lo, f_hi) / P (returned: how many).
struct pf_front {
    uint8_t flag[KVM_PF_LIST];       // per tile: bit 0 some cell visible to some row, bit 1 all to all
    uint16_t list[KVM_PF_LIST];      // tile - t_begin, bit 15: every cell live and visible to every row, so no mask
    uint32_t mm[2][8], cnt[KVM_PF_LIST / 64];
};
template <typename COPY_Q>
__device__ __forceinline__ uint32_t pf_tiles(const pf_args &a, uint32_t row, uint32_t t_begin, uint32_t f_lo, uint32_t f_hi,
                                             pf_front &fr, uint32_t &qlim, COPY_Q &&copy_q) {
    const int tid = (int)opaque((int)threadIdx.x), l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // ---- the loads of the prologue, all issued before any is used: the lane's
    // row position, the tiles' cells, the Q rows' copies
    const bool live_row = row < a.n_rows;
    const int32_t qp = a.q_pos[(live_row ? row : 0u) / a.G];
    const uint32_t n_seg_t = a.n_tiles - t_begin < KVM_PF_LIST ? a.n_tiles - t_begin : KVM_PF_LIST;
    // a wave looks at 4 tiles at a time, 4 cells a lane (36,864 cells at once)
    constexpr uint32_t NL = 18, TPB = NL * 32;
    const uint32_t t_lane = (uint32_t)(4 * w + (l >> 4));
    kvm_u32x4 cells[NL];
    auto load_cells = [&](uint32_t t0) {
#pragma unroll
        for (uint32_t i = 0; i < NL; ++i) {
            const uint32_t t = t0 + 32 * i + t_lane;
            const uint64_t tile = t_begin + (t < n_seg_t ? t : 0u);
            cells[i] = *(const kvm_u32x4 *)(a.cell_pos + tile * 64 + 4 * (l & 15));
        }
    };
    load_cells(0);
    copy_q();
    __builtin_amdgcn_sched_barrier(0);

    // ---- a cell is visible to the lane's row iff (unsigned)position < qlim
    qlim = live_row && qp >= 0 ? (uint32_t)qp + 1u : 0u;
    const uint32_t mn = kvm_wave_min_u32(live_row ? qlim : 0xffffffffu), mx = ~kvm_wave_min_u32(~qlim);
    if (l == 0) {
        fr.mm[0][w] = mn;
        fr.mm[1][w] = mx;
    }
    KVM_LDS_BARRIER();
    uint32_t wg_min = fr.mm[0][0], wg_max = fr.mm[1][0];
#pragma unroll
    for (int i = 1; i < 8; ++i) {
        wg_min = min(wg_min, fr.mm[0][i]);
        wg_max = max(wg_max, fr.mm[1][i]);
    }

    // ---- the piece's tiles: the segment's tiles that some row here can see,
    // in order, and of these the share [f_lo, f_hi) / P.  fr.list holds tile -
    // t_begin and bit 15: every cell live and visible to every row, so no mask.
    for (uint32_t t0 = 0;;) {
#pragma unroll
        for (uint32_t i = 0; i < NL; ++i) {
            const uint32_t t = t0 + 32 * i + t_lane;
            const kvm_u32x4 c = cells[i];
            const uint32_t lo = min(min(c[0], c[1]), min(c[2], c[3])), hi = max(max(c[0], c[1]), max(c[2], c[3]));
            const uint32_t some = (uint32_t)(__builtin_amdgcn_ballot_w64(lo < wg_max) >> (l & 48)) & 0xffffu;
            const uint32_t all = (uint32_t)(__builtin_amdgcn_ballot_w64(hi < wg_min) >> (l & 48)) & 0xffffu;
            if (t < n_seg_t && (l & 15) == 0) fr.flag[t] = (uint8_t)((some != 0) | (all == 0xffffu) << 1);
        }
        t0 += TPB;
        if (t0 >= n_seg_t) break;
        load_cells(t0);
    }
    KVM_LDS_BARRIER();
    uint32_t n_t;
    {
        const uint32_t n_it = (n_seg_t + 511) / 512;
        auto flag = [&](uint32_t it) { return 512 * it + tid < n_seg_t ? (uint32_t)fr.flag[512 * it + tid] : 0u; };
        for (uint32_t it = 0; it < n_it; ++it) {
            const uint64_t bal = __builtin_amdgcn_ballot_w64(flag(it) & 1u);
            if (l == 0) fr.cnt[8 * it + w] = __popcll(bal);
        }
        KVM_LDS_BARRIER();
        // every wave scans the counts of all (at most 16 x 8 of them)
        const uint32_t c0 = (uint32_t)l < 8 * n_it ? fr.cnt[l] : 0u, c1 = (uint32_t)l + 64 < 8 * n_it ? fr.cnt[l + 64] : 0u;
        const uint32_t i0 = kvm_wave_incl_scan(c0), half = __builtin_amdgcn_readlane(i0, 63);
        const uint32_t i1 = n_it > 8 ? kvm_wave_incl_scan(c1) : 0u, total = half + (n_it > 8 ? __builtin_amdgcn_readlane(i1, 63) : 0u);
        const uint32_t lo = total * f_lo / a.P, hi = total * f_hi / a.P;     // P <= 2^16
        n_t = hi - lo;
        for (uint32_t it = 0; it < n_it; ++it) {
            const uint32_t f = flag(it), x = 8 * it + w;
            const uint64_t bal = __builtin_amdgcn_ballot_w64(f & 1u);
            const uint32_t base = x < 64 ? __builtin_amdgcn_readlane(i0 - c0, x) : half + __builtin_amdgcn_readlane(i1 - c1, x - 64);
            const uint32_t rank = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
            if ((f & 1u) && rank >= lo && rank < hi) fr.list[rank - lo] = (uint16_t)((512 * it + tid) | (f >> 1) << 15);
        }
        KVM_LDS_BARRIER();
    }
    return n_t;
}

template <int D, int SRC, bool BF16>
__global__ void __launch_bounds__(512) k_pf_attn(pf_args a) {
    // LDS operand rings: K runs KR-1 k-steps ahead of its MFMAs, V VR-1
    // operands ahead (the first ones in flight during the softmax)
    constexpr int KR = 3, VR = 3;
    constexpr int ROWS = 256;
    constexpr int KS = D / 16, DT = D / 32, NB = D / 32;
    constexpr uint32_t TILE_B = 128u * D;                 // bytes of an f16 K (or V) tile
    constexpr uint32_t MEM = 4u * TILE_B;                 // two K/V buffers
    // Q in LDS: units of 16 bytes of a row, of these at a time, and where: beside
    // the first tile's copies if it fits there
    constexpr uint32_t Q_UNITS = D * (BF16 ? 2 : 4) / 16, Q_UC = Q_UNITS * ROWS * 16 <= MEM ? Q_UNITS : Q_UNITS / 2;
    constexpr bool Q_EARLY = Q_UC * ROWS * 16 <= 2 * TILE_B;
    constexpr uint32_t Q_OFS = Q_EARLY ? 2 * TILE_B : 0;
    static_assert(Q_UC * ROWS * 16 <= MEM && (Q_UNITS == Q_UC || Q_UNITS == 2 * Q_UC), "Q passes");
    __shared__ __align__(16) uint8_t s_mem[MEM];
    __shared__ pf_front s_front;
    __shared__ __align__(16) int32_t s_cp[2][64];         // the tiles' cell positions
    const int tid = threadIdx.x, l = tid & 63, m2 = l & 31;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

    const uint32_t lds_mem = (uint32_t)(uintptr_t)(kvm_lds_ptr)&s_mem[0];

    // Consecutive hardware workgroup ids go round robin over the 8 XCDs; regroup
    // them so one XCD runs consecutive shares, whose K/V tiles its L2 holds.
    uint32_t p = blockIdx.x;
    if (a.longest) p = pf_longest(a, p);
    else if ((a.P & 7u) == 0) p = (p & 7u) * (a.P >> 3) + (p >> 3);
    const uint32_t sh0 = p * a.U, sh1 = sh0 + a.U;
    const uint32_t u_first = sh0 / a.P, u_last = (sh1 - 1) / a.P;

    for (uint32_t u = u_first; u <= u_last; ++u) {
        const uint32_t u0 = u * a.P;
        const uint32_t f_lo = max(sh0, u0) - u0, f_hi = min(sh1 - u0, a.P);
        const uint32_t seg = u % a.n_seg, rest = u / a.n_seg;
        const uint32_t rt_i = __builtin_amdgcn_readfirstlane(pf_row_tile(a, rest % a.n_row_tiles)), h = __builtin_amdgcn_readfirstlane(rest / a.n_row_tiles);
        const bool whole = f_lo == 0 && f_hi == a.P && a.n_seg == 1;

        const uint32_t row = rt_i * ROWS + 32 * w + m2;
        const uint32_t t_begin = seg * KVM_PF_LIST;
        uint32_t qlim;
        auto dma_q = [&](int pass) { pf_copy_q<D, ROWS, Q_UC, BF16>(a, rt_i, h, pass, lds_mem + Q_OFS, w, l); };
        const uint32_t n_t = pf_tiles(a, row, t_begin, f_lo, f_hi, s_front, qlim, [&]() { dma_q(0); });
        auto entry = [&](uint32_t k) { return (uint32_t)s_front.list[k < n_t ? k : n_t - 1]; };

        // Q rows as f16 B operands: lane (g2, m2) holds Q[row m2][16ks + 8 g2 .. +7]
        kvm_f16x8 qop[KS];
        auto take_q = [&](int pass) {
            const uint32_t le = opaque(l), r = 32 * w + (le & 31u), sw = r % Q_UC;
            const uint8_t *qr = s_mem + Q_OFS + r * (Q_UC * 16);
            constexpr int KP = KS * Q_UC / Q_UNITS;       // k-steps of a pass
#pragma unroll
            for (int i = 0; i < KP; ++i) {
                const int ks = pass * KP + i;
                kvm_u32x4 x[BF16 ? 1 : 2];
#pragma unroll
                for (int j = 0; j < (BF16 ? 1 : 2); ++j)
                    x[j] = *(const kvm_u32x4 *)(qr + ((((BF16 ? 1 : 2) * (2 * i + (le >> 5)) + j) ^ sw) * 16));
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t y = x[BF16 ? 0 : j >> 2][BF16 ? j >> 1 : j & 3];
                    const float v = __uint_as_float(!BF16 ? y : j & 1 ? y & 0xffff0000u : y << 16);
                    qop[ks][j] = (_Float16)v;
                }
            }
        };
        // (the caller has waited for its own copies)
        auto load_q = [&]() {
            KVM_LDS_BARRIER();
            take_q(0);
            if constexpr (Q_UNITS != Q_UC) {
                KVM_LDS_BARRIER();
                dma_q(1);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                KVM_LDS_BARRIER();
                take_q(1);
            }
            KVM_LDS_BARRIER();
        };
        kvm_f32x16 O[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) O[dt][r] = 0.0f;
        float ms = -INFINITY, lp = 0.0f;        // running max of the row (times c), lane's share of its sum
        const float c = a.c;
        // a wave of padding rows only copies
        const bool active = rt_i * ROWS + 32u * w < a.n_rows;

        // operand addresses of a lane: K row m2 is key m2 with bits 2 and 3 swapped
        auto k_lane = [&](uint32_t x) {
            const uint32_t key = (x & 0x13) | (x & 4) << 1 | (x & 8) >> 1;
            return ((key >> 4) * NB * 64 + 16 * (x >> 5) + (key & 15)) * 16;
        };
        auto v_lane = [&](uint32_t x) { return ((x >> 4 & 1) * 64 + 16 * (x >> 5) + (x & 15)) * 16; };

        // S^T of one 32-key sub tile: K operand ks at sk + ..., KR - 1 ahead
        auto scores = [&](const uint8_t *sk) {
            kvm_f32x16 S;
#pragma unroll
            for (int r = 0; r < 16; ++r) S[r] = 0.0f;
            kvm_f16x8 kr[KR];
            auto ld = [&](int ks) { return *(const kvm_f16x8 *)(sk + (ks >> 1) * 1024 + (ks & 1) * 512); };
#pragma unroll
            for (int i = 0; i < KR - 1; ++i) kr[i] = ld(i);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                if (ks + KR - 1 < KS) kr[(ks + KR - 1) % KR] = ld(ks + KR - 1);
                __builtin_amdgcn_sched_barrier(0);
                S = __builtin_amdgcn_mfma_f32_32x32x16_f16(kr[ks % KR], qop[ks], S, 0, 0, 0);
                PF_PIN(S);
            }
            return S;
        };
        // mask, running maximum; returns the maximum that P is formed against
        auto settle = [&](kvm_f32x16 &S, bool masked, const int32_t *cp) {
            if (masked) {
                asm volatile("" ::: "memory");            // keep the mask on this (rare) path
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const kvm_u32x4 x = *(const kvm_u32x4 *)(cp + 16 * (i >> 1) + 8 * (opaque(l) >> 5) + 4 * (i & 1));
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (!(x[r] < qlim)) S[4 * i + r] = -INFINITY;
                }
            }
            float x = S[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) x = fmaxf(x, S[r]);
            x = kvm_max_xor32(x);
            const bool up = fmaf(x, c, -ms) > KVM_PF_LAZY;   // false for a row with nothing visible yet
            if (__builtin_amdgcn_ballot_w64(up) != 0) {
                const float mnew = up ? x * c : ms;
                const float alpha = up ? __builtin_amdgcn_exp2f(ms - mnew) : 1.0f;
                ms = mnew;
                lp *= alpha;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) O[dt] *= alpha;
            }
            return ms == -INFINITY ? 0.0f : ms;
        };
        // O^T += V^T P^T: operand i = (key half i / DT, dim tile i % DT); the
        // second half's probabilities are formed between the first half's MFMAs
        auto ldv = [&](const uint8_t *sv, int i) { return *(const kvm_f16x8 *)(sv + (i % DT) * 2048 + (i / DT) * 512); };
        auto accumulate = [&](const uint8_t *sv, const kvm_f32x16 &S, float msr, kvm_f16x8 (&vr)[VR]) {
            kvm_f16x8 pb[2];
            float sum = 0.0f;
            auto prob = [&](int r) {
                // the row sum takes p before its rounding to the fp16 operand:
                // within 2^-11 of it per element
                const float x = __builtin_amdgcn_exp2f(fmaf(S[r], c, -msr));
                pb[r >> 3][r & 7] = (_Float16)x;
                sum += x;
            };
#pragma unroll
            for (int r = 0; r < 8; ++r) prob(r);
#pragma unroll
            for (int i = 0; i < 2 * DT; ++i) {
                if (i + VR - 1 < 2 * DT) vr[(i + VR - 1) % VR] = ldv(sv, i + VR - 1);
                __builtin_amdgcn_sched_barrier(0);
                O[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vr[i % VR], pb[i / DT], O[i % DT], 0, 0, 0);
                if (i < DT) {
#pragma unroll
                    for (int j = 0; j < 8 / DT; ++j) prob(8 + i * (8 / DT) + j);
                }
                PF_PIN(O[i % DT]);
            }
            lp += sum;
        };
        // Copies go global -> LDS directly (global_load_lds_dwordx4: lane l writes
        // 16 bytes at M0 + offset + 16 l), issued from asm so the compiler adds no
        // wait for them; the loops wait for them themselves before each barrier.
        // The asm restores M0, which the compiler reserves.
        const uint32_t lds_cp = (uint32_t)(uintptr_t)(kvm_lds_ptr)&s_cp[0][0];
        auto dma_cp = [&](uint32_t t, uint32_t buf) {
            const int32_t *src = a.cell_pos + (uint64_t)t * 64;
            uint32_t m0_saved;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, %3\n\ts_mov_b32 m0, %0"
                         : "=&s"(m0_saved) : "v"(4u * opaque(l)), "s"(lds_cp + buf * 256u), "s"(src) : "memory");
        };

        if (n_t != 0) {
            // Wave w copies bytes [CW w, CW (w+1)) of the tile's K and of its V in
            // CW / 1 KB copies under one M0 value (the immediate offset moves the
            // global and the LDS address alike).  A window's f16 V tile holds the
            // two key halves of a dim side by side, so its copies read every
            // second unit of a dim tile.  Wave 0 also copies the cell positions.
            constexpr uint32_t CW = TILE_B / 8;
            static_assert(CW == 4096 || CW == 2048, "copy layout");
            const uint32_t wofs = __builtin_amdgcn_readfirstlane(CW * w), loff = 16u * l;
            const uint8_t *k_head = a.k + (uint64_t)h * a.n_tiles * TILE_B + wofs;
            const uint8_t *v_head = a.v + (uint64_t)h * a.n_tiles * TILE_B +
                                    (SRC == PF_F16 ? (w >> 2) * 16u + (w & 3) * 2u * CW : wofs);
            const uint32_t voff = SRC == PF_F16 ? 32u * l : loff;
            constexpr uint32_t VS = SRC == PF_F16 ? 1024u : 0u;     // global bytes a V copy moves beyond the LDS's
            auto dma_tile = [&](uint32_t t, uint32_t buf) {
                const uint8_t *kb = k_head + (uint64_t)t * TILE_B, *vb = v_head + (uint64_t)t * TILE_B;
                const uint32_t dk = lds_mem + buf * (2 * TILE_B) + wofs, dv = dk + TILE_B;
                uint32_t m0_saved;
                if constexpr (CW == 4096) {
                    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
                                 "global_load_lds_dwordx4 %1, %5\n\t"
                                 "global_load_lds_dwordx4 %1, %5 offset:1024\n\t"
                                 "global_load_lds_dwordx4 %1, %5 offset:2048\n\t"
                                 "global_load_lds_dwordx4 %1, %5 offset:3072\n\t"
                                 "s_mov_b32 m0, %4\n\ts_nop 0\n\t"
                                 "global_load_lds_dwordx4 %2, %6\n\t"
                                 "global_load_lds_dwordx4 %2, %7 offset:1024\n\t"
                                 "global_load_lds_dwordx4 %2, %8 offset:2048\n\t"
                                 "global_load_lds_dwordx4 %2, %9 offset:3072\n\t"
                                 "s_mov_b32 m0, %0"
                                 : "=&s"(m0_saved) : "v"(loff), "v"(voff), "s"(dk), "s"(dv), "s"(kb), "s"(vb),
                                   "s"(vb + VS), "s"(vb + 2 * VS), "s"(vb + 3 * VS) : "memory");
                } else {
                    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
                                 "global_load_lds_dwordx4 %1, %5\n\t"
                                 "global_load_lds_dwordx4 %1, %5 offset:1024\n\t"
                                 "s_mov_b32 m0, %4\n\ts_nop 0\n\t"
                                 "global_load_lds_dwordx4 %2, %6\n\t"
                                 "global_load_lds_dwordx4 %2, %7 offset:1024\n\t"
                                 "s_mov_b32 m0, %0"
                                 : "=&s"(m0_saved) : "v"(loff), "v"(voff), "s"(dk), "s"(dv), "s"(kb), "s"(vb),
                                   "s"(vb + VS) : "memory");
                }
                if (w == 0) dma_cp(t, buf);
            };
            // list entries k and k+1 are in registers at the top of tile k; entry
            // k+2 is read during tile k
            uint32_t e_cur = entry(0), e_nxt = entry(1);
            const uint32_t t_0 = t_begin + (__builtin_amdgcn_readfirstlane(e_cur) & 0x7fffu);
            if constexpr (Q_EARLY) dma_tile(t_0, 0);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            load_q();
            if constexpr (!Q_EARLY) {
                dma_tile(t_0, 0);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                KVM_LDS_BARRIER();
            }
            const uint32_t k_ofs = k_lane(l), v_ofs = v_lane(l);
            for (uint32_t k = 0; k < n_t; ++k) {
                const uint32_t b = k & 1u;
                const uint32_t e = __builtin_amdgcn_readfirstlane(e_cur), en = __builtin_amdgcn_readfirstlane(e_nxt);
                e_cur = en;
                e_nxt = entry(k + 2);
                dma_tile(t_begin + (en & 0x7fffu), b ^ 1u);       // next tile, in flight during this one
                const bool masked = (e >> 15) == 0;
                const uint8_t *sk = s_mem + b * (2 * TILE_B) + k_ofs, *sv = s_mem + b * (2 * TILE_B) + TILE_B + v_ofs;
                if (active) {
#pragma unroll
                    for (int sub = 0; sub < 2; ++sub) {
                        kvm_f32x16 S = scores(sk + sub * 2 * NB * 1024);
                        kvm_f16x8 vr[VR];
#pragma unroll
                        for (int i = 0; i < VR - 1; ++i) vr[i] = ldv(sv + sub * (TILE_B / 2), i);
                        const float msr = settle(S, masked, &s_cp[b][32 * sub]);
                        accumulate(sv + sub * (TILE_B / 2), S, msr, vr);
                    }
                }
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next tile's copies
                __syncthreads();
            }
        }

        if (n_t == 0) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // Q's copies
            KVM_LDS_BARRIER();
        }

        // ---- results: quad i of O: dims 8 i + 4 g2 .. + 3 of the lane's row.  (The lane
        // and its row are formed again here: kept through the loop they take registers
        // that O needs.)
        const float lr = kvm_add_xor32(lp);
        const uint32_t le = opaque(l), me = le & 31u, ge = le >> 5, row_e = rt_i * ROWS + 32 * w + me;
        auto quad = [&](int i) {
            return kvm_f32x4{O[i >> 2][4 * (i & 3)], O[i >> 2][4 * (i & 3) + 1], O[i >> 2][4 * (i & 3) + 2], O[i >> 2][4 * (i & 3) + 3]};
        };
        if (whole) {
            if (row_e < a.n_rows) {
                const float inv = lr > 0.0f ? 1.0f / lr : 0.0f;
                float *o = a.out + ((uint64_t)(row_e / a.G) * a.n_head + h * a.G + row_e % a.G) * D + 4 * ge;
#pragma unroll
                for (int i = 0; i < DT * 4; ++i) *(kvm_f32x4 *)(o + 8 * i) = lr == 0.0f ? kvm_f32x4{0.f, 0.f, 0.f, 0.f} : quad(i) * inv;
            }
        } else if (active) {
            const uint64_t slot = pf_slot(a.U, a.P, a.n_seg, p, u, u_first);
            float *o = a.ws_o + (slot * ROWS + 32 * w) * D + 4 * le;
#pragma unroll
            for (int i = 0; i < DT * 4; ++i) *(kvm_f32x4 *)(o + 256 * i) = quad(i);
            if (ge == 0) {
                float *o_ml = a.ws_ml + (slot * ROWS + 32 * w + me) * 2;
                o_ml[0] = ms;
                o_ml[1] = lr;
            }
        }
        if (u != u_last) __syncthreads();       // the LDS is the next piece's
    }
}

// Units of 128 rows, two roles.  Waves 0 - 3, one a SIMD, have 32 rows each and take
// every key of a tile; waves 4 - 7 bring tile k + 1 into one LDS buffer while tile k in
// the other is worked on, one barrier a tile: an f16 window's by copies, a quantised
// one's through registers, loaded two tiles ahead and written as f16 operands.  What bounds it is the attention waves'
// chain (~3,900 cycles a tile of 256 dims, of which 2,048 on the matrix cores): the
// softmax of a 32-key sub tile is taken between the MFMAs of the next scores or of
// the P V before.  (Converting between the MFMAs of eight attention waves took 5,300:
// their LDS writes, 64 bytes a cycle, held up the operand reads.  37 tokens x 32,768
// cells 61.6 -> 52.3 us, 64 x 4,096 of 8 heads x 128 28 -> 22.5.)
template <int D, int SRC, bool BF16>
__global__ void __launch_bounds__(512) k_pf_attn_split(pf_args a) {
    static_assert(SRC == PF_F16 || SRC == PF_QUANT, "a window is converted ahead for 256-row units only");
    constexpr int ROWS = 128;
    constexpr int KS = D / 16, DT = D / 32, NB = D / 32;  // k-steps of a score; MFMAs of a sub tile's P V: 2 DT = KS
    constexpr uint32_t TILE_B = 128u * D;                 // bytes of an f16 K (or V) tile
    constexpr uint32_t KRAW = 64u * D + 64u * NB * 2u, VRAW = 32u * D + NB * 128u;    // quantised tiles
    constexpr uint32_t MEM = 4u * TILE_B;                 // two K/V buffers
    constexpr uint32_t Q_UNITS = D * (BF16 ? 2 : 4) / 16, Q_UC = Q_UNITS;
    constexpr bool Q_EARLY = Q_UNITS * ROWS * 16 <= 2 * TILE_B;      // Q fits beside the first tile
    constexpr uint32_t Q_OFS = Q_EARLY ? 2 * TILE_B : 0;
    static_assert(Q_UNITS * ROWS * 16 <= MEM, "Q in LDS");
    // Operand rings: R1 where a softmax is under way (registers), R0 elsewhere.  At
    // 256 dims there are none left to keep the softmax's steps where they are
    // written, so the compiler gathers the exponentials.
    constexpr std::integral_constant<int, 6> R0;
    constexpr std::integral_constant<int, D == 256 ? 2 : 4> R1;
    constexpr bool PINS = D == 128;
    __shared__ __align__(16) uint8_t s_mem[MEM];
    __shared__ pf_front s_front;
    __shared__ __align__(16) int32_t s_cp[2][64];         // the tiles' cell positions
    const int tid = threadIdx.x, l = tid & 63, g2 = l >> 5, m2 = l & 31;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), rg = w & 3;
    const bool consumer = w < 4;
    const uint32_t lds_mem = (uint32_t)(uintptr_t)(kvm_lds_ptr)&s_mem[0];
    uint32_t p = blockIdx.x;
    if (a.longest) p = pf_longest(a, p);
    else if ((a.P & 7u) == 0) p = (p & 7u) * (a.P >> 3) + (p >> 3);       // as k_pf_attn
    const uint32_t sh0 = p * a.U, sh1 = sh0 + a.U;
    const uint32_t u_first = sh0 / a.P, u_last = (sh1 - 1) / a.P;

    for (uint32_t u = u_first; u <= u_last; ++u) {
        const uint32_t u0 = u * a.P;
        const uint32_t f_lo = max(sh0, u0) - u0, f_hi = min(sh1 - u0, a.P);
        const uint32_t seg = u % a.n_seg, rest = u / a.n_seg;
        const uint32_t rt_i = __builtin_amdgcn_readfirstlane(pf_row_tile(a, rest % a.n_row_tiles)), h = __builtin_amdgcn_readfirstlane(rest / a.n_row_tiles);
        const bool whole = f_lo == 0 && f_hi == a.P && a.n_seg == 1;
        const uint32_t row = rt_i * ROWS + 32 * rg + m2;
        const uint32_t t_begin = seg * KVM_PF_LIST;
        uint32_t qlim;
        const uint32_t n_t = pf_tiles(a, row, t_begin, f_lo, f_hi, s_front, qlim, [&]() {
            pf_copy_q<D, ROWS, Q_UC, BF16>(a, rt_i, h, 0, lds_mem + Q_OFS, w, l);
        });
        // Both roles take the same barriers: one when Q is in LDS (two if the first
        // tile has to wait for it to be read), one when the first tile is ready, and
        // one a tile.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        KVM_LDS_BARRIER();
        if (consumer) {
            // ======== consumers: S^T = K Q^T, softmax, O^T += V^T P^T of 32 rows
            const float c = a.c;
            kvm_f32x16 O[DT];
            float ms = -INFINITY, lp = 0.0f;        // running max of the row (times c), lane's share of its sum
            // Q rows as f16 B operands: lane (g2, m2) holds Q[row m2][16ks + 8 g2 .. +7]
            kvm_f16x8 qop[KS];
            {
                const uint32_t lq = opaque(l), r = 32 * rg + (lq & 31u), sw = r % Q_UNITS;
                const uint8_t *qr = s_mem + Q_OFS + r * (Q_UNITS * 16);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    kvm_u32x4 x[BF16 ? 1 : 2];
#pragma unroll
                    for (int j = 0; j < (BF16 ? 1 : 2); ++j)
                        x[j] = *(const kvm_u32x4 *)(qr + ((((BF16 ? 1 : 2) * (2 * ks + (lq >> 5)) + j) ^ sw) * 16));
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const uint32_t y = x[BF16 ? 0 : j >> 2][BF16 ? j >> 1 : j & 3];
                        qop[ks][j] = (_Float16)__uint_as_float(!BF16 ? y : j & 1 ? y & 0xffff0000u : y << 16);
                    }
                }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) O[dt][r] = 0.0f;
            // operand addresses of a lane: K row m2 is key m2 with bits 2 and 3 swapped
            const uint32_t key = (m2 & 0x13) | (m2 & 4) << 1 | (m2 & 8) >> 1;
            const uint32_t k_ofs = ((key >> 4) * NB * 64 + 16 * g2 + (key & 15)) * 16;
            const uint32_t v_ofs = ((m2 >> 4) * 64 + 16 * g2 + (m2 & 15)) * 16;
            if constexpr (!Q_EARLY) KVM_LDS_BARRIER();

            // S^T of one 32-key sub tile: K operand ks at sk + ..., KR - 1 ahead;
            // between(ks) follows MFMA ks
            auto scores = [&](auto ring, const uint8_t *sk, auto &&between) {
                constexpr int KR = decltype(ring)::value;
                kvm_f32x16 S;
#pragma unroll
                for (int r = 0; r < 16; ++r) S[r] = 0.0f;
                kvm_f16x8 kr[KR];
                auto ld = [&](int ks) { return *(const kvm_f16x8 *)(sk + (ks >> 1) * 1024 + (ks & 1) * 512); };
#pragma unroll
                for (int i = 0; i < KR - 1; ++i) kr[i] = ld(i);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    if (ks + KR - 1 < KS) kr[(ks + KR - 1) % KR] = ld(ks + KR - 1);
                    __builtin_amdgcn_sched_barrier(0);
                    S = __builtin_amdgcn_mfma_f32_32x32x16_f16(kr[ks % KR], qop[ks], S, 0, 0, 0);
                    between(ks);
                    PF_PIN(S);
                }
                return S;
            };
            // O^T += V^T P^T: operand i = (key half i / DT, dim tile i % DT)
            auto accumulate = [&](auto ring, const uint8_t *sv, const kvm_f16x8 (&pb)[2], auto &&between) {
                constexpr int VR = decltype(ring)::value;
                kvm_f16x8 vr[VR];
                auto ld = [&](int i) { return *(const kvm_f16x8 *)(sv + (i % DT) * 2048 + (i / DT) * 512); };
#pragma unroll
                for (int i = 0; i < VR - 1; ++i) vr[i] = ld(i);
#pragma unroll
                for (int i = 0; i < 2 * DT; ++i) {
                    if (i + VR - 1 < 2 * DT) vr[(i + VR - 1) % VR] = ld(i + VR - 1);
                    __builtin_amdgcn_sched_barrier(0);
                    O[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vr[i % VR], pb[i / DT], O[i % DT], 0, 0, 0);
                    between(i);
                    PF_PIN(O[i % DT]);
                }
            };
            auto mask = [&](kvm_f32x16 &S, const int32_t *cp) {
                asm volatile("" ::: "memory");            // keep the mask on this (rare) path
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const kvm_u32x4 x = *(const kvm_u32x4 *)(cp + 16 * (i >> 1) + 8 * (opaque(l) >> 5) + 4 * (i & 1));
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (!(x[r] < qlim)) S[4 * i + r] = -INFINITY;
                }
            };
            // The softmax of a sub tile in KS steps, taken between another's MFMAs:
            // the maximum (KS / 4 steps), the running maximum's move (one step), the
            // probabilities (KS / 2 steps).
            float x = 0.0f, msr = 0.0f, alpha = 1.0f, sum = 0.0f;
            bool moved = false;
            auto soft = [&](const kvm_f32x16 &S, kvm_f16x8 (&pb)[2], int i) {
                constexpr int NM = KS / 4, EM = 16 / NM, EP = 16 / (KS / 2);
                if (i < NM) {
#pragma unroll
                    for (int r = 0; r < EM; ++r) x = i == 0 && r == 0 ? S[0] : fmaxf(x, S[EM * i + r]);
                    if constexpr (PINS) asm volatile("" : "+v"(x));
                } else if (i == NM) {
                    x = kvm_max_xor32(x);
                    const bool up = fmaf(x, c, -ms) > KVM_PF_LAZY;   // false for a row with nothing visible yet
                    moved = __builtin_amdgcn_ballot_w64(up) != 0;
                    const float mnew = up ? x * c : ms;
                    alpha = up ? __builtin_amdgcn_exp2f(ms - mnew) : 1.0f;
                    ms = mnew;
                    msr = ms == -INFINITY ? 0.0f : ms;
                    sum = 0.0f;
                } else if (i >= KS / 2) {
#pragma unroll
                    for (int j = 0; j < EP; ++j) {
                        // the row sum takes p before its rounding to the fp16 operand:
                        // within 2^-11 of it per element
                        const int r = EP * (i - KS / 2) + j;
                        const float y = __builtin_amdgcn_exp2f(fmaf(S[r], c, -msr));
                        pb[r >> 3][r & 7] = (_Float16)y;
                        sum += y;
                        if constexpr (PINS) asm volatile("" : "+v"(sum));
                    }
                    if constexpr (PINS) asm volatile("" : "+v"(pb[(EP * (i - KS / 2)) >> 3]));
                }
            };
            // what the moved maximum asks of the sums so far
            auto settle = [&]() {
                if (moved) {
                    asm volatile("" ::: "memory");        // keep it on this (rare) path
                    lp *= alpha;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) O[dt] *= alpha;
                }
                lp += sum;
            };
            auto nothing = [](int) {};

            KVM_LDS_BARRIER();                            // the first tile is in LDS
            const bool active = rt_i * ROWS + 32u * rg < a.n_rows;    // not a wave of padding rows
            uint32_t e_nxt = n_t ? s_front.list[0] : 0u;
            for (uint32_t k = 0; k < n_t; ++k) {
                if (!active) {
                    KVM_LDS_BARRIER();
                    continue;
                }
                const bool masked = (__builtin_amdgcn_readfirstlane(e_nxt) >> 15) == 0;
                e_nxt = s_front.list[k + 1 < n_t ? k + 1 : k];
                const uint8_t *sk = s_mem + (k & 1u) * (2 * TILE_B) + k_ofs, *sv = s_mem + (k & 1u) * (2 * TILE_B) + TILE_B + v_ofs;
                kvm_f16x8 pb[2];
                kvm_f32x16 S0 = scores(R0, sk, nothing);
                if (masked) mask(S0, &s_cp[k & 1u][0]);
                kvm_f32x16 S1 = scores(R1, sk + 2 * NB * 1024, [&](int i) { soft(S0, pb, i); });
                settle();
                if (masked) mask(S1, &s_cp[k & 1u][32]);
                kvm_f16x8 pb1[2];
                accumulate(R1, sv, pb, [&](int i) { soft(S1, pb1, i); });
                settle();
                accumulate(R0, sv + TILE_B / 2, pb1, nothing);
                KVM_LDS_BARRIER();
            }
            // ---- results: quad i of O: dims 8 i + 4 g2 .. + 3 of the lane's row
            const float lr = kvm_add_xor32(lp);
            const uint32_t le = opaque(l), me = le & 31u, ge = le >> 5, row_e = rt_i * ROWS + 32 * rg + me;
            auto quad = [&](int i) {
                return kvm_f32x4{O[i >> 2][4 * (i & 3)], O[i >> 2][4 * (i & 3) + 1], O[i >> 2][4 * (i & 3) + 2], O[i >> 2][4 * (i & 3) + 3]};
            };
            if (whole) {
                if (row_e < a.n_rows) {
                    const float inv = lr > 0.0f ? 1.0f / lr : 0.0f;
                    float *o = a.out + ((uint64_t)(row_e / a.G) * a.n_head + h * a.G + row_e % a.G) * D + 4 * ge;
#pragma unroll
                    for (int i = 0; i < DT * 4; ++i) *(kvm_f32x4 *)(o + 8 * i) = lr == 0.0f ? kvm_f32x4{0.f, 0.f, 0.f, 0.f} : quad(i) * inv;
                }
            } else if (rt_i * ROWS + 32 * rg < a.n_rows) {
                const uint64_t slot = pf_slot(a.U, a.P, a.n_seg, p, u, u_first);
                float *o = a.ws_o + (slot * ROWS + 32 * rg) * D + 4 * le;
#pragma unroll
                for (int i = 0; i < DT * 4; ++i) *(kvm_f32x4 *)(o + 256 * i) = quad(i);
                if (ge == 0) {
                    float *o_ml = a.ws_ml + (slot * ROWS + 32 * rg + me) * 2;
                    o_ml[0] = ms;
                    o_ml[1] = lr;
                }
            }
        } else {
            // ======== producers: tile k + 1 into one buffer while the consumers work
            // on tile k in the other
            const int pw = w - 4;
            auto tile = [&](uint32_t k) { return t_begin + (__builtin_amdgcn_readfirstlane((uint32_t)s_front.list[k < n_t ? k : n_t - 1]) & 0x7fffu); };
            auto cells_to = [&](uint32_t t) { return a.cell_pos[(uint64_t)t * 64 + l]; };
            if constexpr (SRC == PF_F16) {
                // Copies go global -> LDS directly (global_load_lds_dwordx4: lane l
                // writes 16 bytes at M0 + 16 l), issued from asm so the compiler adds
                // no wait for them; the wait is before the barrier.  The asm restores
                // M0, which the compiler reserves.  A window's f16 V tile holds the two
                // key halves of a dim side by side, so its copies read every second
                // unit of a dim tile.
                constexpr int NC = (int)TILE_B / 4096;    // 1 KB copies of a wave, of K and of V
                const uint8_t *k_head = a.k + (uint64_t)h * a.n_tiles * TILE_B, *v_head = a.v + (uint64_t)h * a.n_tiles * TILE_B;
                auto copy = [&](uint32_t voff, uint32_t dst, const uint8_t *src) {
                    uint32_t m0_saved;
                    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                                 "global_load_lds_dwordx4 %1, %3\n\ts_mov_b32 m0, %0"
                                 : "=&s"(m0_saved) : "v"(voff), "s"(dst), "s"(src) : "memory");
                };
                auto copy_tile = [&](uint32_t t, uint32_t buf) {
                    const uint32_t dst = lds_mem + buf * (2 * TILE_B);
                    const uint8_t *kt = k_head + (uint64_t)t * TILE_B, *vt = v_head + (uint64_t)t * TILE_B;
#pragma unroll
                    for (int i = 0; i < NC; ++i) copy(16u * opaque(l), dst + (pw * NC + i) * 1024u, kt + (pw * NC + i) * 1024u);
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        const uint32_t x = pw * NC + i;   // key half, dim tile
                        copy(32u * opaque(l), dst + TILE_B + x * 1024u, vt + (x % (D / 16)) * 2048u + (x / (D / 16)) * 16u);
                    }
                };
                if constexpr (!Q_EARLY) KVM_LDS_BARRIER();
                if (n_t != 0) {
                    const uint32_t t = tile(0);
                    copy_tile(t, 0);
                    if (pw == 0) s_cp[0][l] = cells_to(t);
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                KVM_LDS_BARRIER();
                for (uint32_t k = 0; k < n_t; ++k) {
                    if (k + 1 < n_t) {
                        const uint32_t t = tile(k + 1);
                        copy_tile(t, (k + 1) & 1u);
                        if (pw == 0) s_cp[(k + 1) & 1u][l] = cells_to(t);
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    }
                    KVM_LDS_BARRIER();
                }
            } else {
                // The quantised tile goes through registers (two sets: tiles k + 2 and
                // k + 3 are in flight while tile k + 1 is converted).  Thread (pw, l): K
                // units 4 j + pw (lane l of (sub, block pair)), V dim tiles VJ pw + j.
                constexpr int KJ = D / 64, VJ = D / 64, VB = VJ / 2;
                struct raw_tile {
                    kvm_u32x4 k[KJ];
                    uint32_t kd[KJ][2];
                    kvm_u32x2 v[VJ];
                    kvm_u32x4 vs[VB][2];
                    int32_t cp;
                };
                raw_tile rt[2] = {};
                const uint8_t *k_head = a.k + (uint64_t)h * a.n_tiles * KRAW, *v_head = a.v + (uint64_t)h * a.n_tiles * VRAW;
                auto load = [&](raw_tile &r, uint32_t t) {
                    const uint32_t ln = opaque(l);
                    const uint8_t *kt = k_head + (uint64_t)t * KRAW, *vt = v_head + (uint64_t)t * VRAW;
#pragma unroll
                    for (int j = 0; j < KJ; ++j) {
                        const uint32_t sp = 4 * j + pw, s = sp / (NB / 2), pr = sp % (NB / 2);
                        r.k[j] = *(const kvm_u32x4 *)(kt + (sp * 64 + ln) * 16);
                        r.kd[j][0] = *(const uint16_t *)(kt + kvm_kd_off(D, 16 * s + (ln & 15), 2 * pr));
                        r.kd[j][1] = *(const uint16_t *)(kt + kvm_kd_off(D, 16 * s + (ln & 15), 2 * pr + 1));
                    }
#pragma unroll
                    for (int j = 0; j < VJ; ++j) r.v[j] = *(const kvm_u32x2 *)(vt + ((VJ * pw + j) * 64 + ln) * 8);
#pragma unroll
                    for (int b = 0; b < VB; ++b)
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks)
                            r.vs[b][ks] = *(const kvm_u32x4 *)(vt + 32 * D + (((VB * pw + b) * 2 + ks) * 4 + (ln >> 4)) * 16);
                    r.cp = cells_to(t);
                };
                auto convert = [&](const raw_tile &r, uint32_t buf) {
                    uint8_t *dk = s_mem + buf * (2 * TILE_B) + 16 * opaque(l), *dv = dk + TILE_B;
#pragma unroll
                    for (int j = 0; j < KJ; ++j) {
                        const uint32_t sp = 4 * j + pw, s = sp / (NB / 2), pr = sp % (NB / 2);
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            *(kvm_f16x8 *)(dk + (s * NB + 2 * pr + i) * 1024) = pf_q8(r.k[j][2 * i], r.k[j][2 * i + 1], r.kd[j][i]);
                    }
#pragma unroll
                    for (int j = 0; j < VJ; ++j)
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks)
                            *(kvm_f16x8 *)(dv + ks * (TILE_B / 2) + (VJ * pw + j) * 1024) = pf_q4(r.v[j][ks], r.vs[j / 2][ks]);
                    if (pw == 0) s_cp[buf][l] = r.cp;
                };
                if (n_t != 0) {
                    load(rt[0], tile(0));
                    load(rt[1], tile(1));
                }
                if constexpr (!Q_EARLY) KVM_LDS_BARRIER();
                if (n_t != 0) {
                    convert(rt[0], 0);
                }
                KVM_LDS_BARRIER();
                if (2 < n_t) load(rt[0], tile(2));
                auto step = [&](raw_tile &r, uint32_t k) {
                    if (k + 1 < n_t) convert(r, (k + 1) & 1u);
                    if (k + 3 < n_t) load(r, tile(k + 3));
                    KVM_LDS_BARRIER();
                };
                uint32_t k = 0;
                for (; k + 2 <= n_t; k += 2) {
                    step(rt[1], k);
                    step(rt[0], k + 1);
                }
                if (k < n_t) step(rt[1], k);
            }
        }

        if (u != u_last) __syncthreads();       // the LDS is the next piece's
    }
}

// Merge the pieces of a unit's 32-row group: a lane has 4 dims of a row.  WS waves
// share the pieces, each with NP pieces' loads in flight, and meet in LDS: what
// bounds a unit of many pieces is the round trips of its loads.
template <int D, int ROWS, int WS, int NP>
__global__ void __launch_bounds__(256) k_pf_combine(pf_args a) {
    constexpr uint32_t IB = 4 / WS;
    const uint32_t l = threadIdx.x & 63u, wv = threadIdx.x >> 6, ws = wv % WS, i = blockIdx.z * IB + wv / WS;
    const uint32_t rg = blockIdx.y, m2 = l & 31u, rt_i = pf_row_tile(a, blockIdx.x % a.n_row_tiles), h = blockIdx.x / a.n_row_tiles;
    const uint32_t row = rt_i * ROWS + 32 * rg + m2;
    // the unit's pieces: workgroups q0 .. q1 of each of its segments
    const uint32_t u0 = blockIdx.x * a.n_seg, u1 = u0 + a.n_seg;
    float M = -INFINITY, L = 0.0f;
    kvm_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (rt_i * ROWS + 32 * rg >= a.n_rows) return;
    for (uint32_t u = u0; u < u1; ++u) {
        const uint32_t q0 = u * a.P / a.U, q1 = ((u + 1) * a.P - 1) / a.U;
        if (q0 == q1 && a.n_seg == 1) return;             // whole: the attention wrote it
        // u is the first unit of every workgroup after q0
        const uint32_t s0 = pf_slot(a.U, a.P, a.n_seg, q0, u, q0 * a.U / a.P);
        for (uint32_t q = q0; q <= q1; q += NP * WS) {
            kvm_f32x4 x[NP];
            float m[NP], s[NP];
#pragma unroll
            for (uint32_t j = 0; j < NP; ++j) {
                const uint32_t qj = q + WS * j + ws, pj = min(qj, q1);
                const uint64_t slot = pj == q0 ? s0 : pf_slot(a.U, a.P, a.n_seg, pj, u, u);
                x[j] = *(const kvm_f32x4 *)(a.ws_o + (slot * ROWS + 32 * rg) * D + 256 * i + 4 * l);
                const kvm_f32x2 ml = *(const kvm_f32x2 *)(a.ws_ml + (slot * ROWS + 32 * rg + m2) * 2);
                m[j] = qj <= q1 ? ml[0] : -INFINITY;
                s[j] = ml[1];
            }
            if (q + NP * WS > q1 + 1) {
                // past q1 its piece was read again: an infinity there times the weight 0 is no number
#pragma unroll
                for (uint32_t j = 0; j < NP; ++j)
                    if (q + WS * j + ws > q1) x[j] = kvm_f32x4{0.f, 0.f, 0.f, 0.f};
            }
            float mb = M;
#pragma unroll
            for (uint32_t j = 0; j < NP; ++j) mb = fmaxf(mb, m[j]);
            const float keep = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - mb);
            L *= keep;
            acc *= keep;
#pragma unroll
            for (uint32_t j = 0; j < NP; ++j) {
                const float wgt = m[j] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m[j] - mb);
                L += m[j] == -INFINITY ? 0.0f : s[j] * wgt;
                acc += x[j] * wgt;
            }
            M = mb;
        }
    }
    if constexpr (WS > 1) {
        __shared__ __align__(16) float s_x[WS][64][4];
        __shared__ float s_m[WS][64], s_l[WS][64];
        *(kvm_f32x4 *)s_x[ws][l] = acc;
        s_m[ws][l] = M;
        s_l[ws][l] = L;
        __syncthreads();
        if (ws != 0) return;
        float mb = M;
#pragma unroll
        for (int j = 1; j < WS; ++j) mb = fmaxf(mb, s_m[j][l]);
        M = mb;
        L = 0.0f;
        acc = kvm_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < WS; ++j) {
            const float wgt = s_m[j][l] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(s_m[j][l] - mb);
            L += s_l[j][l] * wgt;
            acc += *(const kvm_f32x4 *)s_x[j][l] * wgt;
        }
    }
    if (row >= a.n_rows) return;
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    if (M == -INFINITY) acc = kvm_f32x4{0.f, 0.f, 0.f, 0.f};      // nothing visible: not 0 times what its tiles hold
    *(kvm_f32x4 *)(a.out + ((uint64_t)(row / a.G) * a.n_head + h * a.G + row % a.G) * D + 8 * i + 4 * (l >> 5)) = acc * inv;
}

// The copies global -> LDS take 16-byte aligned sources: a buffer that is not is
// copied to the workspace first.
__global__ void __launch_bounds__(256) k_pf_align(const uint8_t *src, uint8_t *dst, uint64_t n16) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n16) return;
    kvm_u32x4 x;
    __builtin_memcpy(&x, src + 16 * i, 16);
    *(kvm_u32x4 *)(dst + 16 * i) = x;
}

template <int D, int ROWS, int SRC>
static void pf_attn(const pf_args &a, hipStream_t stream) {
    auto go = [&](auto bf16) {
        constexpr bool B = decltype(bf16)::value;
        if constexpr (ROWS == 256) hipLaunchKernelGGL((k_pf_attn<D, SRC, B>), dim3(a.P), dim3(512), 0, stream, a);
        else hipLaunchKernelGGL((k_pf_attn_split<D, SRC, B>), dim3(a.P), dim3(512), 0, stream, a);
    };
    if (a.q_bf16) go(std::true_type{});
    else go(std::false_type{});
    if (a.n_seg == 1 && a.U % a.P == 0) return;           // every unit whole
    // The form by the most pieces of a unit (of one of its segments): a call's time, us,
    // with (waves, loads in flight) = (1, 2), (1, 4), (1, 8), (4, 4), (4, 8).
    //    2 pieces, 32 units of 128 dims   40.4  40.6  41.1  42.2  44.0
    //    2, 64 units (shares) of 128      33.1  33.4  34.9  38.7  43.7
    //    4, 12 units of 256 dims          36.1  35.9  36.6  36.8  38.1
    //    8, 4 units of 256 dims           25.5  24.8  24.5  24.8  25.3
    //    8, 2 units of 128 dims           15.4  14.7  14.3  14.4  14.8
    //   16, 2 units of 128 dims           16.1  14.8  14.2  13.5  14.0
    //   16, 12 units of 256 dims          25.0  24.1  24.3  24.1  24.9
    //   32, 1 unit of 128 dims            17.8  15.7  14.6  12.9  12.4
    //   64, 4 units of 256 dims           33.9  29.4  27.4  25.7  26.0
    // (A kernel trace does not show it: there every launch takes 4.5 us and more.)
    const dim3 g1(a.n_row_tiles * a.H, ROWS / 32, D / 32), g4(a.n_row_tiles * a.H, ROWS / 32, D / 8), t(256);
    const uint32_t n = a.P % a.U == 0 ? a.P / a.U : a.P / a.U + 2;
    if (n <= 2) hipLaunchKernelGGL((k_pf_combine<D, ROWS, 1, 2>), g1, t, 0, stream, a);
    else if (n <= 4) hipLaunchKernelGGL((k_pf_combine<D, ROWS, 1, 4>), g1, t, 0, stream, a);
    else if (n <= 8) hipLaunchKernelGGL((k_pf_combine<D, ROWS, 1, 8>), g1, t, 0, stream, a);
    else if (n <= 16) hipLaunchKernelGGL((k_pf_combine<D, ROWS, 4, 4>), g4, t, 0, stream, a);
    else hipLaunchKernelGGL((k_pf_combine<D, ROWS, 4, 8>), g4, t, 0, stream, a);
}

template <int D>
static void pf_launch(const pf_args &a, const pf_stage_args &sa, int src, uint32_t rows, uint32_t n_cu, hipStream_t stream) {
    if (src == PF_QUANT) return pf_attn<D, 128, PF_QUANT>(a, stream);
    if (src == PF_F16) return rows == 256 ? pf_attn<D, 256, PF_F16>(a, stream) : pf_attn<D, 128, PF_F16>(a, stream);
    // (8 workgroups of 4 waves a CU)
    if ((uint64_t)sa.n_tiles * a.H >= 8 * n_cu) hipLaunchKernelGGL((k_pf_stage<D, true>), dim3(sa.n_tiles, a.H), dim3(256), 0, stream, sa);
    else hipLaunchKernelGGL((k_pf_stage<D, false>), dim3(sa.n_tiles, a.H), dim3(256), 0, stream, sa);
    pf_attn<D, 256, PF_STAGED>(a, stream);
}

// ---- the launch's shape, from estimated costs (us)
// A 64-cell tile of a unit, as measured at D 256; at D 128 half of it is taken, where
// 1.1 - 1.25 (128 rows) and 2.0 - 2.2 (256) are measured: the lines below were found
// with these values.
static double pf_tile_us(uint32_t D, int src, uint32_t rows) {
    return (rows == 256 ? 3.3 : src == PF_QUANT ? 1.75 : 1.6) * D / 256;
}

// Workgroups that U units of n_tiles tiles are dealt to: equal shares to one per CU
// (LDS), or one whole unit each.  The same number s for every unit, so that none has
// two pieces (a second piece costs its workgroup another start and end, PF_START us:
// 100 tokens over 32 tiles, 20 units, took 39.9 us on 256 workgroups, 29.3 on 220),
// unless so many CUs would idle that the second piece is cheaper.  Each piece is
// written and read once more, `piece` us of all (500 tokens over 16 tiles of 128
// dims, 32 units: 30.2 us in 256 pieces, 22.8 in 128): over few tiles that costs more
// than a last round of whole units that does not fill the chip (64 heads on 8 x 128,
// 1,500 tokens, 376 units: over 2,048 cells 112 us in shares, 92.6 whole; over 8,192
// 399 and 426).  More units than CUs even out over the chip, so `seen` counts there:
// the tiles that a unit sees on the average, if the chunk is the window's last cells.
#define PF_START 8.0
static uint32_t pf_shares(uint64_t U, uint32_t n_tiles, double seen, double t, double piece, uint32_t n_cu) {
    double best = t * (U > n_cu ? seen : n_tiles) * U / n_cu;
    if (U % n_cu) best += PF_START + piece * (U < n_cu ? n_cu + U : 2.0 * n_cu);
    uint32_t P = n_cu;
    for (uint64_t s = 1; s * U <= n_cu && s <= n_tiles; ++s) {
        const double c = t * kvm_cdiv(n_tiles, s) + (s > 1 ? piece * (s * U) : 0.0);
        if (c < best) {
            best = c;
            P = (uint32_t)(s * U);
        }
    }
    // Whole units, longest first: the shortest fill a part of the last round's gap (0.6 as
    // measured: 32 heads on 8 x 128, 3,000 tokens over 8,192 cells, 376 units, 360 us in
    // shares and 369 whole; alone in the window 130 and 101).
    const double least = 2 * seen - n_tiles, gap = kvm_cdiv(U, n_cu) - (double)U / n_cu;
    if (U > n_cu && U < 65536 && t * std::max((double)n_tiles, seen * U / n_cu + 0.6 * gap * least) < best) P = (uint32_t)U;
    return P;
}
// A piece's partial output, written and read at the rate that such launches reach.
static double pf_piece_us(uint32_t D, uint64_t n_rows, uint32_t row_tiles) {
    return (double)n_rows / row_tiles * D * 8 / 3.2e6;
}

// Rows of a unit, and with them the kernel: 256 (k_pf_attn; a quantised window is
// converted ahead) once a workgroup would have PF_LONG tiles of 128 rows, 128
// (k_pf_attn_split) below.  Full windows, us with 256 and with 128 rows: 1,500 tokens x
// 512 tiles, 4 heads x 256, 1,055 and 1,215; 1,024 x 128, 210 and 236; 400 x 256, 179 and
// 190; 400 x 128, 106 and 106; 1,024 x 64, 120 and 122; 200 x 256, 114 and 106; on an f16
// window of 8 x 128, 1,024 x 256, 261 and 285; 1,024 x 32, 51 and 44.  What is live in the
// window is not known here: chunks that start a large one would rather have 128 rows
// (1,024 tokens alone in 8,192 cells of 8 x 128: 44 and 29, full 150 and 160).
// - PF_TIGHT instead, where the 256-row units fill the chip with one or two workgroups
//   each: the last row tiles then bound the call, and smaller units leave their
//   workgroups less (1,024 x 64, 8 x 128, 128 units: 87 and 84, and in a chunk that
//   is alone in the window 43 and 29; 2,048 x 32, 256 units: 70 and 58; from twice
//   that many tiles on 256 rows win, 1,024 x 128: 147 and 160).
// - A quantised window keeps 128 rows up to PF_FEW row tiles of 256: converting it
//   ahead costs more than so few of them save (32 heads, no groups, 128 dims: 200
//   x 256, one row tile, 144 and 98; 1,024 x 128, four, 182 and 166; 1,500 x 128,
//   six, 241 and 243).
#define PF_LONG 64.0
#define PF_TIGHT 112.0
#define PF_FEW 4u

struct pf_shape {
    uint32_t src, rows, n_row_tiles, n_seg, U, P;
    uint64_t slots;
};
static int pf_shape_of(bool quant, uint32_t D, uint32_t H, uint32_t n_tiles, uint32_t n_tokens, uint32_t G, uint32_t n_cu,
                       pf_shape *s) {
    const uint64_t n_rows = (uint64_t)n_tokens * G;
    s->n_seg = kvm_cdiv(n_tiles, KVM_PF_LIST);
    const uint64_t rt256 = kvm_cdiv(n_rows, 256), wgs = rt256 * H <= n_cu ? n_cu / (rt256 * H) : 0;      // workgroups a unit
    const bool tight = (wgs == 1 || wgs == 2) && wgs * rt256 * H * 8 >= 7u * n_cu;
    const bool long_work = (double)kvm_cdiv(n_rows, 128) * H * n_tiles / n_cu >= (tight ? PF_TIGHT : PF_LONG) &&
                           !(quant && rt256 <= PF_FEW);
    s->rows = long_work ? 256u : 128u;
    s->src = !quant ? PF_F16 : long_work ? PF_STAGED : PF_QUANT;
    s->n_row_tiles = (uint32_t)kvm_cdiv(n_rows, s->rows);
    const uint64_t units = (uint64_t)s->n_row_tiles * H * s->n_seg;
    if (units > (1u << 30)) return KVM_ERANGE;
    s->U = (uint32_t)units;
    const uint32_t seg_tiles = kvm_cdiv(n_tiles, s->n_seg);
    const double own = std::min(1.0, (double)n_tokens / ((double)n_tiles * KVM_TILE_CELLS));
    uint64_t P = pf_shares(units, seg_tiles, seg_tiles * (1.0 - own / 2), pf_tile_us(D, s->src, s->rows),
                           pf_piece_us(D, n_rows, s->n_row_tiles), n_cu);
    // KVM_PF_SPLITS in the environment fixes the pieces per unit
    if (const char *e = getenv("KVM_PF_SPLITS")) {
        const int v = atoi(e);
        if (v >= 1 && v <= 8) P = units * v < 65536u ? units * v : 65536u;
    }
    if (P * units > 0xffffffffu) P = 0xffffffffu / units;
    s->P = (uint32_t)P;
    s->slots = pf_slots(s->U, s->P, s->n_seg);
    return KVM_OK;
}

// The launch's shape and the slot of a piece, for tests on the host (not part of the ABI).
extern "C" int kvm_fa_prefill_shape(int k_type, uint32_t head_dim, uint32_t n_head_kv, uint32_t n_cells,
                                    uint32_t n_tokens, uint32_t n_head, uint32_t n_cu, uint32_t out[7]) {
    pf_shape s{};
    const int rc = pf_shape_of(kvm_k_quant(k_type), head_dim, n_head_kv, n_cells / KVM_TILE_CELLS,
                               n_tokens, n_head / n_head_kv, n_cu, &s);
    const uint32_t v[7] = {s.src, s.rows, s.n_row_tiles, s.n_seg, s.U, s.P, (uint32_t)s.slots};
    for (int i = 0; i < 7; ++i) out[i] = v[i];
    return rc;
}
extern "C" uint32_t kvm_fa_prefill_slots(uint32_t U, uint32_t P, uint32_t n_seg) { return (uint32_t)pf_slots(U, P, n_seg); }
extern "C" uint32_t kvm_fa_prefill_slot(uint32_t U, uint32_t P, uint32_t n_seg, uint32_t p, uint32_t u) {
    return pf_slot(U, P, n_seg, p, u, (uint32_t)((uint64_t)p * U / P));
}

extern "C" int kvm_fa_prefill(kvm_state *st, const kvm_window *w, const void *q, int q_type,
                              const int32_t *q_pos, uint32_t n_tokens, uint32_t n_head, float scale,
                              float *out) {
    if (!st || !w || !q || !q_pos || !out) return kvm_fail(st, KVM_EINVAL, "fa_prefill: null argument");
    int rc = kvm_window_check(w);
    if (rc) return kvm_fail(st, rc, "fa_prefill: bad window");
    if (q_type != KVM_TYPE_F32 && q_type != KVM_TYPE_BF16) return kvm_fail(st, KVM_EUNSUPPORTED, "fa_prefill: q type %d", q_type);
    if (!w->n_head_kv || n_head % w->n_head_kv) return kvm_fail(st, KVM_EINVAL, "fa_prefill: head counts");
    if (n_tokens == 0) return KVM_OK;
    const uint32_t G = n_head / w->n_head_kv;
    // Up to 32 rows per kv head the decode kernel's tile fits the whole query.
    if ((uint64_t)n_tokens * G <= 32) return kvm_fa_prefill_chunked(st, w, q, q_type, q_pos, n_tokens, n_head, scale, out);

    const uint32_t D = w->head_dim, H = w->n_head_kv, n_tiles = w->n_cells / KVM_TILE_CELLS;
    const uint64_t n_rows = (uint64_t)n_tokens * G;
    if (n_rows > (1u << 30)) return kvm_fail(st, KVM_ERANGE, "fa_prefill: %u tokens", n_tokens);
    pf_shape sh{};
    if (pf_shape_of(kvm_k_quant(w->k_type), D, H, n_tiles, n_tokens, G, st->n_cu, &sh))
        return kvm_fail(st, KVM_ERANGE, "fa_prefill: %u tokens", n_tokens);
    const int src = (int)sh.src;
    const uint32_t rows = sh.rows;

    pf_args a{};
    a.n_tiles = n_tiles;
    a.n_seg = sh.n_seg;
    a.H = H;
    a.G = G;
    a.n_head = n_head;
    a.n_rows = (uint32_t)n_rows;
    a.n_row_tiles = sh.n_row_tiles;
    a.U = sh.U;
    a.P = sh.P;
    a.c = scale * 1.4426950408889634f;
    a.q_bf16 = q_type == KVM_TYPE_BF16;
    a.longest = a.U == a.P && a.P > st->n_cu && a.n_seg == 1;
    a.q = q;
    a.q_pos = q_pos;
    a.out = out;
    a.cell_pos = w->cell_pos;
    a.k = (const uint8_t *)w->k;
    a.v = (const uint8_t *)w->v;

    // workspace: the pieces, and for PF_STAGED the f16 K and V operand tiles
    auto up256 = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t kv_bytes = src == PF_STAGED ? up256((size_t)H * n_tiles * 64 * D * 2) : 0;
    const size_t part_o = (size_t)sh.slots * rows * D * 4, part_ml = (size_t)sh.slots * rows * 8;
    // aligned copies (all sizes are multiples of 16)
    struct { const uint8_t **p; size_t bytes; } src_buf[3] = {
        {(const uint8_t **)&a.q, (size_t)n_tokens * n_head * D * (a.q_bf16 ? 2 : 4)},
        {&a.k, src == PF_F16 ? (size_t)H * n_tiles * 128 * D : 0},
        {&a.v, src == PF_F16 ? (size_t)H * n_tiles * 128 * D : 0}};
    size_t copies = 0;
    for (auto &b : src_buf) {
        if (!((uintptr_t)*b.p & 15)) b.bytes = 0;
        copies += up256(b.bytes);
    }
    const size_t total = 2 * kv_bytes + copies + part_o + part_ml;
    uint8_t *ws = nullptr;
    if (total) {
        ws = (uint8_t *)kvm_workspace(st, total);
        if (!ws) return kvm_fail(st, KVM_ENOMEM, "fa_prefill: workspace of %zu bytes", total);
    }
    pf_stage_args sa{};
    if (src == PF_STAGED) {
        sa.k = a.k;
        sa.v = a.v;
        sa.cell_pos = a.cell_pos;
        sa.kh = ws;
        sa.vh = ws + kv_bytes;
        sa.n_tiles = n_tiles;
        a.k = sa.kh;
        a.v = sa.vh;
    }
    KVM_HIP(st, hipSetDevice(st->device));
    uint8_t *at = ws + 2 * kv_bytes;
    for (auto &b : src_buf) {
        if (!b.bytes) continue;
        hipLaunchKernelGGL(k_pf_align, dim3(kvm_cdiv(b.bytes / 16, 256)), dim3(256), 0, st->stream, *b.p, at, (uint64_t)(b.bytes / 16));
        *b.p = at;
        at += up256(b.bytes);
    }
    a.ws_o = (float *)at;
    a.ws_ml = (float *)(at + part_o);

    if (D == 256) pf_launch<256>(a, sa, src, rows, st->n_cu, st->stream);
    else pf_launch<128>(a, sa, src, rows, st->n_cu, st->stream);
    KVM_LAUNCH_CHECK(st, "fa_prefill");
    return KVM_OK;
}
