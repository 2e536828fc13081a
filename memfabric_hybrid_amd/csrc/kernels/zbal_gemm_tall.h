/*
 * The grouped GEMM for experts with many rows, 8-bit modes: 320 rows x 256 channels x 128 K-bytes per step, eight waves, one
 * persistent workgroup per CU.
 *
 * What bounds it: no single unit. A step's MFMAs, the LDS reads that feed them and the transfers that refill the LDS each
 * take about half of it, and what is lost is lost where they wait for one another; the more they overlap, the lower the
 * clock that the power limit leaves (W8A8, 4096 tokens over 32 experts: MFMAs in 60 / 52 % of the cycles at 1.85 / 1.93 GHz, fp8 50 /
 * 45 % at 1.88 / 1.95). As built / slabs always in the L2 / no transfers / no stores of the second GEMM's rows, us: fp8 965 / 879 / 863
 * and 514 / 486 / 449 / 455, W8A8 893 / 812 / 760 and 461 / 423 / 382 / 388. Hence:
 *
 *  - The waves are two row groups x four channel ranges. A wave keeps the four weight fragments of a step in registers and
 *    streams its ten activation fragments past them, so that every fragment is read once (four row groups of five sub-tiles
 *    had no registers for a step's weights and read them twice).
 *  - A stage of the LDS is handed back in two parts. The weights and the first 128 rows have been read by the middle of a
 *    step, the other rows by its end, and each part is refilled for the step after next as soon as the barrier there has been
 *    passed: every transfer has at least one whole step to arrive, in two stages.
 *  - Either barrier stands in front of a sub-tile whose operands are in registers already; behind it the first fragments of
 *    the next part are asked for, and that sub-tile's MFMAs run while they come. At the end of a step the weight fragments
 *    are replaced one by one, each after its last MFMA.
 *  - One K loop for every number of rows: a sub-tile that has none is branched over. (One loop for each number, as in the
 *    kernels with fewer sub-tiles, costs registers where the loops meet: hundreds of them spilled here.)
 *  - fp8's activation scales come as four steps of 64 rows per transfer. As one step of them, every lane on a line of its own,
 *    they kept the address unit busy for a third of its time (first GEMM 1.15 against 1.02 ms).
 *  - The tiles of a workgroup are worked out 32 at a time, one per lane.
 */
#ifndef ZBAL_GEMM_TALL_H_
#define ZBAL_GEMM_TALL_H_

#include "zbal_gemm_tile.h"

namespace {

template <int MODE> struct TallShape {
    static constexpr int TM = 320, THREADS = 512, RG = 2, COL_GROUPS = 4, NT = 4, MTM = 10;
    static constexpr int HALF = 4;                              /* sub-tiles per wave in the first part: 128 rows of the tile */
    static constexpr int A_BYTES = TM * BKB, STAGE_BYTES = A_BYTES + BN * 128;
    static constexpr int MAX_KB = 256, MAX_EXPERTS = 512, TABLE = 32;
    static constexpr int SA_FLOATS = MODE == MODE_FP8 ? TM * 4 : 0;                      /* four steps' block scales, [row][step] */
    static constexpr int SC_FLOATS = MODE == MODE_FP8 ? MAX_KB : 256 + TM;               /* fp8: weight block scales, twice 128; W8A8: channel and token scales */
    static constexpr int LDS_BYTES = 2 * (STAGE_BYTES + SA_FLOATS * 4 + SC_FLOATS * 4) + TM * 4 + TABLE * 16 + (MAX_EXPERTS + 1) * 4;
    static_assert(LDS_BYTES <= 160 * 1024, "tile does not fit the LDS");
};

/*
 * The tables end the number of experts. fp8's scales travel as four steps of a row: rows of fewer are read along with a
 * neighbour's, which wants a tile without the first or the last row of all.
 */
template <int MODE> inline bool tall_accepts(const GemmParams &p)
{
    const int kb = p.K / 128;
    if (kb < 2 || p.experts > TallShape<MODE>::MAX_EXPERTS) return false;
    return MODE != MODE_FP8 || (kb <= TallShape<MODE>::MAX_KB && (kb >= 4 || p.max_rows > TallShape<MODE>::TM));
}

/*
 * fp8: K whose steps leave one over from groups of four, make less than one group, or are more than the weight block scales have
 * room for twice, take a kernel of their own (ANY_K), because what it asks in every step costs the others: 1024 rows per expert,
 * 32 experts of 7168 x 4096 / 2048 x 7168, 990 -> 1010 / 532 -> 550 us. Those K in the 256-row shape -> in ANY_K, first GEMM 4096 wide,
 * second 7168: 32 experts, K 1152, 256 rows 73 -> 57 us, 512 rows 113 -> 100, 1800 rows 338 -> 325; K 5248, 256 rows 335 -> 223, 1024
 * rows 818 -> 757; K 256, 512 rows 51 -> 44; second, K 640, 512 rows 157 -> 126, K 384 126 -> 98; 8 experts, K 17408, 300 rows 454 -> 278.
 */
inline bool tall_wants_any_k(int kb) { return kb < 4 || kb % 4 == 1 || kb > 128; }

template <int MODE, bool GMM1, int OUT_DT, bool ANY_K = false>
__global__ void __launch_bounds__(512, 2)
grouped_gemm_tall_kernel(GemmParams p)
{
    static_assert(MODE == MODE_W8A8 || MODE == MODE_FP8, "8-bit modes");
    static_assert(!ANY_K || MODE == MODE_FP8, "W8A8 has no scales by step");
    using S = TallShape<MODE>;
    constexpr Shared SH = SHARED_ON_DEMAND;
    constexpr int TM = S::TM, RG = S::RG, NT = S::NT, MTM = S::MTM, H = S::HALF, A_BYTES = S::A_BYTES, STAGE_BYTES = S::STAGE_BYTES;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    float *lds_sa = reinterpret_cast<float *>(smem + 2 * STAGE_BYTES);
    float *lds_sc = lds_sa + 2 * S::SA_FLOATS;
    float *lds_rowmax = lds_sc + 2 * S::SC_FLOATS;                          /* [TM], zero between the epilogues */
    int *lds_tiles = reinterpret_cast<int *>(lds_rowmax + TM);              /* [TABLE][4]: expert and channel tile, first row, end, - */
    int *lds_mtp = lds_tiles + S::TABLE * 4;                                /* [experts + 1] row tiles before expert e */

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / S::COL_GROUPS, wn = wave % S::COL_GROUPS;
    const int n_tiles = GMM1 ? (p.N / 2) / 128 : p.N / BN;
    const int K = p.K, KB = K / 128, I = p.N / 2, E = p.experts;

    if (wave == 0) {
        int run = 0;
        for (int base = 0; base < E; base += 64) {
            const int e = base + lane;
            const int mt = e < E ? (p.row_off[e + 1] - first_row_of<SH>(p, e) + TM - 1) / TM : 0;
            int incl = mt;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int o = __shfl_up(incl, off, 64);
                if (lane >= off) incl += o;
            }
            if (e < E) lds_mtp[e] = run + incl - mt;
            run += __shfl(incl, 63, 64);
        }
        if (lane == 0) lds_mtp[E] = run;
    }
    if (tid < TM) lds_rowmax[tid] = 0.0f;
    __syncthreads();

    /*
     * XCD x (workgroups x, x + 8, ...) has a contiguous run of the logical tile order, its workgroups take consecutive tiles of
     * it. Tiles walk an expert in groups of (all its row tiles) x (as many channel tiles as make the group fit the XCD's
     * workgroups), row tile fastest: concurrent tiles share slabs in the L2. An expert's rows are cut evenly, in multiples of 16.
     */
    const int total = __builtin_amdgcn_readfirstlane(lds_mtp[E]) * n_tiles;
    const int chunk = (total + 7) / 8, slots = gridDim.x >> 3;
    const int id0 = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
    const int id_end = ((int)(blockIdx.x & 7) + 1) * chunk < total ? ((int)(blockIdx.x & 7) + 1) * chunk : total;
    if (id0 >= id_end) return;
    /* ANY_K has no registers for what the compiler would work out of `lane` ahead of the loops */
    auto fresh_lane = [&]() __attribute__((always_inline)) {
        int l = lane;
        if constexpr (ANY_K) asm volatile("" : "+v"(l));
        return l;
    };
    /* tiles `from` .. `from` + 31 of this workgroup's sequence, one per lane of wave 0 */
    auto make_table = [&](int from) __attribute__((always_inline)) {
        const int lane_t = fresh_lane();
        int n_tiles_t = n_tiles;
        if constexpr (ANY_K) asm volatile("" : "+s"(n_tiles_t));
        const int id = id0 + (from + lane_t) * slots;
        if (wave != 0 || lane_t >= S::TABLE) return;
        int expert = -1, n_tile = 0, row_begin = 0, row_end = 0;
        if (id < id_end) {
            const int q = id / n_tiles_t;
            int lo = 0, hi = E;                                       /* mtp[lo] <= q < mtp[hi] */
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (lds_mtp[mid] <= q) lo = mid;
                else hi = mid;
            }
            expert = lo;
            const int first = lds_mtp[lo], mt_e = lds_mtp[lo + 1] - first, l = id - first * n_tiles_t;
            int group_n = slots / mt_e;
            group_n = group_n < 1 ? 1 : (group_n > GROUP_N ? GROUP_N : group_n);
            const int per_group = mt_e * group_n, ng = l / per_group, r = l - ng * per_group;
            n_tile = ng * group_n + r / mt_e;
            const int first_row = first_row_of<SH>(p, expert), end_row = p.row_off[expert + 1];
            const int height = (((end_row - first_row + mt_e - 1) / mt_e) + 15) & ~15;
            row_begin = first_row + r % mt_e * height;
            row_end = row_begin + height < end_row ? row_begin + height : end_row;
        }
        *reinterpret_cast<i32x4 *>(lds_tiles + lane_t * 4) = i32x4{expert, n_tile, row_begin, row_end};
    };
    struct Tile {
        int expert, n_tile, row_begin, row_end, last_rel;
        const uint8_t *a;            /* slab 0 */
        const uint8_t *w[2];
        const float *sa;
    };
    auto tile_at = [&](int i) -> Tile {
        const i32x4 v = *reinterpret_cast<const i32x4 *>(lds_tiles + (i & (S::TABLE - 1)) * 4);
        Tile t;
        t.expert = __builtin_amdgcn_readfirstlane(v[0]);
        t.n_tile = __builtin_amdgcn_readfirstlane(v[1]);
        t.row_begin = __builtin_amdgcn_readfirstlane(v[2]);
        t.row_end = __builtin_amdgcn_readfirstlane(v[3]);
        if (t.expert < 0) return t;
        t.last_rel = t.row_end - 1 - t.row_begin;
        t.a = p.a + (int64_t)t.row_begin * K;
        t.sa = p.a_scale + (int64_t)t.row_begin * KB;
        const int col0 = GMM1 ? t.n_tile : t.n_tile * 2, col1 = GMM1 ? I / 128 + t.n_tile : t.n_tile * 2 + 1;
        const uint8_t *wb = weights_of<uint8_t, SH>(p, t.expert, (int64_t)(p.N / 128) * KB * 16384);
        t.w[0] = wb + (int64_t)col0 * KB * 16384;
        t.w[1] = wb + (int64_t)col1 * KB * 16384;
        return t;
    };
    make_table(0);
    __syncthreads();

    /*
     * Transfers. Part 1 of a slab, six (and sometimes the scales) of every wave: the weights and rows 0-127; part 2, two or
     * three: the other rows. Rows past the tile's end repeat its last one; past row 255 they are left out.
     */
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem) + wave * 1024);
    const uint32_t t_row = 8 * wave + (lane >> 3), t_chunk = ((lane & 7) ^ ((lane >> 3) ^ (wave & 1))) * 16, t_w = wave * 1024 + lane * 16;
    auto bring_w = [&](const Tile &t, int kb, int stage, int j) __attribute__((always_inline)) {
        dma16_sv(t.w[j >> 1] + ((int64_t)kb * 16384 + (j & 1) * 8192), t_w, lds0 + stage * STAGE_BYTES + A_BYTES + j * 8192);
    };
    auto bring_a = [&](const Tile &t, int kb, int stage, int j) __attribute__((always_inline)) {
        if (j == 4 && 256 + 8 * wave > t.last_rel) return;
        uint32_t rel = 64 * j + t_row;
        if (rel > (uint32_t)t.last_rel) rel = t.last_rel;
        dma16_sv(t.a + (int64_t)kb * BKB, __umul24(rel, (uint32_t)K) + t_chunk, lds0 + stage * STAGE_BYTES + j * 8192);
    };
    /*
     * fp8's activation scales come in groups of four steps, to two buffers in turn. The last group of a tile brings the row's
     * last four values, whatever it uses of them. It starts at step `tail`; where four would leave one step over, the last two
     * groups have three and two, because the group after the next may not come before this one has been used up. A row of two
     * or three values comes with the end of the row before it, in the tile of the very first row with the start of the one behind.
     */
    const int tail = !ANY_K ? 0 : (KB % 4 == 1 ? KB - 2 : (KB - 1) & ~3);
    auto starts_group = [&](int kb) __attribute__((always_inline)) { return ANY_K ? kb == tail || (kb < tail && (kb & 3) == 0) : (kb & 3) == 0; };
    /* a step's place among its group's four values */
    auto place = [&](const Tile &t, int kb) __attribute__((always_inline)) {
        return kb < tail ? kb & 3 : (KB < 4 && t.row_begin == 0 ? kb : kb - (KB - 4));
    };
    /* the group that starts with step kb, 64 rows per wave, by waves 0-4 */
    auto bring_sa = [&](const Tile &t, int kb, int half) __attribute__((always_inline)) {
        if (MODE != MODE_FP8 || wave >= TM / 64) return;
        uint32_t rel = wave * 64 + fresh_lane();
        if (rel > (uint32_t)t.last_rel) rel = t.last_rel;
        const int from = ANY_K ? kb - place(t, kb) : (kb + 4 > KB ? KB - 4 : kb);
        dma16_sv(reinterpret_cast<const uint8_t *>(t.sa + from), __umul24(rel, (uint32_t)KB * 4u), lds_addr(lds_sa) + (half * S::SA_FLOATS + wave * 256) * 4);
    };
    /*
     * fp8: the weight block scales of up to 128 steps, for either 128 of the channels, to one of two buffers in turn. With more
     * steps the two are one: the second 128 (`upper`) come beside the tile's first step, the next tile's first 128 once all
     * of this one's have been used. W8A8: what the epilogue scales with (channels at 0, tokens at 256).
     */
    int bufs = ANY_K && KB > 128 ? 1 : 2;
    if constexpr (ANY_K) asm volatile("" : "+s"(bufs));                 /* or the compiler keeps `buf` in a vector register */
    const int second = ANY_K && KB > 128 ? 256 : 128;                   /* where the second 128 channels' start */
    auto bring_scales = [&](const Tile &t, int buf, bool upper = false) __attribute__((always_inline)) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_addr(lds_sc) + buf * S::SC_FLOATS * 4);
        if constexpr (MODE == MODE_FP8) {
            const int stride = p.N / 128;
            const float *base = scales_of<float, SH>(p, t.expert, (int64_t)KB * stride) +
                                (wave < 4 ? (GMM1 ? t.n_tile : t.n_tile * 2) : (GMM1 ? I / 128 + t.n_tile : t.n_tile * 2 + 1));
            const int b = (wave & 3) * 64;
            const int step = b + fresh_lane();
            if ((!ANY_K || (b >= 128) == upper) && step < KB) dma4_sv(base, (uint32_t)step * (uint32_t)stride * 4u, dst + ((wave < 4 ? 0 : second) + b) * 4);
        } else {
            if (wave < TM / 64) {
                const int rel = wave * 64 + lane > t.last_rel ? t.last_rel : wave * 64 + lane;
                dma4_sv(p.a_scale + t.row_begin, (uint32_t)rel * 4u, dst + 1024 + wave * 256);
            }
            if (wave < 4) {
                if (GMM1 || !p.wscale_is_bf16) {
                    const float *ws = scales_of<float, SH>(p, t.expert, p.N);
                    const int at = !GMM1 ? t.n_tile * BN + wave * 64 : (wave < 2 ? t.n_tile * 128 + wave * 64 : I + t.n_tile * 128 + (wave - 2) * 64);
                    dma4_sv(ws + at, lane * 4u, dst + wave * 256);
                } else if (wave < 2) {
                    const uint16_t *ws = scales_of<uint16_t, SH>(p, t.expert, p.N);
                    dma4_sv(reinterpret_cast<const float *>(ws + t.n_tile * BN + wave * 128), lane * 4u, dst + wave * 256);
                }
            }
        }
    };
    /*
     * One part has landed for everybody and nobody reads the one before it any more. Eight younger transfers of this wave at
     * least, the two parts that were asked for since, may stay in flight.
     */
    auto landed = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    /* fragments: row lane % 16 of a 16-row sub-tile, logical chunks 2 * (lane / 16) and the next */
    const int frag_row = lane & 15;
    const int key = (lane & 7) ^ ((lane >> 3) & 1), g2 = (lane >> 4) * 2;
    const int off_lo = frag_row * BKB + ((g2 ^ key) * 16), off_hi = frag_row * BKB + (((g2 + 1) ^ key) * 16);
    auto frag = [&](const uint8_t *at) -> i32x8 {
        const u32x4 lo = *reinterpret_cast<const u32x4 *>(at + off_lo);
        const u32x4 hi = *reinterpret_cast<const u32x4 *>(at + off_hi);
        return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    };
    int stage = 0, half = 0;          /* `half`: which buffer holds this step's fp8 scales */
    auto load_w = [&](int nt) -> i32x8 {
        const int r = GMM1 ? (nt < NT / 2 ? wn * 32 + nt * 16 : 128 + wn * 32 + (nt - NT / 2) * 16) : wn * 64 + nt * 16;
        return frag(smem + stage * STAGE_BYTES + A_BYTES + r * BKB);
    };
    auto load_a = [&](int mt) -> i32x8 { return frag(smem + stage * STAGE_BYTES + (RG * mt + wm) * (16 * BKB)); };
    auto load_sa = [&](int mt, int k4) -> float {
        return MODE == MODE_FP8 ? lds_sa[half * S::SA_FLOATS + ((RG * mt + wm) * 16 + frag_row) * 4 + k4] : 0.0f;
    };

    int seq = 0, buf = 0;
    Tile cur = tile_at(0);
    bring_scales(cur, 0);
    bring_a(cur, 0, 0, 0);
    bring_a(cur, 0, 0, 1);
#pragma unroll
    for (int j = 0; j < 4; ++j) bring_w(cur, 0, 0, j);
    bring_sa(cur, 0, 0);
#pragma unroll
    for (int j = 2; j < 5; ++j) bring_a(cur, 0, 0, j);
    bring_a(cur, 1, 1, 0);
    bring_a(cur, 1, 1, 1);
#pragma unroll
    for (int j = 0; j < 4; ++j) bring_w(cur, 1, 1, j);
    landed();
    i32x8 wf[NT], a[2] = {};
    float sa[2] = {};
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wf[nt] = load_w(nt);
    a[0] = load_a(0);
    sa[0] = load_sa(0, ANY_K ? place(cur, 0) : 0);

    while (true) {
        if ((++seq & (S::TABLE - 1)) == 0) {
            make_table(seq);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        Tile nxt = tile_at(seq);
        const bool more = nxt.expert >= 0;
        if (!more) nxt = cur;                  /* the last slabs' successors: asked for, never read */
        f32x4 accf[MTM][NT];
        i32x4 acci[MTM][NT];
#pragma unroll
        for (int mt = 0; mt < MTM; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                accf[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                acci[mt][nt] = i32x4{0, 0, 0, 0};
            }
        const int mt_act = (((cur.row_end - cur.row_begin + 15) >> 4) - wm + RG - 1) / RG;
        /* GMM1: gate and up have a weight block each; GMM2: the wave's channels are in one */
        const float *sw0_at = lds_sc + buf * S::SC_FLOATS + (!GMM1 && wn >= 2 ? second : 0), *sw1_at = lds_sc + buf * S::SC_FLOATS + second;
        float sw0 = 0.0f, sw1 = 0.0f;
        if constexpr (MODE == MODE_FP8) {
            sw0 = sw0_at[0];
            if (GMM1) sw1 = sw1_at[0];
        }
        /* a row sub-tile's sums; RENEW: the weight fragments are replaced behind their last use */
        auto sub_tile = [&](int mt, const i32x8 af, float s, auto renew_tag) __attribute__((always_inline)) {
            constexpr bool RENEW = decltype(renew_tag)::value;
            if constexpr (MODE == MODE_FP8) {
                const float s0 = s * sw0, s1 = GMM1 ? s * sw1 : s0;
                f32x4 part = mfma_fp8_16x16x128(wf[0], af);
                if (RENEW) wf[0] = load_w(0);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    f32x4 next = part;
                    if (nt + 1 < NT) {
                        next = mfma_fp8_16x16x128(wf[nt + 1], af);
                        if (RENEW) wf[nt + 1] = load_w(nt + 1);
                    }
                    const float sc = GMM1 && nt >= NT / 2 ? s1 : s0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) accf[mt][nt][i] = __builtin_fmaf(part[i], sc, accf[mt][nt][i]);
                    part = next;
                }
            } else {
                /*
                 * A wave with MFMAs to issue goes before the one that asks for fragments and transfers: 32 experts of 7168 x 4096 / 2048 x
                 * 7168, 700 rows per expert 632 -> 623 / 340 -> 329 us, 1024 rows 876 -> 862 / 465 -> 457; 128 of 4096 x 3072 / 1536 x 4096,
                 * 512 rows 865 -> 858 / 440 -> 434. (fp8, whose other wave converts as long: 1 % slower.)
                 */
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acci[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{wf[nt][0], wf[nt][1], wf[nt][2], wf[nt][3]},
                                                                         i32x4{af[0], af[1], af[2], af[3]}, acci[mt][nt], 0, 0, 0);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    acci[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{wf[nt][4], wf[nt][5], wf[nt][6], wf[nt][7]},
                                                                         i32x4{af[4], af[5], af[6], af[7]}, acci[mt][nt], 0, 0, 0);
                    if (RENEW) wf[nt] = load_w(nt);
                }
                __builtin_amdgcn_s_setprio(0);
            }
        };
#pragma clang loop unroll(disable)
        for (int kb = 0; kb < KB; ++kb) {
            const bool in2 = kb + 1 < KB, in1 = kb + 2 < KB;
            const Tile &t2 = in2 ? cur : nxt, &t1 = in1 ? cur : nxt;        /* whose slabs the two parts that are asked for in this step belong to */
            const int kb2 = in2 ? kb + 1 : 0, kb1 = in1 ? kb + 2 : kb + 2 - KB;
            const int st = stage, k4 = ANY_K ? place(cur, kb) : (kb + 4 - (kb & 3) > KB ? kb - (KB - 4) : kb & 3);
            int act = mt_act;
            asm volatile("" : "+s"(act));       /* compared where it is asked for: ten conditions in scalar registers push others out */
            i32x8 az;
            float saz = 0.0f, sw0_n = 0.0f, sw1_n = 0.0f;
#pragma unroll
            for (int mt = 0; mt < H; ++mt) {
                if (mt == H - 1) {
                    landed();
                    if (kb == 0) {             /* everybody is past the last tile's epilogue */
                        if (!ANY_K && more) bring_scales(nxt, buf ^ 1);
                        if constexpr (ANY_K) {
                            if (GMM1 && wave < TM / 64) lds_rowmax[wave * 64 + fresh_lane()] = 0.0f;
                        } else if (GMM1 && tid < TM) lds_rowmax[tid] = 0.0f;
                    }
                    if (ANY_K && (kb == 0 || (KB > 128 && kb == 127))) {
                        const bool upper = KB > 128 && kb == 0;
                        if (upper || more) bring_scales(upper ? cur : nxt, buf ^ (bufs - 1), upper);
                    }
                    az = load_a(H);
                    saz = load_sa(H, k4);
                    if constexpr (MODE == MODE_FP8) {
                        sw0_n = sw0_at[kb2];
                        if (GMM1) sw1_n = sw1_at[kb2];
                    }
                }
                a[(mt + 1) & 1] = load_a(mt + 1 < H ? mt + 1 : H + 1);
                sa[(mt + 1) & 1] = load_sa(mt + 1 < H ? mt + 1 : H + 1, k4);
                /* int8: in front of the sub-tile's MFMAs, fp8: behind them (each the other way round 1-3 % slower) */
                if (MODE != MODE_FP8 && mt < 3) bring_a(t2, kb2, st ^ 1, 2 + mt);
                if (mt < act) sub_tile(mt, a[mt & 1], sa[mt & 1], std::false_type{});
                if (MODE == MODE_FP8 && mt < 3) bring_a(t2, kb2, st ^ 1, 2 + mt);
                __builtin_amdgcn_sched_barrier(0);
            }
            /*
             * Sub-tile H is kept for the end: it covers the change of steps. The transfers go out in twos, the weights, which come
             * from further away, first (all at once 2-3 % slower; activations first, fp8, 1 %).
             */
#pragma unroll
            for (int mt = H + 1; mt < MTM; ++mt) {
                constexpr int FIRST = H + 1;
                const int b = (mt - FIRST) & 1;
                if (mt == FIRST) { bring_w(t1, kb1, st, 0); bring_w(t1, kb1, st, 1); }
                if (mt == FIRST + 1) { bring_w(t1, kb1, st, 2); bring_w(t1, kb1, st, 3); }
                if (mt == FIRST + 2) { bring_a(t1, kb1, st, 0); bring_a(t1, kb1, st, 1); }
                if (mt == FIRST + 3 && MODE == MODE_FP8 && starts_group(kb1)) bring_sa(t1, kb1, half ^ 1);
                if (mt < act) {
                    if (mt + 1 < MTM) {
                        a[b ^ 1] = load_a(mt + 1);
                        sa[b ^ 1] = load_sa(mt + 1, k4);
                    }
                    sub_tile(mt, a[b], sa[b], std::false_type{});
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            stage ^= 1;
            if (ANY_K ? starts_group(kb2) : k4 == 3) half ^= 1;        /* the last group of a tile ends with its last step */
            landed();
            a[0] = load_a(0);
            sa[0] = load_sa(0, ANY_K ? place(t2, kb2) : (kb2 + 4 - (kb2 & 3) > KB ? kb2 - (KB - 4) : kb2 & 3));
            sub_tile(H, az, saz, std::true_type{});
            sw0 = sw0_n;
            sw1 = sw1_n;
            __builtin_amdgcn_sched_barrier(0);
        }
        TileCoord tc;
        tc.expert = cur.expert;
        tc.m_tile = 0;
        tc.n_tile = cur.n_tile;
        int lane_e = lane;
        asm volatile("" : "+v"(lane_e));       /* nothing of the epilogue's stays live across the K loop */
        epilogue<MODE, GMM1, OUT_DT, RG, MTM, NT, SH, true>(p, tc, accf, acci, cur.row_begin, cur.row_end, wm, wn, lane_e, lds_rowmax, TM,
                                                            lds_sc + buf * S::SC_FLOATS);
        if (!more) break;
        cur = nxt;
        buf ^= bufs - 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       /* the LDS goes to another workgroup */
}

} // namespace

#endif /* ZBAL_GEMM_TALL_H_ */
