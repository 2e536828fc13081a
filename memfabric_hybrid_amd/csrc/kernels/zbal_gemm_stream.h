/*
 * The grouped GEMM as a weight stream: the kernel for experts with few or moderately many rows, and for int4 weights with any number.
 *
 * A weight byte is wanted by one wave only, so the weights do not go through LDS: a wave keeps the fragments of the next
 * four slabs (128 K each) of its own 32 channels in flight in registers, in exactly the order the pre-pack stores them
 * (a 16-channel sub-tile of a slab is 2 KiB of consecutive bytes, int4 1 KiB), and nothing in the stream waits for
 * another wave. The activations, which all eight waves read, come in chunks of four slabs through two LDS buffers filled
 * by DMA: one barrier per four slabs. Workgroup tile: TM rows x 256 channels; a wave has all rows of its 32 channels
 * (first GEMM: 16 gate and the matching 16 up columns), so a weight is unpacked once, and the epilogue is that of the
 * kernel that stages the slabs (gemm.hip).
 *
 * With 128 registers per lane and at most 80 KiB of LDS two workgroups are resident per CU: four waves per SIMD to cover
 * each other's waits, 256 KiB of 8-bit weights in flight, one workgroup's start and epilogue behind the other's stream.
 * Workgroups are not persistent: the dispatcher evens out what a fixed sequence of tiles per CU cannot (528 tiles on 256
 * CUs, popular experts).
 *
 * What bounds it: 8-bit weights the HBM stream (6.1-6.6 TB/s), int4 the vector instructions that unpack and scale
 * (active in 43 % of the cycles, MFMA in 16 %, at 32 rows per expert). Layers against the staging kernel on one GPU, other
 * weights on every pass: W8A8, 128 experts of 4096 x 3072 / 1536 x 4096, top-8, 509 tokens 487 -> 461 us, Zipf(1.2)
 * routing 508 -> 457; 64 of 2048 x 2048 / 1024 x 2048, top-6, 200 tokens 111 -> 97. W4A8, 128 experts: 20 tokens 188 -> 166,
 * 509 tokens 320 -> 271, Zipf 397 -> 294, 2048 Zipf 842 -> 562, 16384 (96 rows) 3913 -> 3749.
 * A token or two: the tiles are halved between two workgroups of four waves (SPLIT, see few_tiles in gemm.hip).
 * The taller tiles: W8A8, 128 experts, 2048 tokens 720 -> 657, 1200 tokens Zipf 647 -> 558; fp8, 32 experts, 512 tokens 424 -> 384.
 */
#ifndef ZBAL_GEMM_STREAM_H_
#define ZBAL_GEMM_STREAM_H_

#include "zbal_gemm_tile.h"

namespace {

template <int MODE, int TM, int SPLIT = 1, bool VALUES = false> struct StreamShape {
    /* in the taller tiles the L2 serves the weights: two slabs of look-ahead do, and leave registers for six or eight row sub-tiles */
    static constexpr int PF = TM > (MODE == MODE_FP8 ? 48 : 64) ? 2 : 4;                  /* slabs in flight, and slabs per activation chunk */
    static constexpr int MT_STEP = 4 / PF;                      /* row sub-tiles come in ones, or in twos: then two slabs of them are one transfer of every wave */
    static constexpr int NW = 8 / SPLIT, NT = 2, THREADS = NW * 64;      /* SPLIT workgroups share a tile's channels */
    static constexpr int MTM = TM / 16;
    static constexpr int LOADS = MODE == MODE_W4A8 ? 1 : 2;     /* 16-byte loads per lane, sub-tile and slab */
    static constexpr int WRB = MODE == MODE_W4A8 ? 64 : 128;    /* bytes of a weight row per slab */
    static constexpr int A_BYTES = PF * TM * BKB;               /* one chunk: [slab][row][128 bytes, swizzled] */
    static constexpr int SA_ROWS = TM > 64 ? 128 : 64;
    static constexpr int SA_FLOATS = MODE == MODE_FP8 ? PF * SA_ROWS : 0; /* one chunk's block scales, [slab][row] */
    static constexpr int GS_BYTES = MODE == MODE_W4A8 ? PF * BN * 2 : 0;  /* one chunk's fp16 group scales, [slab][channel] */
    static constexpr int SA_LOADS = PF > NW ? PF / NW : 1;
    static constexpr int ES_FLOATS = MODE == MODE_FP8 ? 2 * 256 : (MODE == MODE_W8A8 ? 256 : 0) + (TM + 63) / 64 * 64;
    /* VALUES, see k_loop: the activations of as many slabs as there is room for, [slab][rows of the sub-tiles that there are][128 bytes, swizzled] */
    static constexpr int A_ALL = VALUES ? 2048 * TM : 2 * A_BYTES;
    static constexpr int LDS_BYTES = A_ALL + 2 * (SA_FLOATS * 4 + GS_BYTES) + ES_FLOATS * 4 + NW * TM * 4;
    static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups per CU");
};

/*
 * W4A8: tiles of 128 rows instead of 64. Shapes as at stream_rows, uniform / Zipf(0.6) / Zipf(1.2) routing, both GEMMs, per cent
 * that 128 rows take more: M 80 rows -9 / +3 / +6, 112 -7 / -4 / +1, 200 -7 / -5 / -3, 640 -5 / -6 / -8, 1024 -8 / -8 / -8; S 64 rows
 * -9 / +20 / +9, 200 -6 / +4 / +2, 250 -1 / -1 / +1, 375 -2 / -4 / -3, 640 -7 / -7 / -8; W 128 rows +4 / 0 / +5, 200 -6 / -3 / -3; 8 experts of
 * 14336 x 4096 200 rows +8 / - / +33; 2 of 4096 x 3072, 70 tiles, +16: from where the taller tiles all but fill the chip (two
 * workgroups per CU) twice, which S does at 250 rows, and once with many rows. Below that 64 rows are no worse than the 96 that ran there before: 700 rows per expert, first /
 * second GEMM, 8 experts of S 48.5 -> 44.8 / 21.5 -> 22.1 us, 8 of M 110.5 -> 111.0 / 48.0 -> 46.1; 900 rows, 8 of S 69.5 -> 55.4 / 30.7 -> 27.4.
 */
inline bool w4a8_taller_tile(int64_t rows, int64_t experts, int n_tiles, int64_t cus)
{
    return rows > 112 * experts && rows * n_tiles >= (rows > 640 * experts ? 2 * 128 : 500) * (cus > 0 ? cus : 256);
}

/*
 * A weight load whose wait is counted by hand. The compiler counts its own loads exactly, but not the LDS-DMA transfers
 * issued from inline asm, so its waits reach that many loads too far: half of what an int4 wave has in flight. The value
 * may only be touched after a wait_w() that names it (tests/test_kernel_asm_checks.py reads the generated code for that);
 * `s_nop 4`: a scalar base fresh from a vector instruction (see dma16_sv).
 */
template <bool STREAM>
__device__ __forceinline__ void load16_sv(u32x4 &v, uint32_t lane_off, const uint8_t *uniform_base)
{
    if constexpr (STREAM) asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %1, %2 nt" : "=v"(v) : "v"(lane_off), "s"(uniform_base));
    else asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(lane_off), "s"(uniform_base));
}
template <int N> __device__ __forceinline__ void wait_w(u32x4 (&w)[2][1])
{
    asm volatile("s_waitcnt vmcnt(%2)" : "+v"(w[0][0]), "+v"(w[1][0]) : "n"(N));
}
template <int N> __device__ __forceinline__ void wait_w(u32x4 (&w)[2][2])
{
    asm volatile("s_waitcnt vmcnt(%4)" : "+v"(w[0][0]), "+v"(w[0][1]), "+v"(w[1][0]), "+v"(w[1][1]) : "n"(N));
}

/* which of them share left-over tiles along K, see the kernel */
template <int MODE, bool GMM1, int SPLIT> constexpr bool stream_shares_k() { return GMM1 && MODE == MODE_W8A8 && SPLIT == 1; }

/*
 * Rows up to which an XCD's tiles that are over, `rest` of them, are shared, all of them or none: the longer the K loop, the more a part
 * saves, and the exchange costs by rows and parts. First W8A8 GEMM, N 2048, an expert per CU and XCD times 1 to 4 and `rest` more, all
 * with the same rows, per cent of the unshared launch, at 2 / 16 / 32 / 64 / 84 rows:
 *   - K 4608: rest 1 -13 ... -4 / -10 ... -3 / -6 ... -2 / +1 ... +2 / +3 ... +5; 4 -13 ... -3 / -9 ... -2 / -4 ... 0 / +2 ... +5 / +4 ... +9; 8 -7 ... -1 /
 *     -3 ... +1 / +2 / +5 ... +11 / +8 ... +16; 10 -7 ... -1 / -4 ... 0 / 0 ... +1 / +4 ... +9 / +6 ... +15;
 *   - K 7168: rest 1 -18 ... -5 / -15 ... -4 / -11 ... -3 / -6 ... -2 / -2 ... +1; 4 -16 ... -4 / -13 ... -3 / -10 ... -2 / -4 ... -1 / 0 ... +1; 8 -12 ... -3 /
 *     -9 ... -2 / -5 ... 0 / +1 ... +3 / +3 ... +7; 10 -9 ... -2 / -7 ... -1 / -4 ... 0 / +1 ... +2 / +2 ... +6;
 *   - K 14336: rest 1 -20 ... -6 / ... / -12 ... -4; 10 -10 ... -2 / ... / -4 ... 0.
 * Beyond ten tiles (two parts each) 0 ... +10. Where only some of the tiles were shared the others were still the last to end: +2 ... +8.
 */
__host__ __device__ inline int shared_rows(int slabs, int rest) { return rest > 10 ? 0 : (slabs - 24) * (11 - rest) / 4; }

/*
 * Workgroups of a launch: every XCD gets one for each tile that it can have (a partial row tile per expert with rows at most),
 * and where tiles are shared one per CU for the parts. (Given to every launch, those for the parts doubled the grid of one token's first
 * GEMM: 256 workgroups more that look their tile up and leave, though no time could be measured for them, 70.0 us a layer.)
 */
template <int MODE, bool GMM1, int TM, int SPLIT>
inline int64_t stream_workgroups(const GemmParams &p, int n_tiles)
{
    const int64_t partial = p.max_rows < p.experts ? p.max_rows : p.experts;
    return 8 * ((p.max_rows / TM + partial) * ((n_tiles * SPLIT + 7) / 8) + (stream_shares_k<MODE, GMM1, SPLIT>() && p.part_sums ? p.part_cus : 0));
}

template <int MODE, bool GMM1, int OUT_DT, int TM, int SPLIT = 1, bool VALUES = false>
__global__ void __launch_bounds__(512 / SPLIT, 4)
grouped_gemm_stream_kernel(GemmParams p)
{
    static_assert(!VALUES || (!GMM1 && MODE != MODE_FP8 && StreamShape<MODE, TM, SPLIT>::PF == 4), "second GEMM of the int modes, lower tiles");
    static_assert(SPLIT == 1 || MODE != MODE_FP8 || !GMM1, "fp8's first GEMM requantises 128 columns, which are one workgroup's");
    using S = StreamShape<MODE, TM, SPLIT, VALUES>;
    constexpr int PF = S::PF, NT = S::NT, MTM = S::MTM, LOADS = S::LOADS, NW = S::NW, WRB = S::WRB;
    constexpr int MAX_PARTS = 4;
    constexpr bool SHARES_K = stream_shares_k<MODE, GMM1, SPLIT>();
    constexpr int W_BLOCK_BYTES = 128 * WRB;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    float *lds_sa = reinterpret_cast<float *>(smem + S::A_ALL);
    uint16_t *lds_gs = reinterpret_cast<uint16_t *>(lds_sa + 2 * S::SA_FLOATS);
    float *lds_es = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(lds_gs) + 2 * S::GS_BYTES);
    float *lds_rowmax = lds_es + S::ES_FLOATS;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_tiles = (GMM1 ? (p.N / 2) / 128 : p.N / BN) * SPLIT;
    const int K = p.K, KB = K / 128, I = p.N / 2, E = p.experts;

    /*
     * This workgroup's tile. A column is one expert with rows and 256 / SPLIT of its channels: the weights one row tile streams. The
     * columns are dealt to the XCDs in turn, so every XCD streams the same bytes whatever the routing (a contiguous run of
     * tiles each left the XCDs of the popular experts, whose row tiles share weights in the L2, idle early); the row tiles
     * of a column follow each other on its XCD. Every wave works the tile out for itself, without a barrier.
     */
    auto nth_expert = [&](int i) { return p.shared_index < 0 ? i : (i == 0 ? p.shared_index : i - 1); };      /* a shared expert has the most rows: first */
    auto rows_of = [&](int base, int &lo, int &hi) {
        lo = hi = 0;
        const int e = nth_expert(base + lane);
        if (base + lane < E) { lo = first_row_of<SHARED_IN_REGISTERS>(p, e); hi = p.row_off[e + 1]; }
    };
    int lo[2], hi[2];                                              /* the first 128 experts, one per lane each: one round trip for all of them */
    rows_of(0, lo[0], hi[0]);
    rows_of(64, lo[1], hi[1]);
    const int xcd = blockIdx.x & 7;
    const int slot = blockIdx.x >> 3;
    auto columns_before = [&](int y) { return (y - xcd + 7) >> 3; };      /* of this XCD, among columns 0 .. y - 1 */
    /* f for 64 experts at a time, one per lane: first of them, and the lane's first row, end row, row tiles, first column and tiles on this XCD; until it is true */
    auto walk = [&](auto f) __attribute__((always_inline)) {
        for (int base = 0, used = 0; base < E; base += 64) {
            int l = lo[0], h = hi[0];
            if (base == 64) { l = lo[1]; h = hi[1]; }
            else if (base > 64) rows_of(base, l, h);
            const int m = (h - l + TM - 1) / TM;
            const uint64_t busy = __ballot(m > 0);
            const int c0 = (used + __builtin_amdgcn_mbcnt_hi((uint32_t)(busy >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)busy, 0))) * n_tiles;
            if (f(base, l, h, m, c0, (columns_before(c0 + n_tiles) - columns_before(c0)) * m)) break;
            used += __popcll(busy);
        }
    };
    int expert = -1, n_tile = 0, m_tile = 0, mt_e = 1, first_row = 0, end_row = 0, tiles = 0;
    auto find_tile = [&](int wanted, bool count_all) __attribute__((always_inline)) {
        expert = -1;
        tiles = 0;
        walk([&](int base, int l, int h, int m, int c0, int mine) {
            const int incl = zb_wave_scan_dpp(mine);
            const uint64_t past = __ballot(tiles + incl > wanted);
            if (past && expert < 0) {
                const int src = __ffsll((long long)past) - 1;
                expert = nth_expert(base + src);
                mt_e = __builtin_amdgcn_readlane(m, src);
                first_row = __builtin_amdgcn_readlane(l, src);
                end_row = __builtin_amdgcn_readlane(h, src);
                const int at = wanted - tiles - __builtin_amdgcn_readlane(incl - mine, src), col = at / mt_e;
                m_tile = at - col * mt_e;
                const int first_col = __builtin_amdgcn_readlane(c0, src);
                n_tile = (columns_before(first_col) + col) * 8 + xcd - first_col;
                if (!count_all) return true;
            }
            tiles += __builtin_amdgcn_readlane(incl, 63);
            return false;
        });
    };
    const bool shares = SHARES_K && p.part_sums != nullptr;
    find_tile(slot, shares);
    /*
     * The memory gives every CU the same, so what is over when all CUs have the same number of tiles (`rest`, at the end) runs on
     * a few CUs, long after the others: 528 tiles of 7168 x 4096 on 256 CUs, 16 tiles alone for the last 30 of 168 us. W8A8: such
     * tiles are shared along K by three or four workgroups each, which leave their int32 sums in memory; the last of them to get there
     * adds the parts up and has the epilogue. Nobody waits for anybody. The words and sums go past the L2s, which are the
     * XCDs' own. Integers add up to the same bits in any parts. fp8's scaled sums do not, and which tiles are over depends on the
     * whole batch's routing: there a token's bits would depend on the tokens beside it (37 tokens 264 -> 247 us, taken back).
     */
    int part_k = 0, parts = 1, piece = 0;
    int64_t part_rows = 0;
    if constexpr (SHARES_K) {
        const int rest = shares ? tiles % p.part_cus : 0, whole = tiles - rest;
        if (rest > 0 && whole > 0 && slot >= whole) {
            int n = p.part_cus / rest, rows = 0;
            if (n > KB / PF) n = KB / PF;
            if (n > MAX_PARTS) n = MAX_PARTS;
            int before = 0;
            walk([&](int, int l, int h, int m, int, int mine) {
                const int incl = zb_wave_scan_dpp(mine), r = h - l;
                int height = r;
                if (m > 1) height = ((r + m - 1) / m + 15) & ~15;
                const int top = __builtin_amdgcn_readfirstlane((int)zb_wave_reduce_dpp<true>(mine > 0 && before + incl > whole ? (float)height : 0.0f));
                if (top > rows) rows = top;
                before += __builtin_amdgcn_readlane(incl, 63);
                return false;
            });
            part_rows = p.part_floats / (256 * rest * n);
            if (rows <= part_rows && rows <= shared_rows(KB, rest)) {
                parts = n;
                part_k = (slot - whole) / rest;
                if (part_k >= parts) return;
                piece = slot - whole - part_k * rest;
                if (part_k > 0) find_tile(whole + piece, false);
            }
        }
    }
    if (expert < 0) return;
    const int part = SPLIT == 1 ? 0 : n_tile % SPLIT, chan = part * NW + wave;      /* which 32 of the tile's 256 channels are this wave's */
    n_tile /= SPLIT;
    const int height = ((end_row - first_row + mt_e - 1) / mt_e + 15) & ~15;      /* even tiles, as in the other kernel */
    const int row_begin = first_row + m_tile * height;
    const int row_end = row_begin + height < end_row ? row_begin + height : end_row;
    const int last_rel = row_end - 1 - row_begin;
    /* slabs of this workgroup: whole chunks */
    const int kb_from = SHARES_K ? KB / PF * part_k / parts * PF : 0, kb_to = SHARES_K ? KB / PF * (part_k + 1) / parts * PF : KB;

    /* the wave's two 16-channel sub-tiles: block rows r0, r0 + 16 .. of one 128-channel block, or the same rows of a gate and an up block */
    const uint8_t *wb = weights_of<uint8_t, SHARED_IN_REGISTERS>(p, expert, (int64_t)(p.N / 128) * KB * W_BLOCK_BYTES);
    const int col0 = GMM1 ? n_tile : n_tile * 2, col1 = GMM1 ? I / 128 + n_tile : n_tile * 2 + 1;
    const uint8_t *w_src[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int r = GMM1 ? chan * 16 : (chan & 3) * 32 + nt * 16;
        const int col = GMM1 ? (nt == 0 ? col0 : col1) : (chan < 4 ? col0 : col1);
        w_src[nt] = uniform_ptr(wb + (int64_t)col * KB * W_BLOCK_BYTES + r * WRB);
    }
    const int frag_row = lane & 15;
    const int key = (lane & 7) ^ ((lane >> 3) & 1), g2 = (lane >> 4) * 2;
    const int off_lo = frag_row * BKB + ((g2 ^ key) * 16), off_hi = frag_row * BKB + (((g2 + 1) ^ key) * 16);
    /*
     * 8-bit weights: a load takes eight whole rows (1 KiB of consecutive bytes), lane (g, i) chunk 2g + i/8 of row i%8, and
     * half_rows() trades between the two loads of a sub-tile what the MFMA wants elsewhere. Half of each of 16 rows per
     * load, as the MFMA has them, asks for every line twice (W8A8, 32 experts of 7168 x 4096, one token: GMM1 80 -> 104 us).
     */
    const int w8_row = lane & 7, w8_chunk = g2 + ((lane >> 3) & 1);
    const int w8_off[2] = {w8_row * BKB + ((w8_chunk ^ w8_row) * 16), (8 + w8_row) * BKB + ((w8_chunk ^ w8_row ^ 1) * 16)};
    const int w4_off = frag_row * 64 + (((lane >> 4) ^ ((frag_row >> 2) & 3)) * 16);

    typedef u32x4 Slabs[PF][NT][LOADS];
    auto load_w = [&](auto stream_tag, Slabs &wr, int s, int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int h = 0; h < LOADS; ++h) {
                load16_sv<decltype(stream_tag)::value>(wr[s][nt][h], LOADS == 1 ? w4_off : w8_off[h], w_src[nt] + (int64_t)kb * W_BLOCK_BYTES);
            }
    };

    /*
     * The activations (and what scales them) of a chunk's PF slabs from kb0 on, to buffer b, in the same number of operations of
     * every wave: D in k_loop, whose waits count them. Rows past the tile's end repeat its last one.
     */
    const uint32_t lds_a0 = lds_addr(smem);
    auto issue_chunk = [&](auto mt_tag, int kb0, int b) __attribute__((always_inline)) {
        constexpr int MT = decltype(mt_tag)::value;
        int lane_x = lane;
        asm volatile("" : "+v"(lane_x));           /* the lane offsets are worked out afresh: there is no register to keep them in */
        const int r = lane_x >> 3;
#pragma unroll
        for (int j = 0; j < (VALUES ? 0 : MT * SPLIT / S::MT_STEP); ++j) {        /* slab s of row block rb */
            const int s = (wave + j * NW) & (PF - 1), rb = (wave + j * NW) / PF;
            int rel = rb * 8 + r;
            const uint32_t chunk16 = ((lane_x & 7) ^ (r ^ (rb & 1))) * 16;
            if (rel > last_rel) rel = last_rel;
            dma16_sv(p.a + (int64_t)row_begin * K + (int64_t)(kb0 + s) * BKB, (uint32_t)rel * (uint32_t)K + chunk16,
                     lds_a0 + b * S::A_BYTES + s * (TM * BKB) + rb * 1024);
        }
        if (MODE == MODE_FP8) {                                    /* 64 rows of slab s; several waves bring the same ones */
#pragma unroll
            for (int j = 0; j < S::SA_LOADS; ++j) {
                const int s = (wave + j * NW) & (PF - 1);
                const int row = (TM > 64 ? (wave / PF & 1) * 64 : 0) + lane_x, rel = row > last_rel ? last_rel : row;
                dma4_sv(p.a_scale + (int64_t)row_begin * KB + kb0 + s, (uint32_t)rel * (uint32_t)KB * 4u,
                        lds_addr(lds_sa) + (b * S::SA_FLOATS + s * S::SA_ROWS + (TM > 64 ? (wave / PF & 1) * 64 : 0)) * 4);
            }
        }
        if (MODE == MODE_W4A8) {
            const uint16_t *gs = scales_of<uint16_t, SHARED_IN_REGISTERS>(p, expert, (int64_t)KB * p.N);
#pragma unroll
            for (int j = 0; j < SPLIT; ++j) {                      /* 128 of the tile's 256 channels of slab sg */
                const int t = wave + j * NW, sg = (t >> 1) & (PF - 1);
                dma4_sv(reinterpret_cast<const float *>(gs + (int64_t)(kb0 + sg) * p.N + ((t & 1) ? col1 : col0) * 128), lane_x * 4u,
                        lds_addr(lds_gs) + b * S::GS_BYTES + sg * (BN * 2) + (t & 1) * 256);
            }
        }
    };

    /*
     * What the epilogue (int modes) or the K loop (fp8) needs of the tile's scales; older than everything else, so there first.
     * (W4A8's epilogue loaded its token scales itself, one round trip per row sub-tile: 4.3 us of a tile's 27 in the second GEMM.)
     */
    if constexpr (MODE != MODE_FP8) {
        const uint32_t dst0 = lds_addr(lds_es);
#pragma unroll
        for (int j = 0; j < SPLIT; ++j) {
            const int t = wave + j * NW;
            if (!VALUES && t < (TM + 63) / 64) {                   /* 64 token scales each */
                const int rel = t * 64 + lane > last_rel ? last_rel : t * 64 + lane;
                dma4_sv(p.a_scale + row_begin, (uint32_t)rel * 4u, dst0 + (MODE == MODE_W8A8 ? 1024 : 0) + t * 256);
            }
            if (MODE == MODE_W8A8 && t >= 4) {
                const int w4 = t - 4;
                if (GMM1 || !p.wscale_is_bf16) {
                    const float *wsb = scales_of<float, SHARED_IN_REGISTERS>(p, expert, p.N);
                    const float *src = !GMM1 ? wsb + n_tile * BN + w4 * 64 : (w4 < 2 ? wsb + n_tile * 128 + w4 * 64 : wsb + I + n_tile * 128 + (w4 - 2) * 64);
                    dma4_sv(src, lane * 4u, dst0 + w4 * 256);
                } else if (w4 < 2) {
                    const uint16_t *wsb = scales_of<uint16_t, SHARED_IN_REGISTERS>(p, expert, p.N);
                    dma4_sv(reinterpret_cast<const float *>(wsb + n_tile * BN + w4 * 128), lane * 4u, dst0 + w4 * 256);
                }
            }
        }
    } else if constexpr (MODE == MODE_FP8) {
        const int sw_stride = p.N / 128;
        const float *base = scales_of<float, SHARED_IN_REGISTERS>(p, expert, (int64_t)KB * sw_stride);
#pragma unroll
        for (int j = 0; j < SPLIT; ++j) {
            const int t = wave + j * NW;
            for (int b = (t & 3) * 64; b < KB; b += 256) {
                if (b + lane < KB)
                    dma4_sv(base + (t < 4 ? col0 : col1), (uint32_t)(b + lane) * (uint32_t)sw_stride * 4u,
                            lds_addr(lds_es) + ((t < 4 ? 0 : 256) + b) * 4);
            }
        }
    }

    f32x4 accf[MTM][NT];
    i32x4 acci[MTM][NT];
#pragma unroll
    for (int mt = 0; mt < MTM; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            accf[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            acci[mt][nt] = i32x4{0, 0, 0, 0};
        }

    i32x4 magic = {0x4b400000, 0x4b400000, 0x4b400000, 0x4b400000};      /* W4A8: see multiply() */
    if constexpr (MODE == MODE_W4A8) asm volatile("" : "+v"(magic));
    /* one slab over the first MT row sub-tiles: fragments of slot s, activations of slab s of buffer b */
    int values_from = 0;           /* VALUES: first slab of those in LDS */
    auto multiply = [&](auto mt_tag, const Slabs &wr, int s, int b, int kb) __attribute__((always_inline)) {
        constexpr int MT = decltype(mt_tag)::value;
        const uint8_t *ab = VALUES ? smem + (kb - values_from) * (MT * 2048) : smem + b * S::A_BYTES + s * (TM * BKB);
        auto load_a = [&](int mt) -> i32x8 {
            const u32x4 lo = *reinterpret_cast<const u32x4 *>(ab + mt * (16 * BKB) + off_lo);
            const u32x4 hi = *reinterpret_cast<const u32x4 *>(ab + mt * (16 * BKB) + off_hi);
            return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        };
        /* fragment of channel sub-tile nt: rows 0-7 of the first load beside rows 8-15 of the second, chunk 2g before chunk 2g + 1 */
        auto half_rows = [&](int nt) -> i32x8 {
            const u32x4 r0 = wr[s][nt][0], r8 = wr[s][nt][LOADS - 1];
            i32x8 w;
#pragma unroll
            for (int i = 0; i < 4; ++i) {      /* row_ror:8, into lanes 8-15 and 0-7 of each 16 */
                w[i] = __builtin_amdgcn_update_dpp((int)r0[i], (int)r8[i], 0x128, 0xf, 0xc, false);
                w[4 + i] = __builtin_amdgcn_update_dpp((int)r8[i], (int)r0[i], 0x128, 0xf, 0x3, false);
            }
            return w;
        };
        if constexpr (MODE == MODE_W8A8) {
            i32x8 w[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) w[nt] = half_rows(nt);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const i32x8 a = load_a(mt);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acci[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{w[nt][0], w[nt][1], w[nt][2], w[nt][3]},
                                                                         i32x4{a[0], a[1], a[2], a[3]}, acci[mt][nt], 0, 0, 0);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acci[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{w[nt][4], w[nt][5], w[nt][6], w[nt][7]},
                                                                         i32x4{a[4], a[5], a[6], a[7]}, acci[mt][nt], 0, 0, 0);
            }
        } else if constexpr (MODE == MODE_FP8) {
            const float sw0 = lds_es[kb], sw1 = lds_es[256 + kb];
            i32x8 w[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                w[nt] = half_rows(nt);
                asm volatile("" : "+v"(w[nt]));
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const i32x8 a = load_a(mt);
                const float sa = lds_sa[b * S::SA_FLOATS + s * S::SA_ROWS + mt * 16 + frag_row];
                /*
                 * As in the W4A8 loop below, the MFMAs first: 150 rows per expert, 32 of 7168 x 4096 / 2048 x 7168, 264 -> 260 / 133 ->
                 * 132 us; 400 rows, 64 of 2048 x 2048 / 1024 x 2048, 168 -> 166 / 88.6 -> 86.4. (W8A8, which has nothing to convert: 0 / +1 %.)
                 */
                f32x4 part[NT];
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) part[nt] = mfma_fp8_16x16x128(w[nt], a);
                __builtin_amdgcn_s_setprio(0);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float sc = sa * ((GMM1 ? nt == 1 : chan >= 4) ? sw1 : sw0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) accf[mt][nt][i] = __builtin_fmaf(part[nt][i], sc, accf[mt][nt][i]);
                }
                asm volatile("" ::: "memory");
            }
        } else {
            /* the arithmetic of the other kernel's W4A8 loop (see there): sums from the bits of 1.5 * 2^23, weights times 16 */
            constexpr float MAGIC = 12582912.0f;
            auto lo4 = [](uint32_t v) -> int { return (int)((v << 4) & 0xf0f0f0f0u); };
            auto hi4 = [](uint32_t v) -> int { return (int)(v & 0xf0f0f0f0u); };
            i32x4 w0[NT], w1[NT];
            float gs[NT][4];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const u32x4 pk = wr[s][nt][0];
                w0[nt] = i32x4{lo4(pk[0]), hi4(pk[0]), lo4(pk[1]), hi4(pk[1])};
                w1[nt] = i32x4{lo4(pk[2]), hi4(pk[2]), lo4(pk[3]), hi4(pk[3])};
                const int r = GMM1 ? nt * 128 + chan * 16 : chan * 32 + nt * 16;
                const u32x2 g = *reinterpret_cast<const u32x2 *>(lds_gs + (b * PF + s) * BN + (lane >> 4) * 8 + zb_block_row_channel(r));
                gs[nt][0] = zb_fp16_to_f32(g[0] & 0xffffu);
                gs[nt][1] = zb_fp16_to_f32(g[0] >> 16);
                gs[nt][2] = zb_fp16_to_f32(g[1] & 0xffffu);
                gs[nt][3] = zb_fp16_to_f32(g[1] >> 16);
#pragma unroll
                for (int i = 0; i < 4; ++i) asm("" : "+v"(gs[nt][i]));
            }
            auto promote = [&](int mt, const i32x4 (&part)[NT]) __attribute__((always_inline)) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) accf[mt][nt][i] = __builtin_fmaf(__int_as_float(part[nt][i]) - MAGIC, gs[nt][i], accf[mt][nt][i]);
            };
            /*
             * In the lower tile, where registers are left: the next sub-tile's activations are asked for ahead of this one's MFMAs, and
             * the sums of the one before are converted behind them. 128 experts of 4096 x 3072 / 1536 x 4096, 200 rows per expert
             * 505 -> 500 / 250 -> 242 us, 600 rows 1312 -> 1303 / 654 -> 635.
             */
            constexpr bool AHEAD = TM <= 64;
            i32x8 a = load_a(0);
            i32x4 before[NT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                i32x4 part[NT];
                i32x8 next = a;
                if (AHEAD && mt + 1 < MT) next = load_a(mt + 1);
                if (AHEAD) __builtin_amdgcn_sched_barrier(0);
                /*
                 * A wave with MFMAs to issue goes before those that convert, whose conversions then run beside them: 1024 rows per
                 * expert, 128 experts of 4096 x 3072 / 1536 x 4096, 2199 -> 2142 / 1060 -> 1037 us; 64 rows 223 -> 225 / 107 -> 105.
                 */
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    part[nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0[nt], i32x4{a[0], a[1], a[2], a[3]}, magic, 0, 0, 0);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    part[nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1[nt], i32x4{a[4], a[5], a[6], a[7]}, part[nt], 0, 0, 0);
                __builtin_amdgcn_s_setprio(0);
                if constexpr (AHEAD) {
                    if (mt > 0) promote(mt - 1, before);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) before[nt] = part[nt];
                    a = next;
                } else {
                    promote(mt, part);
                    if (mt + 1 < MT) a = load_a(mt + 1);
                }
            }
            if constexpr (AHEAD) promote(MT - 1, before);
        }
    };

    const int mt_act = (row_end - row_begin + 15) >> 4;
    auto k_loop = [&](auto mt_tag, auto stream_tag) __attribute__((always_inline)) {
        constexpr int MT = decltype(mt_tag)::value;
        constexpr int L = NT * LOADS;                                   /* loads per slab */
        constexpr int D = (VALUES ? 0 : MT * SPLIT / S::MT_STEP) + (MODE == MODE_W8A8 ? 0 : (MODE == MODE_FP8 ? S::SA_LOADS : SPLIT));      /* transfers per chunk */
        Slabs wr;
        /*
         * VALUES: the int modes' second GEMM with few rows makes the bytes of its rows itself, of the first GEMM's fp32 values and the
         * rows' maxima, instead of a launch between the two (4.7 us, in which nothing streams): a group of slabs at a time, as many as
         * there is room for, the first behind its own requests for weights. See zbalhip_gmm2_takes_values.
         */
        constexpr int GROUP = S::A_ALL / (MT * 2048) / PF * PF, BATCH = MODE == MODE_W8A8 ? 4 : 8;
        uint32_t row_max = 0;
        auto request_values = [&](u32x4 (&v)[BATCH], int first, int from, int pieces, int total) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                const int i = first + j * NW < total ? first + j * NW : total - 1, row = i / pieces;
                load16_sv<false>(v[j], lane * 16, uniform_ptr(p.a + ((int64_t)(row_begin + row) * K + from * 128 + (i - row * pieces) * 256) * 4));
            }
        };
        /* behind the wait, for the compiler */
        auto touch = [&](u32x4 (&v)[BATCH]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < BATCH; ++j) asm volatile("" : "+v"(v[j]));
        };
        auto store_values = [&](const u32x4 (&v)[BATCH], int first, int pieces, int total) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                const int i = first + j * NW;
                if (i >= total) break;
                const int row = i / pieces;
                const float mx = __uint_as_float(__builtin_amdgcn_readlane(row_max, row)), inv = mx == 0.0f ? 0.0f : 1.0f / mx;
                float q[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) q[u] = (__uint_as_float(v[j][u]) * 127.0f) * inv;
                const int slab = (i - row * pieces) * 2 + (lane >> 5), slot = ((lane & 31) >> 2) ^ (row & 7) ^ ((row >> 3) & 1);
                *reinterpret_cast<uint32_t *>(smem + slab * (MT * 2048) + row * BKB + slot * 16 + (lane & 3) * 4) = zb_pack4_i8(q[0], q[1], q[2], q[3]);
            }
        };
        auto bring_values = [&](int from, auto first_tag) __attribute__((always_inline)) {
            constexpr bool FIRST = decltype(first_tag)::value;
            const int slabs = from + GROUP < KB ? GROUP : KB - from, pieces = slabs / 2, total = (last_rel + 1) * pieces;
            values_from = from;
            u32x4 v[BATCH];
            if constexpr (FIRST) {
                const int row = lane <= last_rel ? lane : last_rel;
                asm volatile("s_nop 4\n\tglobal_load_dword %0, %1, %2" : "=v"(row_max) : "v"((uint32_t)row * 4u), "s"(uniform_ptr((const uint8_t *)(p.a_scale + row_begin))));
                request_values(v, wave, from, pieces, total);
#pragma unroll
                for (int s = 0; s < PF; ++s) load_w(stream_tag, wr, s, kb_from + s);
                /* everything but the fragments has landed */
                asm volatile("s_waitcnt vmcnt(%1)" : "+v"(row_max) : "n"(PF * L));
                touch(v);
                if (wave == 0 && lane < TM) lds_es[(MODE == MODE_W8A8 ? 256 : 0) + lane] = __uint_as_float(row_max) * (1.0f / 127.0f);
                store_values(v, wave, pieces, total);
            }
            for (int first = wave + (FIRST ? BATCH * NW : 0); first < total; first += BATCH * NW) {
                request_values(v, first, from, pieces, total);
                asm volatile("s_waitcnt vmcnt(0)");
                touch(v);
                store_values(v, first, pieces, total);
            }
        };
        issue_chunk(mt_tag, kb_from, 0);
        if constexpr (VALUES) {
            bring_values(0, std::true_type{});
        } else {
#pragma unroll
            for (int s = 0; s < PF; ++s) load_w(stream_tag, wr, s, kb_from + s);
        }
        auto next_values = [&](int kb0) __attribute__((always_inline)) {      /* before chunk kb0, behind its barrier */
            if constexpr (VALUES) {
                if (kb0 - values_from == GROUP) {
                    bring_values(kb0, std::false_type{});
                    lds_barrier();
                }
            }
        };
        /* issued since chunk c's transfers: the fragments of its slabs, L each; since slab s's fragments: three more slabs, and D */
        auto begin_chunk = [&]() __attribute__((always_inline)) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(PF * L) : "memory");
        };
        int b = 0, kb0 = kb_from;
        for (; kb0 + PF < kb_to; kb0 += PF) {
            begin_chunk();               /* chunk kb0's activations have landed for everybody, and nobody reads the other buffer any more */
            next_values(kb0);
            issue_chunk(mt_tag, kb0 + PF, b ^ 1);
#pragma unroll
            for (int s = 0; s < PF; ++s) {
                wait_w<(PF - 1) * L + D>(wr[s]);
                multiply(mt_tag, wr, s, b, kb0 + s);
                __builtin_amdgcn_sched_barrier(0);
                load_w(stream_tag, wr, s, kb0 + PF + s);
            }
            b ^= 1;
        }
        begin_chunk();
        next_values(kb0);
        if constexpr (PF == 4) {
            wait_w<3 * L>(wr[0]);
            multiply(mt_tag, wr, 0, b, kb0);
            wait_w<2 * L>(wr[1]);
            multiply(mt_tag, wr, 1, b, kb0 + 1);
        }
        wait_w<L>(wr[PF - 2]);
        multiply(mt_tag, wr, PF - 2, b, kb0 + PF - 2);
        wait_w<0>(wr[PF - 1]);
        multiply(mt_tag, wr, PF - 1, b, kb0 + PF - 1);
    };
    auto k_loop_mt = [&](auto stream_tag) __attribute__((always_inline)) {
        constexpr int ST = S::MT_STEP;
        if constexpr (MTM == 1) k_loop(std::integral_constant<int, 1>{}, stream_tag);
        else if (MTM >= 4 * ST && mt_act > 3 * ST) k_loop(std::integral_constant<int, MTM >= 4 * ST ? 4 * ST : MTM>{}, stream_tag);
        else if (MTM >= 3 * ST && mt_act > 2 * ST) k_loop(std::integral_constant<int, MTM >= 3 * ST ? 3 * ST : MTM>{}, stream_tag);
        else if (MTM >= 2 * ST && mt_act > ST) k_loop(std::integral_constant<int, MTM >= 2 * ST ? 2 * ST : MTM>{}, stream_tag);
        else k_loop(std::integral_constant<int, ST>{}, stream_tag);
    };
    /* weights that the other row tiles of the column want too stay in the L2 for them; the others leave no trace in it */
    if (MTM == 1 || mt_e == 1) k_loop_mt(std::true_type{});
    else k_loop_mt(std::false_type{});
    if constexpr (MODE == MODE_W4A8) {
#pragma unroll
        for (int mt = 0; mt < MTM; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) accf[mt][nt][i] *= 0.0625f;
    }
    if constexpr (SHARES_K) {
        if (parts > 1) {
            /* [row][256] sums of a part; a wave has 32 of the channels, its lane 4 of either 16 */
            int l = lane;
            asm volatile("" : "+v"(l));
            auto sums_at = [&](int part, int mt, int nt) {
                return reinterpret_cast<uint64_t *>(p.part_sums + xcd * p.part_floats + (piece * parts + part) * part_rows * 256 +
                                                    ((mt * 16 + (l & 15)) * 256 + wave * 32 + nt * 16 + (l >> 4) * 4));
            };
            auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
                for (int mt = 0; mt < MTM; ++mt)
                    if (mt * 16 + (l & 15) <= last_rel) {
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) f(mt, nt);
                    }
            };
            each([&](int mt, int nt) __attribute__((always_inline)) {
                const u32x4 v = __builtin_bit_cast(u32x4, acci[mt][nt]);
                uint64_t *at = sums_at(part_k, mt, nt);
                __hip_atomic_store(at, (uint64_t)v[1] << 32 | v[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(at + 1, (uint64_t)v[3] << 32 | v[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            });
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (threadIdx.x == 0)
                *reinterpret_cast<uint32_t *>(lds_rowmax) = __hip_atomic_fetch_add(p.part_done + xcd * p.part_cus + piece, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<uint32_t *>(lds_rowmax)) != (uint32_t)parts - 1) return;
            each([&](int mt, int nt) __attribute__((always_inline)) { acci[mt][nt] = i32x4{0, 0, 0, 0}; });
            for (int part = 0; part < parts; ++part) {
                each([&](int mt, int nt) __attribute__((always_inline)) {
                    uint64_t *at = sums_at(part, mt, nt);
                    const uint64_t v0 = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const uint64_t v1 = __hip_atomic_load(at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const u32x4 v = {(uint32_t)v0, (uint32_t)(v0 >> 32), (uint32_t)v1, (uint32_t)(v1 >> 32)};
                    acci[mt][nt] += __builtin_bit_cast(i32x4, v);
                });
            }
            __syncthreads();               /* lds_rowmax goes to the epilogue */
        }
    }
    TileCoord tc;
    tc.expert = expert;
    tc.m_tile = 0;
    tc.n_tile = n_tile;
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));               /* as in the other kernel: nothing of the epilogue's stays live across the K loop */
    epilogue<MODE, GMM1, OUT_DT, 1, MTM, NT, SHARED_IN_REGISTERS, false, MODE != MODE_FP8, NW>(p, tc, accf, acci, row_begin, row_end, 0, chan, lane_e, lds_rowmax, TM, lds_es);
}

} // namespace

#endif /* ZBAL_GEMM_STREAM_H_ */
