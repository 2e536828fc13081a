/*
 * Grouped (per-expert, ragged-M) quantised GEMM with fused epilogues for gfx950.
 *
 * Operands: activations A [rows, K] one byte per element (int8 or e4m3),
 * expert-major rows delimited by row_off[E+1]; weights W pre-packed
 * [E, N, K] with K contiguous (int4: [E, N, K/2]). Both operands are
 * K-contiguous, so either can feed either MFMA input; the kernel feeds the
 * WEIGHT fragment as the matrix-A input and the ACTIVATION fragment as the
 * matrix-B input, i.e. it computes C^T. With the 16x16 MFMA output layout
 * (lane l holds output column l%16, rows 4*(l/16)+i) every lane then owns ONE
 * token row and FOUR consecutive output channels per instruction, and with
 * the pre-pack's order of the weight rows EIGHT consecutive channels per pair
 * of instructions: per-token scales are one value per lane, per-channel
 * scales 16-byte vectors, gate/up pairs of the SwiGLU sit in the same lane,
 * and results leave as 8-element vectors.
 *
 * Workgroup tile: 64 to 256 token rows x 256 output channels x 128 K-bytes per
 * step, eight waves; in the 256-row shape each wave has 64 rows x 128 channels
 * = 4x8 MFMA tiles (128 accumulator registers). For GMM1 the 256 channels are 128 gate
 * columns j and the matching 128 up columns I+j, so the SwiGLU product and,
 * in the fp8 mode, the complete 1x128 requantisation happen in registers.
 * K slabs go from HBM to LDS by DMA, in a swizzled order that the weights are
 * pre-packed in, one persistent workgroup per CU; the details stand at the
 * kernel below.
 *
 * Tile schedule: workgroup ids are dealt round-robin to the 8 XCDs by the
 * hardware; XCD x takes a contiguous run of the logical tile order and its
 * workgroups take consecutive tiles of it. Logical tiles walk an expert in
 * groups of (all its row tiles) x (8 channel tiles), row tile fastest, so
 * the workgroups resident on an XCD share both their A and their W slabs in
 * that XCD's L2.
 */
#include <atomic>
#include <mutex>
#include <type_traits>

#include "zbal_device.h"
#include "zbal_gemm_stream.h"
#include "zbal_gemm_tall.h"
#include "zbal_gemm_tile.h"
#include "zbal_hip_kernels.h"

namespace {

/* ------------------------------------------------------------------------------------------------------
 * The grouped GEMM kernel (W8A8, fp8, W4A8): TM token rows x 256 channels x 128 K elements per workgroup,
 * eight waves (RG row groups x 8 / RG channel ranges; a wave's rows are the 16-row sub-tiles s with
 * s % RG = its row group), one workgroup per CU.
 *
 * K slabs go from HBM to LDS without passing through registers: every wave issues
 * global_load_lds_dwordx4, which deposits the 64 lanes' 16-byte chunks in 1 KiB of consecutive LDS
 * (lane l at +16*l). A block of 1 KiB holds 8 tile rows of 128 bytes; which global chunk a lane fetches is
 * free, so the chunk stored in slot s of row r is logical chunk s ^ f(r), f(r) = (r & 7) ^ ((r >> 3) & 1).
 * A fragment read touches 16 consecutive rows at the same logical chunk (128-byte pitch); with f every
 * aligned run of 8 rows lands in 8 distinct 16-byte slots and the 16 rows in 16 distinct (row parity, slot)
 * pairs, so the read is free of bank conflicts whether the LDS serves 8 or 16 lanes per pass; plain
 * row-major storage would put all 16 rows on the same slot.
 *
 * TM = 256 with two stages of 64 KiB (the slab for step k+1 is in flight while step k is multiplied) has the arithmetic
 * intensity that many-row experts need, for W4A8 and where the 8-bit modes cannot take the kernel of zbal_gemm_tall.h (a single
 * slab, more than 512 experts). TM = 128 and TM = 64 with three or four stages are for few-row experts, where the job is to stream every
 * weight byte once at HBM speed: two weight slabs or more stay in flight per CU, and the MFMAs of sub-tiles past the
 * expert's end are skipped; W4A8, bound by its vector instructions, also has a 192-row shape. The few-row shapes and
 * that one split a tile over one or two row groups of waves instead of four (FewRows, launch_w4a8).
 * Either way there is one barrier per step.
 *
 * W4A8: the weight slab stays packed in LDS (64 bytes per channel; block layout and nibble order as written by
 * the pre-pack) and is unpacked to int8 * 16 in registers, a shift and two masks per packed dword; the factor 16
 * is divided out of the accumulators, exactly, before the epilogue. Each 128-deep slab is one scale group:
 * its 256 fp16 group scales ride along by DMA and `acc = fma(float(partial), gs, acc)` promotes the int32 partial.
 * ------------------------------------------------------------------------------------------------------ */
constexpr int D_MAX_KB = 256;                 /* K up to 32768 */
constexpr int D_MAX_EXPERTS = 1024;

/* WRB = bytes of one weight row per slab: 128 (8-bit) or 64 (packed int4); RG = row groups of waves */
template <int TM, int NSTAGE, int WRB, int RG>
struct DmaShape {
    static constexpr int NW = 8;                           /* eight waves, two per SIMD */
    static constexpr int ROW_GROUPS = RG;
    static constexpr int COL_GROUPS = NW / RG;             /* the waves of a row group split the tile's 256 channels */
    static constexpr int NT = 16 / COL_GROUPS;             /* 16-channel sub-tiles per wave: 8 or 4 */
    static constexpr int MTM = (TM / 16 + ROW_GROUPS - 1) / ROW_GROUPS;   /* 16-row sub-tiles per wave, at most: 2, 4, 6 or 8 */
    static constexpr int THREADS = NW * 64;
    static constexpr int A_BYTES = TM * BKB;
    static constexpr int W_BYTES = BN * WRB;
    static constexpr int STAGE_BYTES = A_BYTES + W_BYTES;
    static constexpr int HALF_BLOCKS = 128 * WRB / 1024;   /* 1 KiB blocks per 128-channel half: 16 or 8 */
    static constexpr int MAX_EXPERTS = D_MAX_EXPERTS;       /* what the lookup tables hold */
    static constexpr int A_PARTS = (A_BYTES / 1024 + NW - 1) / NW;   /* 1 KiB blocks of the A tile per wave: 1 to 4 */
    static constexpr int W_PARTS = W_BYTES / 1024 / NW;    /* 1 KiB blocks of the W tile per wave (2, 4 or 8) */
    static constexpr int PARTS = W_PARTS > A_PARTS ? W_PARTS : A_PARTS;
    static constexpr bool TWO_PHASE = TM == 256;            /* the tiles of short experts run after all the others (see the kernel) */
    /* two buffers of per-tile scales, floats each: fp8 2 x D_MAX_KB weight block scales; W8A8 256 channel + TM token scales */
    static constexpr int SW_STRIDE = WRB == 64 ? 0 : 2 * D_MAX_KB;      /* W4A8 has its own (lds_gs) */
    static constexpr int SW_BYTES = 2 * SW_STRIDE * 4;
    static_assert(WRB == 64 || (SW_STRIDE >= 2 * D_MAX_KB && SW_STRIDE >= 256 + TM), "scale buffer too small");
    static constexpr int SA_FLOATS = WRB == 64 ? 0 : NSTAGE * TM;      /* the fp8 mode's activation block scales */
    static constexpr int LDS_BYTES = NSTAGE * STAGE_BYTES + SA_FLOATS * 4 + COL_GROUPS * TM * 4 + SW_BYTES +
                                     2 * (MAX_EXPERTS + 1) * 4 + (WRB == 64 ? NSTAGE * BN * 2 : 0) +
                                     (TWO_PHASE ? MAX_EXPERTS * 2 + (MAX_EXPERTS + 1) * 4 : 0);
    static_assert(PARTS >= 2 && (TM % (8 * NW) == 0 || NSTAGE == 2),
                  "the issue schedule hands out parts q * PARTS / 4 .. (q + 1) * PARTS / 4 - 1 of a slab with quarter q of a step");
    static_assert(NW <= HALF_BLOCKS && HALF_BLOCKS % NW == 0, "a wave's W blocks must not straddle a weight half");
    static_assert(LDS_BYTES <= 160 * 1024, "tile does not fit the LDS");
};

/*
 * Wait for the oldest slab in flight with `later` (MOST at most) younger slabs left alone; OPS operations per slab, one
 * more where `extra` (wave-uniform).
 */
template <int MOST, int OPS>
__device__ __forceinline__ void wait_slab(int later, bool extra)
{
    if constexpr (MOST > 0) {
        if (later >= MOST) {
            if (extra) wait_vmcnt<MOST * (OPS + 1)>();
            else wait_vmcnt<MOST * OPS>();
        } else {
            wait_slab<MOST - 1, OPS>(later, extra);
        }
    } else {
        wait_vmcnt<0>();
    }
}

/* what a workgroup needs to know about one tile; every member is wave-uniform and lives in scalar registers */
struct DmaTile {
    bool valid;
    int expert, n_tile, row_begin, row_end, last_rel;
    const uint8_t *a_base;            /* first K-byte of the tile's first activation row */
    const float *sa_base;             /* its fp8 block scales */
    const uint8_t *w_half[2];         /* K slab 0 of the tile's two 128-channel weight block rows */
    const uint16_t *gs_mine;          /* W4A8: fp16 group scales, slab 0, of the weight half this wave brings in (wave % 2) */
};

template <int MODE, bool GMM1, int OUT_DT, int TM, int NSTAGE, int RG, bool WSTREAM, Shared SH>
/*
 * Eight waves, two per SIMD (256 registers each), in every shape. The 128-row shape used to run four waves with the
 * wave tile of the 256-row shape (64 x 128), one per SIMD with nobody to cover its waits; as eight waves of 32 x 128
 * it is faster wherever it is used: decode layer (128 tokens, W8A8) 0.295 -> 0.288 ms, fp8 with 96 rows per expert
 * on 32 experts 0.404 -> 0.342 ms, W4A8 with 32-96 rows per expert first GEMM 9-12 % and second 7-8 % faster.
 */
__global__ void __launch_bounds__(512, 2)
grouped_gemm_dma_kernel(GemmParams p)
{
    static_assert(MODE == MODE_W8A8 || MODE == MODE_FP8 || MODE == MODE_W4A8, "unknown mode");
    constexpr int WRB = MODE == MODE_W4A8 ? 64 : 128;
    using S = DmaShape<TM, NSTAGE, WRB, RG>;
    constexpr int COL_GROUPS = S::COL_GROUPS, NT = S::NT;
    constexpr int NW = S::NW, STAGE_BYTES = S::STAGE_BYTES, A_BYTES = S::A_BYTES, W_PARTS = S::W_PARTS, PARTS = S::PARTS;
    constexpr int HALF_BLOCKS = S::HALF_BLOCKS, W_BLOCK_BYTES = 128 * WRB;     /* one 128-channel block of one slab */
    using Tile = DmaTile;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    float *lds_sa = reinterpret_cast<float *>(smem + NSTAGE * STAGE_BYTES);   /* [NSTAGE][TM] */
    float *lds_rowmax = lds_sa + S::SA_FLOATS;                                 /* [COL_GROUPS][TM] */
    constexpr int SW_STRIDE = S::SW_STRIDE;
    float *lds_sw = lds_rowmax + COL_GROUPS * TM;                                      /* [2 tiles][SW_STRIDE]: fp8 [2][D_MAX_KB] weight block scales */
    int *lds_mtp = reinterpret_cast<int *>(lds_sw + 2 * SW_STRIDE);            /* [experts + 1] tiles of TM rows before expert e */
    int *lds_roff = lds_mtp + (S::MAX_EXPERTS + 1);                            /* [experts + 1] copy of row_off */
    uint16_t *lds_gs = reinterpret_cast<uint16_t *>(lds_roff + (S::MAX_EXPERTS + 1));   /* [NSTAGE][BN] W4A8 group scales (fp16) */
    uint16_t *lds_short = lds_gs + (WRB == 64 ? NSTAGE * BN : 0);                       /* [experts] the short experts, second phase */
    int *lds_cost = reinterpret_cast<int *>(lds_short + S::MAX_EXPERTS);                 /* [experts + 1] 16-row sub-tiles of the main tiles before expert e */
    constexpr bool TWO_PHASE = S::TWO_PHASE;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    /* row group (16-row sub-tile s of a tile belongs to group s % RG) and channel range; wave-uniform, so everything derived from them lives in scalar registers */
    const int wm = wave_u / COL_GROUPS, wn = wave_u % COL_GROUPS;
    const int n_tiles = GMM1 ? (p.N / 2) / 128 : p.N / BN;
    const int K = p.K;
    const int KB = K / 128;
    const int I = p.N / 2;
    const int E = p.experts;

    /*
     * The workgroup is persistent: it walks a fixed sequence of tiles, and the DMA runs NSTAGE-1 slabs ahead of the
     * MFMAs across tile boundaries, so a tile's epilogue and the next tile's first loads overlap. The tile lookup
     * tables are built once, in LDS, so that finding the next tile costs no vector-memory traffic (whose waits would
     * also wait for the slabs in flight).
     */
    /*
     * Tile order. A tile with a few rows keeps most waves idle and runs at the pace of its own loads; in the middle
     * of the sequence it drifts away from the workgroups it shares slabs with, and the L2 stops serving them
     * together (measured on 4096 tokens over 32 experts with 42-row tail tiles in the sequence: 3.6 GB of HBM reads
     * per launch for 1.25 GB of operands, against 1.45 GB when every expert has exactly 1024 rows). Rows are
     * therefore cut into even tiles (fill_tile below), and the experts whose rows fill at most half a tile are kept
     * out of the main sequence and run after it, the longer class first: tiles that run side by side take about the
     * same time.
     */
    int n_short = 0;
    if (wave == 0) {
        int run = 0, run_c = 0;
        for (int base = 0; base < E; base += 64) {
            const int e = base + lane;
            int mt = 0, rows_e = 0;
            if (e < E) {
                const int lo = p.row_off[e];
                rows_e = p.row_off[e + 1] - first_row_of<SH>(p, e);
                mt = (rows_e + TM - 1) / TM;
                if (TWO_PHASE && rows_e <= TM / 2) mt = 0;      /* a short expert's only tile is not a main tile */
                lds_roff[e] = lo;
            }
            /* what the expert's main tiles cost: their number times their height in 16-row sub-tiles (fill_tile cuts them evenly) */
            const int cost = mt > 0 ? mt * ((((rows_e + mt - 1) / mt) + 15) >> 4) : 0;
            int incl = mt, incl_c = cost;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int o = __shfl_up(incl, off, 64), oc = __shfl_up(incl_c, off, 64);
                if (lane >= off) { incl += o; incl_c += oc; }
            }
            if (e < E) {
                lds_mtp[e] = run + incl - mt;
                if (TWO_PHASE) lds_cost[e] = run_c + incl_c - cost;
            }
            run += __shfl(incl, 63, 64);
            run_c += __shfl(incl_c, 63, 64);
        }
        if (lane == 0) {
            lds_mtp[E] = run;
            lds_roff[E] = p.row_off[E];
            if (TWO_PHASE) lds_cost[E] = run_c;
        }
        if (TWO_PHASE) {
            for (int cls = 2; cls >= 1; --cls) {          /* experts of TM/4+1 .. TM/2 rows, then those of 1 .. TM/4 */
                for (int base = 0; base < E; base += 64) {
                    const int e = base + lane;
                    bool mine = false;
                    if (e < E) {
                        const int rows = p.row_off[e + 1] - first_row_of<SH>(p, e);
                        mine = rows > 0 && rows <= TM / 2 && (rows > TM / 4) == (cls == 2);
                    }
                    const uint64_t bal = __ballot(mine);
                    if (mine) lds_short[n_short + __popcll(bal & ((1ull << lane) - 1))] = (uint16_t)e;
                    n_short += __popcll(bal);
                }
            }
            if (lane == 0) lds_rowmax[0] = __int_as_float(n_short);    /* for the other waves; the epilogues use this later */
        }
    }
    __syncthreads();
    if (TWO_PHASE) {
        n_short = __builtin_amdgcn_readfirstlane(__float_as_int(lds_rowmax[0]));
        __syncthreads();
    }
    /*
     * XCD x (workgroups x, x+8, ...) owns a contiguous range of the logical tile order. Where tiles differ in height
     * the ranges are cut at equal cost (16-row sub-tiles), not at equal tile counts: the kernel lasts as long as its
     * slowest XCD.
     */
    const int total = __builtin_amdgcn_readfirstlane(lds_mtp[E]) * n_tiles;
    const int chunk = (total + 7) / 8;
    const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
    auto first_id_of = [&](int x) __attribute__((always_inline)) -> int {
        if (!TWO_PHASE) return x * chunk < total ? x * chunk : total;
        if (x >= 8) return total;
        /* the tile at which the cost before it reaches x/8 of the whole: expert by search, tile within it by division */
        const int64_t target = (int64_t)lds_cost[E] * n_tiles * x / 8;
        int id = total;
        for (int base = 0; base < E; base += 64) {
            const int e = base + lane;
            int64_t lo = INT64_MAX, hi = INT64_MAX;
            if (e < E) { lo = (int64_t)lds_cost[e] * n_tiles; hi = (int64_t)lds_cost[e + 1] * n_tiles; }
            const uint64_t bal = __ballot(lo <= target && target < hi);
            if (bal) {
                const int src = __ffsll((long long)bal) - 1;
                const int ex = base + src;
                const int mt_e = lds_mtp[ex + 1] - lds_mtp[ex];
                const int height = (lds_cost[ex + 1] - lds_cost[ex]) / mt_e;      /* sub-tiles per tile of this expert */
                id = lds_mtp[ex] * n_tiles + (int)((target - (int64_t)lds_cost[ex] * n_tiles) / height);
                break;
            }
        }
        return __builtin_amdgcn_readfirstlane(id);
    };
    const int lid_begin = first_id_of(xcd);
    const int lid_end = first_id_of(xcd + 1);
    /* the short experts' tiles follow as ids total, total + 1, ...: n_short * n_tiles of them, split evenly over the XCDs */
    const int total_b = n_short * n_tiles;
    const int chunk_b = (total_b + 7) / 8;
    const int bid_begin = total + xcd * chunk_b + (blockIdx.x >> 3);
    const int bid_end = total + ((xcd + 1) * chunk_b < total_b ? (xcd + 1) * chunk_b : total_b);
    int lid = lid_begin + (blockIdx.x >> 3);
    if (lid >= lid_end) lid = bid_begin;
    /* the id after `id` in this workgroup's sequence */
    auto next_id = [&](int id) __attribute__((always_inline)) {
        const int n = id + slots;
        return (id < total && n >= lid_end) ? bid_begin : n;
    };

    auto fill_tile = [&](Tile &t, int expert, int n_tile, int m_tile) __attribute__((always_inline)) {
        t.expert = expert;
        t.n_tile = n_tile;
        /*
         * An expert's rows are cut into its ceil(rows / TM) tiles evenly, in multiples of 16: 1066 rows are five tiles
         * of 224, 224, 224, 224 and 170 rows rather than four of 256 and one of 42. The tiles cost what their 16-row
         * sub-tiles cost (the K loop leaves out the absent ones), so this is no more work, and no tile is so short
         * that it runs ahead of the tiles it shares slabs with.
         */
        const int first_row = is_shared<SH>(p, expert) ? launch_args()->shared_row : __builtin_amdgcn_readfirstlane(lds_roff[expert]);
        const int end_row = __builtin_amdgcn_readfirstlane(lds_roff[expert + 1]);
        const int n_row_tiles = (end_row - first_row + TM - 1) / TM;
        const int height = (((end_row - first_row + n_row_tiles - 1) / n_row_tiles) + 15) & ~15;
        t.row_begin = first_row + m_tile * height;
        t.row_end = t.row_begin + height < end_row ? t.row_begin + height : end_row;
        t.last_rel = t.row_end - 1 - t.row_begin;   /* rows past the tile's end re-read its last row: in bounds, and one line */
        t.a_base = p.a + (int64_t)t.row_begin * K;
        t.sa_base = p.a_scale + (int64_t)t.row_begin * KB;
        /* weights come pre-packed as 16 KiB blocks of 128 channels x 128 K-bytes in LDS order ([E][N/128][K/128]) */
        const int col0 = GMM1 ? t.n_tile : t.n_tile * 2, col1 = GMM1 ? I / 128 + t.n_tile : t.n_tile * 2 + 1;
        const uint8_t *wb = weights_of<uint8_t, SH>(p, expert, (int64_t)(p.N / 128) * KB * W_BLOCK_BYTES);
        t.w_half[0] = wb + ((int64_t)col0 * KB) * W_BLOCK_BYTES;
        t.w_half[1] = wb + ((int64_t)col1 * KB) * W_BLOCK_BYTES;
        if (MODE == MODE_W4A8) {      /* fp16 group scales [E][K/128][N]: the slab's 128 scales of each half are 256 bytes */
            const uint16_t *gs = scales_of<uint16_t, SH>(p, expert, (int64_t)KB * p.N);
            t.gs_mine = gs + ((wave_u & 1) ? col1 : col0) * 128;
        }
    };
    auto load_tile = [&](int id, Tile &t) __attribute__((always_inline)) {
        t.valid = id < total ? id < lid_end : id < bid_end;
        if (!t.valid) return;
        if (TWO_PHASE && id >= total) {              /* short expert number (id - total) / n_tiles, channel tile the remainder */
            const int j = (id - total) / n_tiles;
            const int expert = __builtin_amdgcn_readfirstlane((int)lds_short[j]);
            fill_tile(t, expert, id - total - j * n_tiles, 0);
            return;
        }
        const int q = id / n_tiles;                  /* index among all TM-row tiles: expert e has [mtp[e], mtp[e+1]) */
        int expert = 0, first = 0, next = 0;
        for (int base = 0; base < E; base += 64) {
            const int e = base + lane;
            int lo = 0x7fffffff, hi = 0x7fffffff;
            if (e < E) { lo = lds_mtp[e]; hi = lds_mtp[e + 1]; }
            const uint64_t bal = __ballot(lo <= q && q < hi);
            if (bal) {
                const int src = __ffsll((long long)bal) - 1;
                expert = base + src;
                first = __shfl(lo, src, 64);
                next = __shfl(hi, src, 64);
                break;
            }
        }
        expert = __builtin_amdgcn_readfirstlane(expert);
        first = __builtin_amdgcn_readfirstlane(first);
        const int mt_e = __builtin_amdgcn_readfirstlane(next) - first;
        /*
         * Within the expert: groups of (all its row tiles) x (a few channel tiles), row tile fastest, so that concurrent
         * tiles share slabs: as many channel tiles as make the group fit the workgroups of one XCD, GROUP_N at most.
         */
        const int l = id - first * n_tiles;
        int group_n = slots / mt_e;
        group_n = group_n < 1 ? 1 : (group_n > GROUP_N ? GROUP_N : group_n);
        const int per_group = mt_e * group_n;
        const int ng = l / per_group;
        const int r = l - ng * per_group;
        fill_tile(t, expert, ng * group_n + r / mt_e, r % mt_e);
    };

    /*
     * DMA: this wave fills 1 KiB blocks wave + NW*j of the A tile (j < A_PARTS) and of the W tile (j < W_PARTS). An A block is
     * tile rows 8*NW*j + r0 with r0 = 8*wave + lane/8, one swizzled 16-byte chunk per lane; rows past the expert's end
     * are clamped onto its last row. 1 KiB block number b = wave + NW*j of the W tile is block b % HALF_BLOCKS of
     * the weight half b / HALF_BLOCKS, a straight copy. Addresses are a wave-uniform base plus a 32-bit lane offset.
     */
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem) + wave * 1024);     /* this wave's block 0 of stage 0 */
    constexpr int SA_WAVES = (TM + 63) / 64;          /* waves that bring in 64 activation block scales each */
    const uint32_t lds_sa0 = __builtin_amdgcn_readfirstlane(lds_addr(lds_sa) + (wave % SA_WAVES) * 256);
    const bool sa_wave = MODE == MODE_FP8 && wave < SA_WAVES;
    const bool gs_wave = MODE == MODE_W4A8 && wave < 2;            /* wave h brings the group scales of weight half h */
    const uint32_t lds_gs0 = __builtin_amdgcn_readfirstlane(lds_addr(lds_gs) + (wave & 1) * 256);
    /*
     * The tallest shapes have no register to spare for the transfers' lane offsets across a K step: there they are worked
     * out afresh for every transfer from a copy of the lane number that the K loop makes opaque once per step (kept
     * across the loop they were spilled, and a reload waits for the slabs in flight).
     */
    constexpr bool FRESH_OFFSETS = MODE == MODE_W4A8 && TM >= 192;
    int lane_dma = lane;
    /* part j of a slab: the wave's j-th block of the W tile (j < W_PARTS), of the A tile (j < A_PARTS) and, with part 0, the scales */
    auto issue_part = [&](const Tile &t, int kb, int stage, int j) __attribute__((always_inline)) {
        const int lane_x = FRESH_OFFSETS ? lane_dma : lane;
        const int r0 = 8 * wave_u + (lane_x >> 3);
        const uint32_t a_chunk = ((lane_x & 7) ^ ((r0 & 7) ^ ((r0 >> 3) & 1))) * 16;
        const uint32_t w_off = wave_u * 1024 + lane_x * 16;
        const uint32_t dst = lds0 + stage * STAGE_BYTES + j * (NW * 1024);
        if (j < W_PARTS) {
            const uint8_t *wsrc = t.w_half[(NW * j) / HALF_BLOCKS] + ((int64_t)kb * W_BLOCK_BYTES + ((NW * j) % HALF_BLOCKS) * 1024);
            if (WSTREAM) dma16_sv_nt(wsrc, w_off, dst + A_BYTES);
            else dma16_sv(wsrc, w_off, dst + A_BYTES);
        }
        if (j < S::A_PARTS && (TM % (8 * NW) == 0 || 8 * NW * j + 8 * wave_u < TM)) {
            /*
             * An 8-row block past the expert's end moves 16 bytes instead of 1 KiB (one lane): the transfer still
             * counts as one operation of this wave, which keeps the outstanding-operation arithmetic the same for
             * every wave and tile. (The two-stage shapes wait for all of their transfers every step, so there a block
             * past the tile's end is simply not issued.)
             */
            const bool present = 8 * NW * j + 8 * wave_u <= t.last_rel;
            int rel = 8 * NW * j + r0;
            if (rel > t.last_rel) rel = t.last_rel;
            if ((present || lane == 0) && (present || NSTAGE != 2)) dma16_sv(t.a_base + (int64_t)kb * BKB, (uint32_t)rel * (uint32_t)K + a_chunk, dst);
        }
        if (j == 0 && sa_wave) {
            int rel = wave_u * 64 + lane_x;
            const bool in_tile = TM % 64 == 0 || rel < TM;          /* the ring holds TM scales per stage: lanes past that stay out */
            if (rel > t.last_rel) rel = t.last_rel;
            if (in_tile) dma4_sv(t.sa_base + kb, (uint32_t)rel * (uint32_t)KB * 4u, lds_sa0 + stage * TM * 4);
        }
        if (j == 0 && gs_wave)      /* 128 fp16 scales = 64 dwords, one per lane */
            dma4_sv((const float *)(t.gs_mine + (int64_t)kb * p.N), lane_x * 4u, lds_gs0 + stage * (BN * 2));
    };
    auto issue = [&](const Tile &t, int kb, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PARTS; ++j) issue_part(t, kb, stage, j);
    };
    /* the two weight block scales of every K slab of a tile go to LDS by DMA as well: lane = K slab */
    auto issue_sw = [&](const Tile &t, int buf) __attribute__((always_inline)) {
        if (MODE != MODE_FP8) return;
        const int sw_stride = p.N / 128;
        const float *base = scales_of<float, SH>(p, t.expert, (int64_t)KB * sw_stride);
        const int c0 = GMM1 ? t.n_tile : t.n_tile * 2, c1 = GMM1 ? I / 128 + t.n_tile : t.n_tile * 2 + 1;
        for (int b = wave_u * 64; b < KB; b += NW * 64) {
            if (b + lane < KB) {
                const uint32_t off = (uint32_t)(b + lane) * (uint32_t)sw_stride * 4u;
                const uint32_t dst = lds_addr(lds_sw) + (buf * SW_STRIDE + b) * 4;
                dma4_sv(base + c0, off, __builtin_amdgcn_readfirstlane(dst));
                dma4_sv(base + c1, off, __builtin_amdgcn_readfirstlane(dst) + D_MAX_KB * 4);
            }
        }
    };
    /*
     * W8A8: the scales a tile's epilogue needs go to LDS by DMA as well (layout: see the epilogue), into the
     * buffer of the tile's parity, which the fp8 mode uses for its weight block scales. Rows past the tile's end
     * repeat its last row. Issued where the block scales are: older than every slab that follows.
     */
    auto issue_es = [&](const Tile &t, int buf) __attribute__((always_inline)) {
        if (MODE != MODE_W8A8) return;
        const uint32_t dst0 = lds_addr(lds_sw) + buf * SW_STRIDE * 4;
        if (wave_u < (TM + 63) / 64) {
            int rel = wave_u * 64 + lane;
            if (rel > t.last_rel) rel = t.last_rel;
            dma4_sv(p.a_scale + t.row_begin, (uint32_t)rel * 4u, __builtin_amdgcn_readfirstlane(dst0 + 1024 + wave_u * 256));
        }
        if (wave_u < 4) {
            if (GMM1) {
                const float *wsb = scales_of<float, SH>(p, t.expert, p.N);
                const float *src = wave_u < 2 ? wsb + t.n_tile * 128 + wave_u * 64 : wsb + I + t.n_tile * 128 + (wave_u - 2) * 64;
                dma4_sv(src, lane * 4u, __builtin_amdgcn_readfirstlane(dst0 + wave_u * 256));
            } else if (!p.wscale_is_bf16) {
                const float *wsb = scales_of<float, SH>(p, t.expert, p.N);
                dma4_sv(wsb + t.n_tile * BN + wave_u * 64, lane * 4u, __builtin_amdgcn_readfirstlane(dst0 + wave_u * 256));
            } else if (wave_u < 2) {
                const uint16_t *wsb = scales_of<uint16_t, SH>(p, t.expert, p.N);
                dma4_sv(reinterpret_cast<const float *>(wsb + t.n_tile * BN + wave_u * 128), lane * 4u,
                        __builtin_amdgcn_readfirstlane(dst0 + wave_u * 256));
            }
        }
    };
    /* this wave's vector-memory operations per slab: what may stay outstanding while an older slab is awaited */
    constexpr int OPS = W_PARTS + S::A_PARTS;
    const bool extra_op_wave = sa_wave || gs_wave;                  /* one more operation per slab: the scales */

    /* fragment reads: row lane%16 of a 16-row sub-tile, logical chunks 2*(lane/16) and 2*(lane/16)+1 */
    const int frag_row = lane & 15;
    const int key = (lane & 7) ^ ((lane >> 3) & 1), g2 = (lane >> 4) * 2;
    const int off_lo = frag_row * BKB + ((g2 ^ key) * 16), off_hi = frag_row * BKB + (((g2 + 1) ^ key) * 16);
    /* int4: one 16-byte chunk per lane, chunk lane/16 of channel lane%16 of the 16-channel block, at its swizzled slot */
    const int w4_off = frag_row * 64 + (((lane >> 4) ^ ((frag_row >> 2) & 3)) * 16);
    int w_sub[NT], w_ch[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        int r;
        if (GMM1) r = (nt < NT / 2) ? wn * (8 * NT) + nt * 16 : 128 + wn * (8 * NT) + (nt - NT / 2) * 16;
        else r = wn * (16 * NT) + nt * 16;
        w_sub[nt] = A_BYTES + r * WRB;
        w_ch[nt] = zb_block_row_channel(r);       /* tile-local channel held by the sub-tile's first block row */
    }
    const int lane_ch = (lane >> 4) * 8;          /* block rows 4q .. 4q+3 of a sub-tile hold channels 8q .. 8q+3 past that */

    Tile cur, nxt;
    load_tile(lid, cur);
    if (!cur.valid) return;
    int sw_buf = 0;
    issue_sw(cur, sw_buf);
    issue_es(cur, sw_buf);
#pragma unroll
    for (int s = 0; s < NSTAGE - 1; ++s) issue(cur, s, s);        /* the host guarantees KB >= NSTAGE - 1 */
    int stage = 0;
    while (true) {
        lid = next_id(lid);
        load_tile(lid, nxt);

        constexpr int MTM = S::MTM;
        f32x4 accf[MTM][NT];
        i32x4 acci[MTM][NT];
#pragma unroll
        for (int mt = 0; mt < MTM; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                accf[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                acci[mt][nt] = i32x4{0, 0, 0, 0};
            }
        /*
         * The wave's 16-row sub-tiles are rows (RG*mt + wm)*16 .. +15 of the tile, mt = 0 .. MTM-1. Only the first `mt_act` of
         * them hold rows of this tile; a wave with none still moves data and meets the barriers, but skips the math.
         */
        const int tile_subs = (cur.row_end - cur.row_begin + 15) >> 4;
        int mt_act = (tile_subs - wm + RG - 1) / RG;
        mt_act = mt_act < 0 ? 0 : (mt_act > MTM ? MTM : mt_act);
        const float *sw_cur = lds_sw + sw_buf * SW_STRIDE;

        /* the K loop over the wave's first MT row sub-tiles; MT is a compile-time constant so that the loops unroll */
        auto k_loop = [&](auto mt_tag) __attribute__((always_inline)) {
        constexpr int MT = decltype(mt_tag)::value;
        for (int kb = 0; kb < KB; ++kb) {
            /*
             * The slabs after this one that have been asked for, NSTAGE - 2 at most, may stay in flight: there are that
             * many while the sequence goes on (the host guarantees KB >= NSTAGE - 1), fewer at its very end.
             */
            const int later = nxt.valid ? NSTAGE - 2 : KB - 1 - kb;
            wait_slab<NSTAGE - 2, OPS>(later, extra_op_wave);
            __syncthreads();                /* slab kb has landed for everybody; the stage read in the step before is free */
            if constexpr (FRESH_OFFSETS) asm volatile("" : "+v"(lane_dma));
            /*
             * The next tile's weight block scales go into the buffer the tile before this one used. Every wave is
             * past this tile's first barrier now, so none of them still reads that buffer; the transfers are older
             * than every slab issued from here on, so the slab waits cover them.
             */
            if (kb == 0 && nxt.valid) {
                issue_sw(nxt, sw_buf ^ 1);
                issue_es(nxt, sw_buf ^ 1);
            }
            /*
             * That stage takes the slab NSTAGE-1 steps ahead, which may belong to the next tile. It is issued in parts,
             * spread over the first half of this step's MFMAs: a wave that pushes all of its loads at once sits in the
             * memory pipeline's queue while the matrix unit idles.
             */
            const bool ahead_in_tile = kb + NSTAGE - 1 < KB;
            const Tile &ft = ahead_in_tile ? cur : nxt;
            const int fill_kb = ahead_in_tile ? kb + NSTAGE - 1 : kb + NSTAGE - 1 - KB;
            const bool more = ahead_in_tile || nxt.valid;
            const int fill_stage = stage == 0 ? NSTAGE - 1 : stage - 1;
            const uint8_t *sb = smem + stage * STAGE_BYTES;
            const int cur_stage = stage;
            stage = stage + 1 == NSTAGE ? 0 : stage + 1;
            if constexpr (MT == 0) {
                if (more) issue(ft, fill_kb, fill_stage);
                continue;
            }
            auto issue_quarter = [&](int q) __attribute__((always_inline)) {
#pragma unroll
                for (int j = q * PARTS / 4; j < (q + 1) * PARTS / 4; ++j) issue_part(ft, fill_kb, fill_stage, j);
            };
            /* the quarters that go out with channel sub-tile nt: one each with the first four, two each where a wave has only two */
            auto issue_at = [&](int nt) __attribute__((always_inline)) {
                constexpr int EACH = NT < 4 ? 4 / NT : 1;
#pragma unroll
                for (int q = nt * EACH; q < nt * EACH + EACH && q < 4; ++q) issue_quarter(q);
            };
            auto load_w = [&](int nt) -> i32x8 {
                const u32x4 lo = *reinterpret_cast<const u32x4 *>(sb + w_sub[nt] + off_lo);
                const u32x4 hi = *reinterpret_cast<const u32x4 *>(sb + w_sub[nt] + off_hi);
                return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
            };

            if constexpr (MT > 0) {
                i32x8 af[MT];
                i32x8 wf_first = {};
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const uint8_t *ab = sb + ((RG * mt + wm) * 16) * BKB;
                    const u32x4 lo = *reinterpret_cast<const u32x4 *>(ab + off_lo);
                    const u32x4 hi = *reinterpret_cast<const u32x4 *>(ab + off_hi);
                    af[mt] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
                    if (mt == 0 && MODE != MODE_W4A8) {
                        /*
                         * All waves start their fragment reads together after the barrier and the LDS serves them in the
                         * order asked, so the two fragments of the first MFMA are asked for before the rest (measured,
                         * alternating with the unordered build on one GPU: 1 % of the kernel; forcing the order of all of
                         * them is slower).
                         */
                        wf_first = load_w(0);
                        asm volatile("" ::: "memory");
                    }
                }

                if constexpr (MODE == MODE_FP8) {
                    /*
                     * Software pipeline over the 8 x MT (channel sub-tile, row sub-tile) pairs: the MFMA of pair p+1 is
                     * issued before the four scale-and-accumulate FMAs of pair p, so the vector ALU works under the
                     * matrix unit.
                     */
                    const float sw0 = sw_cur[kb], sw1 = sw_cur[D_MAX_KB + kb];
                    float s0[MT], s1[MT];
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        const float sa = lds_sa[cur_stage * TM + (RG * mt + wm) * 16 + frag_row];
                        s0[mt] = sa * sw0;
                        s1[mt] = sa * sw1;
                    }
                    i32x8 wf = wf_first;
                    f32x4 part = mfma_fp8_16x16x128(wf, af[0]);
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        i32x8 wf_n = wf;
                        if (nt + 1 < NT) wf_n = load_w(nt + 1);
                        /* the 256-row fp8 loop hands the slab out in two halves (0.6 % faster, measured against quarters on one GPU; the other loops are slower that way) */
                        if (TM == 256) {
                            if (more && (nt == 0 || nt == 2)) { issue_quarter(nt); issue_quarter(nt + 1); }
                        } else if (more) {
                            issue_at(nt);
                        }
                        const bool second = GMM1 ? (nt >= NT / 2) : (wn >= COL_GROUPS / 2);
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            f32x4 nxt_part = part;
                            if (mt + 1 < MT) nxt_part = mfma_fp8_16x16x128(wf, af[mt + 1]);
                            else if (nt + 1 < NT) nxt_part = mfma_fp8_16x16x128(wf_n, af[0]);
                            const float sc = second ? s1[mt] : s0[mt];
#pragma unroll
                            for (int i = 0; i < 4; ++i) accf[mt][nt][i] = __builtin_fmaf(part[i], sc, accf[mt][nt][i]);
                            part = nxt_part;
                        }
                        wf = wf_n;
                    }
                } else if constexpr (MODE == MODE_W4A8) {
                    /*
                     * The lane's 16 packed bytes are its 32 K values of this slab: dwords 0-1 unpack into the operand of
                     * the first 64-deep MFMA, dwords 2-3 into the second (times 16: the nibble moves to the top of its
                     * byte, which keeps the sign). The pair's int32 sum is promoted with the slab's group scales, and as
                     * in the fp8 mode the MFMAs of pair p+1 are issued before the conversions and FMAs of pair p.
                     */
                    const uint16_t *gsb = lds_gs + cur_stage * BN;
                    auto load_pk = [&](int nt) -> u32x4 { return *reinterpret_cast<const u32x4 *>(sb + w_sub[nt] + w4_off); };
                    auto load_gs = [&](int nt) -> u32x2 { return *reinterpret_cast<const u32x2 *>(gsb + lane_ch + w_ch[nt]); };
                    /*
                     * The sums start at the bits of 1.5 * 2^23: |pair sum| <= 128 * 128 * 128 = 2^21, so the result read as a
                     * float is 1.5 * 2^23 + sum, exactly, and one subtraction makes it the float a conversion would. On
                     * this GPU v_cvt_f32_i32 and v_fma_mix_f32 issue at half the rate of v_sub_f32 and v_fma_f32 (2.1
                     * and 2.0 ns against 1.2 and 1.3 per instruction and SIMD, two waves), and next to nothing of
                     * either hides under an MFMA, so the scales are also widened once per channel sub-tile.
                     */
                    constexpr float MAGIC = 12582912.0f;
                    i32x4 magic = {0x4b400000, 0x4b400000, 0x4b400000, 0x4b400000};
                    asm volatile("" : "+v"(magic));
                    auto lo4 = [](uint32_t v) -> int { return (int)((v << 4) & 0xf0f0f0f0u); };
                    auto hi4 = [](uint32_t v) -> int { return (int)(v & 0xf0f0f0f0u); };
                    auto mfma_pair = [&](const u32x4 &pk, const i32x8 &a) -> i32x4 {
                        const i32x4 w0 = i32x4{lo4(pk[0]), hi4(pk[0]), lo4(pk[1]), hi4(pk[1])};
                        const i32x4 w1 = i32x4{lo4(pk[2]), hi4(pk[2]), lo4(pk[3]), hi4(pk[3])};
                        i32x4 part = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, i32x4{a[0], a[1], a[2], a[3]}, magic, 0, 0, 0);
                        return __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, i32x4{a[4], a[5], a[6], a[7]}, part, 0, 0, 0);
                    };
                    constexpr bool LATE_SCALES = TM == 192;      /* no two registers to spare for fetching the scales ahead */
                    /* the packed chunk and the raw fp16 scales of the next channel sub-tile are fetched one sub-tile ahead */
                    u32x4 pk = load_pk(0);
                    u32x2 gsr = load_gs(0);
                    i32x4 part = mfma_pair(pk, af[0]);
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        u32x4 pkn = pk;
                        u32x2 gsn = gsr;
                        if (nt + 1 < NT) {
                            pkn = load_pk(nt + 1);
                            if (!LATE_SCALES) gsn = load_gs(nt + 1);
                        }
                        if (more) issue_at(nt);
                        float gs[4] = {zb_fp16_to_f32(gsr[0] & 0xffffu), zb_fp16_to_f32(gsr[0] >> 16),
                                       zb_fp16_to_f32(gsr[1] & 0xffffu), zb_fp16_to_f32(gsr[1] >> 16)};
#pragma unroll
                        for (int i = 0; i < 4; ++i) if (TM <= 128) asm("" : "+v"(gs[i]));      /* or the compiler folds the widening into v_fma_mix_f32 */
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            i32x4 nxt_part = part;
                            if (mt + 1 < MT) nxt_part = mfma_pair(pk, af[mt + 1]);
                            else if (nt + 1 < NT) nxt_part = mfma_pair(pkn, af[0]);
#pragma unroll
                            for (int i = 0; i < 4; ++i) accf[mt][nt][i] = __builtin_fmaf(__int_as_float(part[i]) - MAGIC, gs[i], accf[mt][nt][i]);
                            part = nxt_part;
                        }
                        pk = pkn;
                        gsr = LATE_SCALES && nt + 1 < NT ? load_gs(nt + 1) : gsn;
                    }
                } else {
                    /*
                     * int8: lane's 32 K bytes feed two 64-deep MFMAs; the two updates of one accumulator are kept apart.
                     * (Asking for the next weight fragment before the MFMAs of this one was 0.5 % slower here: the
                     * SIMD's other wave covers the read.)
                     */
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const i32x8 wf = nt == 0 ? wf_first : load_w(nt);
                        if (more) issue_at(nt);
                        const i32x4 wf0 = i32x4{wf[0], wf[1], wf[2], wf[3]}, wf1 = i32x4{wf[4], wf[5], wf[6], wf[7]};
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt)
                            acci[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                wf0, i32x4{af[mt][0], af[mt][1], af[mt][2], af[mt][3]}, acci[mt][nt], 0, 0, 0);
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt)
                            acci[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                wf1, i32x4{af[mt][4], af[mt][5], af[mt][6], af[mt][7]}, acci[mt][nt], 0, 0, 0);
                    }
                }
            }
        }
        };
        static_assert(MTM <= 8, "sub-tiles per wave");
        if (MTM >= 8 && mt_act == 8) k_loop(std::integral_constant<int, MTM >= 8 ? 8 : MTM>{});
        else if (MTM >= 7 && mt_act == 7) k_loop(std::integral_constant<int, MTM >= 7 ? 7 : MTM>{});
        else if (MTM >= 6 && mt_act == 6) k_loop(std::integral_constant<int, MTM >= 6 ? 6 : MTM>{});
        else if (MTM >= 5 && mt_act == 5) k_loop(std::integral_constant<int, MTM >= 5 ? 5 : MTM>{});
        else if (MTM >= 4 && mt_act == 4) k_loop(std::integral_constant<int, MTM >= 4 ? 4 : MTM>{});
        else if (MTM >= 3 && mt_act == 3) k_loop(std::integral_constant<int, MTM >= 3 ? 3 : MTM>{});
        else if (MTM >= 2 && mt_act == 2) k_loop(std::integral_constant<int, MTM >= 2 ? 2 : MTM>{});
        else if (mt_act == 1) k_loop(std::integral_constant<int, 1>{});
        else k_loop(std::integral_constant<int, 0>{});
        if constexpr (MODE == MODE_W4A8) {      /* the unpacked weights were 16 x their value; a power of two divides out exactly */
#pragma unroll
            for (int mt = 0; mt < MTM; ++mt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) accf[mt][nt][i] *= 0.0625f;
        }
        TileCoord tc;
        tc.expert = cur.expert;
        tc.m_tile = 0;
        tc.n_tile = cur.n_tile;
        /*
         * The epilogue's lane-derived offsets are worked out afresh per tile from an opaque copy of the lane number:
         * hoisted out of the tile loop they stay live across the K loop, spill, and every reload of a spilled
         * register is a vector-memory operation whose wait also waits for the next tile's slab in flight.
         */
        int lane_e = lane;
        asm volatile("" : "+v"(lane_e));
        epilogue<MODE, GMM1, OUT_DT, RG, S::MTM, NT, SH>(p, tc, accf, acci, cur.row_begin, cur.row_end, wm, wn, lane_e, lds_rowmax, TM,
                                         lds_sw + sw_buf * SW_STRIDE);
        if (!nxt.valid) break;
        cur = nxt;
        sw_buf ^= 1;
    }
}

/*
 * Second pass of the int8 GMM1 epilogue: whole-row requantisation from the fp32 SwiGLU values. A row is a few KiB, so
 * one wave takes one row at a time and every lane asks for its (up to eight) 16-byte pieces of the row before it
 * converts the first. Measured on 131 072 rows of 1536 values (read 805 MB, write 201 MB): 256 threads with one piece
 * in flight per lane 200 us (5.0 TB/s), two waves with four pieces 182 us, one wave with eight 166 us (6.1 TB/s).
 * A small batch waits for round trips: the row and its maximum are asked for together with the number of rows that
 * there are (rows past it hold nothing of use, but are inside the scratch, which has max_rows).
 */
constexpr int kRequantThreads = 64, kRequantPieces = 8;

__global__ void __launch_bounds__(kRequantThreads)
requant_rows_kernel(const float *__restrict__ sgl, const uint32_t *__restrict__ rowmax, const int32_t *__restrict__ row_off,
                    int experts, int shared_row, int max_rows, int I, int8_t *__restrict__ q2, float *__restrict__ scale2)
{
    /* rows [0, total) and, of a shared expert (the last of `experts`), [shared_row, end); shared_row = max_rows without one */
    const int total = row_off[shared_row < max_rows ? experts - 1 : experts], end = row_off[experts];
    const int vecs = I / 4;
    for (int row = blockIdx.x; row < max_rows; row += gridDim.x) {
        const uint32_t mx_bits = rowmax[row];
        const f32x4 *src = reinterpret_cast<const f32x4 *>(sgl + (int64_t)row * I);
        uint32_t *dst = reinterpret_cast<uint32_t *>(q2 + (int64_t)row * I);
        for (int c0 = 0; c0 < vecs; c0 += kRequantThreads * kRequantPieces) {
            f32x4 v[kRequantPieces];
#pragma unroll
            for (int u = 0; u < kRequantPieces; ++u) {
                const int c = c0 + u * kRequantThreads + (int)threadIdx.x;
                v[u] = c < vecs ? __builtin_nontemporal_load(src + c) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            if (row >= total && (row < shared_row || row >= end)) break;
            const float mx = __uint_as_float(mx_bits), inv = mx == 0.0f ? 0.0f : 1.0f / mx;
            if (c0 == 0 && threadIdx.x == 0) scale2[row] = mx * (1.0f / 127.0f);
#pragma unroll
            for (int u = 0; u < kRequantPieces; ++u) {
                const int c = c0 + u * kRequantThreads + (int)threadIdx.x;
                float q[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) q[i] = (v[u][i] * 127.0f) * inv;
                if (c < vecs) dst[c] = zb_pack4_i8(q[0], q[1], q[2], q[3]);
            }
        }
    }
}

__global__ void fill_u32_kernel(uint32_t *p, int64_t n, uint32_t v)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

/* rows, weight blocks and channel scales move as 16-byte vectors (with tensor lists: the tables; their entries are the caller's) */
inline bool misaligned16(const void *p) { return ((uintptr_t)p & 15) != 0; }

inline unsigned grid_for(int64_t max_rows, int64_t experts, int n_tiles, int tile_m)
{
    int64_t m_tiles = (max_rows + tile_m - 1) / tile_m + experts;   /* each expert adds at most one partial tile */
    int64_t g = m_tiles * n_tiles;
    return (unsigned)((g + 7) / 8 * 8);
}

/* CUs of the current device (a partition of the GPU has fewer than 256); 0 if it cannot be asked */
inline int cu_count()
{
    static std::atomic<int> cus[64];
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0 && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
        cus[dev].store(n, std::memory_order_relaxed);
    return n;
}

/*
 * The kernels need more dynamic LDS than the default limit: raised once per kernel instantiation and device, which
 * cannot be recorded into a graph. zbalhip_gemm_prepare does it for every instantiation ahead of time (the host layer
 * calls it when a communicator is created), so that no first launch falls into a stream capture; a launch that still
 * finds its kernel unprepared does it itself, and fails with a clear error if the stream is capturing.
 * Returns the device's CU count through n_cus.
 */
template <auto KERNEL, int LDS_BYTES>
int32_t prepare_kernel(hipStream_t st, int *n_cus)
{
    static std::mutex mu;          /* one per kernel instantiation: guards its per-device set-up below */
    static int cus[64] = {};
    const void *kern = reinterpret_cast<const void *>(KERNEL);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return ZBALHIP_RT_ERROR;
    std::lock_guard<std::mutex> guard(mu);
    if (cus[dev] == 0) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (st != nullptr && hipStreamIsCapturing(st, &capture) == hipSuccess && capture != hipStreamCaptureStatusNone) {
            zbalhip_set_last_error("grouped GEMM: the first launch on a device must happen outside of a stream capture");
            return ZBALHIP_RT_ERROR;
        }
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return ZBALHIP_RT_ERROR;
        if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) != hipSuccess)
            return ZBALHIP_RT_ERROR;
        cus[dev] = n;
    }
    *n_cus = cus[dev];
    return ZBALHIP_OK;
}

template <int MODE, bool GMM1, int OUT_DT, int TM, int NSTAGE, int RG, bool WSTREAM, Shared SH = SHARED_ON_DEMAND>
int32_t prepare_shape(hipStream_t st, int *n_cus)
{
    using S = DmaShape<TM, NSTAGE, MODE == MODE_W4A8 ? 64 : 128, RG>;
    return prepare_kernel<&grouped_gemm_dma_kernel<MODE, GMM1, OUT_DT, TM, NSTAGE, RG, WSTREAM, SH>, S::LDS_BYTES>(st, n_cus);
}

template <int MODE, bool GMM1, int OUT_DT, int TM, int SPLIT = 1, bool VALUES = false>
int32_t prepare_stream(hipStream_t st, int *n_cus)
{
    return prepare_kernel<&grouped_gemm_stream_kernel<MODE, GMM1, OUT_DT, TM, SPLIT, VALUES>, StreamShape<MODE, TM, SPLIT, VALUES>::LDS_BYTES>(st, n_cus);
}

template <int MODE, bool GMM1, int OUT_DT, bool ANY_K = false>
int32_t prepare_tall(hipStream_t st, int *n_cus)
{
    return prepare_kernel<&grouped_gemm_tall_kernel<MODE, GMM1, OUT_DT, ANY_K>, TallShape<MODE>::LDS_BYTES>(st, n_cus);
}

/* launched with one persistent workgroup per CU, or fewer when there are not that many tiles */
template <int MODE, bool GMM1, int OUT_DT, bool ANY_K = false>
int32_t launch_tall(const GemmParams &p, int n_tiles, hipStream_t st)
{
    using S = TallShape<MODE>;
    int n_cus = 0;
    const int32_t rc = prepare_tall<MODE, GMM1, OUT_DT, ANY_K>(st, &n_cus);
    if (rc != ZBALHIP_OK) return rc;
    unsigned grid = grid_for(p.max_rows, p.experts, n_tiles, S::TM);
    const unsigned resident = (unsigned)(n_cus + 7) / 8 * 8;
    if (grid > resident) grid = resident;
    grouped_gemm_tall_kernel<MODE, GMM1, OUT_DT, ANY_K><<<grid, S::THREADS, S::LDS_BYTES, st>>>(p);
    return zbalhip_check_launch();
}

template <int MODE, bool GMM1, int OUT_DT, int TM, int NSTAGE, int RG, bool WSTREAM = false, Shared SH = SHARED_ON_DEMAND>
int32_t launch_dma_shape(const GemmParams &p, int n_tiles, hipStream_t st)
{
    using S = DmaShape<TM, NSTAGE, MODE == MODE_W4A8 ? 64 : 128, RG>;
    int n_cus = 0;
    const int32_t rc = prepare_shape<MODE, GMM1, OUT_DT, TM, NSTAGE, RG, WSTREAM, SH>(st, &n_cus);
    if (rc != ZBALHIP_OK) return rc;
    unsigned grid = grid_for(p.max_rows, p.experts, n_tiles, TM);
    const unsigned resident = (unsigned)(n_cus + 7) / 8 * 8;
    if (grid > resident) grid = resident;
    grouped_gemm_dma_kernel<MODE, GMM1, OUT_DT, TM, NSTAGE, RG, WSTREAM, SH><<<grid, S::THREADS, S::LDS_BYTES, st>>>(p);
    return zbalhip_check_launch();
}

template <int MODE, bool GMM1, int OUT_DT, int TM, int SPLIT = 1, bool VALUES = false>
int32_t launch_stream(const GemmParams &p, int n_tiles, hipStream_t st)
{
    using S = StreamShape<MODE, TM, SPLIT, VALUES>;
    int n_cus = 0;
    const int32_t rc = prepare_stream<MODE, GMM1, OUT_DT, TM, SPLIT, VALUES>(st, &n_cus);
    if (rc != ZBALHIP_OK) return rc;
    const unsigned blocks = (unsigned)stream_workgroups<MODE, GMM1, TM, SPLIT>(p, n_tiles);
    grouped_gemm_stream_kernel<MODE, GMM1, OUT_DT, TM, SPLIT, VALUES><<<blocks, S::THREADS, S::LDS_BYTES, st>>>(p);
    return zbalhip_check_launch();
}

/*
 * The shapes with few rows: rows, stages, row groups of waves. The few-row kernels are weight streams, and what a step
 * costs beside the transfer of its slab is the waves' own work after the barrier, so the waves split the channels
 * rather than the rows: with two row groups (W4A8's first GEMM: one) a weight fragment is read from LDS, and unpacked,
 * by two waves instead of four, and a tile of 16 or 32 rows keeps all eight waves busy instead of two or four.
 */
template <int MODE, bool GMM1> struct FewRows {
    static constexpr int RG_W4 = GMM1 ? 1 : 2;
    static constexpr int RG = MODE == MODE_W4A8 ? RG_W4 : 2;
    static constexpr int STAGES_64 = MODE == MODE_W4A8 ? 4 : 3;
};

/*
 * Row tiles of the streaming kernel: the lower one while most experts' rows fit it (four slabs of weights in flight, as the
 * memory wants it), the taller one beyond (two; the L2 serves the row tiles of an expert together). The registers end them:
 * fp8's block scales leave no room for a fourth sub-tile in the lower one, W8A8's second GEMM and W4A8 have room for eight.
 * W4A8 is bound by vector issue, and a weight unpacked for 128 rows instead of 96 is a tenth of a row's instructions less: 1024 rows
 * per expert, 128 experts of 4096 x 3072 / 1536 x 4096, 2050 -> 1984 / 1008 -> 964 us.
 */
template <int MODE, bool GMM1> struct StreamRows {
    static constexpr int LOW = MODE == MODE_FP8 ? 48 : 64;
    static constexpr int TALL = (MODE == MODE_W8A8 && !GMM1) || MODE == MODE_W4A8 ? 128 : 96;
};

/*
 * Where the streaming kernel takes over from the kernel above (K in whole chunks of its four slabs only), by rows per
 * expert on average; 0: it does not. Layers in us with it against without, uniform / Zipf(1.2) routing, 128 experts of
 * 4096 x 3072 / 1536 x 4096 (M), 64 of 2048 x 2048 / 1024 x 2048 (S), 32 of 7168 x 4096 / 2048 x 7168 (W):
 *   - W4A8: always (M 128 rows -12 / -190, 250 -81 / -184), see w4a8_taller_tile;
 *   - W8A8 first GEMM, 96 rows: 75 M -23 / -52, W -7 / -20, 128 M -35 / -23, W -17 / -4, 187 M +3 / -64, S -8 / -41,
 *     250 M +35 / -46, W +22 / -27, 375 S -9 / -33, 512 M +90 / +17; second, 128 rows: 75 M -12 / -37, 128 M -27 / -32,
 *     250 W -13 / -18, 375 M -25 / -21, 512 M +14 / -24;
 *   - fp8 first GEMM: 75 W -7 / -29, 128 W -21 / -13, 187 S +2 / -27, 250 W +39 / -37, 375 S 0 / -23, 768 S +27 / 0; second:
 *     75 W -10 / -25, 250 W -13 / -29, 500 W +9 / +17, 768 S -3 / -17.
 * Beyond, the many-row shapes' arithmetic intensity wins, the sooner the longer K is. Long K loops whose tiles fill whole
 * rounds of CUs run at the memory's rate in both kernels (W, 512 tiles: 6.6 TB/s), and there popular experts of up to 128
 * rows are one tile in the other: 128 tokens Zipf W8A8 +11.
 * With every expert as popular as the next, row counts just past a tile's height cost: two tiles of 50 rows where the other
 * kernel has one of 128 (or 320). Both GEMMs of nine shapes, 8 to 256 experts, 2048 to 8192 wide, 1024 to 14336 deep,
 * 8 to 400 rows, both kernels in turn in one process, uniform / Zipf(0.6) / Zipf(1.2) routing, per cent:
 *   - first GEMM, K > 2048: 84 rows 0 / -11 / -15; 88-108 rows W8A8 +6 (up to +31) / -9 / -12, 88-112 fp8 +12 (+34) / -7 / -13:
 *     left to the other; 120-160 rows W8A8 -4 / -12 / -18, fp8 -3 / -12 / -22; W8A8 190-200 rows +5 (+15) / -11 / -22: hence 184;
 *   - many tiles (256 experts: 4096 in the first GEMM, 7168 in the second), where both run at the memory's rate longer: first
 *     fp8 GEMM 112-150 rows +10 / -2 / -20, second GEMM 200-320 rows W8A8 +7 / +1 / -16, fp8 +13 / +3 / -22;
 *   - second fp8 GEMM, K 14336, 8 experts: 160-190 rows +34 / +25 / +33 (a third row tile on a few CUs, and K is long); from
 *     200 to 350, where the other kernel's tile is 320 rows, -27 / -25 / -25, 400 rows (a fifth row tile) +27 / -14 / -12;
 *   - W4A8 -2 ... -50 throughout.
 * Against the many-row kernel of zbal_gemm_tall.h (nine shapes, 112 to 600 rows, uniform / Zipf(0.6) / Zipf(1.2), per cent that it
 * takes more): the lines lie where it wins with every routing. First GEMM 200 rows W8A8 -16 / +1 / +13, fp8 -24 / 0 / +18,
 * 400 rows -10 / -9 / +2, -16 / -12 / +2; second 300 rows W8A8 -3 / -2 / +13, fp8 -11 / -9 / +10, 400 rows fp8 -15 / -11 / +2;
 * K 1024, 64 experts, fp8: 500 rows -16 / -5 / +11, 600 rows -10 / -12 / -5, 800 rows Zipf(1.2) -13 (until then the line was 800).
 */
template <int MODE, bool GMM1>
inline int stream_rows(const GemmParams &p, int n_tiles)
{
    using R = StreamRows<MODE, GMM1>;
    const int64_t rows = p.max_rows, e = p.experts, tiles = e * n_tiles;
    if (p.K % 512 != 0) return 0;
    if (MODE == MODE_W4A8) return w4a8_taller_tile(rows, e, n_tiles, cu_count()) ? R::TALL : R::LOW;
    const bool many_tiles = tiles >= 4096;
    const int64_t low = MODE == MODE_W8A8 ? 48 : 36;
    int64_t tall = many_tiles && !GMM1 ? 192 : 400;
    if (GMM1 && p.K > 2048) {
        if (p.K >= 6144 && rows <= 40 * e) {
            const int64_t cus = cu_count(), round = cus > 0 ? (tiles + cus - 1) / cus * cus : tiles;
            if (tiles * 8 >= round * 7) return 0;
        }
        if (rows > 87 * e && rows <= (MODE == MODE_W8A8 ? 108 : 112) * e) return 0;
        tall = MODE == MODE_W8A8 ? 184 : (many_tiles ? 87 : 160);
    }
    if (MODE == MODE_FP8 && !GMM1) {
        if (p.K > 8192) {
            if (rows > 150 * e && rows <= 192 * e) return 0;
            tall = 352;
        }
        if (p.K <= 1024 && !many_tiles) tall = 520;
    }
    return rows <= low * e ? R::LOW : (rows <= tall * e ? R::TALL : 0);
}

/*
 * A token or two: where the experts that can have rows make tiles for half of the CUs at most, two workgroups share each of
 * them, four waves and half of the channels to either, because what one CU takes from memory (30 GB/s) is the limit then.
 * Tiles of 16 rows, since there are hardly more. Rows in all, us for whole tiles -> halves (quarters):
 *   - 8 of 32 experts, 7168 x 4096, 128 tiles: W8A8 first GEMM 49.7 -> 41.9 (43.1); second, 224 tiles of 2048 x 7168: 19.3 (19.5);
 *     beyond the half of the CUs (one token with a shared expert is 9 of 33): 144 tiles 50.3 -> 57.7, 160 52.2 -> 59.2; second, 140 tiles
 *     14.2 -> 15.3, fp8 14.5 -> 15.3; W4A8, 4096 x 3072 / 1536 x 4096, 144 tiles 20.7 -> 21.9 / 7.3 -> 7.9;
 *   - 8 of 128, 4096 x 3072 / 1536 x 4096, 96 / 128 tiles: W8A8 30.7 -> 22.9 (24.7) / 11.8 -> 10.2 (10.4), W4A8 19.9 -> 18.1
 *     (20.4) / 7.9 -> 6.8 (7.4); 16 rows, 192 / 256 tiles: W8A8 36.6 (37.9) / 17.4 (17.1), W4A8 23.5 (24.8) / 10.3 (10.2);
 *   - 6 of 64, 2048 x 2048 / 1024 x 2048, 48 tiles: W8A8 18.5 -> 14.6 (14.0) / 8.0 -> 6.0 (5.1), W4A8 14.4 -> 14.0 (14.9) /
 *     5.9 -> 5.1 (5.0), fp8 second 8.2 -> 6.0 (5.5); 12 rows, 96 tiles: fp8 second 8.6 -> 6.9, W4A8 14.4 (14.5) / 6.2 -> 5.3.
 */
inline bool few_tiles(const GemmParams &p, int n_tiles)
{
    const int64_t rows = p.max_rows, e = p.experts, busy = rows < e ? rows : e;
    return p.K % 512 == 0 && busy * n_tiles * 2 <= cu_count() && (rows <= 16 || rows <= 8 * e);
}

/* every shape a launch of (MODE, GMM1, OUT_DT) can take */
template <int MODE, bool GMM1, int OUT_DT>
int32_t prepare_mode()
{
    using F = FewRows<MODE, GMM1>;
    int n = 0;
    int32_t rc = prepare_shape<MODE, GMM1, OUT_DT, 256, 2, 4, false>(nullptr, &n);
    if (rc == ZBALHIP_OK) rc = prepare_shape<MODE, GMM1, OUT_DT, 128, 3, F::RG, false>(nullptr, &n);
    if (rc == ZBALHIP_OK) rc = prepare_shape<MODE, GMM1, OUT_DT, 64, F::STAGES_64, F::RG, true>(nullptr, &n);
    if (rc == ZBALHIP_OK) rc = prepare_stream<MODE, GMM1, OUT_DT, StreamRows<MODE, GMM1>::LOW>(nullptr, &n);
    if (rc == ZBALHIP_OK) rc = prepare_stream<MODE, GMM1, OUT_DT, StreamRows<MODE, GMM1>::TALL>(nullptr, &n);
    if constexpr (!(MODE == MODE_FP8 && GMM1)) {
        if (rc == ZBALHIP_OK) rc = prepare_stream<MODE, GMM1, OUT_DT, 16, 2>(nullptr, &n);
    }
    if constexpr (MODE != MODE_FP8 && !GMM1) {
        if (rc == ZBALHIP_OK) rc = prepare_stream<MODE, GMM1, OUT_DT, 16, 2, true>(nullptr, &n);
        if (rc == ZBALHIP_OK) rc = prepare_stream<MODE, GMM1, OUT_DT, 32, 1, true>(nullptr, &n);
    }
    if constexpr (MODE == MODE_W4A8) {
        if (rc == ZBALHIP_OK) rc = prepare_shape<MODE, GMM1, OUT_DT, 128, 3, 2, false>(nullptr, &n);
        if (rc == ZBALHIP_OK) rc = prepare_shape<MODE, GMM1, OUT_DT, 192, 3, 2, false>(nullptr, &n);
    } else {
        if (rc == ZBALHIP_OK) rc = prepare_shape<MODE, GMM1, OUT_DT, 256, 2, 4, false, SHARED_NONE>(nullptr, &n);
        if (rc == ZBALHIP_OK) rc = prepare_tall<MODE, GMM1, OUT_DT>(nullptr, &n);
        if constexpr (MODE == MODE_FP8) {
            if (rc == ZBALHIP_OK) rc = prepare_tall<MODE, GMM1, OUT_DT, true>(nullptr, &n);
        }
        if (rc == ZBALHIP_OK) rc = prepare_shape<MODE, GMM1, OUT_DT, 128, 3, F::RG, true>(nullptr, &n);
    }
    return rc;
}

/*
 * Shape choice from what the host knows (the row counts themselves live on the device). With few rows per expert the
 * GEMM is a weight-streaming job and takes the three-stage 128-row shape (which needs two K slabs to fill its
 * pipeline); with many it needs the arithmetic intensity of taller tiles. The 128-row shape was timed against the 320-row one (of
 * four row groups of waves) that the many-row kernel has replaced, on 7168 x 4096 / 2048 x 7168 experts (W4A8: 4096 x 3072 / 1536 x 4096, 128 experts) with 32
 * and with 256 experts, random routing; rows per expert on average, first / second GEMM, 128-row against tall
 * (W4A8: 256-row) shape in ms:
 *   - fp8, 32 experts: 128 rows 0.247 / 0.136 against 0.256 / 0.145; 192 rows 0.298 / 0.160 against 0.278 / 0.166;
 *     256 rows 0.369 / 0.194 against 0.306 / 0.188. 256 experts: 128 rows 1.889 / 0.961 against 1.877 / 1.088;
 *     192 rows 2.314 / 1.204 against 2.108 / 1.148;
 *   - W8A8, 32 experts: 128 rows 0.243 / 0.129 against 0.254 / 0.138; 192 rows 0.289 / 0.146 against 0.275 / 0.150;
 *     256 rows 0.342 / 0.174 against 0.303 / 0.163. 256 experts: 128 rows 1.788 / 0.892 against 1.799 / 0.931;
 *     192 rows 2.197 / 1.093 against 2.016 / 1.106.
 */
template <int MODE, bool GMM1>
inline int64_t few_rows_limit(const GemmParams &p, int n_tiles)
{
    if (GMM1) return 128;
    const bool few_tiles = (int64_t)p.experts * n_tiles <= 1024;
    return (MODE == MODE_FP8 && !few_tiles) ? 128 : 192;
}

/*
 * W4A8 where the streaming kernel does not run (K no multiple of 512): the smaller the slab (16 KiB of weights), the more a step's own work shows, and the compute-bound sizes are
 * bound by vector instructions, a quarter of which unpack weights once per row group of waves. Shapes by rows per
 * expert on average, first / second GEMM in us on 4096 x 3072 / 1536 x 4096, 128 experts, random routing, one GPU,
 * old (four row groups, 128 or 256 rows) against now:
 *   - up to 48: 64 rows, 4 stages, streaming hint: 1 row 152 / 82 -> 104 / 58, 4 rows 222 / 108 -> 155 / 78, 32 rows
 *     263 / 127 -> 197 / 102, 44 rows 278 / 135 -> 213 / 109 (53 rows: 244 / 124, the next shape 242 / 118);
 *   - up to 100: 128 rows, 3 stages: 64 rows 308 / 145 -> 255 / 124, 96 rows 362 / 166 -> 316 / 150;
 *   - up to 640: 192 rows, 3 stages, two row groups: 112 rows 436 / 186 -> 368 / 169, 128 rows 440 / 197 -> 380 / 174,
 *     256 rows 757 / 329 -> 697 / 329, 512 rows 1289 / 585 -> 1237 / 571; except where most experts just miss one tile
 *     of it and make two of half the height, which the 128-row shape does cheaper (187 rows, 64 experts of 2048 x 2048
 *     / 1024 x 2048: 145 / 60 against 128 / 54);
 *   - beyond: 256 rows (1024 rows: 2456 / 1098 against 2507 / 1185).
 */
template <bool GMM1, int OUT_DT>
int32_t launch_w4a8(const GemmParams &p, int n_tiles, hipStream_t st)
{
    using F = FewRows<MODE_W4A8, GMM1>;
    const int64_t rows = p.max_rows, e = p.experts;
    if (rows <= 48 * e && p.K >= 128 * (F::STAGES_64 - 1))
        return launch_dma_shape<MODE_W4A8, GMM1, OUT_DT, 64, F::STAGES_64, F::RG, true>(p, n_tiles, st);
    if (p.K >= 256) {
        if (rows <= 100 * e) return launch_dma_shape<MODE_W4A8, GMM1, OUT_DT, 128, 3, F::RG>(p, n_tiles, st);
        if (rows > 160 * e && rows <= 224 * e) return launch_dma_shape<MODE_W4A8, GMM1, OUT_DT, 128, 3, 2>(p, n_tiles, st);
        if (rows <= 640 * e) return launch_dma_shape<MODE_W4A8, GMM1, OUT_DT, 192, 3, 2>(p, n_tiles, st);
    }
    return launch_dma_shape<MODE_W4A8, GMM1, OUT_DT, 256, 2, 4>(p, n_tiles, st);
}

template <int MODE, bool GMM1, int OUT_DT>
int32_t launch_dma(const GemmParams &p, int n_tiles, hipStream_t st)
{
    using R = StreamRows<MODE, GMM1>;
    const int stream = stream_rows<MODE, GMM1>(p, n_tiles);
    if constexpr (!(MODE == MODE_FP8 && GMM1)) {
        if (few_tiles(p, n_tiles)) return launch_stream<MODE, GMM1, OUT_DT, 16, 2>(p, n_tiles, st);
    }
    if (stream == R::LOW) return launch_stream<MODE, GMM1, OUT_DT, R::LOW>(p, n_tiles, st);
    if (stream == R::TALL) return launch_stream<MODE, GMM1, OUT_DT, R::TALL>(p, n_tiles, st);
    if constexpr (MODE == MODE_W4A8) {
        return launch_w4a8<GMM1, OUT_DT>(p, n_tiles, st);
    } else {
        using F = FewRows<MODE, GMM1>;
        const int64_t rows = p.max_rows, e = p.experts;
        if (rows <= few_rows_limit<MODE, GMM1>(p, n_tiles) * e && p.K >= 256) {
            /*
             * Where nearly every expert has a single row tile its weight slabs are read once: they are requested with the
             * streaming hint. Measured on 32 experts of 7168 x 4096 / 2048 x 7168, without / with, rows per expert:
             * fp8 25 rows 165 / 91 -> 147 / 85 us, 64 rows 177 / 100 -> 153 / 99, 100 rows 194 / 109 -> 180 / 112, 128 rows
             * 284 / 132 -> 288 / 146; W8A8 64 rows 195 / 100 -> 175 / 97, on 128 experts of 4096 x 3072 / 1536 x 4096
             * 81 rows 367 / 180 -> 348 / 170, 128 rows 453 / 216 -> 523 / 238 (row tiles that share slabs through the L2).
             */
            const int64_t stream_limit = GMM1 ? 100 : (MODE == MODE_W8A8 ? 96 : 84);
            /*
             * A handful of rows: half the tile height, so the transfers of absent rows shrink as well (one row: 55.9 / 22.8
             * -> 54.8 / 21.2 us on the experts above, 22.9 / 11.1 -> 21.6 / 9.8 on 64 of 2048 x 2048 / 1024 x 2048; equal from
             * 4 to 32 rows). The limit leaves room for popular experts, whose rows would make several tiles of 64.
             */
            if (rows <= 8 * e) return launch_dma_shape<MODE, GMM1, OUT_DT, 64, F::STAGES_64, F::RG, true>(p, n_tiles, st);
            if (rows <= stream_limit * e) return launch_dma_shape<MODE, GMM1, OUT_DT, 128, 3, F::RG, true>(p, n_tiles, st);
            return launch_dma_shape<MODE, GMM1, OUT_DT, 128, 3, F::RG>(p, n_tiles, st);
        }
        /*
         * Many rows: at every count against what ran there before (320-row tiles on four row groups of waves, fp8 beyond 1536 rows
         * per expert the 256-row shape below), both GEMMs, 32 experts of 7168 x 4096 / 2048 x 7168, 64 of 2048 x 2048 /
         * 1024 x 2048, 8 of 4096 x 28672 / 14336 x 4096, 250 to 2300 rows per expert: fp8 -8 / -11 % (0 ... -21), W8A8
         * -10 / -8 % (+1 ... -15). 1024 rows of the first: fp8 1047 / 596 -> 935 / 543 us, W8A8 974 / 519 -> 905 / 468. The kernel for
         * any fp8 K, 256 to 1800 rows per expert, thirty shapes with K from 256 to 32768: -10 % (+5 ... -24).
         */
        if (tall_accepts<MODE>(p)) {
            if constexpr (MODE == MODE_FP8) {
                if (tall_wants_any_k(p.K / 128)) return launch_tall<MODE, GMM1, OUT_DT, true>(p, n_tiles, st);
            }
            return launch_tall<MODE, GMM1, OUT_DT>(p, n_tiles, st);
        }
        /*
         * This shape's K loop has no scalar register to spare for a shared expert's tensors, and with this many rows per
         * expert the fused layer's takes turns with the routed ones: 2048 rows fp8, first GEMM 2.01 ms with the shared
         * expert's branches, 1.95 without.
         */
        if (p.shared_index < 0) return launch_dma_shape<MODE, GMM1, OUT_DT, 256, 2, 4, false, SHARED_NONE>(p, n_tiles, st);
        return launch_dma_shape<MODE, GMM1, OUT_DT, 256, 2, 4>(p, n_tiles, st);
    }
}

/* the second GEMM of the int modes from the first one's fp32 values (zbalhip_gmm2_takes_values) */
template <int MODE, int OUT_DT>
int32_t launch_values(const GemmParams &p, int n_tiles, hipStream_t st)
{
    if (few_tiles(p, n_tiles)) return launch_stream<MODE, false, OUT_DT, 16, 2, true>(p, n_tiles, st);
    return launch_stream<MODE, false, OUT_DT, 32, 1, true>(p, n_tiles, st);
}

} // namespace

/*
 * The requantisation launch is saved, but every channel tile of an expert makes its rows' bytes again, the more of them the
 * longer a row and the more rows. Layers, us: 7168 x 4096 / 2048 x 7168, 32 experts, W8A8, 1 row per 4 experts 76.2 -> 73.7, 1 row per
 * expert 188 -> 182, 2.3 rows 236 -> 232, 3 rows 238 -> 238, 8 rows 242.5 -> 243.5, Zipf(1.2) 242 -> 246; 128 of 4096 x 3072 /
 * 1536 x 4096, W4A8, 1 token 37.9 -> 34.4, 3 rows 211 -> 207, 8 rows 226 -> 228; 64 of 2048 x 2048 / 1024 x 2048, W8A8, 1 token
 * 32.3 -> 29.4, 2 rows 74.2 -> 71.7, 4.7 rows Zipf 76.8 -> 75.3.
 */
extern "C" int32_t zbalhip_gmm2_takes_values(int64_t experts, int64_t max_rows, int64_t k, int32_t mode)
{
    return (mode == MODE_W8A8 || mode == MODE_W4A8) && k > 0 && k % 512 == 0 && max_rows * k <= 5120 * experts;
}

/* the shared expert that rides along: one expert more, its rows from max_rows on (`shared` null: none) */
static void with_shared(GemmParams &p, const zbalhip_shared_expert_t *shared, int64_t out_row_bytes)
{
    p.shared_index = -1;
    if (!shared) return;
    p.shared_index = p.experts;
    p.shared_row = p.max_rows;
    p.experts += 1;
    p.max_rows += (int)shared->rows;
    p.shared_w = (const uint8_t *)shared->weight;
    p.shared_wscale = shared->scale;
    p.shared_out = (void *)((uintptr_t)shared->out - (uintptr_t)p.shared_row * (uintptr_t)out_row_bytes);
}

/*
 * Memory for tiles shared along K (W8A8; null: none). Which of them are is the kernel's business (shared_rows), but not with a K up to
 * 4096: there the exchange took more than it saved where tiles of any height were shared (64 experts of 2048 x 2048, 100 tokens
 * Zipf(1.2), layer 79 -> 81 us, 128 of 4096 x 3072, 64 tokens 314 -> 317), and what lower ones would give has not been measured.
 */
static void with_parts(GemmParams &p, void *parts, int64_t bytes)
{
    const int64_t cus = cu_count() / 8, floats = (bytes / 4 - ZBALHIP_PART_WORDS) / 8 / 4 * 4;
    if (p.K <= 4096) return;
    if (!parts || cus <= 0 || 8 * cus > ZBALHIP_PART_WORDS || floats <= 0) return;
    p.part_done = (uint32_t *)parts;
    p.part_sums = (float *)(p.part_done + ZBALHIP_PART_WORDS);
    p.part_floats = floats;
    p.part_cus = (int)cus;
}

static bool shared_is_valid(const zbalhip_shared_expert_t *shared, int64_t experts, bool needs_out)
{
    if (!shared) return true;
    return experts < 1024 && shared->rows > 0 && shared->weight && shared->scale && !misaligned16(shared->weight) &&
           !misaligned16(shared->scale) && (!needs_out || (shared->out && !misaligned16(shared->out)));
}

extern "C" int32_t zbalhip_gmm1_swiglu_quant_parts(const void *a, const float *a_scale, const void *w1, const void *w1scale,
                                                   const int32_t *row_off, int64_t experts, int64_t max_rows, int64_t k,
                                                   int64_t n1, int32_t mode, void *q2, float *scale2, float *sgl_ws,
                                                   const zbalhip_shared_expert_t *shared, void *parts, int64_t parts_bytes, void *stream)
{
    const int w_is_list = (mode & ZBALHIP_WEIGHTS_AS_LISTS) != 0;
    const bool rowmax_cleared = (mode & ZBALHIP_ROWMAX_CLEARED) != 0, values = (mode & ZBALHIP_SWIGLU_VALUES) != 0;
    mode &= ~(ZBALHIP_WEIGHTS_AS_LISTS | ZBALHIP_ROWMAX_CLEARED | ZBALHIP_SWIGLU_VALUES);
    if (values && mode == MODE_FP8) return ZBALHIP_INVALID;
    if (!a || !a_scale || !w1 || !w1scale || !row_off || !q2 || !scale2) return ZBALHIP_INVALID;
    if (mode < MODE_W8A8 || mode > MODE_W4A8) return ZBALHIP_INVALID;
    if (misaligned16(a) || misaligned16(w1) || misaligned16(w1scale) || misaligned16(q2) || misaligned16(sgl_ws)) return ZBALHIP_INVALID;
    if (experts <= 0 || experts > 1024 || max_rows < 0 || k <= 0 || k % 128 != 0 || k > 128 * 256 || n1 <= 0 || n1 % 256 != 0)
        return ZBALHIP_INVALID;
    if (!shared_is_valid(shared, experts, false)) return ZBALHIP_INVALID;
    if (max_rows == 0) return ZBALHIP_OK;
    hipStream_t st = (hipStream_t)stream;
    GemmParams p = {};
    p.a = (const uint8_t *)a; p.a_scale = a_scale; p.w = (const uint8_t *)w1; p.wscale = w1scale; p.row_off = row_off;
    p.experts = (int)experts; p.max_rows = (int)max_rows; p.K = (int)k; p.N = (int)n1;
    p.out = q2; p.out_scale = scale2; p.sgl_ws = sgl_ws; p.w_is_list = w_is_list;
    with_shared(p, shared, 0);
    if (misaligned16(parts) || (parts && parts_bytes < 0)) return ZBALHIP_INVALID;
    if (mode == MODE_W8A8) with_parts(p, parts, parts_bytes);
    const int n_tiles = (int)(n1 / 2 / 128);
    if (mode == MODE_FP8) return launch_dma<MODE_FP8, true, ZDT_BF16>(p, n_tiles, st);
    if (!sgl_ws) return ZBALHIP_INVALID;
    /* the row maxima live behind the SwiGLU values in the same scratch allocation */
    p.rowmax = (uint32_t *)(sgl_ws + (int64_t)p.max_rows * (n1 / 2));
    if (!rowmax_cleared) fill_u32_kernel<<<(unsigned)((p.max_rows + 255) / 256), 256, 0, st>>>(p.rowmax, p.max_rows, 0u);
    const int32_t rc = mode == MODE_W8A8 ? launch_dma<MODE_W8A8, true, ZDT_BF16>(p, n_tiles, st)
                                         : launch_dma<MODE_W4A8, true, ZDT_BF16>(p, n_tiles, st);
    if (rc != ZBALHIP_OK || values) return rc;
    const int rb = p.max_rows < 16384 ? p.max_rows : 16384;
    requant_rows_kernel<<<(unsigned)rb, kRequantThreads, 0, st>>>(sgl_ws, p.rowmax, row_off, p.experts, shared ? p.shared_row : p.max_rows,
                                                                  p.max_rows, (int)(n1 / 2), (int8_t *)q2, scale2);
    return zbalhip_check_launch();
}

extern "C" int32_t zbalhip_gmm1_swiglu_quant_shared(const void *a, const float *a_scale, const void *w1, const void *w1scale,
                                                    const int32_t *row_off, int64_t experts, int64_t max_rows, int64_t k,
                                                    int64_t n1, int32_t mode, void *q2, float *scale2, float *sgl_ws,
                                                    const zbalhip_shared_expert_t *shared, void *stream)
{
    return zbalhip_gmm1_swiglu_quant_parts(a, a_scale, w1, w1scale, row_off, experts, max_rows, k, n1, mode, q2, scale2, sgl_ws,
                                           shared, nullptr, 0, stream);
}

extern "C" int32_t zbalhip_gmm1_swiglu_quant(const void *a, const float *a_scale, const void *w1, const void *w1scale,
                                             const int32_t *row_off, int64_t experts, int64_t max_rows, int64_t k,
                                             int64_t n1, int32_t mode, void *q2, float *scale2, float *sgl_ws,
                                             void *stream)
{
    return zbalhip_gmm1_swiglu_quant_shared(a, a_scale, w1, w1scale, row_off, experts, max_rows, k, n1, mode, q2, scale2, sgl_ws,
                                            nullptr, stream);
}

extern "C" int32_t zbalhip_gmm2_dequant_shared(const void *a, const float *a_scale, const void *w2, const void *wscale,
                                               int32_t wscale_dtype, const int32_t *row_off, int64_t experts,
                                               int64_t max_rows, int64_t k, int64_t n, int32_t mode, int32_t out_dtype,
                                               void *y, const zbalhip_shared_expert_t *shared, void *stream)
{
    const int w_is_list = (mode & ZBALHIP_WEIGHTS_AS_LISTS) != 0;
    const bool values = (mode & ZBALHIP_SWIGLU_VALUES) != 0;
    mode &= ~(ZBALHIP_WEIGHTS_AS_LISTS | ZBALHIP_SWIGLU_VALUES);
    if (values && (mode == MODE_FP8 || k % 512 != 0)) return ZBALHIP_INVALID;
    if (!a || !a_scale || !w2 || !wscale || !row_off || !y) return ZBALHIP_INVALID;
    if (mode < MODE_W8A8 || mode > MODE_W4A8) return ZBALHIP_INVALID;
    if (misaligned16(a) || misaligned16(w2) || misaligned16(wscale) || misaligned16(y)) return ZBALHIP_INVALID;
    if (out_dtype != ZDT_BF16 && out_dtype != ZDT_FP16) return ZBALHIP_INVALID;
    if (experts <= 0 || experts > 1024 || max_rows < 0 || k <= 0 || k % 128 != 0 || k > 128 * 256 || n <= 0 || n % BN != 0)
        return ZBALHIP_INVALID;
    if (mode == MODE_W8A8 && wscale_dtype != ZDT_FP32 && wscale_dtype != ZDT_BF16) return ZBALHIP_INVALID;
    if (!shared_is_valid(shared, experts, true)) return ZBALHIP_INVALID;
    if (max_rows == 0) return ZBALHIP_OK;
    hipStream_t st = (hipStream_t)stream;
    GemmParams p = {};
    p.a = (const uint8_t *)a; p.a_scale = a_scale; p.w = (const uint8_t *)w2; p.wscale = wscale; p.row_off = row_off;
    p.experts = (int)experts; p.max_rows = (int)max_rows; p.K = (int)k; p.N = (int)n;
    p.wscale_is_bf16 = (wscale_dtype == ZDT_BF16);
    p.w_is_list = w_is_list;
    p.out = y;
    with_shared(p, shared, n * 2);
    const int n_tiles = (int)(n / BN);
    const bool bf = out_dtype == ZDT_BF16;
    if (values) {
        if (mode == MODE_W8A8) return bf ? launch_values<MODE_W8A8, ZDT_BF16>(p, n_tiles, st) : launch_values<MODE_W8A8, ZDT_FP16>(p, n_tiles, st);
        return bf ? launch_values<MODE_W4A8, ZDT_BF16>(p, n_tiles, st) : launch_values<MODE_W4A8, ZDT_FP16>(p, n_tiles, st);
    }
    if (mode == MODE_W8A8)
        return bf ? launch_dma<MODE_W8A8, false, ZDT_BF16>(p, n_tiles, st) : launch_dma<MODE_W8A8, false, ZDT_FP16>(p, n_tiles, st);
    if (mode == MODE_FP8)
        return bf ? launch_dma<MODE_FP8, false, ZDT_BF16>(p, n_tiles, st) : launch_dma<MODE_FP8, false, ZDT_FP16>(p, n_tiles, st);
    return bf ? launch_dma<MODE_W4A8, false, ZDT_BF16>(p, n_tiles, st) : launch_dma<MODE_W4A8, false, ZDT_FP16>(p, n_tiles, st);
}

extern "C" int32_t zbalhip_gmm2_dequant(const void *a, const float *a_scale, const void *w2, const void *wscale,
                                        int32_t wscale_dtype, const int32_t *row_off, int64_t experts,
                                        int64_t max_rows, int64_t k, int64_t n, int32_t mode, int32_t out_dtype,
                                        void *y, void *stream)
{
    return zbalhip_gmm2_dequant_shared(a, a_scale, w2, wscale, wscale_dtype, row_off, experts, max_rows, k, n, mode, out_dtype, y,
                                       nullptr, stream);
}

extern "C" int32_t zbalhip_gemm_prepare(void)
{
    /* once per device and process: later calls (every communicator that is created makes one) cost one device query */
    static std::atomic<bool> prepared[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return ZBALHIP_RT_ERROR;
    if (prepared[dev].load(std::memory_order_acquire)) return ZBALHIP_OK;
    int32_t rc = prepare_mode<MODE_W8A8, true, ZDT_BF16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_FP8, true, ZDT_BF16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_W4A8, true, ZDT_BF16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_W8A8, false, ZDT_BF16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_W8A8, false, ZDT_FP16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_FP8, false, ZDT_BF16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_FP8, false, ZDT_FP16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_W4A8, false, ZDT_BF16>();
    if (rc == ZBALHIP_OK) rc = prepare_mode<MODE_W4A8, false, ZDT_FP16>();
    if (rc == ZBALHIP_OK) prepared[dev].store(true, std::memory_order_release);
    return rc;
}
