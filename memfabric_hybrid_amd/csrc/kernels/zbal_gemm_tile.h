/*
 * What the grouped-GEMM kernels share: the parameter block, one expert's weights, the LDS-DMA transfers and the fused
 * epilogues.
 */
#ifndef ZBAL_GEMM_TILE_H_
#define ZBAL_GEMM_TILE_H_

#include "zbal_device.h"
#include "zbal_hip_kernels.h"

namespace {

constexpr int BN = 256;          /* output channels per workgroup tile */
constexpr int BKB = 128;         /* K bytes of an activation row per slab (128 int8/e4m3 elements) */
constexpr int GROUP_N = 8;       /* channel tiles per schedule group, at most */

enum { MODE_W8A8 = 1, MODE_FP8 = 2, MODE_W4A8 = 3 };

struct GemmParams {
    const uint8_t *a;        /* [rows, K] */
    const float *a_scale;    /* [rows] or [rows, K/128] */
    const uint8_t *w;        /* pre-packed blocks, [E][N/128][K/128] x 16 KiB (8-bit) or 8 KiB (int4) */
    const void *wscale;
    const int32_t *row_off;  /* [E+1] */
    int experts;
    int max_rows;            /* rows the A / output buffers hold */
    int K;
    int N;                   /* weight rows per expert (N1 for GMM1) */
    int wscale_is_bf16;
    int w_is_list;           /* `w` and `wscale` are device tables of `experts` addresses, one expert's tensor each */
    void *out;               /* GMM1: q2 bytes; GMM2: y */
    float *out_scale;        /* GMM1: scale2 (fp8 mode) */
    float *sgl_ws;           /* GMM1 int8 modes: fp32 SwiGLU values [rows, N/2] */
    uint32_t *rowmax;        /* GMM1 int8 modes: per-row absmax bits */
    /*
     * A shared expert in the same launch: the last of `experts`, with tensors of its own. Its rows start at shared_row,
     * behind all rows that the routed experts can have, and end at row_off[experts]. shared_index is -1 without one.
     */
    int shared_index, shared_row;
    const uint8_t *shared_w;
    const void *shared_wscale;
    void *shared_out;        /* GMM2: where row 0 would be if row shared_row is the first */
    /*
     * For the streaming kernel's tiles that several workgroups share along K (W8A8's first GEMM; null: none do): 8 * part_cus
     * words that are zero when the launch starts, and room for part_floats sums of every XCD's tiles.
     */
    uint32_t *part_done;
    float *part_sums;
    int64_t part_floats;
    int part_cus;            /* CUs per XCD */
};

/*
 * First element of expert e's weights or scales: base + e * stride, or entry e of the address table. The table is
 * read through the constant address space: a scalar load, which does not queue behind the slabs in flight.
 */
template <typename T>
__device__ __forceinline__ const T *expert_base(const void *base, int is_list, int expert, int64_t stride_elems)
{
    if (is_list) {
        typedef const uint64_t __attribute__((address_space(4))) *table_t;
        return (const T *)(uintptr_t)((table_t)(uintptr_t)base)[expert];
    }
    return (const T *)base + (int64_t)expert * stride_elems;
}

/*
 * How a kernel knows of a shared expert. The staged kernel's K loop takes all scalar registers, and the shared expert's
 * tensors, kept in some through it, pushed others out into lanes of vector registers (9 to 31 more of them; fp8 2048 rows, 256-row
 * shape: first GEMM +3.5 %, second +1.5 %): it reads them where a tile of the shared expert needs them, from the launch's
 * arguments in memory. The streaming kernel has registers left, and its one tile would wait for the reads (W4A8 +0.5 %).
 */
enum Shared { SHARED_NONE, SHARED_ON_DEMAND, SHARED_IN_REGISTERS };

/* GemmParams is the kernels' only parameter */
using LaunchArgs = const GemmParams __attribute__((address_space(4))) *;
__device__ __forceinline__ LaunchArgs launch_args()
{
    auto *args = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));                     /* not hoisted */
    return (LaunchArgs)args;
}

template <Shared SH> __device__ __forceinline__ bool is_shared(const GemmParams &p, int expert)
{
    return SH != SHARED_NONE && expert == p.shared_index;
}
template <typename T, Shared SH> __device__ __forceinline__ const T *weights_of(const GemmParams &p, int expert, int64_t stride)
{
    if (is_shared<SH>(p, expert)) return (const T *)(SH == SHARED_ON_DEMAND ? launch_args()->shared_w : p.shared_w);
    return expert_base<T>(p.w, p.w_is_list, expert, stride);
}
template <typename T, Shared SH> __device__ __forceinline__ const T *scales_of(const GemmParams &p, int expert, int64_t stride)
{
    if (is_shared<SH>(p, expert)) return (const T *)(SH == SHARED_ON_DEMAND ? launch_args()->shared_wscale : p.shared_wscale);
    return expert_base<T>(p.wscale, p.w_is_list, expert, stride);
}
template <Shared SH> __device__ __forceinline__ int first_row_of(const GemmParams &p, int expert)
{
    if constexpr (SH == SHARED_ON_DEMAND) return is_shared<SH>(p, expert) ? launch_args()->shared_row : p.row_off[expert];
    else return is_shared<SH>(p, expert) ? p.shared_row : p.row_off[expert];
}

struct TileCoord {
    int expert, m_tile, n_tile;
};

__device__ __forceinline__ f32x4 mfma_fp8_16x16x128(const i32x8 &wfrag, const i32x8 &afrag)
{
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    /* cbsz = blgp = 0 selects e4m3 for both inputs; scale exponents 0 leave the product unscaled */
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wfrag, afrag, zero, 0, 0, 0, 0, 0, 0);
}

/*
 * A barrier for what is in LDS, with the slabs in flight left alone whatever the compiler takes a barrier to wait for (its
 * __syncthreads() waits for no more on gfx950, and the staged kernel's step has one).
 */
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

/* four consecutive bytes -> one dword store helpers */
__device__ __forceinline__ uint32_t pack4_e4m3(float a, float b, float c, float d)
{
    return zb_cvt_pk_e4m3(a, b) | (zb_cvt_pk_e4m3(c, d) << 16);
}

/*
 * Shared epilogue. The calling wave holds, for sub-tile (mt, nt), block rows nt*16 + 4*(lane/16) + i of its weight
 * rows, for token row (RG*mt + wm)*16 + lane%16 of the tile (RG = row groups of waves; a wave's 16-row sub-tiles
 * are dealt round-robin over the row groups, so a tile that is not full leaves every SIMD the same share). The pre-pack put channels 32*(nt/2) + 8*(lane/16) + 4*(nt%2) + i in
 * those rows (zb_block_row_channel), so the sub-tiles nt = 2s and 2s+1 together are eight consecutive channels.
 * A wave's NT channel sub-tiles are 16 * NT consecutive channels (GMM1: 8 * NT gate and the matching 8 * NT up columns).
 * `lds_rowmax` is [COL_GROUPS][tile_rows] floats of scratch for the row maxima of the workgroup's channel ranges (GMM1 only;
 * all of the tile's but where several workgroups share it);
 * ONE_MAX: [tile_rows], zero before, which takes the maximum over the channel ranges itself.
 */
template <int MODE, bool GMM1, int OUT_DT, int RG, int MTM, int NT, Shared SH, bool ONE_MAX = false, bool ROW_SCALES = MODE == MODE_W8A8,
          int COL_GROUPS = 16 / NT>
__device__ __forceinline__ void epilogue(const GemmParams &p, const TileCoord &tc, f32x4 (&accf)[MTM][NT],
                                         i32x4 (&acci)[MTM][NT], int row_begin, int row_end, int wm, int wn, int lane,
                                         float *lds_rowmax, int tile_rows, const float *es)
{
    /*
     * W8A8: `es` is this tile's scales in LDS, brought there by DMA while the tile was multiplied: [0, 256) the
     * channel scales of the tile's 256 weight rows (fp32, or 256 bf16 in the first 512 bytes), [256, 256 +
     * tile_rows) the per-token scales of its rows. A global load here is waited for with a count that also waits
     * for the next tile's slabs, which are already in flight (decode: 5-6 % of both GEMMs). ROW_SCALES: the per-token scales
     * are there. The W4A8 mode of the staged kernel, whose channel scales travel with the slabs and which has no registers to
     * spare, loads its per-token scales here, all of them before it uses the first.
     */
    float xs_loaded[MTM];
    if constexpr (MODE == MODE_W4A8 && !ROW_SCALES) {
#pragma unroll
        for (int mt = 0; mt < MTM; ++mt) {
            const int row = row_begin + (RG * mt + wm) * 16 + (lane & 15);
            xs_loaded[mt] = p.a_scale[row < p.max_rows ? row : p.max_rows - 1];
        }
    }
    const float *es_row = es + (MODE == MODE_W8A8 ? 256 : 0);
    const int frag_row = lane & 15;
    const int I = p.N / 2;
    const int q8 = (lane >> 4) * 8;
    if constexpr (!GMM1) {
        uint16_t *y = (uint16_t *)p.out;
        if (is_shared<SH>(p, tc.expert)) y = (uint16_t *)(SH == SHARED_ON_DEMAND ? launch_args()->shared_out : p.shared_out);
#pragma unroll
        for (int mt = 0; mt < MTM; ++mt) {
            const int row = row_begin + (RG * mt + wm) * 16 + frag_row;
            if (row >= row_end) continue;
            float xs = 1.0f;
            if (ROW_SCALES) xs = es_row[(RG * mt + wm) * 16 + frag_row];
            else if (MODE == MODE_W4A8) xs = xs_loaded[mt];
#pragma unroll
            for (int s = 0; s < NT / 2; ++s) {    /* sub-tiles 2s and 2s+1: eight consecutive channels from n */
                const int nl = wn * (16 * NT) + s * 32 + q8;       /* within the tile */
                const int n = tc.n_tile * BN + nl;
                float ws[8];
                if constexpr (MODE == MODE_W8A8) {
                    if (p.wscale_is_bf16) {
                        const u32x4 v = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint16_t *>(es) + nl);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            ws[2 * i] = zb_bf16_to_f32(v[i] & 0xffffu);
                            ws[2 * i + 1] = zb_bf16_to_f32(v[i] >> 16);
                        }
                    } else {
                        const float *wsp = es + nl;
                        const f32x4 v0 = *reinterpret_cast<const f32x4 *>(wsp), v1 = *reinterpret_cast<const f32x4 *>(wsp + 4);
#pragma unroll
                        for (int i = 0; i < 4; ++i) { ws[i] = v0[i]; ws[4 + i] = v1[i]; }
                    }
                }
                float d[8];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int nt = 2 * s + h;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (MODE == MODE_W8A8) d[4 * h + i] = ((float)acci[mt][nt][i] * ws[4 * h + i]) * xs;
                        else if constexpr (MODE == MODE_FP8) d[4 * h + i] = accf[mt][nt][i];
                        else d[4 * h + i] = accf[mt][nt][i] * xs;
                    }
                }
                *reinterpret_cast<u32x4 *>(y + (int64_t)row * p.N + n) =
                    u32x4{zb_pack2_half<OUT_DT>(d[0], d[1]), zb_pack2_half<OUT_DT>(d[2], d[3]),
                          zb_pack2_half<OUT_DT>(d[4], d[5]), zb_pack2_half<OUT_DT>(d[6], d[7])};
            }
        }
    } else {
        /* SwiGLU on gate sub-tile nt and up sub-tile nt + NT/2: columns j = n_tile*128 + 32*(t/2) + q8 + 4*(t%2) + i with t = wn*NT/2 + nt */
        constexpr int UP = NT / 2;
        const int group = wn % COL_GROUPS;         /* of this workgroup's */
        float sg[MTM][UP][4];
        float rmax[MTM];
#pragma unroll
        for (int mt = 0; mt < MTM; ++mt) {
            /*
             * A 16-row sub-tile past the tile's end holds nothing (the K loop left it out as well): its SwiGLU, which is
             * most of this epilogue's arithmetic (an exact exp and a division per value in the int modes), is skipped.
             * Wave-uniform. Few-row tiles spent 10 us here per tile before, one seventh of the decode kernel.
             */
            if ((RG * mt + wm) * 16 >= row_end - row_begin) continue;
            const int row = row_begin + (RG * mt + wm) * 16 + frag_row;
            float xs = 1.0f;
            if (ROW_SCALES) xs = es_row[(RG * mt + wm) * 16 + frag_row];
            else if (MODE == MODE_W4A8) xs = xs_loaded[mt];
            rmax[mt] = 0.0f;
#pragma unroll
            for (int nt = 0; nt < UP; ++nt) {
                const int t = wn * UP + nt, jl = (t >> 1) * 32 + q8 + (t & 1) * 4;       /* within the tile's 128 SwiGLU columns */
                float g[4], u[4];
                if constexpr (MODE == MODE_W8A8) {
                    const f32x4 wg = *reinterpret_cast<const f32x4 *>(es + jl);             /* gate scales, then up scales */
                    const f32x4 wu = *reinterpret_cast<const f32x4 *>(es + 128 + jl);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        g[i] = ((float)acci[mt][nt][i] * wg[i]) * xs;
                        u[i] = ((float)acci[mt][nt + UP][i] * wu[i]) * xs;
                    }
                } else if constexpr (MODE == MODE_FP8) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) { g[i] = accf[mt][nt][i]; u[i] = accf[mt][nt + UP][i]; }
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) { g[i] = accf[mt][nt][i] * xs; u[i] = accf[mt][nt + UP][i] * xs; }
                }
                /*
                 * The int modes' exact exp and division: a wave whose values are all of ordinary size takes the short form
                 * (any NaN, infinity or |g| > 80 in it: the general one).
                 */
                bool far = false;
                if constexpr (MODE != MODE_FP8) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) far |= !(fabsf(g[i]) <= kSiluNear);
                    far = __builtin_amdgcn_ballot_w64(far) != 0;
                }
                float left[4];
                if (MODE != MODE_FP8 && far) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) left[i] = g[i] / (1.0f + zb_expf(-g[i]));
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        /* fp8: e4m3 keeps 3 mantissa bits, the hardware exp2 / reciprocal approximations (1 ulp) are ample */
                        if constexpr (MODE == MODE_FP8)
                            left[i] = g[i] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g[i] * -1.44269504088896341f));
                        else left[i] = zb_silu_near(g[i]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float s = left[i] * u[i];
                    sg[mt][nt][i] = s;
                    rmax[mt] = fmaxf(rmax[mt], fabsf(s));
                }
                if constexpr (MODE != MODE_FP8) {
                    if (row < row_end)
                        *reinterpret_cast<f32x4 *>(p.sgl_ws + (int64_t)row * I + tc.n_tile * 128 + jl) =
                            f32x4{sg[mt][nt][0], sg[mt][nt][1], sg[mt][nt][2], sg[mt][nt][3]};
                }
            }
            /* the four lane groups (lane/16) hold different columns of the same row */
            rmax[mt] = zb_max_of_rows(rmax[mt]);
            if (lane < 16) {
                float *at = lds_rowmax + (RG * mt + wm) * 16 + lane;
                if (ONE_MAX) atomicMax(reinterpret_cast<uint32_t *>(at), __float_as_uint(rmax[mt]));      /* not negative, no NaN: ordered as integers */
                else at[group * tile_rows] = rmax[mt];
            }
        }
        lds_barrier();
        /*
         * One wave per row group raises the rows' maxima; the others, whose values are stored already, are done. (All of them
         * reduced the maxima and stored after the barrier before: first GEMM at 1024 rows per expert, 128 experts of 4096 x 3072,
         * W8A8 1781 -> 1715 us, W4A8 2199 -> 2158.)
         */
        if (MODE != MODE_FP8 && group != 0) return;
#pragma unroll
        for (int mt = 0; mt < MTM; ++mt) {
            const int lr = (RG * mt + wm) * 16 + frag_row;
            const int row = row_begin + lr;
            float amax_tile = lds_rowmax[lr];
#pragma unroll
            for (int g = 1; g < (ONE_MAX ? 1 : COL_GROUPS); ++g) amax_tile = fmaxf(amax_tile, lds_rowmax[g * tile_rows + lr]);
            if (row >= row_end) continue;
            if constexpr (MODE == MODE_FP8) {
                const float amax = fmaxf(amax_tile, 1e-4f);
                const float mult = 448.0f / amax;
                uint8_t *q2 = (uint8_t *)p.out;
                uint32_t q[UP];
#pragma unroll
                for (int nt = 0; nt < UP; ++nt)
                    q[nt] = pack4_e4m3(sg[mt][nt][0] * mult, sg[mt][nt][1] * mult, sg[mt][nt][2] * mult, sg[mt][nt][3] * mult);
                uint8_t *q2row = q2 + (int64_t)row * I + tc.n_tile * 128;
                if constexpr (UP == 1) {
                    *reinterpret_cast<uint32_t *>(q2row + (wn >> 1) * 32 + q8 + (wn & 1) * 4) = q[0];
                } else {
#pragma unroll
                    for (int s = 0; s < UP / 2; ++s)      /* sub-tiles 2s and 2s+1: eight consecutive columns */
                        *reinterpret_cast<u32x2 *>(q2row + wn * (8 * NT) + s * 32 + q8) = u32x2{q[2 * s], q[2 * s + 1]};
                }
                if (wn == 0 && lane < 16) p.out_scale[(int64_t)row * (I / 128) + tc.n_tile] = amax * (1.0f / 448.0f);
            } else {
                if (lane < 16) atomicMax(&p.rowmax[row], __float_as_uint(amax_tile));
            }
        }
    }
}

/* the pointer as scalar registers; a no-op where the compiler already knows it is wave-uniform */
template <typename T>
__device__ __forceinline__ const T *uniform_ptr(const T *p)
{
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const T *)(((uint64_t)hi << 32) | lo);
}

/*
 * One LDS-DMA transfer with the address split the way the instruction wants it: a wave-uniform 64-bit base in
 * scalar registers plus a 32-bit offset per lane, and the wave's LDS destination in M0. Spelled out because
 * the compiler otherwise keeps a 64-bit vector address per transfer alive across the whole K loop.
 *
 * The base often reaches the asm through v_readfirstlane. A scalar register written by a vector instruction must not
 * be read by a vector-memory instruction within five wait states, and the compiler, which inserts such waits for its
 * own instructions, does not look inside the asm text. So the text brings them along: the move to M0 is one,
 * `s_nop 3` the other four. (With no wait state at all the load used the register's old contents and the kernel
 * faulted; the two states of an `s_nop 0` ran clean, but the documented figure is five.)
 */
__device__ __forceinline__ void dma16_sv(const uint8_t *uniform_base, uint32_t lane_off, uint32_t lds_wave_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_wave_addr), "v"(lane_off), "s"(uniform_ptr(uniform_base))
                 : "memory", "m0");
}

/*
 * The same with the streaming hint, for weight slabs that no other workgroup asks for again (experts with a single
 * row tile: each slab is read once). Measured on the few-row shape: the decode layer 5 % faster, the weight stream of
 * a 128-token fp8 layer 5.3 -> 5.9 TB/s; on slabs that several row tiles share it costs 3-9 %, and decided tile by
 * tile inside the kernel it cost registers, so the launcher decides per launch (WSTREAM).
 */
__device__ __forceinline__ void dma16_sv_nt(const uint8_t *uniform_base, uint32_t lane_off, uint32_t lds_wave_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(lds_wave_addr), "v"(lane_off), "s"(uniform_ptr(uniform_base))
                 : "memory", "m0");
}

__device__ __forceinline__ void dma4_sv(const float *uniform_base, uint32_t lane_off_bytes, uint32_t lds_wave_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(lds_wave_addr), "v"(lane_off_bytes), "s"(uniform_ptr(uniform_base))
                 : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_addr(const void *p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
}


/* wait until at most N of this wave's vector-memory operations are outstanding (they complete in order) */
template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

} // namespace

#endif /* ZBAL_GEMM_TILE_H_ */
