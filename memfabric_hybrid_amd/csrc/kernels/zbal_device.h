/*
 * Device-side helpers shared by the gfx950 kernels: scalar format
 * conversions, the fixed expf used by the SwiGLU epilogue, wave64 reductions
 * and the launch-error plumbing of the C ABI.
 *
 * The kernels are compiled with -ffp-contract=off: a product followed by a
 * sum rounds twice unless written as __builtin_fmaf().
 */
#ifndef ZBAL_DEVICE_H_
#define ZBAL_DEVICE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#define ZBALHIP_OK 0
#define ZBALHIP_INVALID (-2)
#define ZBALHIP_RT_ERROR (-11)

/* zbal_datatype_t values used by the kernels */
#define ZDT_INT8 0
#define ZDT_INT16 1
#define ZDT_INT32 2
#define ZDT_INT64 3
#define ZDT_FP16 6
#define ZDT_FP32 7
#define ZDT_BF16 8

#define ZBAL_WAVE 64

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int32_t i32x2 __attribute__((ext_vector_type(2)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

/* thread-local last-error text of the library (zbal_get_last_error_msg), for launchers that refuse a call */
void zbalhip_set_last_error(const char *text);

static inline int32_t zbalhip_check_launch()
{
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? ZBALHIP_OK : ZBALHIP_RT_ERROR;
}

/*
 * kernel<<<grid, block, lds, st>>>(args...) without its detour: the compiler's form stacks the launch shape for a stub to take off again
 * before it calls hipLaunchKernel. Host time of a launch 3.39 -> 3.24 us; a low-latency dispatch and its combine, which are bound by it,
 * 11.2 -> 10.9 (7 tokens bf16), a reduce-scatter of 8 x 100003 fp16 4.05 -> 3.92. For the launches that small calls make.
 */
template <typename T> struct ZbSame { using type = T; };
template <typename... P>
static inline void zb_launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st, typename ZbSame<P>::type... args)
{
    const void *at[] = {static_cast<const void *>(&args)...};
    (void)hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, const_cast<void **>(at), lds, st);
}

/* ---- scalar formats ------------------------------------------------------ */

__device__ __forceinline__ float zb_bf16_to_f32(uint32_t h) { return __uint_as_float(h << 16); }

/* two floats -> two bf16 in one dword: v_cvt_pk_bf16_f32, round to nearest even, NaN stays a quiet NaN */
__device__ __forceinline__ uint32_t zb_pack2_bf16(float lo, float hi)
{
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

__device__ __forceinline__ uint32_t zb_f32_to_bf16(float f) { return zb_pack2_bf16(f, 0.0f) & 0xffffu; }

__device__ __forceinline__ float zb_fp16_to_f32(uint32_t h)
{
    _Float16 v;
    uint16_t s = (uint16_t)h;
    __builtin_memcpy(&v, &s, 2);
    return (float)v;
}

__device__ __forceinline__ uint32_t zb_f32_to_fp16(float f)
{
    /*
     * The empty asm keeps the compiler from folding a preceding fp32 multiply into v_fma_mixlo_f16, which
     * rounds the exact product straight to fp16; the result must be the fp32-rounded product rounded again.
     */
    asm volatile("" : "+v"(f));
    _Float16 v = (_Float16)f; /* v_cvt_f16_f32: round to nearest even */
    uint16_t s;
    __builtin_memcpy(&s, &v, 2);
    return s;
}

template <int DT> __device__ __forceinline__ float zb_half_to_f32(uint32_t h)
{
    if constexpr (DT == ZDT_FP16) return zb_fp16_to_f32(h);
    else return zb_bf16_to_f32(h);
}

template <int DT> __device__ __forceinline__ uint32_t zb_f32_to_half(float f)
{
    if constexpr (DT == ZDT_FP16) return zb_f32_to_fp16(f);
    else return zb_f32_to_bf16(f);
}

/* two values rounded to DT, `lo` in the low half of the dword */
template <int DT> __device__ __forceinline__ uint32_t zb_pack2_half(float lo, float hi)
{
    if constexpr (DT == ZDT_FP16) return zb_f32_to_fp16(lo) | (zb_f32_to_fp16(hi) << 16);
    else return zb_pack2_bf16(lo, hi);
}

/* two floats -> two e4m3 codes in the low 16 bits (v_cvt_pk_fp8_f32, OCP format on gfx950); inputs pre-clamped */
__device__ __forceinline__ uint32_t zb_cvt_pk_e4m3(float a, float b)
{
    a = fminf(fmaxf(a, -448.0f), 448.0f);
    b = fminf(fmaxf(b, -448.0f), 448.0f);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false) & 0xffffu;
}

/*
 * Four floats -> four int8 in a dword: clamped to [-128, 127], rounded to nearest even by the addition of 1.5 * 2^23, which leaves the
 * integer in the low bits. A NaN gives -128 (the median of a NaN and two numbers is the smaller number).
 */
__device__ __forceinline__ uint32_t zb_pack4_i8(float a, float b, float c, float d)
{
    constexpr float MAGIC = 12582912.0f;
    const uint32_t ai = __float_as_uint(__builtin_amdgcn_fmed3f(a, -128.0f, 127.0f) + MAGIC), bi = __float_as_uint(__builtin_amdgcn_fmed3f(b, -128.0f, 127.0f) + MAGIC);
    const uint32_t ci = __float_as_uint(__builtin_amdgcn_fmed3f(c, -128.0f, 127.0f) + MAGIC), di = __float_as_uint(__builtin_amdgcn_fmed3f(d, -128.0f, 127.0f) + MAGIC);
    const uint32_t ab = __builtin_amdgcn_perm(bi, ai, 0x0c0c0400), cd = __builtin_amdgcn_perm(di, ci, 0x04000c0c);
    return ab | cd;
}

/*
 * exp() of the SwiGLU epilogue: Cody-Waite reduction by ln2, a degree-6
 * polynomial in fmaf form and scaling by two exact powers of two. The same
 * operation sequence is what the CPU oracle evaluates, so both sides agree
 * bit for bit (the hardware v_exp_f32 is an approximation and would not).
 */
__device__ __forceinline__ float zb_expf(float x)
{
    if (!(x == x)) return x;
    if (x > 88.72284f) return __builtin_inff();
    if (x < -103.97208f) return 0.0f;
    float n = __builtin_rintf(x * 1.44269504088896341f);
    float r = __builtin_fmaf(n, -0.693145751953125f, x);
    r = __builtin_fmaf(n, -1.42860682030941723e-06f, r);
    float p = 1.3888889e-03f;
    p = __builtin_fmaf(p, r, 8.3333333e-03f);
    p = __builtin_fmaf(p, r, 4.1666668e-02f);
    p = __builtin_fmaf(p, r, 1.6666667e-01f);
    p = __builtin_fmaf(p, r, 0.5f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_fmaf(p, r, 1.0f);
    int ni = (int)n;
    int n1 = ni / 2, n2 = ni - n1;
    float s1 = __uint_as_float((uint32_t)(n1 + 127) << 23);
    float s2 = __uint_as_float((uint32_t)(n2 + 127) << 23);
    return (p * s1) * s2;
}

/*
 * g / (1 + zb_expf(-g)) for |g| <= 80, bit for bit (tests/test_gpu_gemm_shapes.py compares every such float; only -0 comes out as +0): the
 * same reduction and polynomial, where exp(-g) is a normal number, so one addition to the exponent scales it, rounding to
 * an integer is adding and subtracting 1.5 * 2^23, and the quotient needs neither range scaling nor a second correction.
 * 17 vector instructions without a branch, so the four values of a lane overlap; the general form takes about 50, and its
 * three range checks are branches that run one value after the other. Layers: W4A8 16384 tokens over 128 experts of
 * 4096 x 3072 3.60 -> 3.53 ms, W8A8 8192 tokens 1.65 -> 1.61; W8A8 4096 tokens over 32 of 7168 x 4096 1.61 -> 1.59.
 */
constexpr float kSiluNear = 80.0f;
__device__ __forceinline__ float zb_silu_near(float g)
{
    constexpr float MAGIC = 12582912.0f;
    const float t = g * -1.44269504088896341f + MAGIC;
    const float n = t - MAGIC;
    float r = __builtin_fmaf(n, -0.693145751953125f, -g);
    r = __builtin_fmaf(n, -1.42860682030941723e-06f, r);
    float p = 1.3888889e-03f;
    p = __builtin_fmaf(p, r, 8.3333333e-03f);
    p = __builtin_fmaf(p, r, 4.1666668e-02f);
    p = __builtin_fmaf(p, r, 1.6666667e-01f);
    p = __builtin_fmaf(p, r, 0.5f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_fmaf(p, r, 1.0f);
    const float d = 1.0f + __uint_as_float((__float_as_uint(t) << 23) + __float_as_uint(p));
    const float y = __builtin_amdgcn_rcpf(d);
    const float q = g * y;
    return __builtin_fmaf(__builtin_fmaf(-d, q, g), y, q);
}

/*
 * Expert ids, read where the caller has them: an int32 array (stride 1) or an int64 one (stride 2), so that int64 ids
 * need no converting launch in front of the kernel. IDS_FULL: an int64 id outside of int32 is no expert (-1);
 * otherwise its low word counts, which is what converting the array first would have left.
 */
enum { IDS_I32 = 0, IDS_LOW = 1, IDS_FULL = 2 };
struct ExpertIds {
    const int32_t *p;
    int kind;
    __device__ __forceinline__ int stride() const { return kind == IDS_I32 ? 1 : 2; }
    __device__ __forceinline__ int32_t of_words(uint32_t lo, uint32_t hi) const { return kind == IDS_FULL && hi != 0u ? -1 : (int32_t)lo; }
    __device__ __forceinline__ int32_t operator[](int64_t i) const
    {
        if (kind == IDS_I32) return p[i];
        const u32x2 w = reinterpret_cast<const u32x2 *>(p)[i];
        return of_words(w[0], w[1]);
    }
    /* ids i .. i + 3, one or two loads that need no more than the array's alignment */
    __device__ __forceinline__ i32x4 four(int64_t i) const
    {
        typedef u32x4 __attribute__((aligned(4))) words_t;
        if (kind == IDS_I32) return __builtin_bit_cast(i32x4, (u32x4)*reinterpret_cast<const words_t *>(p + i));
        const u32x4 a = *reinterpret_cast<const words_t *>(p + 2 * i), b = *reinterpret_cast<const words_t *>(p + 2 * i + 4);
        return i32x4{of_words(a[0], a[1]), of_words(a[2], a[3]), of_words(b[0], b[1]), of_words(b[2], b[3])};
    }
};
inline ExpertIds expert_ids(const void *p, bool is_i64, bool full = false)
{
    return {(const int32_t *)p, !is_i64 ? IDS_I32 : (full ? IDS_FULL : IDS_LOW)};
}

/* ---- wave64 reductions ------------------------------------------------------ */

__device__ __forceinline__ float zb_wave_max(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, ZBAL_WAVE));
    return v;
}

/*
 * Wave-wide reductions on the data-parallel-primitive path (no LDS round trips: six dependent vector instructions
 * instead of six ds_bpermute latencies). Lanes swap within quads, mirror within 8 and 16, then rows 1 and 3 take
 * the totals of rows 0 and 2 and the upper half takes lane 31's; lane 63 ends with the result, which is broadcast.
 */
template <bool IS_MAX> __device__ __forceinline__ float zb_wave_reduce_dpp(float x)
{
    const int ident = IS_MAX ? (int)0xff800000u : 0;       /* -inf or +0 for the lanes a step does not write */
    auto step = [&](auto ctrl_tag, auto mask_tag) __attribute__((always_inline)) {
        constexpr int CTRL = decltype(ctrl_tag)::value, MASK = decltype(mask_tag)::value;
        const float o = __int_as_float(__builtin_amdgcn_update_dpp(ident, __float_as_int(x), CTRL, MASK, 0xf, false));
        x = IS_MAX ? fmaxf(x, o) : x + o;
    };
    step(std::integral_constant<int, 0xB1>{}, std::integral_constant<int, 0xf>{});     /* quad_perm [1,0,3,2] */
    step(std::integral_constant<int, 0x4E>{}, std::integral_constant<int, 0xf>{});     /* quad_perm [2,3,0,1] */
    step(std::integral_constant<int, 0x141>{}, std::integral_constant<int, 0xf>{});    /* row_half_mirror */
    step(std::integral_constant<int, 0x140>{}, std::integral_constant<int, 0xf>{});    /* row_mirror */
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});    /* row_bcast:15 into rows 1 and 3 */
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});    /* row_bcast:31 into rows 2 and 3 */
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

/* sum over the wave, in every lane */
__device__ __forceinline__ int32_t zb_wave_sum_dpp(int32_t x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, false);     /* the steps of zb_wave_reduce_dpp */
    x += __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return __builtin_amdgcn_readlane(x, 63);
}

/* inclusive sum over the lanes up to this one */
__device__ __forceinline__ int32_t zb_wave_scan_dpp(int32_t x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);     /* row_shr:1, 2, 4, 8 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);     /* row_bcast:15 into rows 1 and 3 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);     /* row_bcast:31 into rows 2 and 3 */
    return x;
}

/* max over the lanes l, l ^ 16, l ^ 32 and l ^ 48, in all of them: the swaps leave every lane with both values of a pair */
__device__ __forceinline__ float zb_max_of_rows(float v)
{
    u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

/* max over groups of 2^LOG2 consecutive lanes */
template <int LOG2> __device__ __forceinline__ float zb_group_max(float v)
{
#pragma unroll
    for (int off = (1 << LOG2) >> 1; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, ZBAL_WAVE));
    return v;
}

/* block-wide max through LDS; `red` holds one float per wave; all threads receive the result */
__device__ __forceinline__ float zb_block_max(float v, float *red)
{
    v = zb_wave_max(v);
    const int lane = threadIdx.x & (ZBAL_WAVE - 1), wave = threadIdx.x / ZBAL_WAVE;
    const int nwaves = (blockDim.x + ZBAL_WAVE - 1) / ZBAL_WAVE;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float r = red[0];
    for (int i = 1; i < nwaves; ++i) r = fmaxf(r, red[i]);
    return r;
}

/*
 * Pre-packed weight blocks: which channel of a 128-channel block sits in block row r. Rows 16t .. 16t+15 feed one
 * MFMA of the grouped GEMM and rows 4q .. 4q+3 of it come out in the lanes 16q .. 16q+15; the permutation (within
 * groups of 32 rows) gives those lanes channels 8q .. 8q+3 of the group from the even operand t and 8q+4 .. 8q+7
 * from the odd one, eight consecutive channels per lane.
 */
__host__ __device__ __forceinline__ constexpr int zb_block_row_channel(int r)
{
    return (r & ~31) | (((r & 15) >> 2) << 3) | (((r >> 4) & 1) << 2) | (r & 3);
}

#endif /* ZBAL_DEVICE_H_ */
