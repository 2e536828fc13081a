/*
 * N-buffer reduction: out[j] = op over p of in[p][j], the local compute under
 * reduce-scatter / all-reduce. A single pass: every lane streams one 16-byte
 * vector from each of the N inputs (N independent loads in flight), folds
 * them in buffer order (floating types in fp32) and writes one 16-byte
 * vector, so HBM traffic is (N + 1) x the slice size — the reference's
 * copy-then-atomic-accumulate scheme re-reads and re-writes the output slice
 * once per peer.
 */
#include <string.h>

#include "zbal_device.h"
#include "zbal_hip_kernels.h"

namespace {

struct ReducePtrs {
    const void *p[ZBALHIP_MAX_REDUCE_PEERS];
    unsigned long long *trace;      /* device trace ring or null */
    uint32_t trace_points;
    uint32_t trace_frame;
};

/*
 * One record into this workgroup's block of the ring (reference ZBAL_PROF_RECORD, zbal_kernel_trace.h:22-42):
 * bump the block's index word, then write the record there. Called by one lane of workgroups below
 * ZBALHIP_TRACE_UNITS; the ring is host memory, so the stores are made visible to the host with a system fence.
 */
__device__ __forceinline__ void trace_record(const ReducePtrs &in, bool end)
{
    if (in.trace == nullptr || in.trace_frame == 0 || blockIdx.x >= ZBALHIP_TRACE_UNITS || threadIdx.x != 0) return;
    unsigned long long *blk = in.trace + (uint64_t)blockIdx.x * in.trace_points;
    unsigned long long idx = blk[ZBALHIP_TRACE_IDX_OFF] + 1;
    if (idx <= ZBALHIP_TRACE_REC_OFF) idx = ZBALHIP_TRACE_REC_OFF;
    if (idx >= in.trace_points) return;
    const unsigned long long ts = (unsigned long long)wall_clock64() & ((1ull << ZBALHIP_TRACE_FRAME_SHIFT) - 1);
    blk[idx] = ((unsigned long long)in.trace_frame << ZBALHIP_TRACE_FRAME_SHIFT) | ((end ? 1ull : 0ull) << ZBALHIP_TRACE_BE_SHIFT) | ts;
    blk[ZBALHIP_TRACE_IDX_OFF] = idx;
    __threadfence_system();
}

enum { OP_PROD = 0, OP_SUM = 1, OP_MAX = 2, OP_MIN = 3 };

template <int OP, typename A> __device__ __forceinline__ A fold(A a, A b)
{
    if constexpr (OP == OP_PROD) return a * b;
    else if constexpr (OP == OP_SUM) return a + b;
    else if constexpr (OP == OP_MAX) return a > b ? a : b;
    else return a < b ? a : b;
}

/* Element traits: how many per 16 bytes, and how to unpack to / pack from the accumulation type. */
template <int DT> struct Elem;
template <> struct Elem<ZDT_FP32> { typedef float acc_t; static constexpr int per = 4; };
template <> struct Elem<ZDT_BF16> { typedef float acc_t; static constexpr int per = 8; };
template <> struct Elem<ZDT_FP16> { typedef float acc_t; static constexpr int per = 8; };
template <> struct Elem<ZDT_INT32> { typedef uint32_t acc_t; static constexpr int per = 4; };
template <> struct Elem<ZDT_INT16> { typedef int32_t acc_t; static constexpr int per = 8; };
template <> struct Elem<ZDT_INT8> { typedef int32_t acc_t; static constexpr int per = 16; };
template <> struct Elem<ZDT_INT64> { typedef int64_t acc_t; static constexpr int per = 2; };

template <int DT> __device__ __forceinline__ void unpack(const u32x4 &v, typename Elem<DT>::acc_t *o)
{
    if constexpr (DT == ZDT_FP32) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = __uint_as_float(v[i]);
    } else if constexpr (DT == ZDT_BF16 || DT == ZDT_FP16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[2 * i] = zb_half_to_f32<DT>(v[i] & 0xffffu);
            o[2 * i + 1] = zb_half_to_f32<DT>(v[i] >> 16);
        }
    } else if constexpr (DT == ZDT_INT32) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = v[i];
    } else if constexpr (DT == ZDT_INT16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[2 * i] = (int32_t)(int16_t)(v[i] & 0xffffu);
            o[2 * i + 1] = (int32_t)(int16_t)(v[i] >> 16);
        }
    } else if constexpr (DT == ZDT_INT8) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) o[4 * i + j] = (int32_t)(int8_t)((v[i] >> (8 * j)) & 0xffu);
    } else {
        o[0] = (int64_t)(((uint64_t)v[1] << 32) | v[0]);
        o[1] = (int64_t)(((uint64_t)v[3] << 32) | v[2]);
    }
}

template <int DT> __device__ __forceinline__ u32x4 pack(const typename Elem<DT>::acc_t *a)
{
    u32x4 v;
    if constexpr (DT == ZDT_FP32) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = __float_as_uint(a[i]);
    } else if constexpr (DT == ZDT_BF16 || DT == ZDT_FP16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = zb_pack2_half<DT>(a[2 * i], a[2 * i + 1]);
    } else if constexpr (DT == ZDT_INT32) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = a[i];
    } else if constexpr (DT == ZDT_INT16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = ((uint32_t)a[2 * i] & 0xffffu) | ((uint32_t)a[2 * i + 1] << 16);
    } else if constexpr (DT == ZDT_INT8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t w = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) w |= ((uint32_t)a[4 * i + j] & 0xffu) << (8 * j);
            v[i] = w;
        }
    } else {
        v[0] = (uint32_t)(uint64_t)a[0]; v[1] = (uint32_t)((uint64_t)a[0] >> 32);
        v[2] = (uint32_t)(uint64_t)a[1]; v[3] = (uint32_t)((uint64_t)a[1] >> 32);
    }
    return v;
}

/* integer sum / product wrap modulo 2^bits; done in unsigned arithmetic */
template <int DT, int OP>
__device__ __forceinline__ typename Elem<DT>::acc_t fold_elem(typename Elem<DT>::acc_t a, typename Elem<DT>::acc_t b)
{
    typedef typename Elem<DT>::acc_t A;
    if constexpr (DT == ZDT_INT64 && (OP == OP_SUM || OP == OP_PROD)) {
        return (A)fold<OP, uint64_t>((uint64_t)a, (uint64_t)b);
    } else if constexpr (DT == ZDT_INT32 && (OP == OP_MAX || OP == OP_MIN)) {
        return (A)fold<OP, int32_t>((int32_t)a, (int32_t)b);
    } else if constexpr ((DT == ZDT_INT16 || DT == ZDT_INT8) && (OP == OP_SUM || OP == OP_PROD)) {
        /* keep intermediate values inside the element width so that wrapping matches the element type */
        const uint32_t r = fold<OP, uint32_t>((uint32_t)a, (uint32_t)b);
        return DT == ZDT_INT16 ? (A)(int16_t)r : (A)(int8_t)r;
    } else {
        return fold<OP, A>(a, b);
    }
}

/* one element of a buffer, as the fold wants it, and back */
template <int DT> __device__ __forceinline__ typename Elem<DT>::acc_t load_elem(const void *p, int64_t j)
{
    typedef typename Elem<DT>::acc_t A;
    if constexpr (DT == ZDT_FP32) return ((const float *)p)[j];
    else if constexpr (DT == ZDT_INT32) return (A)((const uint32_t *)p)[j];
    else if constexpr (DT == ZDT_INT64) return ((const int64_t *)p)[j];
    else if constexpr (DT == ZDT_INT8) return (A)((const int8_t *)p)[j];
    else if constexpr (DT == ZDT_INT16) return (A)((const int16_t *)p)[j];
    else return zb_half_to_f32<DT>(((const uint16_t *)p)[j]);
}
template <int DT> __device__ __forceinline__ void store_elem(void *out, int64_t j, typename Elem<DT>::acc_t v)
{
    if constexpr (DT == ZDT_FP32) ((float *)out)[j] = v;
    else if constexpr (DT == ZDT_INT32) ((uint32_t *)out)[j] = (uint32_t)v;
    else if constexpr (DT == ZDT_INT64) ((int64_t *)out)[j] = v;
    else if constexpr (DT == ZDT_INT8) ((int8_t *)out)[j] = (int8_t)v;
    else if constexpr (DT == ZDT_INT16) ((int16_t *)out)[j] = (int16_t)v;
    else ((uint16_t *)out)[j] = (uint16_t)zb_f32_to_half<DT>(v);
}

/* [0, head) element by element, then nvec 16-byte vectors of the output, then the rest up to count element by element */
struct ReduceSpan {
    int64_t count, nvec;
    int head;
    int chunk;                      /* consecutive blocks per XCD and turn, 0: blocks in order */
};

constexpr int kMaxReduceThreads = 1024;
typedef u32x4 __attribute__((aligned(1))) u32x4_any_offset;      /* global loads may sit at any byte */

/*
 * The output's vectors are aligned; ANY_OFFSET: the inputs' need not be, and are read with vector loads that are only
 * aligned to their elements (reduce-scatter slices of odd length: 2 x 10^8 halves 287 us element by element, as this was
 * done before, 148 so; loads from the dword below, shifted into place, are slower again, 1 ms, for the registers they
 * take over 16 inputs). The few elements around the vectors belong to the last block, so there is one launch whatever
 * the offsets and the length.
 */
template <int DT, int OP, int N, bool ANY_OFFSET>
__global__ void __launch_bounds__(kMaxReduceThreads)
reduce_kernel(ReducePtrs in, int n_in, ReduceSpan sp, void *__restrict__ out_base)
{
    typedef typename Elem<DT>::acc_t A;
    constexpr int PER = Elem<DT>::per, ESZ = 16 / PER;
    const int64_t skip = (int64_t)sp.head * ESZ;
    typedef std::conditional_t<ANY_OFFSET, u32x4_any_offset, u32x4> vec_in;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    u32x4 *out = reinterpret_cast<u32x4 *>((char *)out_base + skip);
    int64_t b = blockIdx.x;
    if (sp.chunk) {                 /* gridDim.x is a multiple of 8 * chunk then */
        const int64_t turn = b / (8 * sp.chunk), r = b - turn * (8 * sp.chunk);
        b = turn * (8 * sp.chunk) + (r & 7) * sp.chunk + (r >> 3);
    }
    trace_record(in, false);
    for (int64_t i = b * blockDim.x + threadIdx.x; i < sp.nvec; i += stride) {
        u32x4 v[N];
#pragma unroll
        for (int p = 0; p < N; ++p)
            if (N != ZBALHIP_MAX_REDUCE_PEERS || p < n_in)
                v[p] = __builtin_nontemporal_load(reinterpret_cast<const vec_in *>((const char *)in.p[p] + skip) + i);
        A acc[PER], cur[PER];
        unpack<DT>(v[0], acc);
#pragma unroll
        for (int p = 1; p < N; ++p) {
            if (N != ZBALHIP_MAX_REDUCE_PEERS || p < n_in) {
                unpack<DT>(v[p], cur);
#pragma unroll
                for (int e = 0; e < PER; ++e) acc[e] = fold_elem<DT, OP>(acc[e], cur[e]);
            }
        }
        out[i] = pack<DT>(acc);      /* inputs are streamed (non-temporal loads); the plain store measured 5% faster than a non-temporal one */
    }
    if (blockIdx.x == gridDim.x - 1) {
        const int64_t rest = sp.head + sp.nvec * PER, n = sp.head + (sp.count - rest);
        for (int64_t k = threadIdx.x; k < n; k += blockDim.x) {
            const int64_t j = k < sp.head ? k : rest + (k - sp.head);
            A acc = load_elem<DT>(in.p[0], j);
            for (int p = 1; p < n_in; ++p) acc = fold_elem<DT, OP>(acc, load_elem<DT>(in.p[p], j));
            store_elem<DT>(out_base, j, acc);
        }
    }
    trace_record(in, true);
}

template <int DT, int OP>
int32_t launch_reduce(const ReducePtrs &ptrs, int n_in, int64_t count, void *out, bool same_offset, hipStream_t st)
{
    constexpr int PER = Elem<DT>::per, ESZ = 16 / PER;
    ReduceSpan sp = {};
    const unsigned mis = (unsigned)((uintptr_t)out & 15u);
    const int64_t head = mis ? (16 - mis) / ESZ : 0;
    sp.count = count;
    sp.head = (int)(head < count ? head : count);
    sp.nvec = (count - sp.head) / PER;
    /*
     * One 16-byte vector per thread: short-lived workgroups stream faster (6.2 TB/s for 8 x 256 MiB) than a capped grid
     * with a grid-stride loop (5.3 TB/s); the loop only serves huge counts. From 8 Mi vectors on (128 MiB of output):
     * workgroups of 1024, and each XCD takes 512 KiB in a row of every buffer, so that it needs fewer pages at a time
     * (three sets of 8 x 256 MiB in turn, more than the address caches hold: 423 -> 408 us; 256 threads in order 423,
     * 1024 in order 416, 256 KiB and 2 MiB in a row 430).
     */
    const bool big = sp.nvec >= (8ll << 20);
    const int threads = big ? kMaxReduceThreads : 256;
    int64_t blocks = (sp.nvec + threads - 1) / threads;
    const int64_t cap = 1 << 22;
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    if (big) {
        sp.chunk = 32;
        blocks = (blocks + 255) / 256 * 256;
    }
#define ZB_REDUCE(N, ANY) zb_launch(reduce_kernel<DT, OP, N, ANY>, (unsigned)blocks, threads, 0, st, ptrs, n_in, sp, out)
    if (!same_offset) ZB_REDUCE(ZBALHIP_MAX_REDUCE_PEERS, true);
    else if (n_in == 1) ZB_REDUCE(1, false);
    else if (n_in == 2) ZB_REDUCE(2, false);
    else if (n_in == 4) ZB_REDUCE(4, false);
    else if (n_in == 8) ZB_REDUCE(8, false);
    else ZB_REDUCE(ZBALHIP_MAX_REDUCE_PEERS, false);
#undef ZB_REDUCE
    return zbalhip_check_launch();
}

template <int DT> int32_t dispatch_op(const ReducePtrs &ptrs, int n_in, int64_t count, int op, void *out, hipStream_t st)
{
    /* every base must hold whole elements; where it sits relative to a 16-byte boundary picks the path */
    constexpr int ESZ = 16 / Elem<DT>::per;
    const unsigned mis = (unsigned)((uintptr_t)out & 15u);
    if (mis % ESZ) return ZBALHIP_INVALID;
    bool same = true;
    for (int p = 0; p < n_in; ++p) {
        const unsigned m = (unsigned)((uintptr_t)ptrs.p[p] & 15u);
        if (m % ESZ) return ZBALHIP_INVALID;
        same = same && m == mis;
    }
    switch (op) {
        case OP_PROD: return launch_reduce<DT, OP_PROD>(ptrs, n_in, count, out, same, st);
        case OP_SUM: return launch_reduce<DT, OP_SUM>(ptrs, n_in, count, out, same, st);
        case OP_MAX: return launch_reduce<DT, OP_MAX>(ptrs, n_in, count, out, same, st);
        case OP_MIN: return launch_reduce<DT, OP_MIN>(ptrs, n_in, count, out, same, st);
        default: return ZBALHIP_INVALID;
    }
}

} // namespace

extern "C" int32_t zbalhip_trace_alloc(int64_t points, uint64_t **host_ring, uint64_t **device_ring)
{
    if (points <= ZBALHIP_TRACE_REC_OFF || points > (1 << 24) || !host_ring || !device_ring) return ZBALHIP_INVALID;
    const size_t bytes = (size_t)points * ZBALHIP_TRACE_UNITS * sizeof(uint64_t);
    void *h = nullptr, *d = nullptr;
    if (hipHostMalloc(&h, bytes, hipHostMallocMapped) != hipSuccess) return ZBALHIP_RT_ERROR;
    memset(h, 0, bytes);
    if (hipHostGetDevicePointer(&d, h, 0) != hipSuccess) {
        (void)hipHostFree(h);
        return ZBALHIP_RT_ERROR;
    }
    *host_ring = (uint64_t *)h;
    *device_ring = (uint64_t *)d;
    return ZBALHIP_OK;
}

extern "C" int32_t zbalhip_trace_sync(void) { return hipDeviceSynchronize() == hipSuccess ? ZBALHIP_OK : ZBALHIP_RT_ERROR; }

extern "C" int32_t zbalhip_trace_free(uint64_t *host_ring)
{
    if (!host_ring) return ZBALHIP_INVALID;
    if (hipDeviceSynchronize() != hipSuccess) return ZBALHIP_RT_ERROR;
    return hipHostFree(host_ring) == hipSuccess ? ZBALHIP_OK : ZBALHIP_RT_ERROR;
}

extern "C" int32_t zbalhip_reduce(const void *const *in, int32_t n_in, int64_t count, int32_t dtype, int32_t op,
                                  void *out, int32_t trace_frame, uint64_t *trace_ring, int64_t trace_points, void *stream)
{
    if (!in || !out || n_in <= 0 || n_in > ZBALHIP_MAX_REDUCE_PEERS || count <= 0) return ZBALHIP_INVALID;
    if (trace_frame < 0 || trace_frame >= (1 << (ZBALHIP_TRACE_BE_SHIFT - ZBALHIP_TRACE_FRAME_SHIFT))) return ZBALHIP_INVALID;
    if (trace_ring != nullptr && (trace_points <= ZBALHIP_TRACE_REC_OFF || trace_points > (1 << 24))) return ZBALHIP_INVALID;
    ReducePtrs ptrs;
    for (int p = 0; p < ZBALHIP_MAX_REDUCE_PEERS; ++p) ptrs.p[p] = p < n_in ? in[p] : nullptr;
    ptrs.trace = trace_frame ? (unsigned long long *)trace_ring : nullptr;
    ptrs.trace_points = trace_ring ? (uint32_t)trace_points : 0;
    ptrs.trace_frame = (uint32_t)trace_frame;
    for (int p = 0; p < n_in; ++p)
        if (!in[p]) return ZBALHIP_INVALID;
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case ZDT_INT8: return dispatch_op<ZDT_INT8>(ptrs, n_in, count, op, out, st);
        case ZDT_INT16: return dispatch_op<ZDT_INT16>(ptrs, n_in, count, op, out, st);
        case ZDT_INT32: return dispatch_op<ZDT_INT32>(ptrs, n_in, count, op, out, st);
        case ZDT_INT64: return dispatch_op<ZDT_INT64>(ptrs, n_in, count, op, out, st);
        case ZDT_FP16: return dispatch_op<ZDT_FP16>(ptrs, n_in, count, op, out, st);
        case ZDT_BF16: return dispatch_op<ZDT_BF16>(ptrs, n_in, count, op, out, st);
        case ZDT_FP32: return dispatch_op<ZDT_FP32>(ptrs, n_in, count, op, out, st);
        default: return ZBALHIP_INVALID;
    }
}
