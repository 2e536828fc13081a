/*
 * Weighted combine (gather-reduce): out[t,:] = round(sum_k w[t,k] * y[row(t,k),:]).
 *
 * One workgroup per output token (small batches: per piece of a token's row,
 * so that every CU has work). Each lane owns 16-byte chunks (8 elements)
 * of the row; for a chunk it issues the loads of up to eight picks back to
 * back so that eight 16-byte requests per lane are in flight, then folds
 * them into fp32 accumulators in pick order with a separately rounded
 * multiply and add, and stores one rounded 16-byte chunk. HBM traffic is
 * K row reads plus one row write per token.
 */
#include "zbal_device.h"
#include "zbal_hip_kernels.h"

namespace {

constexpr int kThreads = 256;
constexpr int kMaxTopk = 32;
constexpr int kGroup = 8;

/*
 * Where the rows are read from: expert e's rows sit in the window of rank e / e_loc, at the slot
 * base[e * ranks + my_rank] that this rank's dispatch wrote them to (reference zbal_kernel_combine_normal.h:437-494).
 * One GPU: the windows are local allocations; over xGMI they would be mapped peer memory. rows_cap: rows per window.
 */
struct PeerSource {
    const uint16_t *y[ZBALHIP_MAX_REDUCE_PEERS];
    int ranks, my_rank, e_loc;
    int64_t rows_cap;
};

/*
 * U chunks per lane and pass. Every wave resolves the token's picks itself, one lane per pick, and takes them from
 * there as scalars: no LDS, no barrier between the loads of a pick's address and the row loads. BASES: one rank of at most 64 *
 * BASES experts, whose bases are asked for one per lane beside the picks and taken from the lane that has them, instead of by a
 * load that depends on the pick (0: such a load). The kernel alone, hidden 7168, 32 experts, rows in the cache / from memory: 7 tokens
 * 4.0 -> 3.8 / 4.8 -> 4.8 us, 128 tokens 4.5 -> 4.2 / 6.4 -> 5.8, 4096 tokens 91.3 -> 90.4 / 93.4 -> 92.2.
 */
template <int DT, int U, int BASES>
__global__ void __launch_bounds__(kThreads)
combine_kernel(PeerSource src, const int32_t *__restrict__ base, int base_inclusive,
               const float *__restrict__ w, ExpertIds topk_idx,
               const int32_t *__restrict__ rank_in_expert, int hidden, int topk, int experts,
               uint16_t *__restrict__ out)
{
    const int t = blockIdx.x;
    /*
     * Rank -2 (or a negative rank on a valid expert id) belongs to a token that the layout masked out (x_active_mask):
     * such a token's output row is left as it is. Rank -1 on an invalid expert id is a pick that goes nowhere: the
     * token's row is still written, from its other picks, or as zeros if it has none.
     */
    const int k = threadIdx.x & 63;
    bool keep = false, masked = false;
    const uint16_t *row_ptr = nullptr;
    float wk = 0.0f;
    int e = -1;
    int32_t rk = -1, bases[BASES > 0 ? BASES : 1], first = 0;
    if (k < topk) {
        e = topk_idx[(int64_t)t * topk + k];
        rk = rank_in_expert[(int64_t)t * topk + k];
        wk = w[(int64_t)t * topk + k];
    }
    if constexpr (BASES > 0) {
        /* inclusive: expert e starts where e - 1 ends */
#pragma unroll
        for (int j = 0; j < BASES; ++j) {
            const int i = j * 64 + k - (base_inclusive ? 1 : 0);
            bases[j] = i >= 0 && i < experts ? base[i] : 0;
        }
#pragma unroll
        for (int j = 0; j < BASES; ++j) {
            const int32_t b = __shfl(bases[j], e & 63, 64);
            if ((e >> 6) == j) first = b;
        }
    }
    if (k < topk) {
        if (rk == -2) masked = true;
        else if (e >= 0 && e < experts) {
            if (rk < 0) masked = true;
            else {
                const int slot = e * src.ranks + src.my_rank;
                /* running sums start anew with every rank's block of `experts` entries (low-latency counts) */
                const int32_t b = BASES > 0 ? first : base_inclusive ? (slot % experts == 0 ? 0 : base[slot - 1]) : base[slot];
                const int64_t row = (int64_t)b + rk;
                if (row < src.rows_cap) {            /* never read past the window */
                    keep = true;
                    row_ptr = src.y[src.ranks == 1 ? 0 : e / src.e_loc] + row * hidden;
                }
            }
        }
    }
    const uint64_t kept = __ballot(keep);
    if (__ballot(masked) != 0) return;
    const uint32_t ptr_lo = (uint32_t)(uint64_t)row_ptr, ptr_hi = (uint32_t)((uint64_t)row_ptr >> 32);
    auto pick_ptr = [&](int p) __attribute__((always_inline)) {
        const uint32_t lo = __builtin_amdgcn_readlane(ptr_lo, p), hi = __builtin_amdgcn_readlane(ptr_hi, p);
        return reinterpret_cast<const u32x4 *>(((uint64_t)hi << 32) | lo);
    };
    /* blockIdx.y: a small batch spreads each row over several workgroups, so that the whole chip takes part */
    const int nchunk_all = hidden / 8;
    const int per_split = (nchunk_all + gridDim.y - 1) / gridDim.y;
    const int c_begin = blockIdx.y * per_split;
    const int c_end = c_begin + per_split < nchunk_all ? c_begin + per_split : nchunk_all;
    for (int c0 = c_begin + threadIdx.x; c0 < c_end; c0 += U * blockDim.x) {
        float acc[U][8];
#pragma unroll
        for (int j = 0; j < U; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[j][i] = 0.0f;
        for (uint64_t left = kept; left != 0;) {
            /* the group's row loads are issued back to back, then folded in pick order */
            u32x4 v[kGroup][U];
            float wu[kGroup];
            uint64_t m = left;
#pragma unroll
            for (int u = 0; u < kGroup; ++u) {
                if (m == 0) break;
                const int p = __ffsll((long long)m) - 1;
                m &= m - 1;
                wu[u] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wk), p));
                const u32x4 *row = pick_ptr(p);
#pragma unroll
                for (int j = 0; j < U; ++j)
                    if (U == 1 || c0 + j * (int)blockDim.x < c_end) v[u][j] = __builtin_nontemporal_load(row + c0 + j * blockDim.x);
            }
#pragma unroll
            for (int u = 0; u < kGroup; ++u) {
                if (left == 0) break;
                left &= left - 1;
#pragma unroll
                for (int j = 0; j < U; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float lo = zb_half_to_f32<DT>(v[u][j][i] & 0xffffu) * wu[u];
                        const float hi = zb_half_to_f32<DT>(v[u][j][i] >> 16) * wu[u];
                        acc[j][2 * i] = acc[j][2 * i] + lo;
                        acc[j][2 * i + 1] = acc[j][2 * i + 1] + hi;
                    }
            }
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int c = c0 + j * blockDim.x;
            if (U > 1 && c >= c_end) break;
            u32x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = zb_pack2_half<DT>(acc[j][2 * i], acc[j][2 * i + 1]);
            __builtin_nontemporal_store(o, reinterpret_cast<u32x4 *>(out + (int64_t)t * hidden + (int64_t)c * 8));
        }
    }
}

} // namespace

extern "C" int32_t zbalhip_combine(const void *const *y, int32_t ranks, int32_t my_rank, int64_t y_rows, int32_t dtype,
                                   const int32_t *base, int32_t base_is_inclusive, const float *w, const int32_t *topk_idx,
                                   const int32_t *send_token_idx, int64_t tokens, int64_t hidden, int64_t topk,
                                   int64_t experts, void *out, void *stream)
{
    if (!y || !base || !w || !topk_idx || !send_token_idx || !out) return ZBALHIP_INVALID;
    if (dtype != ZDT_BF16 && dtype != ZDT_FP16) return ZBALHIP_INVALID;
    if (tokens < 0 || hidden <= 0 || hidden % 8 != 0 || topk <= 0 || topk > kMaxTopk || experts <= 0)
        return ZBALHIP_INVALID;
    const ExpertIds ids = expert_ids(topk_idx, (base_is_inclusive & ZBALHIP_IDS_ARE_I64) != 0);
    base_is_inclusive &= ~ZBALHIP_IDS_ARE_I64;
    if (ranks <= 0 || ranks > ZBALHIP_MAX_REDUCE_PEERS || my_rank < 0 || my_rank >= ranks || experts % ranks != 0 || y_rows < 0)
        return ZBALHIP_INVALID;
    PeerSource src = {};
    for (int r = 0; r < ranks; ++r) {
        if (!y[r]) return ZBALHIP_INVALID;
        src.y[r] = (const uint16_t *)y[r];
    }
    src.ranks = ranks;
    src.my_rank = my_rank;
    src.e_loc = (int)(experts / ranks);
    src.rows_cap = y_rows;
    if (tokens == 0) return ZBALHIP_OK;
    /*
     * Fewer tokens than four for each of the 256 CUs: the rows are cut into pieces of at least half a chunk per lane of a full workgroup, so that a row is
     * not read in two or more passes by the few workgroups that there are. Where the line lay at two per CU -> four, the kernel alone: 300
     * tokens x 7168 9.55 -> 9.12 us, 512 14.7 -> 13.9, 900 24.4 -> 23.7, 400 x 4096 7.77 -> 7.54, 1021 15.4 -> 15.05; 512 and 1500 x 2048, 2000 x
     * 4096 the same. At eight per CU 1021 x 4096 16.0, 1500 x 2048 9.8 -> 10.6.
     */
    int splits = 1;
    while (tokens * splits < 1024 && splits < 8 && hidden / 8 / (splits * 2) >= kThreads / 2) splits *= 2;
    const int64_t per_split = (hidden / 8 + splits - 1) / splits;
    int threads = (int)((per_split + 63) / 64 * 64);
    /*
     * Large batches take two chunks per lane and pass: 16 row loads in flight per lane. 4096 tokens x 7168 98.6 -> 93.1 us,
     * 8192 x 4096 118 -> 101 (of 8 picks each); 1021 x 4096 14.4 -> 16.0, with too few workgroups left to fill the chip.
     */
    const bool two = tokens >= 2048;
    if (two) threads = (int)(((per_split + 1) / 2 + 63) / 64 * 64);
    if (threads > kThreads) threads = kThreads;
    const dim3 grid((unsigned)tokens, (unsigned)splits);
    hipStream_t st = (hipStream_t)stream;
#define ZB_GO_BASES(DT, U, BASES)                                                                                     \
    zb_launch(combine_kernel<DT, U, BASES>, grid, threads, 0, st, src, base, base_is_inclusive, w, ids, send_token_idx, \
                                                           (int)hidden, (int)topk, (int)experts, (uint16_t *)out)
#define ZB_GO(DT, U)                                                                                                  \
    do {                                                                                                              \
        if (ranks == 1 && experts <= 64) ZB_GO_BASES(DT, U, 1);                                                       \
        else if (ranks == 1 && experts <= 128) ZB_GO_BASES(DT, U, 2);                                                 \
        else ZB_GO_BASES(DT, U, 0);                                                                                   \
    } while (0)
    if (dtype == ZDT_BF16) { if (two) ZB_GO(ZDT_BF16, 2); else ZB_GO(ZDT_BF16, 1); }
    else { if (two) ZB_GO(ZDT_FP16, 2); else ZB_GO(ZDT_FP16, 1); }
#undef ZB_GO_BASES
#undef ZB_GO
    return zbalhip_check_launch();
}
