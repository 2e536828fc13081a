/*
 * Routing and layout kernels: softmax top-k router, per-expert histogram with
 * stable per-pick ranks, and the count scans that turn the histogram into row
 * offsets.
 *
 * The stable rank of a pick (its position among earlier picks of the same
 * expert, in flat (t,k) order) is computed without atomics on the result:
 * blocks own contiguous token ranges, each counts the picks before its own
 * range, and inside a block picks are ranked 64 at a time with wave ballots
 * (lanes holding the same expert find each other by intersecting one ballot
 * per index bit).
 */
#include <time.h>

#include "zbal_device.h"
#include "zbal_hip_kernels.h"
#include "zbal_layout_rank.h"

#define ZB_MAX_EXPERTS 1024
#define ZB_FUSED_THREADS 1024

namespace {

struct LayoutPlan {
    int nblk;
    int tokens_per_block;
};

inline LayoutPlan plan_layout(int64_t tokens, int64_t topk, int max_blocks)
{
    LayoutPlan p;
    int64_t want = (tokens * topk + 1023) / 1024;
    if (want < 1) want = 1;
    if (want > max_blocks) want = max_blocks;
    int64_t tpb = (tokens + want - 1) / want;
    if (tpb < 1) tpb = 1;
    p.tokens_per_block = (int)tpb;
    p.nblk = (int)((tokens + tpb - 1) / tpb);
    if (p.nblk < 1) p.nblk = 1;
    return p;
}

/*
 * What a layout launch writes; every pointer may be null. send_token_idx [T, K]; incl_i32 [E] running sums; row_off
 * [E + 1] exclusive offsets; counts_i32 / counts_i64 [E]; nums_typed [E] counts (type 1) or running sums (type 0);
 * tokens_per_rank [ranks]: tokens with a pick of one of the rank's experts; token_in_rank [T, ranks]: 1 where the token
 * has such a pick, else 0.
 */
struct LayoutOutputs {
    int32_t *send_token_idx, *incl_i32, *row_off, *counts_i32;
    int64_t *counts_i64, *nums_typed;
    int32_t *tokens_per_rank, *token_in_rank;
    int ranks, token_nums_type;
};

/* bit r of the returned mask: the token's picks [i0, i0 + topk) include an expert of rank first_rank + r (r < 32) */
__device__ __forceinline__ uint32_t token_ranks(const ExpertIds &idx, int64_t i0, int topk, int experts, int e_loc, int first_rank)
{
    uint32_t mask = 0;
    for (int k0 = 0; k0 < topk; k0 += 8) {
        int e[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) e[k] = k0 + k < topk ? idx[i0 + k0 + k] : -1;      /* requested together */
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (e[k] < 0 || e[k] >= experts) continue;
            const int r = (e_loc == experts ? 0 : e[k] / e_loc) - first_rank;
            if (r >= 0 && r < 32) mask |= 1u << r;
        }
    }
    return mask;
}

/*
 * One rank, up to 64 picks per token: a wave takes as many whole tokens as it has lanes for and reads their picks in a row; one
 * ballot says which tokens have a valid one. (A thread per token, its picks a line apart from the next thread's, was
 * through after 10 us of the launch at 4096 tokens, the ranking blocks after 7.) Returns this thread's share of the count.
 */
template <bool WIDE>        /* int64 ids */
__device__ __forceinline__ int32_t tokens_of_one_rank(const ExpertIds &idx, int tokens, int topk, int experts, int32_t *token_in_rank)
{
    constexpr int U = 8;                                  /* picks in flight per lane */
    const int lane = threadIdx.x & 63, per_wave = 64 / topk, group = lane / topk;
    const int step = per_wave * (blockDim.x >> 6);
    const uint64_t mine = group < per_wave ? (~0ull >> (64 - topk)) << (group * topk) : 0ull;
    const int64_t last = (int64_t)tokens * topk - 1;
    int32_t n = 0;
    for (int t0 = (threadIdx.x >> 6) * per_wave; t0 < tokens; t0 += U * step) {
        u32x2 w[U];                            /* words, not ids: what is worked out under a condition waits for its load there */
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int64_t i = (int64_t)(t0 + u * step) * topk + lane;
            i = i < last ? i : last;
            if (WIDE) w[u] = reinterpret_cast<const u32x2 *>(idx.p)[i];
            else w[u] = u32x2{(uint32_t)idx.p[i], 0u};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = WIDE ? idx.of_words(w[u][0], w[u][1]) : (int)w[u][0];
            const uint64_t valid = __ballot(e >= 0 && e < experts);
            const int t = t0 + u * step + group;
            if (lane == group * topk && group < per_wave && t < tokens) {
                const int32_t any = (valid & mine) != 0;
                n += any;
                if (token_in_rank) token_in_rank[t] = any;
            }
        }
    }
    return n;
}

/*
 * One count per (token, rank) no matter how many of the token's picks land there, 32 ranks per pass; by one block. With one
 * rank it writes token_in_rank as well.
 */
__device__ __forceinline__ void count_tokens_per_rank(const ExpertIds &idx, int tokens, int topk, int experts, int e_loc,
                                                      const LayoutOutputs &o, int32_t *rcnt)
{
    for (int r = threadIdx.x; r < o.ranks; r += blockDim.x) rcnt[r] = 0;
    __syncthreads();
    if (o.ranks == 1 && topk <= 64) {
        const int32_t mine = zb_wave_sum_dpp(idx.kind == IDS_I32 ? tokens_of_one_rank<false>(idx, tokens, topk, experts, o.token_in_rank)
                                                                 : tokens_of_one_rank<true>(idx, tokens, topk, experts, o.token_in_rank));
        if ((threadIdx.x & 63) == 0 && mine) atomicAdd(&rcnt[0], mine);
    } else for (int first = 0; first < o.ranks; first += 32) {
        int32_t mine = 0;                       /* ranks == 1: counted in a register */
        for (int t = threadIdx.x; t < tokens; t += blockDim.x) {
            uint32_t mask = token_ranks(idx, (int64_t)t * topk, topk, experts, e_loc, first);
            if (o.ranks == 1) {
                mine += (int32_t)(mask & 1u);
                if (o.token_in_rank) o.token_in_rank[t] = (int32_t)(mask & 1u);
            } else
                for (; mask; mask &= mask - 1) atomicAdd(&rcnt[first + __ffs((int)mask) - 1], 1);
        }
        if (o.ranks == 1) {
            mine = zb_wave_sum_dpp(mine);
            if ((threadIdx.x & 63) == 0 && mine) atomicAdd(&rcnt[0], mine);
        }
    }
    __syncthreads();
    if (o.tokens_per_rank)
        for (int r = threadIdx.x; r < o.ranks; r += blockDim.x) o.tokens_per_rank[r] = rcnt[r];
}

/*
 * The whole layout in one launch: every block first counts the picks that precede its own range (the index array is a
 * few hundred KiB and sits in L2, so reading it again per block is cheaper than a launch) and ranks its own picks. One
 * block more counts all of them and scans the counts into the offsets, one more the tokens per rank (RANKS). The counts go
 * to several copies of a counter, a lane's by its number, so that lanes with the same expert seldom meet at one address.
 * (4096 tokens of 8 int64 picks over 32 experts 12.2 -> 10.2 us, 6 of them counting; 1021 over 128 experts 8.8 -> 6.6.)
 * With per-rank counts on 4096 tokens of 8 int64 picks over 32 experts this replaces a histogram, a ranking and a scan
 * launch (4.7 + 20.3 + 6.1 us; the ranking blocks summed up to 49 histograms one after the other) and five elementwise
 * launches that worked token_in_rank out.
 */
template <bool RANKS>
__global__ void __launch_bounds__(ZB_FUSED_THREADS)
layout_fused_kernel(ExpertIds idx, int tokens, int topk, int experts, int tpb, int nbits,
                    const uint8_t *__restrict__ active_mask, LayoutOutputs o)
{
    __shared__ int32_t run[ZB_MAX_EXPERTS];
    __shared__ __align__(16) int32_t copies[ZB_MAX_EXPERTS];
    __shared__ int32_t wsum[ZB_FUSED_THREADS / 64];
    __shared__ int32_t s_active;
    __shared__ __align__(16) uint8_t cnt[ZB_FUSED_THREADS / 64 * ZB_MAX_EXPERTS];
    const int e_loc = RANKS ? experts / o.ranks : experts;
    const int ranges = (int)gridDim.x - (RANKS ? 2 : 1);
    const bool totals = (int)blockIdx.x == ranges;              /* counts every pick, ranks none */
    if (RANKS && (int)blockIdx.x > ranges) {
        if (o.tokens_per_rank || o.ranks == 1) count_tokens_per_rank(idx, tokens, topk, experts, e_loc, o, run);
        return;
    }
    const int log_copies = experts <= 64 ? 4 : (experts <= 128 ? 3 : (experts <= 256 ? 2 : (experts <= 512 ? 1 : 0)));
    copies[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_active = 0;
    __syncthreads();
    /*
     * x_active_mask (one bool per token): the reference processes the first sum(mask) tokens and nothing else
     * (TokenActiveMaskCal, fused_deep_moe/gemm/kernel/...swiglu_quant_multistage_workspace.h:836-863). Picks of
     * the other tokens get rank -2 here: the permute kernel skips every negative rank, and the combine kernel leaves
     * the output row of such a token alone. (-1 is a pick with an invalid expert id in a token that is routed: the
     * combine still writes that token's row, from its other picks or as zeros.)
     */
    int active = tokens;
    if (active_mask) {
        int part = 0;
        for (int t = threadIdx.x; t < tokens; t += blockDim.x) part += active_mask[t] != 0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
        if ((threadIdx.x & 63) == 0 && part) atomicAdd(&s_active, part);
        __syncthreads();
        active = s_active;
    }
    int tok0 = totals ? tokens : (int)blockIdx.x * tpb;
    int tok1 = totals ? tokens : tok0 + tpb;
    if (tok1 > tokens) tok1 = tokens;
    if (RANKS && o.token_in_rank && o.ranks > 1)
        for (int i = tok0 * o.ranks + threadIdx.x; i < tok1 * o.ranks; i += blockDim.x) {
            const int t = i / o.ranks;
            o.token_in_rank[i] = (int)(token_ranks(idx, (int64_t)t * topk, topk, experts, e_loc, i - t * o.ranks) & 1u);
        }
    for (int64_t i = (int64_t)(tok0 > active ? tok0 : active) * topk + threadIdx.x; i < (int64_t)tok1 * topk; i += blockDim.x)
        o.send_token_idx[i] = -2;
    if (tok0 > active) tok0 = active;
    if (tok1 > active) tok1 = active;
    const int64_t p0 = (int64_t)tok0 * topk, p1 = (int64_t)tok1 * topk;
    const int own = first_pick(idx, p0, p1);
    auto count = [&](int e) __attribute__((always_inline)) {
        if (e >= 0 && e < experts) atomicAdd(&copies[(e << log_copies) + (threadIdx.x & ((1 << log_copies) - 1))], 1);
    };
    const int per = 4 / idx.stride();                /* ids per 16-byte load */
    const int64_t nvec = ((uintptr_t)idx.p & 15) == 0 ? p0 / per : 0;
    /* up to sixteen 16-byte loads per lane are requested before the first is counted: a chain of round trips otherwise */
    constexpr int U = 16;
    for (int64_t v0 = threadIdx.x; v0 < nvec; v0 += U * (int64_t)blockDim.x) {
        u32x4 raw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t v = v0 + u * (int64_t)blockDim.x;
            raw[u] = v < nvec ? *reinterpret_cast<const u32x4 *>(idx.p + v * 4) : u32x4{~0u, ~0u, ~0u, ~0u};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (v0 + u * (int64_t)blockDim.x >= nvec) break;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (idx.kind != IDS_I32 && (j & 1)) continue;
                count(idx.kind == IDS_I32 ? (int)raw[u][j] : idx.of_words(raw[u][j], raw[u][j | 1]));
            }
        }
    }
    for (int64_t i = nvec * per + threadIdx.x; i < p0; i += blockDim.x) count(idx[i]);
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += blockDim.x) {
        int32_t sum = 0;
        if (log_copies >= 2) {
            i32x4 c[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                c[j] = j < 1 << (log_copies - 2) ? *reinterpret_cast<const i32x4 *>(copies + (e << log_copies) + 4 * j) : i32x4{0, 0, 0, 0};
            c[0] += c[1] + c[2] + c[3];
            sum = c[0][0] + c[0][1] + c[0][2] + c[0][3];
        } else
            for (int c = 0; c < 1 << log_copies; ++c) sum += copies[(e << log_copies) + c];
        run[e] = sum;
    }
    __syncthreads();
    if (!totals) {
        rank_picks<ZB_FUSED_THREADS / 64, false>(idx, p0, p1, own, experts, nbits, run, cnt, o.send_token_idx);
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int32_t carry = 0;
    for (int base = 0; base < experts; base += ZB_FUSED_THREADS) {
        const int e = base + threadIdx.x;
        const int32_t c = e < experts ? run[e] : 0;
        int32_t s = zb_wave_scan_dpp(c);
        if (lane == 63) wsum[wave] = s;
        __syncthreads();
        s += carry;
#pragma unroll
        for (int w = 0; w < ZB_FUSED_THREADS / 64; ++w) {
            const int32_t of_wave = wsum[w];
            s += w < wave ? of_wave : 0;
            carry += of_wave;
        }
        __syncthreads();
        if (e < experts) {
            if (o.incl_i32) o.incl_i32[e] = s;
            if (o.row_off) { o.row_off[e] = s - c; if (e == experts - 1) o.row_off[experts] = s; }
            if (o.counts_i32) o.counts_i32[e] = c;
            if (o.counts_i64) o.counts_i64[e] = c;
            if (o.nums_typed) o.nums_typed[e] = o.token_nums_type == 0 ? (int64_t)s : (int64_t)c;
        }
    }
}

/*
 * The part of the layout that needs no other block: the picks of a token range are ranked among themselves
 * (send_token_idx = position among the range's picks of the same expert) and the range's histogram is left in
 * hist[range][experts]. The permute kernel that follows turns the histograms into offsets on its own (dispatch.hip,
 * table mode), so this launch is all there is in front of it: no counting of the ranges before, no scan.
 * A range is worked on by `subs` blocks, each ranking one slice of it; a block counts the picks of the slices before
 * its own itself (LDS atomics: a fraction of what ranking them costs), so no block waits for another, and the block of
 * the last slice ends up with the whole range's histogram and writes it.
 */
template <bool SLICED>
__global__ void __launch_bounds__(ZB_FUSED_THREADS)
layout_ranges_kernel(ExpertIds idx, int tokens, int topk, int experts, int tpb, int subs_arg, int nbits,
                     const uint8_t *__restrict__ active_mask, int32_t *__restrict__ send_token_idx,
                     int32_t *__restrict__ hist)
{
    __shared__ int32_t run[ZB_MAX_EXPERTS];
    __shared__ int32_t s_active;
    __shared__ __align__(16) uint8_t cnt[ZB_FUSED_THREADS / 64 * ZB_MAX_EXPERTS];
    for (int e = threadIdx.x; e < experts; e += blockDim.x) run[e] = 0;
    if (threadIdx.x == 0) s_active = 0;
    __syncthreads();
    int active = tokens;
    if (active_mask) {          /* the first sum(mask) tokens are routed, the picks of the others get rank -2 (layout_fused_kernel) */
        int part = 0;
        for (int t = threadIdx.x; t < tokens; t += blockDim.x) part += active_mask[t] != 0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
        if ((threadIdx.x & 63) == 0 && part) atomicAdd(&s_active, part);
        __syncthreads();
        active = s_active;
    }
    const int subs = SLICED ? subs_arg : 1;
    const int range = SLICED ? blockIdx.x / subs : blockIdx.x, sub = SLICED ? blockIdx.x - range * subs : 0;
    int tok0 = range * tpb;
    int tok1 = tok0 + tpb;
    if (tok1 > tokens) tok1 = tokens;
    int sl0 = tok0, sl1 = tok1;
    if (SLICED) {
        const int tps = (tpb + subs - 1) / subs;            /* tokens per slice */
        sl0 = tok0 + sub * tps;
        sl1 = sl0 + tps;
        if (sl0 > tok1) sl0 = tok1;
        if (sl1 > tok1) sl1 = tok1;
    }
    for (int64_t i = (int64_t)(sl0 > active ? sl0 : active) * topk + threadIdx.x; i < (int64_t)sl1 * topk; i += blockDim.x)
        send_token_idx[i] = -2;
    if (tok0 > active) tok0 = active;
    if (sl0 > active) sl0 = active;
    if (sl1 > active) sl1 = active;
    if (SLICED) {       /* the picks of this range in front of the slice: counted only */
        for (int64_t i = (int64_t)tok0 * topk + threadIdx.x; i < (int64_t)sl0 * topk; i += blockDim.x) {
            const int e = idx[i];
            if (e >= 0 && e < experts) atomicAdd(&run[e], 1);
        }
        __syncthreads();
    }
    const int64_t p0 = (int64_t)sl0 * topk, p1 = (int64_t)sl1 * topk;
    rank_picks<ZB_FUSED_THREADS / 64>(idx, p0, p1, first_pick(idx, p0, p1), experts, nbits, run, cnt, send_token_idx);
    /* rank_picks ends on a barrier: run[] counts the range up to this slice's end; the last slice's block has it all */
    if (!SLICED || sub == subs - 1)
        for (int e = threadIdx.x; e < experts; e += blockDim.x) hist[(int64_t)range * experts + e] = run[e];
}

/* where a notify launch leaves the counts for a host that waits for them: pinned memory that the GPU writes directly */
struct HostCounts {
    int64_t counts[ZB_MAX_EXPERTS];
    uint64_t ready;                /* the number of the launch that wrote the counts, stored after them */
};

/*
 * Notify for a group of one rank, one block: the offsets are the exclusive running sum of the counts. With `host` the
 * counts also go to pinned host memory, followed by a flag, so that a caller who has to know them spins on that word
 * instead of queueing a copy behind the kernel and waiting for the stream.
 */
__global__ void __launch_bounds__(ZB_MAX_EXPERTS)
notify_one_kernel(const int32_t *__restrict__ tokens_per_expert, int experts, int topk, int32_t *__restrict__ recv_data,
                  int32_t *__restrict__ put_offset, int64_t *__restrict__ recv_tokens_per_expert,
                  int32_t *__restrict__ total, int32_t *__restrict__ balance, HostCounts *host, uint64_t launch)
{
    __shared__ int32_t wsum[ZB_MAX_EXPERTS / 64];
    const int e = threadIdx.x;
    const int32_t c = e < experts ? tokens_per_expert[e] : 0;
    if (host && e < experts) host->counts[e] = c;
    int32_t s = c;
    const int lane = e & 63, wave = e >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        int32_t o = __shfl_up(s, off, 64);
        if (lane >= off) s += o;
    }
    if (lane == 63) wsum[wave] = s;
    if (host) __threadfence_system();
    __syncthreads();
    if (host && e == 0) __hip_atomic_store(&host->ready, launch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    int32_t add = 0;
    for (int w = 0; w < wave; ++w) add += wsum[w];
    s += add;
    if (e < experts) {
        recv_data[e] = c;
        put_offset[e] = s - c;
        recv_tokens_per_expert[e] = c;
        if (e == experts - 1) {
            *total = s;
            const int32_t bs = s / topk;
            balance[0] = bs > 0 ? 0 : -1;
            balance[1] = bs > 0 ? bs - 1 : -1;
        }
    }
}

/*
 * Notify for a group of R ranks, from the point of view of rank `me` (reference zbal_kernel_notify_dispatch.h
 * ReorderRecvDataOutput :356-378, BuildTotalRecvTokens :531-564, BuildRecvTokenPerExp :566-596,
 * BuildBalanceMatrix :421-498 without re-balancing). counts.p[s] is rank s's tokens-per-expert vector, read where
 * it lies in that rank's window. For every destination rank r the offsets are the exclusive running sum of
 * counts[s][r * E_loc + le] taken local expert by local expert and, within an expert, source rank by source rank.
 * One block, one thread per (local expert, source rank) pair of a destination rank.
 */
struct CountsOfRanks {
    const int32_t *p[ZBALHIP_MAX_REDUCE_PEERS];
};

__global__ void __launch_bounds__(ZB_MAX_EXPERTS)
notify_ranks_kernel(CountsOfRanks counts, int ranks, int me, int experts, int topk, int32_t *__restrict__ recv_data,
                    int32_t *__restrict__ put_offset, int32_t *__restrict__ total_recv,
                    int64_t *__restrict__ recv_tokens_per_expert, int32_t *__restrict__ balance)
{
    __shared__ int32_t wsum[ZB_MAX_EXPERTS / 64];
    __shared__ int32_t rank_total[ZBALHIP_MAX_REDUCE_PEERS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
    const int e_loc = experts / ranks;
    for (int i = tid; i < ranks * experts; i += blockDim.x) recv_data[i] = counts.p[i / experts][i % experts];
    if (tid < ranks) rank_total[tid] = 0;
    __syncthreads();
    for (int r = 0; r < ranks; ++r) {
        const int le = tid / ranks, s = tid - le * ranks;
        const int32_t c = tid < experts ? counts.p[s][r * e_loc + le] : 0;
        int32_t incl = c;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t o = __shfl_up(incl, off, 64);
            if (lane >= off) incl += o;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int32_t add = 0, all = 0;
        for (int w = 0; w < nwaves; ++w) {
            if (w < wave) add += wsum[w];
            all += wsum[w];
        }
        if (tid < experts) put_offset[r * experts + tid] = incl + add - c;
        if (r == me && tid == 0) *total_recv = all;
        /* what source rank s sends in all: the sum over destination ranks of its share */
        if (tid < experts && c) atomicAdd(&rank_total[s], c);
        __syncthreads();
    }
    for (int le = tid; le < e_loc; le += blockDim.x) {
        int64_t sum = 0;
        for (int s = 0; s < ranks; ++s) sum += counts.p[s][me * e_loc + le];
        recv_tokens_per_expert[le] = sum;
    }
    for (int i = tid; i < ranks * 2 * ranks; i += blockDim.x) {
        const int row = i / (2 * ranks), col = i - row * 2 * ranks;
        const int32_t bs = rank_total[row] / topk;
        int32_t v = -1;
        if (bs > 0 && col == 2 * row) v = 0;
        if (bs > 0 && col == 2 * row + 1) v = bs - 1;
        balance[i] = v;
    }
}

/*
 * Counts of the low-latency dispatch for a group of R ranks, from the point of view of rank `me` (reference
 * zbal_kernel_dispatch_low_latency.h: every rank's per-expert counts gathered into allExpertTokenNums :344-345,
 * ReorderRecvDataOutput :690-713, WaitNotify :641-688). ids.p[s] is rank s's [tokens, topk] expert ids, read where
 * they lie in that rank's window (the reference's ranks push their counts to each other and wait for flags; on one
 * GPU the inputs of all modelled ranks are in place before any of them is launched). all_counts[s * E + e] = picks
 * of expert e by rank s; ep_recv_counts[r * E + le * R + s] = INCLUSIVE running sum, per destination rank r, over
 * its local experts le and, within an expert, the source ranks s (a consumer takes index i's start from entry i - 1,
 * 0 at the start of a rank's block); expert_token_nums[le] = rows rank `me` receives for its local expert le
 * (type 1) or their running sum (type 0). One block, one thread per (local expert, source rank) pair.
 */
struct IdsOfRanks {
    const int32_t *p[ZBALHIP_MAX_REDUCE_PEERS];
};

__global__ void __launch_bounds__(ZB_MAX_EXPERTS)
ll_counts_kernel(IdsOfRanks ids, int ranks, int me, int tokens, int topk, int experts, int token_nums_type,
                 int32_t *__restrict__ all_counts, int32_t *__restrict__ ep_recv_counts,
                 int64_t *__restrict__ expert_token_nums)
{
    __shared__ int32_t hist[ZB_MAX_EXPERTS];
    __shared__ int32_t mine[ZB_MAX_EXPERTS];
    __shared__ int32_t wsum[ZB_MAX_EXPERTS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
    const int n = tokens * topk, e_loc = experts / ranks;
    for (int s = 0; s < ranks; ++s) {
        for (int e = tid; e < experts; e += blockDim.x) hist[e] = 0;
        __syncthreads();
        for (int i = tid; i < n; i += blockDim.x) {
            const int e = ids.p[s][i];
            if (e >= 0 && e < experts) atomicAdd(&hist[e], 1);
        }
        __syncthreads();
        for (int e = tid; e < experts; e += blockDim.x) all_counts[s * experts + e] = hist[e];
        __syncthreads();
    }
    for (int r = 0; r < ranks; ++r) {
        const int le = tid / ranks, s = tid - le * ranks;
        const int32_t c = tid < experts ? all_counts[s * experts + r * e_loc + le] : 0;
        int32_t incl = c;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t o = __shfl_up(incl, off, 64);
            if (lane >= off) incl += o;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        for (int w = 0; w < wave && w < nwaves; ++w) incl += wsum[w];
        if (tid < experts) {
            ep_recv_counts[r * experts + tid] = incl;
            if (r == me) mine[tid] = incl;
        }
        __syncthreads();
    }
    for (int le = tid; le < e_loc; le += blockDim.x) {
        const int32_t hi = mine[(le + 1) * ranks - 1], lo = le ? mine[le * ranks - 1] : 0;
        expert_token_nums[le] = token_nums_type == 0 ? (int64_t)hi : (int64_t)(hi - lo);
    }
}

/* ---- router ----------------------------------------------------------------- */

/*
 * One wave per token; lane l holds logits l, l + 64, ... (PER_LANE of them: the launcher picks the smallest
 * instantiation that covers `experts`, the arithmetic and its order are the same in all of them).
 */
/*
 * Up to 64 experts: one logit per lane. A lane's pick position is its rank: the number of logits that are larger, or equal with a
 * lower index (the order K rounds of arg-max with ties to the lower index produce). With few experts to a pick the ranks come from
 * one pass over the experts, with the logit of expert m read from lane m as a scalar (0.035 us an expert of a lone wave); with more than
 * four, where that is longer, from rounds of arg-max as in the general kernel below (0.19 us each). The kernel alone, ranks / rounds: 1
 * token, 64 experts, top-6 4.11 / 2.36 us, top-8 4.13 / 2.70, 48 experts 3.51 / 2.37, 32 experts, top-8 2.97 / 2.82; 8192 tokens, 64 experts 9.0
 * / 5.4, 32 experts, top-8 5.9 / 6.1. Maximum and sums run on the DPP path. Same formulas as the general kernel
 * (p = exp(l - max) / sum; weight = p / sum of the picked p), sums taken in a different order.
 */
__global__ void __launch_bounds__(256)
topk_route_small_kernel(const float *__restrict__ logits, int tokens, int experts, int topk, void *__restrict__ topk_idx,
                        int idx_is_i64, float *__restrict__ topk_w)
{
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (t >= tokens) return; /* whole waves leave together */
    const bool mine = lane < experts;
    const float v = mine ? logits[(int64_t)t * experts + lane] : -__builtin_inff();
    const float mx = zb_wave_reduce_dpp<true>(v);
    const float ex = mine ? zb_expf(v - mx) : 0.0f;
    const float sum = zb_wave_reduce_dpp<false>(ex);
    int rank = 0;
    if (experts > 4 * topk) {
        float left = v;
        uint64_t avail = experts == 64 ? ~0ull : (1ull << experts) - 1;
        rank = topk;
        for (int k = 0; k < topk; ++k) {
            const float best = zb_wave_reduce_dpp<true>(left);
            const uint64_t owners = __ballot(v == best) & avail;
            if (owners == 0) break;              /* only NaNs are left */
            const int owner = __ffsll((long long)owners) - 1;
            avail &= ~(1ull << owner);
            if (lane == owner) { rank = k; left = -__builtin_inff(); }
        }
    } else {
        for (int m = 0; m < experts; ++m) {
            const float s = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), m));
            rank += (s > v || (s == v && m < lane)) ? 1 : 0;
        }
    }
    /* a NaN is no pick; slots for which there is no logit get what the general kernel leaves there, an id that no expert has */
    const bool number = mine && v == v, picked = number && rank < topk;
    const int numbers = __popcll(__ballot(number));
    const float p = ex / sum;
    const float wsum = zb_wave_reduce_dpp<false>(picked ? p : 0.0f);
    auto put = [&](int slot, int expert, float w) __attribute__((always_inline)) {
        if (idx_is_i64) static_cast<int64_t *>(topk_idx)[(int64_t)t * topk + slot] = expert;
        else static_cast<int32_t *>(topk_idx)[(int64_t)t * topk + slot] = expert;
        topk_w[(int64_t)t * topk + slot] = w;
    };
    if (picked) put(rank, lane, p / wsum);
    if (numbers < topk && lane >= numbers && lane < topk) put(lane, 0x7fffffff, __builtin_nanf(""));
}

template <int PER_LANE>
__global__ void __launch_bounds__(256)
topk_route_kernel(const float *__restrict__ logits, int tokens, int experts, int topk, void *__restrict__ topk_idx,
                  int idx_is_i64, float *__restrict__ topk_w)
{
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (t >= tokens) return; /* whole waves leave together */
    const float *l = logits + (int64_t)t * experts;
    float v[PER_LANE];
    float mx = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
        const int e = j * 64 + lane;
        v[j] = (e < experts) ? l[e] : -__builtin_inff();
        mx = fmaxf(mx, v[j]);
    }
    mx = zb_wave_reduce_dpp<true>(mx);
    float part = 0.0f;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
        const int e = j * 64 + lane;
        if (e < experts) part += zb_expf(v[j] - mx);
    }
    const float sum = zb_wave_reduce_dpp<false>(part);

    /*
     * K rounds of arg-max, each without an LDS round trip: the largest remaining logit by a DPP reduction of the
     * lanes' own best, then its owner by one ballot per logit slot, lowest slot and lowest lane first (the lowest
     * expert index among equal logits, as a sequential scan would pick). Who has been picked is a scalar mask, and a lane's picked
     * logit is minus infinity from then on, so a round asks no lane what it has left: 128 experts, top-8, 1 token 3.83 -> 3.54 us, 16384
     * 14.8 -> 13.1, 256 experts, 4096 tokens 8.3 -> 7.0, 1024 experts, top-16 45 -> 25.
     */
    uint64_t avail[PER_LANE]; /* the experts that have not been picked, 64 by 64 */
    float left[PER_LANE];     /* and their logits */
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
        const int n = experts - j * 64;
        avail[j] = n >= 64 ? ~0ull : (n > 0 ? (1ull << n) - 1 : 0);
        left[j] = v[j];
    }
    float picked = 0.0f; /* lane k keeps the k-th logit (topk <= 32) */
    int myidx = 0;
    for (int k = 0; k < topk; ++k) {
        float best = left[0];
#pragma unroll
        for (int j = 1; j < PER_LANE; ++j) best = fmaxf(best, left[j]);
        best = zb_wave_reduce_dpp<true>(best);
        int bidx = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < PER_LANE; ++j) {
            const uint64_t owners = __ballot(v[j] == best) & avail[j];
            if (bidx == 0x7fffffff && owners) {
                const int owner = __ffsll((long long)owners) - 1;
                bidx = j * 64 + owner;
                avail[j] &= ~(1ull << owner);
                if (lane == owner) left[j] = -__builtin_inff();
            }
        }
        if (lane == k) { picked = best; myidx = bidx; }
    }
    /*
     * One exp and one quotient for all picks, summed in their order: the kernel alone, 16384 tokens, 128 experts, top-8, logits in
     * the cache / from memory 15.6 / 16.6 us; in every round 20.5 / 21.4 (17 to 19 between a layer's other kernels, on their clock).
     */
    const float myw = zb_expf(picked - mx) / sum;
    float wsum = 0.0f;
    for (int k = 0; k < topk; ++k) wsum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(myw), k));
    if (lane < topk) {
        if (idx_is_i64) static_cast<int64_t *>(topk_idx)[(int64_t)t * topk + lane] = myidx;
        else static_cast<int32_t *>(topk_idx)[(int64_t)t * topk + lane] = myidx;
        topk_w[(int64_t)t * topk + lane] = myw / wsum;
    }
}

__global__ void fill_i32_kernel(int32_t *p, int64_t n, int32_t v)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

inline int ceil_log2(int64_t v)
{
    int b = 0;
    while ((1ll << b) < v) ++b;
    return b;
}

} // namespace

static int32_t launch_fused_layout(const ExpertIds &idx, int64_t tokens, int64_t experts, int64_t topk,
                                   const uint8_t *active_mask, const LayoutOutputs &o, hipStream_t st)
{
    const LayoutPlan p = plan_layout(tokens, topk, 64);
    if (o.tokens_per_rank || o.token_in_rank)
        zb_launch(layout_fused_kernel<true>, p.nblk + 2, ZB_FUSED_THREADS, 0, st, idx, (int)tokens, (int)topk, (int)experts,
                                                                     p.tokens_per_block, ceil_log2(experts), active_mask, o);
    else
        zb_launch(layout_fused_kernel<false>, p.nblk + 1, ZB_FUSED_THREADS, 0, st, idx, (int)tokens, (int)topk, (int)experts,
                                                                      p.tokens_per_block, ceil_log2(experts), active_mask, o);
    return zbalhip_check_launch();
}

/* Used by the other translation units of the library (fused path, low-latency dispatch): ranks + offsets in one launch */
int32_t zbalhip_layout_fused_internal(const ExpertIds &idx, int64_t tokens, int64_t experts, int64_t topk,
                                      int32_t token_nums_type, const uint8_t *active_mask, int32_t *send_token_idx,
                                      int32_t *incl_i32, int32_t *row_off, int64_t *counts_i64, int64_t *nums_typed,
                                      hipStream_t st)
{
    LayoutOutputs o = {};
    o.send_token_idx = send_token_idx;
    o.incl_i32 = incl_i32;
    o.row_off = row_off;
    o.counts_i64 = counts_i64;
    o.nums_typed = nums_typed;
    o.token_nums_type = token_nums_type;
    return launch_fused_layout(idx, tokens, experts, topk, active_mask, o, st);
}

/* ranks within token ranges + one histogram per range, for the permute kernel's table mode; returns the ranges' size */
int32_t zbalhip_layout_ranges_internal(const ExpertIds &idx, int64_t tokens, int64_t experts, int64_t topk,
                                       const uint8_t *active_mask, int32_t *send_token_idx, int32_t *hist, int nblk,
                                       int tokens_per_block, hipStream_t st)
{
    /*
     * Ranking costs a block about 0.2 + 0.017 x experts microseconds per 1024 picks (32 experts: 5.0 us for 5248
     * picks; 128 experts: 21 us for 8192): slices of so many picks that a block is through in about five.
     */
    int64_t slice_picks = 1024 * (int64_t)(5.0 / (0.2 + 0.017 * (double)experts));
    if (slice_picks < 1024) slice_picks = 1024;
    int64_t subs = ((int64_t)tokens_per_block * topk + slice_picks - 1) / slice_picks;
    subs = subs < 1 ? 1 : (subs > 8 ? 8 : subs);
    if (subs > tokens_per_block) subs = tokens_per_block;
    if (subs == 1)
        zb_launch(layout_ranges_kernel<false>, (unsigned)nblk, ZB_FUSED_THREADS, 0, st,
            idx, (int)tokens, (int)topk, (int)experts, tokens_per_block, 1, ceil_log2(experts), active_mask, send_token_idx, hist);
    else
        zb_launch(layout_ranges_kernel<true>, (unsigned)(nblk * subs), ZB_FUSED_THREADS, 0, st,
            idx, (int)tokens, (int)topk, (int)experts, tokens_per_block, (int)subs, ceil_log2(experts), active_mask,
            send_token_idx, hist);
    return zbalhip_check_launch();
}

int32_t zbalhip_ll_counts_internal(const int32_t *const *ids, int ranks, int me, int64_t tokens, int64_t topk,
                                   int64_t experts, int32_t token_nums_type, int32_t *all_counts, int32_t *ep_recv_counts,
                                   int64_t *expert_token_nums, hipStream_t st)
{
    IdsOfRanks all = {};
    for (int r = 0; r < ranks; ++r) all.p[r] = ids[r];
    const int threads = (int)((experts + 63) / 64 * 64);
    ll_counts_kernel<<<1, threads, 0, st>>>(all, ranks, me, (int)tokens, (int)topk, (int)experts, token_nums_type, all_counts,
                                            ep_recv_counts, expert_token_nums);
    return zbalhip_check_launch();
}

static bool layout_args_ok(int64_t tokens, int64_t experts, int64_t topk)
{
    return tokens >= 0 && tokens <= 0x7fffffff / (topk > 0 ? topk : 1) && experts > 0 && experts <= ZB_MAX_EXPERTS &&
           topk > 0;
}

extern "C" int32_t zbalhip_fill_i32(int32_t *p, int64_t n, int32_t value, void *stream)
{
    if (n < 0 || (n > 0 && !p)) return ZBALHIP_INVALID;
    if (n == 0) return ZBALHIP_OK;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    fill_i32_kernel<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(p, n, value);
    return zbalhip_check_launch();
}

extern "C" int32_t zbalhip_topk_route(const float *logits, int64_t tokens, int64_t experts, int64_t topk,
                                      void *topk_idx, int32_t idx_is_i64, float *topk_w, void *stream)
{
    if (!logits || !topk_idx || !topk_w || tokens < 0 || experts <= 0 || experts > ZB_MAX_EXPERTS || topk <= 0 ||
        topk > 32 || topk > experts)
        return ZBALHIP_INVALID;
    if (tokens == 0) return ZBALHIP_OK;
    const int wpb = 4;
    const int64_t blocks = (tokens + wpb - 1) / wpb;
    const dim3 grid((unsigned)blocks), block(wpb * 64);
    hipStream_t st = (hipStream_t)stream;
    if (experts <= 64) zb_launch(topk_route_small_kernel, grid, block, 0, st, logits, (int)tokens, (int)experts, (int)topk, topk_idx, idx_is_i64, topk_w);
    else if (experts <= 128) zb_launch(topk_route_kernel<2>, grid, block, 0, st, logits, (int)tokens, (int)experts, (int)topk, topk_idx, idx_is_i64, topk_w);
    else if (experts <= 256) zb_launch(topk_route_kernel<4>, grid, block, 0, st, logits, (int)tokens, (int)experts, (int)topk, topk_idx, idx_is_i64, topk_w);
    else zb_launch(topk_route_kernel<ZB_MAX_EXPERTS / 64>, grid, block, 0, st, logits, (int)tokens, (int)experts, (int)topk, topk_idx, idx_is_i64, topk_w);
    return zbalhip_check_launch();
}

extern "C" int32_t zbalhip_dispatch_layout(const void *topk_idx, int32_t idx_is_i64, int64_t tokens, int64_t experts,
                                           int64_t topk, int32_t ranks, int32_t *tokens_per_rank,
                                           int32_t *tokens_per_expert, int32_t *send_token_idx, int32_t *scratch,
                                           void *stream)
{
    if (!scratch) return ZBALHIP_INVALID;
    return zbalhip_dispatch_layout_in_rank(topk_idx, idx_is_i64, tokens, experts, topk, ranks, tokens_per_rank,
                                           tokens_per_expert, send_token_idx, nullptr, stream);
}

extern "C" int32_t zbalhip_dispatch_layout_in_rank(const void *topk_idx, int32_t idx_is_i64, int64_t tokens,
                                                   int64_t experts, int64_t topk, int32_t ranks,
                                                   int32_t *tokens_per_rank, int32_t *tokens_per_expert,
                                                   int32_t *send_token_idx, int32_t *token_in_rank, void *stream)
{
    if (!topk_idx || !tokens_per_rank || !tokens_per_expert || !send_token_idx) return ZBALHIP_INVALID;
    if (!layout_args_ok(tokens, experts, topk) || ranks <= 0 || ranks > experts || experts % ranks != 0)
        return ZBALHIP_INVALID;
    if (token_in_rank && tokens > 0x7fffffff / ranks) return ZBALHIP_INVALID;
    LayoutOutputs o = {};
    o.send_token_idx = send_token_idx;
    o.counts_i32 = tokens_per_expert;
    o.tokens_per_rank = tokens_per_rank;
    o.token_in_rank = token_in_rank;
    o.ranks = ranks;
    return launch_fused_layout(expert_ids(topk_idx, idx_is_i64 != 0, true), tokens, experts, topk, nullptr, o, (hipStream_t)stream);
}

extern "C" int32_t zbalhip_dispatch_layout_static(const void *topk_idx, int32_t idx_is_i64, int64_t tokens, int64_t experts,
                                                  int64_t topk, int32_t ranks, int32_t *tokens_per_rank,
                                                  int32_t *tokens_per_expert, int32_t *send_token_idx, void *stream)
{
    if (!topk_idx || !tokens_per_rank || !tokens_per_expert || !send_token_idx) return ZBALHIP_INVALID;
    if (experts > ZBALHIP_LAYOUT_STATIC_MAX_EXPERTS) {
        zbalhip_set_last_error("zbalhip_dispatch_layout_static: more than 1024 experts (the limit of the static scratch that the layout once had)");
        return ZBALHIP_INVALID;
    }
    return zbalhip_dispatch_layout_in_rank(topk_idx, idx_is_i64, tokens, experts, topk, ranks, tokens_per_rank,
                                           tokens_per_expert, send_token_idx, nullptr, stream);
}

static int32_t launch_notify(const int32_t *const *tokens_per_expert, int32_t ranks, int32_t my_rank, int64_t experts,
                             int64_t topk, int32_t *recv_data, int32_t *put_offset, int32_t *total_recv,
                             int64_t *recv_tokens_per_expert, int32_t *balance_matrix, HostCounts *host, uint64_t launch,
                             hipStream_t st)
{
    if (!tokens_per_expert || !recv_data || !put_offset || !total_recv || !recv_tokens_per_expert || !balance_matrix)
        return ZBALHIP_INVALID;
    if (experts <= 0 || experts > ZB_MAX_EXPERTS || topk <= 0) return ZBALHIP_INVALID;
    if (ranks <= 0 || ranks > ZBALHIP_MAX_REDUCE_PEERS || my_rank < 0 || my_rank >= ranks || experts % ranks != 0)
        return ZBALHIP_INVALID;
    for (int r = 0; r < ranks; ++r)
        if (!tokens_per_expert[r]) return ZBALHIP_INVALID;
    const int threads = (int)((experts + 63) / 64 * 64);
    if (ranks == 1) {
        zb_launch(notify_one_kernel, 1, threads, 0, st, tokens_per_expert[0], (int)experts, (int)topk, recv_data, put_offset,
                                                 recv_tokens_per_expert, total_recv, balance_matrix, host, launch);
        return zbalhip_check_launch();
    }
    CountsOfRanks counts = {};
    for (int r = 0; r < ranks; ++r) counts.p[r] = tokens_per_expert[r];
    notify_ranks_kernel<<<1, threads, 0, st>>>(counts, ranks, my_rank, (int)experts, (int)topk, recv_data, put_offset,
                                               total_recv, recv_tokens_per_expert, balance_matrix);
    return zbalhip_check_launch();
}

extern "C" int32_t zbalhip_dispatch_notify(const int32_t *const *tokens_per_expert, int32_t ranks, int32_t my_rank,
                                           int64_t experts, int64_t topk, int32_t *recv_data, int32_t *put_offset,
                                           int32_t *total_recv, int64_t *recv_tokens_per_expert, int32_t *balance_matrix,
                                           void *stream)
{
    return launch_notify(tokens_per_expert, ranks, my_rank, experts, topk, recv_data, put_offset, total_recv,
                         recv_tokens_per_expert, balance_matrix, nullptr, 0, (hipStream_t)stream);
}

extern "C" int32_t zbalhip_host_counts_alloc(void **block)
{
    if (!block) return ZBALHIP_INVALID;
    if (hipHostMalloc(block, sizeof(HostCounts), hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess)
        return ZBALHIP_RT_ERROR;
    static_cast<HostCounts *>(*block)->ready = 0;
    return ZBALHIP_OK;
}

extern "C" int32_t zbalhip_host_counts_free(void *block)
{
    return block == nullptr || hipHostFree(block) == hipSuccess ? ZBALHIP_OK : ZBALHIP_RT_ERROR;
}

extern "C" int32_t zbalhip_dispatch_notify_counts(const int32_t *const *tokens_per_expert, int32_t ranks, int32_t my_rank,
                                                  int64_t experts, int64_t topk, int32_t *recv_data, int32_t *put_offset,
                                                  int32_t *total_recv, int64_t *recv_tokens_per_expert,
                                                  int32_t *balance_matrix, void *block, uint64_t *ticket, void *stream)
{
    if (!block || !ticket) return ZBALHIP_INVALID;
    hipStream_t st = (hipStream_t)stream;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (st != nullptr && hipStreamIsCapturing(st, &capture) == hipSuccess && capture != hipStreamCaptureStatusNone) {
        zbalhip_set_last_error("NotifyDispatch failed as the counts cannot be read back while the stream is being captured");
        return ZBALHIP_RT_ERROR;
    }
    HostCounts *host = static_cast<HostCounts *>(block);
    *ticket = ranks == 1 ? host->ready + 1 : 0;
    const int32_t rc = launch_notify(tokens_per_expert, ranks, my_rank, experts, topk, recv_data, put_offset, total_recv,
                                     recv_tokens_per_expert, balance_matrix, host, *ticket, st);
    if (rc != ZBALHIP_OK || ranks == 1) return rc;
    const size_t bytes = (size_t)(experts / ranks) * sizeof(int64_t);
    return hipMemcpyAsync(host->counts, recv_tokens_per_expert, bytes, hipMemcpyDeviceToHost, st) == hipSuccess ? ZBALHIP_OK : ZBALHIP_RT_ERROR;
}

extern "C" int32_t zbalhip_host_counts_wait(void *block, uint64_t ticket, int64_t n, int64_t *host_counts, void *stream)
{
    if (!block || !host_counts || n < 0 || n > ZB_MAX_EXPERTS) return ZBALHIP_INVALID;
    HostCounts *host = static_cast<HostCounts *>(block);
    bool arrived = false;
    if (ticket != 0) {
        /*
         * The flag arrives a few microseconds after the kernels in front of the notify have run. A stream with long work
         * queued is not spun on for more than a millisecond; the runtime's wait takes over, and reports a stream that
         * will never get there.
         */
        timespec t0, t1;
        clock_gettime(CLOCK_MONOTONIC, &t0);
        for (int spin = 0;; ++spin) {
            arrived = __atomic_load_n(&host->ready, __ATOMIC_ACQUIRE) == ticket;
            if (arrived) break;
            __builtin_ia32_pause();
            if ((spin & 63) != 63) continue;
            clock_gettime(CLOCK_MONOTONIC, &t1);
            if ((t1.tv_sec - t0.tv_sec) * 1000000000ll + (t1.tv_nsec - t0.tv_nsec) > 1000000) break;
        }
    }
    if (!arrived) {
        if (hipStreamSynchronize((hipStream_t)stream) != hipSuccess) return ZBALHIP_RT_ERROR;
        if (ticket != 0 && __atomic_load_n(&host->ready, __ATOMIC_ACQUIRE) != ticket) return ZBALHIP_RT_ERROR;
    }
    for (int64_t e = 0; e < n; ++e) host_counts[e] = host->counts[e];
    return ZBALHIP_OK;
}
