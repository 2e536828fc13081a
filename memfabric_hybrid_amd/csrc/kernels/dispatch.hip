/*
 * Expert-major permutation with fused per-token quantisation.
 *
 * One workgroup owns one source token: the row is read from HBM once (two
 * 16-byte loads per lane per 16 elements), reduced to its absmax (whole row
 * for int8, per 128 columns for e4m3), quantised once in registers and then
 * stored to each of the token's K destination rows with 16-byte stores, so
 * HBM traffic is the algorithmic minimum of one read and K quantised writes.
 * With per-expert smooth scales the quantised row differs per pick and is
 * recomputed per pick from the registers.
 */
#include "zbal_device.h"
#include "zbal_hip_kernels.h"

int32_t zbalhip_layout_ranges_internal(const ExpertIds &idx, int64_t tokens, int64_t experts, int64_t topk,
                                       const uint8_t *active_mask, int32_t *send_token_idx, int32_t *hist, int nblk,
                                       int tokens_per_block, hipStream_t st);

int32_t zbalhip_ll_counts_internal(const int32_t *const *ids, int ranks, int me, int64_t tokens, int64_t topk,
                                   int64_t experts, int32_t token_nums_type, int32_t *all_counts, int32_t *ep_recv_counts,
                                   int64_t *expert_token_nums, hipStream_t st);

int32_t zbalhip_layout_fused_internal(const ExpertIds &idx, int64_t tokens, int64_t experts, int64_t topk,
                                      int32_t token_nums_type, const uint8_t *active_mask, int32_t *send_token_idx,
                                      int32_t *incl_i32, int32_t *row_off, int64_t *counts_i64, int64_t *nums_typed,
                                      hipStream_t st);

namespace {

constexpr int kThreads = 256;
constexpr int kElemsPerLane = 16;

enum { QM_COPY = 0, QM_INT8_EPS = 1, QM_FP8 = 2, QM_INT8_NOEPS = 3 };

/*
 * Where the rows go. Expert e belongs to rank e / e_loc, whose receive window is dest[that rank] (and scale[that
 * rank] for the quantisation scales); on one GPU the windows are local allocations, over xGMI they would be
 * mapped peer memory, the kernel is the same. Offsets are looked up as base[e * ranks + my_rank]: the slot of
 * this sender in the receiver's expert-major, then source-rank order (reference
 * zbal_kernel_notify_dispatch.h:356-378, zbal_kernel_dispatch_normal.h:528-533). rows_cap is the number of rows
 * each window holds; a pick that would land past it is dropped rather than written out of bounds.
 */
struct PeerRows {
    uint8_t *dest[ZBALHIP_MAX_REDUCE_PEERS];
    float *scale[ZBALHIP_MAX_REDUCE_PEERS];
    int ranks, my_rank, e_loc;
    int64_t rows_cap;
};

__device__ __forceinline__ int64_t pick_row(const int32_t *__restrict__ base, int base_inclusive, const PeerRows &pr, int e,
                                            int32_t rank_in_expert)
{
    /* running sums start anew with every destination rank's block of `experts` entries (low-latency counts) */
    const int slot = e * pr.ranks + pr.my_rank;
    const int32_t b = base_inclusive ? (slot % (pr.e_loc * pr.ranks) == 0 ? 0 : base[slot - 1]) : base[slot];
    const int64_t row = (int64_t)b + rank_in_expert;
    return row < pr.rows_cap ? row : -1;
}

/*
 * Small batches: the permute kernel works the layout out itself, with no layout launch in front of it and no dependency
 * between workgroups. A pick's destination row is the number of picks that sort before it (lower expert, or the same
 * expert and an earlier pick), so with at most kInlineMaxPicks picks in all every workgroup reads the whole index array
 * (a few KiB that sit in L2) and each thread compares its share of the picks with those of the workgroup's token, in
 * registers; the counts meet in LDS behind the one barrier that the row's absmax needs anyway. (A histogram in LDS, its
 * scan and the ranks, with a barrier after each, took 10.4 us where this takes 6: 128 tokens of 8 picks, 32 experts.)
 * One workgroup more works the layout's outputs out and does nothing else.
 */
constexpr int kInlineMaxPicks = 4096;
constexpr int kCountByAll = 512;              /* from so many picks on the count wants more threads than a short row has pieces */
constexpr int kInlineMaxTopk = 32;
constexpr int kInlineMaxExperts = 1024;

struct InlineLayout {
    const uint8_t *active_mask;   /* optional: only the first sum(mask) tokens are routed */
    int tokens, token_nums_type;
    int32_t *expand_idx;          /* [T, K] */
    int32_t *incl_i32;            /* [E] running sums */
    int32_t *row_off;             /* [E + 1] exclusive offsets */
    int64_t *counts_i64;          /* [E] */
    int64_t *nums_typed;          /* [E] counts (type 1) or running sums (type 0) */
    int part_shift;               /* log2 of how many workgroups share a token's picks, see inline_part_shift */
};

/* the token of an inline-mode workgroup and which of its picks are this workgroup's: [begin, end) */
struct PickRange {
    int token, begin, end, part;
};
__device__ __forceinline__ PickRange picks_of_block(const InlineLayout &il, int topk)
{
    const int b = (int)blockIdx.x - 1, part = b & ((1 << il.part_shift) - 1);
    return {b >> il.part_shift, (topk * part) >> il.part_shift, (topk * (part + 1)) >> il.part_shift, part};
}

/* how many tokens the mask routes (all of them without one); `s` is one word of LDS; holds barriers if there is a mask */
__device__ __forceinline__ int active_tokens(const uint8_t *mask, int tokens, int32_t *s)
{
    if (mask == nullptr) return tokens;
    if (threadIdx.x == 0) *s = 0;
    __syncthreads();
    int part = 0;
    for (int t = threadIdx.x; t < tokens; t += blockDim.x) part += mask[t] != 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
    if ((threadIdx.x & 63) == 0 && part) atomicAdd(s, part);
    __syncthreads();
    return *s;
}

/* a shared expert: every active token's row once more, row t at first_row + t (end null: none) */
struct SharedRows {
    int64_t first_row;
    int32_t *end;                 /* first_row + active tokens goes here */
    const float *smooth;          /* [H], where the routed experts have smooth scales */
};

/* the layout's outputs, by one workgroup; any of them may be null */
__device__ __forceinline__ void write_inline_layout(const ExpertIds &idx, int topk, int experts, const InlineLayout &il,
                                                    const SharedRows &sh, int32_t *s_hist, int32_t *s_tmp)
{
    const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = tid >> 6;
    for (int e = tid; e < experts; e += nthr) s_hist[e] = 0;
    const int active = active_tokens(il.active_mask, il.tokens, s_tmp), n = active * topk;
    if (sh.end && tid == 0) *sh.end = (int32_t)(sh.first_row + active);
    __syncthreads();
    for (int i0 = tid; i0 < n; i0 += 4 * nthr) {
        int ev[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) ev[u] = i0 + u * nthr < n ? idx[i0 + u * nthr] : -1;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (ev[u] >= 0 && ev[u] < experts) atomicAdd(&s_hist[ev[u]], 1);
    }
    __syncthreads();
    /* a thread owns `chunk` consecutive experts */
    const int chunk = (experts + nthr - 1) / nthr, b0 = tid * chunk;
    int32_t sum = 0;
    for (int j = 0; j < chunk; ++j)
        if (b0 + j < experts) sum += s_hist[b0 + j];
    int32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int32_t o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    if (lane == 63) s_tmp[1 + wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += s_tmp[1 + w];
    int32_t run = incl - sum;
    for (int j = 0; j < chunk && b0 + j < experts; ++j) {
        const int e = b0 + j;
        const int32_t c = s_hist[e];
        if (il.row_off) il.row_off[e] = run;
        if (il.incl_i32) il.incl_i32[e] = run + c;
        if (il.counts_i64) il.counts_i64[e] = c;
        if (il.nums_typed) il.nums_typed[e] = il.token_nums_type == 0 ? (int64_t)(run + c) : (int64_t)c;
        run += c;
        if (e == experts - 1 && il.row_off) il.row_off[experts] = run;
    }
}

/* a token's picks, one per lane (lane k holds pick k, every wave a copy): expert and destination row, -1 where not routed */
struct LanePicks {
    int e;
    int32_t row;
};

/*
 * This wave's part of the counts: lane k returns, for pick k of token r.token, (picks of lower experts) << 16 | (picks that
 * sort before it), over the wave's share of the picks [0, n), for the picks of the range. my_e: lane k's pick. KG: picks per pass
 * over the array.
 */
template <int KG>
__device__ __forceinline__ int32_t count_before(const ExpertIds &idx, const PickRange &r, int topk, int experts, int n, int my_e)
{
    const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63;
    int32_t result = 0;
    for (int k0 = r.begin; k0 < r.end; k0 += KG) {
        int32_t first[KG], self[KG], below[KG], before[KG];
#pragma unroll
        for (int k = 0; k < KG; ++k) {
            const int e = __builtin_amdgcn_readlane(my_e, (k0 + k) & 63);
            first[k] = e << 13;                        /* keys: expert << 13 | pick, kInlineMaxPicks < 2^13 */
            self[k] = first[k] | (r.token * topk + k0 + k);
            below[k] = before[k] = 0;
        }
        auto count = [&](int e, int i) __attribute__((always_inline)) {
            const int key = e >= 0 && e < experts ? (e << 13 | i) : 0x7fffffff;
#pragma unroll
            for (int k = 0; k < KG; ++k) {
                below[k] += key < first[k] ? 1 : 0;
                before[k] += key < self[k] ? 1 : 0;
            }
        };
        /*
         * Four picks in a row per load, four loads in flight: a workgroup has few waves and next to none beside it on its CU, so the
         * count takes as long as its round trips to the L2. Low-latency dispatch, kernel alone (with as many threads as kCountByAll
         * wants): 2048 wide, 512 tokens of 6 picks, rows as they are 11.2 -> 9.2 us, 300 tokens, int8 9.9 -> 7.4; dispatch and combine,
         * 512 tokens, int8: 7168 wide, 8 picks 30.3 -> 27.1, 4096 wide 23.2 -> 20.4, 2048 wide 17.8 -> 14.6.
         */
        const int whole = n & ~3;
        for (int i0 = tid * 4; i0 < whole; i0 += 16 * nthr) {
            i32x4 e[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) e[u] = i0 + u * 4 * nthr < whole ? idx.four(i0 + u * 4 * nthr) : i32x4{-1, -1, -1, -1};
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (u > 0 && whole <= u * 4 * nthr) break;
#pragma unroll
                for (int j = 0; j < 4; ++j) count(e[u][j], i0 + u * 4 * nthr + j);
            }
        }
        if (whole + tid < n) count(idx[whole + tid], whole + tid);
#pragma unroll
        for (int k = 0; k < KG; ++k) {
            const int32_t sum = zb_wave_sum_dpp(below[k] << 16 | before[k]);
            if (lane == k0 + k) result = sum;
        }
    }
    return result;
}

/*
 * Large batches: the layout launch in front of the permute only ranks the picks within token ranges and leaves one
 * histogram per range (layout_ranges_kernel); what is left of the layout -- how many picks of an expert the ranges
 * before a token's own hold, and the experts' first rows -- every permute workgroup works out for itself from that
 * small table while its row is on its way from HBM: no workgroup of either launch waits for another, and the layout
 * launch is a third of what it was. Workgroup 0 also writes the offsets and counts the stages after the permute read.
 */
constexpr int kTableMaxEntries = 2048;        /* ranges x experts */
constexpr int kTableMaxExperts = 256;         /* one expert per thread in the scan */

struct RangeTable {
    const int32_t *hist;          /* [ranges][experts] */
    int ranges, tokens_per_range;
    int32_t *expand_idx;          /* [T, K]: in, the rank within the range; out, the rank within the expert */
    int32_t *row_off;             /* [E + 1] */
    int64_t *counts_i64;          /* [E] */
};

constexpr int kTablePerThread = kTableMaxEntries / kThreads;

/* the table's entries tid, tid + kThreads, ...: requested before the row, so that they arrive first (a wave's loads return in order) */
__device__ __forceinline__ void table_request(const RangeTable &rt, int experts, int32_t (&tabv)[kTablePerThread])
{
    const int n = rt.ranges * experts;
#pragma unroll
    for (int j = 0; j < kTablePerThread; ++j) {
        const int i = j * kThreads + (int)threadIdx.x;
        tabv[j] = i < n ? rt.hist[i] : 0;
    }
}

/* On return s_first[e] = first row of expert e, s_before[e] = picks of expert e in the ranges before `range`. */
__device__ __forceinline__ void table_layout(const RangeTable &rt, const int32_t (&tabv)[kTablePerThread], int range,
                                             int experts, bool writer, int32_t *s_tab, int32_t *s_first, int32_t *s_before,
                                             int32_t *s_tmp)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int j = 0; j < kTablePerThread; ++j) s_tab[j * kThreads + tid] = tabv[j];
    __syncthreads();
    int32_t c = 0;
    if (tid < experts) {
        int32_t bef = 0;
        for (int r = 0; r < rt.ranges; ++r) {
            const int32_t v = s_tab[r * experts + tid];
            c += v;
            if (r < range) bef += v;
        }
        s_before[tid] = bef;
    }
    int32_t incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int32_t o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    if (lane == 63) s_tmp[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += s_tmp[w];
    if (tid < experts) {
        s_first[tid] = incl - c;
        if (writer) {
            rt.row_off[tid] = incl - c;
            if (rt.counts_i64) rt.counts_i64[tid] = c;
            if (tid == experts - 1) rt.row_off[experts] = incl;
        }
    }
    __syncthreads();
}

/* 16 consecutive 16-bit elements (two 16-byte loads) as fp32 */
template <int XDT> __device__ __forceinline__ void cvt16(const u32x4 &a, const u32x4 &b, float (&v)[16])
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = zb_half_to_f32<XDT>(a[i] & 0xffffu);
        v[2 * i + 1] = zb_half_to_f32<XDT>(a[i] >> 16);
        v[8 + 2 * i] = zb_half_to_f32<XDT>(b[i] & 0xffffu);
        v[8 + 2 * i + 1] = zb_half_to_f32<XDT>(b[i] >> 16);
    }
}

__device__ __forceinline__ u32x4 pack16_i8(const float (&v)[16], float s)
{
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = zb_pack4_i8(v[4 * i] * s, v[4 * i + 1] * s, v[4 * i + 2] * s, v[4 * i + 3] * s);
    return o;
}

__device__ __forceinline__ u32x4 pack16_e4m3(const float (&v)[16], float mult)
{
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = zb_cvt_pk_e4m3(v[4 * i] * mult, v[4 * i + 1] * mult);
        const uint32_t hi = zb_cvt_pk_e4m3(v[4 * i + 2] * mult, v[4 * i + 3] * mult);
        o[i] = lo | (hi << 16);
    }
    return o;
}

/*
 * SLOTS = ceil(H / 16 / blockDim): 16-element segments each lane keeps in registers.
 * QM: quant flavour. SMOOTH: per-expert fp32 multipliers [E,H] (int8 only).
 */
enum { LM_GIVEN = 0, LM_INLINE = 1, LM_TABLE = 2, LM_COUNTS = 3 };     /* where ranks and offsets come from */

/*
 * Notify and dispatch of a group of one rank in one launch: the offsets are the running sum of at most 1024 counts, which
 * every wave of the permute kernel works out for itself while its row is on its way (a launch of its own in front took
 * 2-5 us of the GPU and 3 us of the host: 24.3 -> 21.5 us for the whole exchange of 64 to 512 tokens). The first wave of
 * all writes what a notify launch would. Where the host waits for the counts, a launch of its own has them there sooner
 * (26 us for that exchange, 28 with the notify riding along), and it is what runs then.
 */
struct NotifyOut {
    const int32_t *counts;        /* [experts] */
    int32_t *recv_data, *put_offset, *total, *balance;
    int64_t *recv_per_expert;
};
constexpr int kCountsPerLane = kInlineMaxExperts / 64;

/* lane l's counts: experts l * per .. (l + 1) * per - 1, per = ceil(experts / 64) */
__device__ __forceinline__ void request_counts(const NotifyOut &no, int experts, int32_t (&c)[kCountsPerLane])
{
    const int per = (experts + 63) / 64, e0 = (threadIdx.x & 63) * per;
#pragma unroll
    for (int j = 0; j < kCountsPerLane; ++j) c[j] = j < per && e0 + j < experts ? no.counts[e0 + j] : 0;
}

/* s_off[e] = first row of expert e; every wave writes all of it, the same values, and reads only what it has written itself */
__device__ __forceinline__ void counts_to_offsets(const NotifyOut &no, int experts, int topk, bool writer,
                                                  const int32_t (&c)[kCountsPerLane], int32_t *s_off)
{
    const int lane = threadIdx.x & 63, per = (experts + 63) / 64, e0 = lane * per;
    int32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kCountsPerLane; ++j) sum += c[j];
    int32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int32_t o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    int32_t run = incl - sum;
#pragma unroll
    for (int j = 0; j < kCountsPerLane; ++j) {
        const int e = e0 + j;
        if (j >= per || e >= experts) continue;
        s_off[e] = run;
        if (writer) {
            no.recv_data[e] = c[j];
            no.put_offset[e] = run;
            no.recv_per_expert[e] = c[j];
            if (e == experts - 1) {
                const int32_t total = run + c[j], bs = total / topk;
                *no.total = total;
                no.balance[0] = bs > 0 ? 0 : -1;
                no.balance[1] = bs > 0 ? bs - 1 : -1;
            }
        }
        run += c[j];
    }
}

/*
 * Picks k0 + lane of token t where ranks and offsets come from a layout launch. The index and rank loads go out before
 * the row's, the offset's (which depends on them) after: resolve_given takes them up.
 */
struct GivenPicks {
    int e;
    int32_t rank;
};
__device__ __forceinline__ GivenPicks request_given(const ExpertIds &idx, const int32_t *__restrict__ rank_in_expert, int t, int topk, int k)
{
    GivenPicks g = {-1, -1};
    if (k < topk) {
        g.e = idx[(int64_t)t * topk + k];
        g.rank = rank_in_expert[(int64_t)t * topk + k];
    }
    return g;
}
__device__ __forceinline__ LanePicks resolve_given(const GivenPicks &g, const int32_t *__restrict__ base, int base_inclusive,
                                                   int experts, const PeerRows &pr)
{
    LanePicks p = {g.e, -1};
    /* rank < 0: the layout masked this token out */
    if (g.e >= 0 && g.e < experts && g.rank >= 0) p.row = (int32_t)pick_row(base, base_inclusive, pr, g.e, g.rank);
    return p;
}

/* the same with the offsets in LDS (LM_COUNTS) */
__device__ __forceinline__ LanePicks resolve_counts(const GivenPicks &g, const int32_t *s_off, int experts, const PeerRows &pr)
{
    LanePicks p = {g.e, -1};
    if (g.e >= 0 && g.e < experts && g.rank >= 0) {
        const int64_t row = (int64_t)s_off[g.e] + g.rank;
        if (row < pr.rows_cap) p.row = (int32_t)row;
    }
    return p;
}

/* window of the rank that owns expert e */
__device__ __forceinline__ int window_of(const PeerRows &pr, int e) { return pr.ranks == 1 ? 0 : e / pr.e_loc; }

/*
 * The workgroup's token (or its share of one) in inline mode, in two halves with one barrier of the caller's between them: the wave's counts
 * go to LDS, their sums come back as destination rows. Writes the token's expand_idx.
 */
__device__ __forceinline__ void inline_counts(const ExpertIds &idx, const PickRange &r, int topk, int experts, int active, int my_e,
                                              const InlineLayout &il, int32_t (*s_cnt)[kInlineMaxTopk])
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int32_t c = il.part_shift > 0 ? count_before<2>(idx, r, topk, experts, active * topk, my_e)
                                        : count_before<8>(idx, r, topk, experts, active * topk, my_e);
    if (lane < topk) s_cnt[wave][lane] = c;
}
__device__ __forceinline__ LanePicks inline_rows(const PickRange &r, int topk, int experts, int active, int my_e, const InlineLayout &il,
                                                 const PeerRows &pr, int32_t (*s_cnt)[kInlineMaxTopk])
{
    const int lane = threadIdx.x & 63, nwaves = (blockDim.x + 63) >> 6;
    LanePicks p = {my_e, -1};
    if (lane >= r.begin && lane < r.end) {
        int32_t c = 0;
        for (int w = 0; w < nwaves; ++w) c += s_cnt[w][lane];
        const bool valid = my_e >= 0 && my_e < experts, routed = valid && r.token < active;
        const int32_t row = c & 0xffff, rank = r.token >= active ? -2 : (valid ? row - (c >> 16) : -1);
        if (routed && row < pr.rows_cap) p.row = row;
        if (threadIdx.x < 64) il.expand_idx[(int64_t)r.token * topk + lane] = rank;
    }
    return p;
}

template <int XDT, int QM, int SLOTS, bool SMOOTH, int LM>
__global__ void __launch_bounds__(kThreads)
permute_quant_kernel(const uint16_t *__restrict__ x, ExpertIds topk_idx,
                     const int32_t *__restrict__ rank_in_expert, const int32_t *__restrict__ base, int base_inclusive,
                     const float *__restrict__ smooth, int hidden, int topk, int experts, PeerRows pr, InlineLayout il,
                     RangeTable rt, SharedRows sh, NotifyOut no, uint32_t *__restrict__ clear_words, int64_t clear_count)
{
    constexpr bool INLINE = LM == LM_INLINE, TABLE = LM == LM_TABLE, COUNTS = LM == LM_COUNTS;
    __shared__ float red[kThreads / 64];
    __shared__ int32_t s_off[INLINE || COUNTS ? kInlineMaxExperts : (TABLE ? kTableMaxExperts : 1)];
    __shared__ int32_t s_before[TABLE ? kTableMaxExperts : 1], s_tab[TABLE ? kTableMaxEntries : 1];
    __shared__ int32_t s_cnt[kThreads / 64][kInlineMaxTopk], s_tmp[8];
    const int lane = threadIdx.x & 63;
    const int nseg = hidden / kElemsPerLane;
    /* words the next stage wants at zero (the row maxima the int modes' first GEMM accumulates into) */
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < clear_count; i += (int64_t)gridDim.x * blockDim.x)
        clear_words[i] = 0u;
    if (INLINE && blockIdx.x == 0) {
        write_inline_layout(topk_idx, topk, experts, il, sh, s_off, s_tmp);
        return;
    }
    const PickRange mine = INLINE ? picks_of_block(il, topk) : PickRange{(int)blockIdx.x, 0, topk, 0};
    const int t = mine.token;
    if (!INLINE && sh.end && t == 0) {
        const int n = active_tokens(il.active_mask, il.tokens, s_tmp);
        if (threadIdx.x == 0) *sh.end = (int32_t)(sh.first_row + n);
    }
    /*
     * Where the token's picks go is worked out by one lane per pick, in every wave, while the row is on its way (the
     * picks' index, rank and offset loads depend on each other: done pick after pick inside the store loop they cost
     * topk round trips to L2 per workgroup).
     */
    GivenPicks given = {-1, -1};
    if (INLINE) given.e = lane < topk ? topk_idx[(int64_t)t * topk + lane] : -1;
    else given = request_given(topk_idx, TABLE ? rt.expand_idx : rank_in_expert, t, topk, lane);
    int32_t tabv[TABLE ? kTablePerThread : 1];
    if constexpr (TABLE) table_request(rt, experts, tabv);
    int32_t cnt[COUNTS ? kCountsPerLane : 1];
    if constexpr (COUNTS) request_counts(no, experts, cnt);
    /* the row is requested here (streamed: it is read once) and first used after the picks are resolved: the two latencies overlap */
    u32x4 raw[SLOTS][2];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
        const int seg = s * blockDim.x + threadIdx.x;
        raw[s][0] = raw[s][1] = u32x4{0u, 0u, 0u, 0u};
        if (seg < nseg) {
            raw[s][0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x + (int64_t)t * hidden + (int64_t)seg * 16));
            raw[s][1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x + (int64_t)t * hidden + (int64_t)seg * 16 + 8));
        }
    }
    LanePicks picks = {-1, -1};
    int active = 0;
    if constexpr (INLINE) {
        active = active_tokens(il.active_mask, il.tokens, s_tmp);
        inline_counts(topk_idx, mine, topk, experts, active, given.e, il, s_cnt);
    } else if constexpr (TABLE) {
        table_layout(rt, tabv, t / rt.tokens_per_range, experts, t == 0, s_tab, s_off, s_before, s_tmp);
        picks.e = given.e;
        if (given.e >= 0 && given.e < experts && given.rank >= 0) {       /* rank < 0: the layout masked this token out */
            const int32_t rk = s_before[given.e] + given.rank, row = s_off[given.e] + rk;
            if (threadIdx.x < 64) rt.expand_idx[(int64_t)t * topk + lane] = rk;   /* the rank within the expert: what the combine reads */
            if (row < pr.rows_cap) picks.row = row;
        }
    } else if constexpr (COUNTS) {
        counts_to_offsets(no, experts, topk, t == 0 && threadIdx.x < 64, cnt, s_off);
        picks = resolve_counts(given, s_off, experts, pr);
    } else {
        picks = resolve_given(given, base, base_inclusive, experts, pr);
    }
    float v[SLOTS][16];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) cvt16<XDT>(raw[s][0], raw[s][1], v[s]);
    constexpr bool ROW_MAX = QM != QM_FP8 && !SMOOTH;
    if constexpr (ROW_MAX) {
        float amax = 0.0f;
#pragma unroll
        for (int s = 0; s < SLOTS; ++s)
#pragma unroll
            for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[s][i]));
        amax = zb_wave_reduce_dpp<true>(amax);
        if (lane == 0) red[threadIdx.x >> 6] = amax;
    }
    if constexpr (ROW_MAX || INLINE) __syncthreads();
    if constexpr (INLINE) picks = inline_rows(mine, topk, experts, active, given.e, il, pr, s_cnt);
    /* rank -2: the layout masked the token out */
    const bool shares = sh.end && (INLINE ? mine.part == 0 && t < active : __builtin_amdgcn_readlane(given.rank, 0) != -2);
    /* f(pick's expert, window, row) for every routed pick of the token, and for the shared expert (-1); wave-uniform */
    auto for_each_pick = [&](auto f) __attribute__((always_inline)) {
        for (int k0 = 0; k0 < topk; k0 += 64) {
            if (COUNTS && k0 > 0)
                picks = resolve_counts(request_given(topk_idx, rank_in_expert, t, topk, k0 + lane), s_off, experts, pr);
            else if (!INLINE && !TABLE && k0 > 0)
                picks = resolve_given(request_given(topk_idx, rank_in_expert, t, topk, k0 + lane), base, base_inclusive, experts, pr);
            const int n = INLINE ? mine.end : (topk - k0 < 64 ? topk - k0 : 64);
            for (int k = INLINE ? mine.begin : 0; k < n; ++k) {
                const int32_t row = __builtin_amdgcn_readlane(picks.row, k);
                if (row < 0) continue;
                const int e = __builtin_amdgcn_readlane(picks.e, k);
                f(e, window_of(pr, e), (int64_t)row);
            }
        }
        if (shares) f(-1, 0, sh.first_row + t);
    };

    if constexpr (QM == QM_FP8) {
        /* eight consecutive lanes share one 128-column block */
        u32x4 q[SLOTS];
        float sc[SLOTS];
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[s][i]));
            amax = zb_group_max<3>(amax);
            amax = fmaxf(amax, 1e-4f);
            const float mult = 448.0f / amax;
            q[s] = pack16_e4m3(v[s], mult);
            sc[s] = amax * (1.0f / 448.0f);
        }
        const int nblk128 = hidden / 128;
        for_each_pick([&](int, int win, int64_t row) __attribute__((always_inline)) {
            uint8_t *dest = pr.dest[win];
            float *dest_scale = pr.scale[win];
#pragma unroll
            for (int s = 0; s < SLOTS; ++s) {
                const int seg = s * blockDim.x + threadIdx.x;
                if (seg < nseg) {
                    *reinterpret_cast<u32x4 *>(dest + row * hidden + (int64_t)seg * 16) = q[s];
                    if ((seg & 7) == 0) dest_scale[row * nblk128 + (seg >> 3)] = sc[s];
                }
            }
        });
    } else if constexpr (!SMOOTH) {
        float amax = red[0];
        for (int w = 1; w < (int)((blockDim.x + 63) >> 6); ++w) amax = fmaxf(amax, red[w]);
        float sq, stored;
        if (QM == QM_INT8_NOEPS && amax == 0.0f) { sq = 0.0f; stored = 0.0f; }
        else {
            sq = (QM == QM_INT8_EPS) ? 127.0f / (amax + 1e-12f) : 127.0f / amax;
            stored = 1.0f / sq;
        }
        u32x4 q[SLOTS];
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) q[s] = pack16_i8(v[s], sq);
        for_each_pick([&](int, int win, int64_t row) __attribute__((always_inline)) {
            uint8_t *dest = pr.dest[win];
#pragma unroll
            for (int s = 0; s < SLOTS; ++s) {
                const int seg = s * blockDim.x + threadIdx.x;
                if (seg < nseg)
                    *reinterpret_cast<u32x4 *>(dest + row * hidden + (int64_t)seg * 16) = q[s];
            }
            if (threadIdx.x == 0) pr.scale[win][row] = stored;
        });
    } else {
        for_each_pick([&](int e, int win, int64_t row) __attribute__((always_inline)) {
            uint8_t *dest = pr.dest[win];
            const float *sm = e < 0 ? sh.smooth : smooth + (int64_t)e * hidden;
            float sv[SLOTS][16];
            float amax = 0.0f;
#pragma unroll
            for (int s = 0; s < SLOTS; ++s) {
                const int seg = s * blockDim.x + threadIdx.x;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float m = (seg < nseg) ? sm[seg * 16 + i] : 0.0f;
                    sv[s][i] = v[s][i] * m;
                    amax = fmaxf(amax, fabsf(sv[s][i]));
                }
            }
            amax = zb_block_max(amax, red);
            float sq, stored;
            if (amax == 0.0f) { sq = 0.0f; stored = 0.0f; }
            else { sq = 127.0f / amax; stored = 1.0f / sq; }
#pragma unroll
            for (int s = 0; s < SLOTS; ++s) {
                const int seg = s * blockDim.x + threadIdx.x;
                if (seg < nseg) {
                    const u32x4 q = pack16_i8(sv[s], sq);
                    *reinterpret_cast<u32x4 *>(dest + row * hidden + (int64_t)seg * 16) = q;
                }
            }
            if (threadIdx.x == 0) pr.scale[win][row] = stored;
        });
    }
}

/* plain row copy (no quantisation): 16-byte chunks of 8 elements, UNROLL of them per lane and pass */
template <int LM, int UNROLL>
__global__ void __launch_bounds__(kThreads)
permute_copy_kernel(const uint16_t *__restrict__ x, ExpertIds topk_idx,
                    const int32_t *__restrict__ rank_in_expert, const int32_t *__restrict__ base, int base_inclusive,
                    int hidden, int topk, int experts, PeerRows pr, InlineLayout il, NotifyOut no)
{
    constexpr bool INLINE = LM == LM_INLINE, COUNTS = LM == LM_COUNTS;
    __shared__ int32_t s_off[INLINE || COUNTS ? kInlineMaxExperts : 1], s_cnt[kThreads / 64][kInlineMaxTopk], s_tmp[8];
    if (INLINE && blockIdx.x == 0) {
        write_inline_layout(topk_idx, topk, experts, il, SharedRows{}, s_off, s_tmp);
        return;
    }
    const PickRange mine = INLINE ? picks_of_block(il, topk) : PickRange{(int)blockIdx.x, 0, topk, 0};
    const int t = mine.token, lane = threadIdx.x & 63;
    const int nchunk = hidden / 8;
    const u32x4 *src = reinterpret_cast<const u32x4 *>(x + (int64_t)t * hidden);
    GivenPicks given = {-1, -1};
    if (INLINE) given.e = lane < topk ? topk_idx[(int64_t)t * topk + lane] : -1;
    else given = request_given(topk_idx, rank_in_expert, t, topk, lane);
    int32_t cnt[COUNTS ? kCountsPerLane : 1];
    if constexpr (COUNTS) request_counts(no, experts, cnt);
    u32x4 v[UNROLL];
    auto load = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int c = c0 + u * blockDim.x + threadIdx.x;
            if (c < nchunk) v[u] = __builtin_nontemporal_load(src + c);
        }
    };
    load(0);
    LanePicks first;
    if constexpr (INLINE) {
        const int active = active_tokens(il.active_mask, il.tokens, s_tmp);
        inline_counts(topk_idx, mine, topk, experts, active, given.e, il, s_cnt);
        __syncthreads();
        first = inline_rows(mine, topk, experts, active, given.e, il, pr, s_cnt);
    } else if constexpr (COUNTS) {
        counts_to_offsets(no, experts, topk, t == 0 && threadIdx.x < 64, cnt, s_off);
        first = resolve_counts(given, s_off, experts, pr);
    } else {
        first = resolve_given(given, base, base_inclusive, experts, pr);
    }
    for (int c0 = 0; c0 < nchunk; c0 += blockDim.x * UNROLL) {
        if (c0 > 0) load(c0);
        LanePicks picks = first;
        for (int k0 = 0; k0 < topk; k0 += 64) {
            if (COUNTS && k0 > 0)
                picks = resolve_counts(request_given(topk_idx, rank_in_expert, t, topk, k0 + lane), s_off, experts, pr);
            else if (!INLINE && k0 > 0)
                picks = resolve_given(request_given(topk_idx, rank_in_expert, t, topk, k0 + lane), base, base_inclusive, experts, pr);
            const int n = INLINE ? mine.end : (topk - k0 < 64 ? topk - k0 : 64);
            for (int k = INLINE ? mine.begin : 0; k < n; ++k) {
                const int32_t row = __builtin_amdgcn_readlane(picks.row, k);
                if (row < 0) continue;
                u32x4 *dest = reinterpret_cast<u32x4 *>(pr.dest[window_of(pr, __builtin_amdgcn_readlane(picks.e, k))] + (int64_t)row * hidden * 2);
#pragma unroll
                for (int u = 0; u < UNROLL; ++u) {
                    const int c = c0 + u * blockDim.x + threadIdx.x;
                    if (c < nchunk) dest[c] = v[u];       /* (non-temporal stores: 4096 x 7168 3-5 % slower) */
                }
            }
        }
    }
}

/* what a permute launch does besides permuting: work out the layout itself (small batches), clear words for the next stage */
struct PermuteExtras {
    const InlineLayout *inline_layout;     /* null: ranks and offsets come from the layout launch */
    uint32_t *clear_words;
    int64_t clear_count;
    const RangeTable *range_table;         /* non-null: ranks within token ranges + the ranges' histograms (large batches) */
    SharedRows shared;
    const uint8_t *active_mask;            /* with a shared expert, whatever the layout comes from */
    const NotifyOut *notify = nullptr;     /* offsets from counts, and what a notify launch writes */
};

/*
 * Fewer tokens than half of the CUs: up to eight workgroups, as many as make one for each of the 256 CUs, share a token's picks. Each reads
 * the row and its scale for itself, but counts for its own picks and stores their rows only, and that is what a lone workgroup spends its
 * time on (one token of 8 picks, 7168 wide, int8: 1.5 us of 4.5 each, a CU storing 50 GB/s). The kernel alone: 1 token 5.31 -> 3.68 us,
 * 7 tokens 5.53 -> 3.83 (rows as they are 5.05 -> 3.31), 32 of 4096, 128 experts 5.29 -> 3.75, 64 of 7168 5.94 -> 4.80, of 2048 4.64 -> 3.40,
 * 128 6.58 -> 6.33; two per CU: 64 tokens 6.37, 128 6.96, 512 12.6 -> 15.5.
 */
inline int inline_part_shift(int64_t tokens)
{
    int shift = 0;
    while (shift < 3 && tokens << (shift + 1) <= 256) ++shift;
    return shift;
}

template <int XDT, int QM, bool SMOOTH>
int32_t launch_quant(const void *x, const ExpertIds &topk_idx, const int32_t *rank_in_expert, const int32_t *base,
                     int base_inclusive, const float *smooth, int64_t tokens, int64_t hidden, int64_t topk,
                     int64_t experts, const PeerRows &pr, const PermuteExtras &ex, hipStream_t st)
{
    const int nseg = (int)(hidden / kElemsPerLane);
    int threads = (nseg + 63) / 64 * 64;
    if (threads > kThreads) threads = kThreads;
    if (ex.range_table) threads = kThreads;       /* the table's scan gives every expert a thread */
    if (ex.inline_layout && tokens * topk > kCountByAll) threads = kThreads;
    const int slots = (nseg + threads - 1) / threads;
    InlineLayout il = ex.inline_layout ? *ex.inline_layout : InlineLayout{};
    if (ex.inline_layout) il.part_shift = inline_part_shift(tokens);
    else {
        il.active_mask = ex.active_mask;
        il.tokens = (int)tokens;
    }
    const RangeTable rt = ex.range_table ? *ex.range_table : RangeTable{};
    const NotifyOut no = ex.notify ? *ex.notify : NotifyOut{};
    constexpr bool NOTIFIES = !SMOOTH && QM != QM_INT8_NOEPS;      /* the quantisations of the normal-mode dispatch */
#define ZB_LAUNCH_I(S, LMV)                                                                                       \
    zb_launch(permute_quant_kernel<XDT, QM, S, SMOOTH, LMV>, (unsigned)(LMV == LM_INLINE ? (tokens << il.part_shift) + 1 : tokens), threads, 0, st, \
        (const uint16_t *)x, topk_idx, rank_in_expert, base, base_inclusive, smooth, (int)hidden, (int)topk,       \
        (int)experts, pr, il, rt, ex.shared, no, ex.clear_words, ex.clear_count)
#define ZB_LAUNCH(S)                                                                                              \
    do {                                                                                                          \
        if (ex.inline_layout) ZB_LAUNCH_I(S, LM_INLINE);                                                          \
        else if (ex.range_table) ZB_LAUNCH_I(S, LM_TABLE);                                                        \
        else if (NOTIFIES && ex.notify) ZB_LAUNCH_I(S, (NOTIFIES ? LM_COUNTS : LM_GIVEN));                         \
        else ZB_LAUNCH_I(S, LM_GIVEN);                                                                            \
    } while (0)
    if (slots <= 1) ZB_LAUNCH(1);
    else if (slots <= 2) ZB_LAUNCH(2);
    else if (slots <= 4) ZB_LAUNCH(4);
    else return ZBALHIP_INVALID;
#undef ZB_LAUNCH
#undef ZB_LAUNCH_I
    return zbalhip_check_launch();
}

} // namespace

/*
 * Shared by the three public launchers. quant: QM_* flavour. `base` is the
 * exclusive (or inclusive) per-expert row offset table on the device; `pr`
 * says where each rank's rows go.
 */
static int32_t permute_launch(const void *x, int32_t x_dtype, const ExpertIds &topk_idx, const int32_t *rank_in_expert,
                              const int32_t *base, int base_inclusive, const float *smooth, int64_t tokens,
                              int64_t hidden, int64_t topk, int64_t experts, int quant, const PeerRows &pr, hipStream_t st,
                              const PermuteExtras &ex = PermuteExtras{})
{
    if (x_dtype != ZDT_BF16 && x_dtype != ZDT_FP16) return ZBALHIP_INVALID;
    if (hidden <= 0 || hidden > 16 * kThreads * 4 || topk <= 0 || tokens < 0) return ZBALHIP_INVALID;
    if (tokens == 0) return ZBALHIP_OK;
    if (quant == QM_COPY) {
        if (hidden % 8 != 0 || ex.range_table || ex.clear_count) return ZBALHIP_INVALID;
        const int nchunk = (int)(hidden / 8);
        int threads = (nchunk + 63) / 64 * 64;
        if (threads > kThreads) threads = kThreads;
        if (ex.inline_layout && tokens * topk > kCountByAll) threads = kThreads;
        if (ex.inline_layout) {
            InlineLayout il = *ex.inline_layout;
            il.part_shift = inline_part_shift(tokens);
            zb_launch(permute_copy_kernel<LM_INLINE, 4>, (unsigned)(tokens << il.part_shift) + 1, threads, 0, st,
                (const uint16_t *)x, topk_idx, rank_in_expert, base, base_inclusive, (int)hidden, (int)topk, (int)experts, pr,
                il, NotifyOut{});
        }
        else if (ex.notify)
            zb_launch(permute_copy_kernel<LM_COUNTS, 4>, (unsigned)tokens, threads, 0, st,
                (const uint16_t *)x, topk_idx, rank_in_expert, base, base_inclusive, (int)hidden, (int)topk, (int)experts, pr,
                InlineLayout{}, *ex.notify);
        else
            zb_launch(permute_copy_kernel<LM_GIVEN, 4>, (unsigned)tokens, threads, 0, st,
                (const uint16_t *)x, topk_idx, rank_in_expert, base, base_inclusive, (int)hidden, (int)topk, (int)experts, pr,
                InlineLayout{}, NotifyOut{});
        return zbalhip_check_launch();
    }
    if (hidden % 16 != 0 || (quant == QM_FP8 && hidden % 128 != 0)) return ZBALHIP_INVALID;
    const bool bf = (x_dtype == ZDT_BF16);
#define ZB_GO(QMV, SM)                                                                                               \
    return bf ? launch_quant<ZDT_BF16, QMV, SM>(x, topk_idx, rank_in_expert, base, base_inclusive, smooth, tokens,  \
                                                 hidden, topk, experts, pr, ex, st)                                  \
              : launch_quant<ZDT_FP16, QMV, SM>(x, topk_idx, rank_in_expert, base, base_inclusive, smooth, tokens,  \
                                                 hidden, topk, experts, pr, ex, st)
    if (quant == QM_FP8) { ZB_GO(QM_FP8, false); }
    if (quant == QM_INT8_EPS) { ZB_GO(QM_INT8_EPS, false); }
    if (quant == QM_INT8_NOEPS) {
        if (smooth) { ZB_GO(QM_INT8_NOEPS, true); }
        ZB_GO(QM_INT8_NOEPS, false);
    }
#undef ZB_GO
    return ZBALHIP_INVALID;
}

/* the permute kernel can work the layout out itself when the batch is this small (InlineLayout above) */
static bool layout_fits_inline(int64_t tokens, int64_t topk, int64_t experts)
{
    return tokens > 0 && tokens * topk <= kInlineMaxPicks && topk <= kInlineMaxTopk &&
           experts <= kInlineMaxExperts;
}

/* one rank that owns every expert: all rows go to `dest` */
static PeerRows single_window(void *dest, float *dest_scale, int64_t experts, int64_t rows_cap)
{
    PeerRows pr = {};
    pr.dest[0] = (uint8_t *)dest;
    pr.scale[0] = dest_scale;
    pr.ranks = 1;
    pr.my_rank = 0;
    pr.e_loc = (int)experts;
    pr.rows_cap = rows_cap;
    return pr;
}

extern "C" int32_t zbalhip_dispatch_normal(const void *x, int32_t x_dtype, const int32_t *topk_idx,
                                           const int32_t *send_token_idx, const int32_t *put_offset, int64_t tokens,
                                           int64_t hidden, int64_t topk, int64_t experts, int32_t quant_mode,
                                           void *const *dest, float *const *dest_scale, int32_t ranks, int32_t my_rank,
                                           int64_t dest_rows, void *stream)
{
    if (!x || !topk_idx || !send_token_idx || !put_offset || !dest) return ZBALHIP_INVALID;
    const ExpertIds ids = expert_ids(topk_idx, (quant_mode & ZBALHIP_IDS_ARE_I64) != 0);
    quant_mode &= ~ZBALHIP_IDS_ARE_I64;
    if (experts <= 0 || quant_mode < 0 || quant_mode > 2) return ZBALHIP_INVALID;
    if (ranks <= 0 || ranks > ZBALHIP_MAX_REDUCE_PEERS || my_rank < 0 || my_rank >= ranks || experts % ranks != 0 || dest_rows < 0)
        return ZBALHIP_INVALID;
    if (quant_mode != 0 && !dest_scale) return ZBALHIP_INVALID;
    PeerRows pr = {};
    for (int r = 0; r < ranks; ++r) {
        if (!dest[r] || (quant_mode != 0 && !dest_scale[r])) return ZBALHIP_INVALID;
        pr.dest[r] = (uint8_t *)dest[r];
        pr.scale[r] = quant_mode != 0 ? dest_scale[r] : nullptr;
    }
    pr.ranks = ranks;
    pr.my_rank = my_rank;
    pr.e_loc = (int)(experts / ranks);
    pr.rows_cap = dest_rows;
    const int q = quant_mode == 0 ? QM_COPY : (quant_mode == 1 ? QM_INT8_EPS : QM_FP8);
    return permute_launch(x, x_dtype, ids, send_token_idx, put_offset, 0, nullptr, tokens, hidden, topk, experts, q, pr,
                          (hipStream_t)stream);
}

extern "C" int32_t zbalhip_dispatch_normal_notified(const void *x, int32_t x_dtype, const int32_t *topk_idx,
                                                    const int32_t *send_token_idx, const zbalhip_notify_t *notify, int64_t tokens,
                                                    int64_t hidden, int64_t topk, int64_t experts, int32_t quant_mode, void *dest,
                                                    float *dest_scale, int64_t dest_rows, void *stream)
{
    if (!x || !topk_idx || !send_token_idx || !notify || !dest) return ZBALHIP_INVALID;
    const ExpertIds ids = expert_ids(topk_idx, (quant_mode & ZBALHIP_IDS_ARE_I64) != 0);
    quant_mode &= ~ZBALHIP_IDS_ARE_I64;
    if (tokens <= 0 || topk <= 0 || experts <= 0 || experts > kInlineMaxExperts || quant_mode < 0 || quant_mode > 2 || dest_rows < 0)
        return ZBALHIP_INVALID;
    if (quant_mode != 0 && !dest_scale) return ZBALHIP_INVALID;
    if (!notify->tokens_per_expert || !notify->recv_data || !notify->put_offset || !notify->total_recv ||
        !notify->recv_tokens_per_expert || !notify->balance_matrix)
        return ZBALHIP_INVALID;
    hipStream_t st = (hipStream_t)stream;
    const NotifyOut no = {notify->tokens_per_expert, notify->recv_data, notify->put_offset, notify->total_recv, notify->balance_matrix,
                          notify->recv_tokens_per_expert};
    const int q = quant_mode == 0 ? QM_COPY : (quant_mode == 1 ? QM_INT8_EPS : QM_FP8);
    PermuteExtras ex = {};
    ex.notify = &no;
    return permute_launch(x, x_dtype, ids, send_token_idx, nullptr, 0, nullptr, tokens, hidden, topk, experts, q,
                          single_window(dest, dest_scale, experts, dest_rows), st, ex);
}

extern "C" int32_t zbalhip_dispatch_low_latency(const void *x, int32_t x_dtype, const int32_t *expert_ids,
                                                int64_t tokens, int64_t hidden, int64_t topk, int64_t experts,
                                                int32_t quant_mode, int32_t token_nums_type, void *expand_x,
                                                float *dynamic_scales, int32_t *expand_idx, int64_t *expert_token_nums,
                                                int32_t *ep_recv_counts, int32_t *scratch, int32_t scratch_blocks,
                                                void *stream)
{
    /* an empty batch has no per-token data: only the counts are written */
    if (!expert_token_nums || !ep_recv_counts || !scratch) return ZBALHIP_INVALID;
    if (tokens > 0 && (!x || !expert_ids || !expand_x || !expand_idx)) return ZBALHIP_INVALID;
    const ExpertIds ids = ::expert_ids(expert_ids, (quant_mode & ZBALHIP_IDS_ARE_I64) != 0);
    quant_mode &= ~ZBALHIP_IDS_ARE_I64;
    if (experts <= 0 || experts > 1024 || topk <= 0 || tokens < 0 || quant_mode < 0 || quant_mode > 2 ||
        scratch_blocks < 1)
        return ZBALHIP_INVALID;
    hipStream_t st = (hipStream_t)stream;
    const int q = quant_mode == 0 ? QM_COPY : (quant_mode == 1 ? QM_INT8_NOEPS : QM_FP8);
    if (tokens > 0 && q != QM_COPY && !dynamic_scales) return ZBALHIP_INVALID;
    if (layout_fits_inline(tokens, topk, experts)) {      /* one launch: the permute kernel derives ranks and counts itself */
        InlineLayout il = {};
        il.tokens = (int)tokens;
        il.token_nums_type = token_nums_type;
        il.expand_idx = expand_idx;
        il.incl_i32 = ep_recv_counts;
        il.nums_typed = expert_token_nums;
        const PermuteExtras ex = {&il, nullptr, 0, nullptr, {}, nullptr};
        return permute_launch(x, x_dtype, ids, expand_idx, ep_recv_counts, 1, nullptr, tokens, hidden, topk, experts, q,
                              single_window(expand_x, dynamic_scales, experts, tokens * topk), st, ex);
    }
    const int32_t rc = zbalhip_layout_fused_internal(ids, tokens, experts, topk, token_nums_type, nullptr, expand_idx,
                                                     ep_recv_counts, nullptr, nullptr, expert_token_nums, st);
    if (rc != ZBALHIP_OK) return rc;
    return permute_launch(x, x_dtype, ids, expand_idx, ep_recv_counts, 1, nullptr, tokens, hidden, topk, experts, q,
                          single_window(expand_x, dynamic_scales, experts, tokens * topk), st);
}

extern "C" int32_t zbalhip_dispatch_low_latency_ranks(const void *x, int32_t x_dtype, const int32_t *const *expert_ids,
                                                      int64_t tokens, int64_t hidden, int64_t topk, int64_t experts,
                                                      int32_t quant_mode, int32_t token_nums_type, void *const *expand_x,
                                                      float *const *dynamic_scales, int32_t ranks, int32_t my_rank,
                                                      int64_t dest_rows, int32_t *expand_idx, int64_t *expert_token_nums,
                                                      int32_t *ep_recv_counts, int32_t *all_counts, void *stream)
{
    if (!expert_ids || !expert_token_nums || !ep_recv_counts || !all_counts) return ZBALHIP_INVALID;
    if (experts <= 0 || experts > 1024 || topk <= 0 || tokens < 0 || tokens * topk > 0x7fffffff || quant_mode < 0 ||
        quant_mode > 2 || dest_rows < 0)
        return ZBALHIP_INVALID;
    if (ranks <= 0 || ranks > ZBALHIP_MAX_REDUCE_PEERS || my_rank < 0 || my_rank >= ranks || experts % ranks != 0)
        return ZBALHIP_INVALID;
    if (tokens > 0 && (!x || !expand_x || !expand_idx || (quant_mode != 0 && !dynamic_scales))) return ZBALHIP_INVALID;
    PeerRows pr = {};
    for (int r = 0; r < ranks; ++r) {
        if (tokens > 0 && (!expert_ids[r] || !expand_x[r] || (quant_mode != 0 && !dynamic_scales[r]))) return ZBALHIP_INVALID;
        pr.dest[r] = tokens > 0 ? (uint8_t *)expand_x[r] : nullptr;
        pr.scale[r] = (tokens > 0 && quant_mode != 0) ? dynamic_scales[r] : nullptr;
    }
    pr.ranks = ranks;
    pr.my_rank = my_rank;
    pr.e_loc = (int)(experts / ranks);
    pr.rows_cap = dest_rows;
    hipStream_t st = (hipStream_t)stream;
    int32_t rc = zbalhip_ll_counts_internal(expert_ids, ranks, my_rank, tokens, topk, experts, token_nums_type, all_counts,
                                            ep_recv_counts, expert_token_nums, st);
    if (rc != ZBALHIP_OK || tokens == 0) return rc;
    /* the rank of each of my picks among my own earlier picks of the same expert */
    const ExpertIds ids = ::expert_ids(expert_ids[my_rank], false);
    rc = zbalhip_layout_fused_internal(ids, tokens, experts, topk, 1, nullptr, expand_idx, nullptr, nullptr,
                                       nullptr, nullptr, st);
    if (rc != ZBALHIP_OK) return rc;
    const int q = quant_mode == 0 ? QM_COPY : (quant_mode == 1 ? QM_INT8_NOEPS : QM_FP8);
    return permute_launch(x, x_dtype, ids, expand_idx, ep_recv_counts, 1, nullptr, tokens, hidden, topk,
                          experts, q, pr, st);
}

static int32_t fused_permute_quant(const void *x, int32_t x_dtype, const int32_t *expert_ids, const float *smooth,
                                   const uint8_t *active_mask, int64_t tokens, int64_t hidden, int64_t topk, int64_t experts,
                                   int32_t mode, void *q1, float *xs, int32_t *expand_idx, int64_t *counts, int32_t *row_off,
                                   uint32_t *clear_words, int64_t clear_count, int32_t *scratch, int32_t scratch_blocks,
                                   const SharedRows &sh, void *stream)
{
    if (!counts || !row_off || clear_count < 0 || (clear_count > 0 && !clear_words)) return ZBALHIP_INVALID;
    if (tokens > 0 && (!x || !expert_ids || !q1 || !xs || !expand_idx)) return ZBALHIP_INVALID;
    const ExpertIds ids = ::expert_ids(expert_ids, (mode & ZBALHIP_IDS_ARE_I64) != 0);
    mode &= ~ZBALHIP_IDS_ARE_I64;
    if (experts <= 0 || experts > 1024 || topk <= 0 || tokens < 0 || (mode != 1 && mode != 2)) return ZBALHIP_INVALID;
    if (mode == 2 && smooth) return ZBALHIP_INVALID;
    if (scratch_blocks < 0 || (scratch_blocks > 0 && !scratch)) return ZBALHIP_INVALID;
    hipStream_t st = (hipStream_t)stream;
    const int q = mode == 2 ? QM_FP8 : QM_INT8_NOEPS;
    if (layout_fits_inline(tokens, topk, experts)) {      /* one launch: the permute kernel derives ranks and offsets itself */
        InlineLayout il = {};
        il.active_mask = active_mask;
        il.tokens = (int)tokens;
        il.token_nums_type = 1;
        il.expand_idx = expand_idx;
        il.row_off = row_off;
        il.counts_i64 = counts;
        const PermuteExtras ex = {&il, clear_words, clear_count, nullptr, sh, nullptr};
        return permute_launch(x, x_dtype, ids, expand_idx, row_off, 0, smooth, tokens, hidden, topk, experts, q,
                              single_window(q1, xs, experts, tokens * topk), st, ex);
    }
    /* large batches with room for the ranges' histograms: a short layout launch, the rest of the layout inside the permute launch */
    int64_t ranges = (tokens * topk + 1023) / 1024;
    if (ranges > scratch_blocks) ranges = scratch_blocks;
    if (ranges > kTableMaxEntries / experts) ranges = kTableMaxEntries / experts;
    if (tokens > 0 && ranges >= 1 && experts <= kTableMaxExperts && topk <= kInlineMaxTopk && tokens * topk <= 0x7fffffff) {
        RangeTable rt = {};
        rt.tokens_per_range = (int)((tokens + ranges - 1) / ranges);
        rt.ranges = (int)((tokens + rt.tokens_per_range - 1) / rt.tokens_per_range);
        rt.hist = scratch;
        rt.expand_idx = expand_idx;
        rt.row_off = row_off;
        rt.counts_i64 = counts;
        const int32_t rc = zbalhip_layout_ranges_internal(ids, tokens, experts, topk, active_mask, expand_idx, scratch,
                                                          rt.ranges, rt.tokens_per_range, st);
        if (rc != ZBALHIP_OK) return rc;
        const PermuteExtras ex = {nullptr, clear_words, clear_count, &rt, sh, active_mask};
        return permute_launch(x, x_dtype, ids, nullptr, nullptr, 0, smooth, tokens, hidden, topk, experts, q,
                              single_window(q1, xs, experts, tokens * topk), st, ex);
    }
    const int32_t rc = zbalhip_layout_fused_internal(ids, tokens, experts, topk, 1, active_mask, expand_idx, nullptr,
                                                     row_off, counts, nullptr, st);
    if (rc != ZBALHIP_OK) return rc;
    if (tokens == 0 && clear_count > 0) return zbalhip_fill_i32((int32_t *)clear_words, clear_count, 0, stream);
    const PermuteExtras ex = {nullptr, clear_words, clear_count, nullptr, sh, active_mask};
    return permute_launch(x, x_dtype, ids, expand_idx, row_off, 0, smooth, tokens, hidden, topk, experts, q,
                          single_window(q1, xs, experts, tokens * topk), st, ex);
}

extern "C" int32_t zbalhip_fused_permute_quant(const void *x, int32_t x_dtype, const int32_t *expert_ids,
                                               const float *smooth, const uint8_t *active_mask, int64_t tokens,
                                               int64_t hidden, int64_t topk,
                                               int64_t experts, int32_t mode, void *q1, float *xs, int32_t *expand_idx,
                                               int64_t *counts, int32_t *row_off, uint32_t *clear_words,
                                               int64_t clear_count, int32_t *scratch, int32_t scratch_blocks, void *stream)
{
    return fused_permute_quant(x, x_dtype, expert_ids, smooth, active_mask, tokens, hidden, topk, experts, mode, q1, xs, expand_idx,
                               counts, row_off, clear_words, clear_count, scratch, scratch_blocks, SharedRows{}, stream);
}

extern "C" int32_t zbalhip_fused_permute_quant_shared(const void *x, int32_t x_dtype, const int32_t *expert_ids,
                                                      const float *smooth, const uint8_t *active_mask, int64_t tokens,
                                                      int64_t hidden, int64_t topk, int64_t experts, int32_t mode, void *q1,
                                                      float *xs, int32_t *expand_idx, int64_t *counts, int32_t *row_off,
                                                      uint32_t *clear_words, int64_t clear_count, int32_t *scratch,
                                                      int32_t scratch_blocks, const float *shared_smooth, void *stream)
{
    if (!row_off || tokens <= 0 || experts <= 0 || (smooth != nullptr) != (shared_smooth != nullptr)) return ZBALHIP_INVALID;
    const SharedRows sh = {tokens * topk, row_off + experts + 1, shared_smooth};
    return fused_permute_quant(x, x_dtype, expert_ids, smooth, active_mask, tokens, hidden, topk, experts, mode, q1, xs, expand_idx,
                               counts, row_off, clear_words, clear_count, scratch, scratch_blocks, sh, stream);
}
