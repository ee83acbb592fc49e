// Input preparation of the fused MoE operator on the GPU: the two steps every caller runs right before it.
//
//   * per-token-group FP8 quantisation of the activations (the reference calls SGLang's
//     sglang_per_token_group_quant_fp8(x, 128), jit_moe.py:142; the kernel consumes the result at
//     fused_moe_w8a8_up_down_acc.cu:793,800-807): scale = max(amax, 1e-10) / 448, q = fp8_rne(clamp(x / scale, +-448));
//   * grouping of the routing slots by expert, padded to the row-block size (SGLang's moe_align_block_size,
//     jit_moe.py:158; consumed at fused_moe_w8a8_up_down_acc.cu:676-679,756-758): flat slot ids in ascending expert
//     order, ascending id within an expert (stable: the result depends on nothing but the input), padding entries
//     equal to numel, one expert id per block (-1 past the padded total), and the padded total.
//
// Both are HBM-bound integer/byte passes: 16-byte loads, no matrix instructions.
#include <mutex>
#include <type_traits>

#include "moe_common.hpp"

namespace alpha_moe {
namespace {

constexpr int kAlignSeg = 1024;        // routing slots per workgroup (segment) of the histogram and placement kernels, and
constexpr int kAlignMaxSeg = 512;      // most segments before they get longer: every workgroup reads all segments' histograms
                                       // (4 Mi slots, 4096 experts: 9.2 ms in 4096 segments, 225 us in 512;
                                       // 600 000 slots, 257 experts: 35 us in 586, 23 in 293)
// Most routing slots one workgroup aligns by itself.  MI355X, one workgroup / two launches, 128 - 512 experts: 3072 slots
// 6.2 - 6.7 / 7.2 - 7.8 us, 4096 7.1 - 7.8 / 7.4 - 7.8, 5120 8.7 - 9.7 / 7.5 - 8.1.
constexpr int kAlignSmall = ALPHA_MOE_ALIGN_SLOTS_WITHOUT_WORKSPACE;
constexpr int kAlignMaxExperts = 4096;

// ---- quantisation ------------------------------------------------------------------------------------------
// A group of 128 values is held by 16 lanes x 8 values; a wavefront works on 4 groups at a time.
template <typename T>
__device__ __forceinline__ void load8(const T *p, float (&v)[8]);

template <>
__device__ __forceinline__ void load8<uint16_t>(const uint16_t *p, float (&v)[8])   // bf16
{
    const v4i raw = *reinterpret_cast<const v4i *>(p);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[2 * i] = __builtin_bit_cast(float, (uint32_t)raw[i] << 16);
        v[2 * i + 1] = __builtin_bit_cast(float, (uint32_t)raw[i] & 0xffff0000u);
    }
}

template <>
__device__ __forceinline__ void load8<float>(const float *p, float (&v)[8])
{
    const v4f a = *reinterpret_cast<const v4f *>(p), b = *reinterpret_cast<const v4f *>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[i] = a[i];
        v[4 + i] = b[i];
    }
}

// The groups of workgroup `part` of `parts`, one at a time: a second group's loads in flight per thread take registers, and
// wavefronts hide the latency as well.  MI355X, cold, bf16, one / two groups in flight: 8192 x 7168 37.9 / 39.9 us (4.7 TB/s),
// 32768 x 7168 148 / 157, 8192 x 2048 15.2 / 15.8; at 333 tokens and fewer both alike.
template <typename T>
__device__ __forceinline__ void quant_groups(const T *__restrict__ x, uint8_t *__restrict__ q, float *__restrict__ scale,
                                             long long n_groups, int part, int parts)
{
    const int sub = threadIdx.x & 15, per = blockDim.x >> 4;
    const long long stride = (long long)parts * per;
    for (long long g = (long long)part * per + (threadIdx.x >> 4); g < n_groups; g += stride) {
        float v[8];
        load8<T>(x + g * 128 + sub * 8, v);
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) m = fmaxf(m, fabsf(v[i]));
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
        const float s = fmaxf(m, kAmaxFloor) / kFp8Max;
        uint2 o;
        o.x = pack_fp8x4(clamp_fp8(v[0] / s), clamp_fp8(v[1] / s), clamp_fp8(v[2] / s), clamp_fp8(v[3] / s));
        o.y = pack_fp8x4(clamp_fp8(v[4] / s), clamp_fp8(v[5] / s), clamp_fp8(v[6] / s), clamp_fp8(v[7] / s));
        *reinterpret_cast<uint2 *>(q + g * 128 + sub * 8) = o;
        if (sub == 0) scale[g] = s;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void quant_group128_kernel(const T *__restrict__ x, uint8_t *__restrict__ q,
                                                             float *__restrict__ scale, long long n_groups)
{
    quant_groups<T>(x, q, scale, n_groups, blockIdx.x, gridDim.x);
}

// ---- alignment ---------------------------------------------------------------------------------------------
// A stable counting sort of the routing slots by expert.  What bounds it is a chain of dependent steps on one workgroup of
// sixteen wavefronts, where every instruction of all of them takes 16 cycles of the chain: round trips and instructions are
// what is saved.  A wavefront ranks 64 consecutive slots among the equal experts of its chunk with a table of lane masks in LDS
// (same_expert; a ballot per bit of the expert id was 72 instructions a chunk), keeps its slots in registers between counting and
// placing, and counts and places a run of slots of its own behind cursors of its own.  MI355X, us in a graph of such calls,
// before (ballots, slots read twice, prefix sums by LDS shuffles, divisions by the block size) / now: 9 slots of 257 experts
// 5.4 / 4.1, 2997 slots 9.1 / 6.4, 4000 slots of 512 experts 11.1 / 7.8; in two launches 18 432 slots 11.1 / 8.4, 73 728 slots
// 11.5 / 9.3, 600 000 slots 27.3 / 22.9, 8192 slots of 128 experts 9.7 / 7.5, 4 Mi slots of 4096 experts 273 / 225.
typedef unsigned long long lanes_t;
constexpr int kMasks = 256;   // entries of a wavefront's table of lane masks: the experts' low eight bits

// LDS accesses of one wavefront complete in order; this keeps the compiler to the written order
__device__ __forceinline__ void lds_order()
{
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// The lanes of this wavefront whose slot has the same expert as this lane's (e < 0: no slot, no lanes); all 64 lanes
// call it.  masks: the wavefront's table, zero before and after (its LDS accesses complete in order).
// Lanes that add to one table entry take turns.  FEW (few experts, many slots: few_experts()) is for inputs on which that is the
// rule and not the exception: up to eight experts a ballot per bit of the id instead, otherwise the first lane's expert - the hot
// one, if there is one - by a ballot and the others by the table.
template <bool FEW>
__device__ __forceinline__ lanes_t same_expert(int e, int id_bits, lanes_t *masks)
{
    lanes_t first = 0;
    bool other = e >= 0;
    if constexpr (FEW) {
        if (id_bits <= 3) {
            lanes_t same = __ballot(e >= 0);
            for (int b = 0; b < id_bits; b++) {
                const bool set = (e >> b) & 1;
                const lanes_t with = __ballot(set);
                same &= set ? with : ~with;
            }
            return e >= 0 ? same : 0;
        }
        const int e0 = __builtin_amdgcn_readfirstlane(e);
        first = __ballot(e == e0);
        first = e == e0 && e >= 0 ? first : 0;
        other = e >= 0 && e != e0;
    }
    lanes_t same = 0;
    if (other) atomicOr(&masks[e & (kMasks - 1)], 1ull << (threadIdx.x & 63));
    lds_order();
    if (other) same = masks[e & (kMasks - 1)];
    lds_order();
    if (other) masks[e & (kMasks - 1)] = 0;
    lds_order();
    for (int b = 8; b < id_bits; b++) {   // the upper bits, one ballot each
        const bool set = (e >> b) & 1;
        const lanes_t with = __ballot(set);
        same &= set ? with : ~with;
    }
    return same | first;
}

__device__ __forceinline__ int expert_of_slot(const int32_t *ids, int i, int end, int E)
{
    const int e = i < end ? ids[i] : -1;
    return e < E ? e : -1;
}

__device__ __forceinline__ lanes_t lanes_below() { return (1ull << (threadIdx.x & 63)) - 1ull; }

// The 64-slot chunks of ids[lo, hi) that a wavefront keeps in registers between counting and placing.
constexpr int kKept = 4;
struct Chunks {
    int e[kKept];
    lanes_t same[kKept];
};

__device__ __forceinline__ void load_chunks(const int32_t *ids, int lo, int hi, int E, Chunks &c)
{
#pragma unroll
    for (int k = 0; k < kKept; k++) c.e[k] = expert_of_slot(ids, lo + k * 64 + (threadIdx.x & 63), hi, E);
}

// counts[at] += n, 16-bit counts, without a round trip.  (Neighbouring wavefronts' counters may share a word.)
__device__ __forceinline__ void add_count(uint16_t *counts, int at, int n)
{
    atomicAdd(reinterpret_cast<unsigned *>(counts) + (at >> 1), (unsigned)n << (16 * (at & 1)));
}

// cursors[e][column] += slots of expert e in ids[lo, hi).  One wavefront, its own column; c holds the first chunks' experts.
template <bool FEW>
__device__ __forceinline__ void count_run(const int32_t *ids, int lo, int hi, int E, int id_bits, lanes_t *masks,
                                          uint16_t *cursors, int column, int n_waves, Chunks &c)
{
    auto count = [&](int e, lanes_t same) {
        if (e >= 0 && (same & lanes_below()) == 0) add_count(cursors, e * n_waves + column, __builtin_popcountll(same));
    };
#pragma unroll
    for (int k = 0; k < kKept; k++)
        if (lo + k * 64 < hi) c.same[k] = same_expert<FEW>(c.e[k], id_bits, masks);
#pragma unroll
    for (int k = 0; k < kKept; k++)
        if (lo + k * 64 < hi) count(c.e[k], c.same[k]);
    for (int base = lo + kKept * 64; base < hi; base += 64) {
        const int e = expert_of_slot(ids, base + (threadIdx.x & 63), hi, E);
        count(e, same_expert<FEW>(e, id_bits, masks));
    }
}

// sorted_ids[start(e) + cursor[e] ...] = the slots of expert e in ids[lo, hi), in order.  One wavefront, its own cursors
// (a chunk's are read before they move on: LDS accesses of a wavefront complete in order).
template <bool FEW, typename Start>
__device__ __forceinline__ void place_run(const int32_t *ids, int lo, int hi, int E, int id_bits, lanes_t *masks, Start start,
                                          uint16_t *cursors, int column, int n_waves, const Chunks &c,
                                          int32_t *sorted_ids)
{
    auto place = [&](int e, lanes_t same) {   // the slot's place
        int at = 0;
        if (e >= 0) at = start(e) + cursors[e * n_waves + column];
        lds_order();
        if (e >= 0 && (same & lanes_below()) == 0) add_count(cursors, e * n_waves + column, __builtin_popcountll(same));
        lds_order();
        return at + __builtin_popcountll(same & lanes_below());
    };
    int at[kKept];
#pragma unroll
    for (int k = 0; k < kKept; k++)
        if (lo + k * 64 < hi) at[k] = place(c.e[k], c.same[k]);
#pragma unroll
    for (int k = 0; k < kKept; k++)
        if (lo + k * 64 < hi && c.e[k] >= 0) sorted_ids[at[k]] = lo + k * 64 + (threadIdx.x & 63);
    for (int base = lo + kKept * 64; base < hi; base += 64) {
        const int i = base + (threadIdx.x & 63);
        const int e = expert_of_slot(ids, i, hi, E);
        const int to = place(e, same_expert<FEW>(e, id_bits, masks));
        if (e >= 0) sorted_ids[to] = i;
    }
}

// cursors[e][w] of the n_waves (2, 4, 8 or 16) wavefronts: counts -> exclusive prefix over the wavefronts; returns the sum
__device__ __forceinline__ int prefix_over_waves(uint16_t *cursors, int e, int n_waves)
{
    int run = 0;
    auto step = [&](unsigned two) {
        const unsigned c0 = two & 0xffffu, c1 = two >> 16, first = run;
        run += (int)(c0 + c1);
        return first | (first + c0) << 16;
    };
    if (n_waves >= 8) {
        v4i *c = reinterpret_cast<v4i *>(cursors + (size_t)e * n_waves);
        v4i a = c[0], b = c[n_waves > 8 ? 1 : 0];
#pragma unroll
        for (int k = 0; k < 4; k++) a[k] = (int)step((unsigned)a[k]);
        c[0] = a;
        if (n_waves > 8) {
#pragma unroll
            for (int k = 0; k < 4; k++) b[k] = (int)step((unsigned)b[k]);
            c[1] = b;
        }
    } else {
        unsigned *c = reinterpret_cast<unsigned *>(cursors + (size_t)e * n_waves);
        const unsigned a = c[0], b = c[n_waves > 2 ? 1 : 0];
        c[0] = step(a);
        if (n_waves > 2) c[1] = step(b);
    }
    return run;
}

// Inclusive prefix sum over the wavefront, in registers (a step is a shift within rows of 16 lanes, or the last lane of the rows
// before; through LDS, as __shfl_up goes, a step is a round trip).
__device__ __forceinline__ int row_inclusive_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // from 1, 2, 4, 8 lanes below in the row
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    return v;
}
__device__ __forceinline__ int wave_inclusive_scan(int v)
{
    v = row_inclusive_scan(v);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // lane 15 of rows 0 and 2 to rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // lane 31 to rows 2 and 3
    return v;
}

// Exclusive prefix sum over the n values of LDS array `vals`, in place; returns their sum.  All 1024 threads call it.
__device__ int block_exclusive_scan(int *vals, int n, int *wave_sums /* [16] */)
{
    const int per = (n + 1023) / 1024;
    const int lo = min((int)threadIdx.x * per, n), hi = min(lo + per, n);
    int sum = 0, incl = 0;
    if (__builtin_amdgcn_readfirstlane(lo < n)) {   // (a wavefront without values leaves the others its cycles)
        for (int i = lo; i < hi; i++) sum += vals[i];
        incl = wave_inclusive_scan(sum);
    }
    if ((threadIdx.x & 63) == 63) wave_sums[threadIdx.x >> 6] = incl;
    lds_barrier();
    const int sums = row_inclusive_scan(wave_sums[threadIdx.x & 15]);   // (of all sixteen wavefronts, in every row)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), total = __builtin_amdgcn_readlane(sums, 15);
    int run = incl - sum + (wave > 0 ? __builtin_amdgcn_readlane(sums, wave - 1) : 0);
    for (int i = lo; i < hi; i++) {
        const int v = vals[i];
        vals[i] = run;
        run += v;
    }
    lds_barrier();
    return total;
}

// v / block_size (a division is some forty instructions, of every wavefront)
__device__ __forceinline__ int blocks_in(int v, int block_size)
{
    return (block_size & (block_size - 1)) == 0 ? v >> __builtin_ctz(block_size) : v / block_size;
}
__device__ __forceinline__ int pad_to(int v, int block_size) { return blocks_in(v + block_size - 1, block_size) * block_size; }

// expert_ids and the padded total from the starts of the experts' padded segments (total behind the last one): thread `tid` of
// `stride` writes its share.
__device__ void write_blocks(const int *start, int E, int block_size, int total, int32_t *expert_ids, int n_blocks,
                             int32_t *ntpp, int tid, int stride)
{
    const int used = blocks_in(total, block_size);
    for (int b = tid; b < n_blocks; b += stride) {
        int e = -1;
        if (b < used) {   // the last expert whose segment starts at or before the block (empty segments start there too)
            int lo = 0, hi = E;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (start[mid] <= b * block_size) lo = mid;
                else hi = mid;
            }
            e = lo;
        }
        expert_ids[b] = e;
    }
    if (tid == 0) ntpp[0] = total;
}

__device__ __forceinline__ void fill_sentinel(int32_t *sorted_ids, int sorted_num, int numel, int tid, int stride)
{
    // 16 bytes per store from the first aligned element on
    const int head = min((int)((0u - (unsigned)(reinterpret_cast<uintptr_t>(sorted_ids) >> 2)) & 3u), sorted_num);
    const int quads = (sorted_num - head) >> 2;
    v4i *body = reinterpret_cast<v4i *>(sorted_ids + head);
    for (int i = tid; i < quads; i += stride) body[i] = (v4i){numel, numel, numel, numel};
    for (int i = tid; i < head; i += stride) sorted_ids[i] = numel;
    for (int i = head + 4 * quads + tid; i < sorted_num; i += stride) sorted_ids[i] = numel;
}

// bytes of the cursors of n_waves wavefronts, whole 16 bytes
__host__ __device__ constexpr size_t cursor_bytes(int n_waves, int E) { return ((size_t)n_waves * E * sizeof(uint16_t) + 15) & ~(size_t)15; }

// One workgroup does everything (up to kAlignSmall slots).  n_waves of its wavefronts count and place `run` slots each.
struct AlignSmall {
    const int32_t *ids;
    int numel, E, id_bits, block_size;
    int32_t *sorted_ids;
    int sorted_num;
    int32_t *expert_ids;
    int n_blocks;
    int32_t *ntpp;
    int n_waves, run;
};
template <bool FEW>
__device__ __forceinline__ void align_small(const AlignSmall &a)
{
    const int32_t *__restrict__ ids = a.ids;
    const int numel = a.numel, E = a.E, id_bits = a.id_bits, block_size = a.block_size, sorted_num = a.sorted_num;
    const int n_waves = a.n_waves, run = a.run;
    int32_t *sorted_ids = a.sorted_ids;
    // [n_waves] tables of lane masks | [E][n_waves] cursors (16 bit, whole 16 bytes) | [16] the scan's sums | [E] starts
    extern __shared__ __attribute__((aligned(16))) uint8_t mem[];
    lanes_t *masks = reinterpret_cast<lanes_t *>(mem);
    uint16_t *cursors = reinterpret_cast<uint16_t *>(masks + n_waves * kMasks);
    const int zero_quads = (int)(cursor_bytes(n_waves, E) + n_waves * kMasks * sizeof(lanes_t)) / 16;
    int *wave_sums = reinterpret_cast<int *>(mem) + 4 * zero_quads, *start = wave_sums + 16;
    const int wave = threadIdx.x >> 6;
    const int lo = wave * run, hi = wave < n_waves ? min(lo + run, numel) : lo;
    Chunks c;
    load_chunks(ids, lo, hi, E, c);
    for (int i = threadIdx.x; i < zero_quads; i += blockDim.x) reinterpret_cast<v4i *>(mem)[i] = (v4i){0, 0, 0, 0};
    masks += wave * kMasks;
    lds_barrier();
    count_run<FEW>(ids, lo, hi, E, id_bits, masks, cursors, wave, n_waves, c);
    // (behind the use of the slots' experts: a load is waited for with everything issued behind it)
    fill_sentinel(sorted_ids, sorted_num, numel, threadIdx.x, blockDim.x);
    lds_barrier();
    for (int e = threadIdx.x; e < E; e += blockDim.x) start[e] = pad_to(prefix_over_waves(cursors, e, n_waves), block_size);
    lds_barrier();
    const int total = block_exclusive_scan(start, E, wave_sums);
    drain_vmem();   // the sentinels are there before any slot is placed
    lds_barrier();
    place_run<FEW>(ids, lo, hi, E, id_bits, masks, [&](int e) { return start[e]; }, cursors, wave, n_waves, c, sorted_ids);
    // (wavefronts without slots take the first blocks)
    write_blocks(start, E, block_size, total, a.expert_ids, a.n_blocks, a.ntpp, blockDim.x - 1 - threadIdx.x, blockDim.x);
}

template <bool FEW>
__global__ __launch_bounds__(1024) void align_small_kernel(const AlignSmall a) { align_small<FEW>(a); }

// Both preparations of a layer call in one launch: workgroup 0 aligns, the others quantise.  Neither needs the other's
// result, and at decode sizes each is 2 - 6 us of latency.
template <typename T, bool FEW>
__global__ __launch_bounds__(1024) void prepare_small_kernel(const AlignSmall a, const T *__restrict__ x,
                                                             uint8_t *__restrict__ q, float *__restrict__ scale,
                                                             long long n_groups)
{
    if (blockIdx.x == 0) align_small<FEW>(a);
    else quant_groups<T>(x, q, scale, n_groups, (int)blockIdx.x - 1, (int)gridDim.x - 1);
}

// Larger inputs, pass 1: one workgroup per segment of `seg` slots writes the segment's expert histogram (16-bit
// counts, two per word); also the sentinel fill.
__device__ __forceinline__ void align_hist(const int32_t *__restrict__ ids, int numel, int E, int *hist, int words,
                                           int32_t *sorted_ids, int sorted_num, int n_seg, int seg)
{
    extern __shared__ int lds[];   // [words]
    for (int i = threadIdx.x; i < words; i += blockDim.x) lds[i] = 0;
    __syncthreads();
    const int lo = blockIdx.x * seg, hi = min(lo + seg, numel);
    for (int i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        const int e = ids[i];
        if (e >= 0 && e < E) atomicAdd(&lds[e >> 1], 1 << (16 * (e & 1)));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < words; i += blockDim.x) hist[(size_t)blockIdx.x * words + i] = lds[i];
    fill_sentinel(sorted_ids, sorted_num, numel, blockIdx.x * blockDim.x + threadIdx.x, n_seg * blockDim.x);
}

__global__ __launch_bounds__(256) void align_hist_kernel(const int32_t *__restrict__ ids, int numel, int E, int *hist,
                                                         int words, int32_t *sorted_ids, int sorted_num, int seg)
{
    align_hist(ids, numel, E, hist, words, sorted_ids, sorted_num, gridDim.x, seg);
}

// Pass 1 and the quantiser in one launch: the first n_seg workgroups count, the others quantise.
template <typename T>
__global__ __launch_bounds__(256) void prepare_hist_kernel(const int32_t *__restrict__ ids, int numel, int E, int *hist,
                                                           int words, int32_t *sorted_ids, int sorted_num, int n_seg, int seg,
                                                           const T *__restrict__ x, uint8_t *__restrict__ q,
                                                           float *__restrict__ scale, long long n_groups)
{
    if ((int)blockIdx.x < n_seg) align_hist(ids, numel, E, hist, words, sorted_ids, sorted_num, n_seg, seg);
    else quant_groups<T>(x, q, scale, n_groups, (int)blockIdx.x - n_seg, (int)gridDim.x - n_seg);
}

// Pass 2, one workgroup per segment: every workgroup adds the histograms up itself (columns of two experts, the segments
// split over the threads that share a column, up to eight of a thread's in flight; a third launch of one workgroup for the sums
// took 17 - 42 us), scans the padded totals and places its segment, each of its n_waves wavefronts a part of it.
// 1024 threads: four times as many as 256 took a quarter of the rounds of dependent round trips (18 432 slots 13 -> 10 us, before
// the rounds themselves were shortened).
template <bool FEW>
__global__ __launch_bounds__(1024) void align_place_kernel(const int32_t *__restrict__ ids, int numel, int E, int id_bits,
                                                           int block_size, const int *__restrict__ hist, int words,
                                                           int32_t *sorted_ids, int32_t *expert_ids, int n_blocks,
                                                           int32_t *ntpp, int n_waves, int seg_slots)
{
    // [n_waves] tables of lane masks | [E][n_waves] cursors (16 bit, whole 16 bytes) | [2 words] starts | [2 words] slots of
    // earlier segments | [16] the scan's sums
    extern __shared__ __attribute__((aligned(16))) uint8_t mem[];
    lanes_t *masks = reinterpret_cast<lanes_t *>(mem);
    uint16_t *cursors = reinterpret_cast<uint16_t *>(masks + n_waves * kMasks);
    int *start = reinterpret_cast<int *>(mem + n_waves * kMasks * sizeof(lanes_t) + cursor_bytes(n_waves, E));
    int *before = start + 2 * words, *wave_sums = before + 2 * words;
    const int wave = threadIdx.x >> 6, n_seg = gridDim.x, seg = blockIdx.x;
    const int run = seg_slots / n_waves;
    const int lo = seg * seg_slots + wave * run, hi = wave < n_waves ? min(lo + run, numel) : lo;
    Chunks c;
    load_chunks(ids, lo, hi, E, c);
    const int zero_quads = (int)(reinterpret_cast<uint8_t *>(wave_sums) - mem) / 16;
    for (int i = threadIdx.x; i < zero_quads; i += blockDim.x) reinterpret_cast<v4i *>(mem)[i] = (v4i){0, 0, 0, 0};
    masks += wave * kMasks;
    lds_barrier();
    const int share = words < (int)blockDim.x ? blockDim.x / words : 1;   // threads of a column
    const int part = words < (int)blockDim.x ? threadIdx.x / words : 0;
    // U segments in flight as long as there are as many, then R, of which those past the end are loaded twice and count nothing
    auto add_up = [&](auto in_flight, auto rest) {
        constexpr int U = decltype(in_flight)::value, R = decltype(rest)::value;
        for (int col = (int)threadIdx.x - part * words; col < words && part < share; col += blockDim.x) {
            int b0 = 0, b1 = 0, t0 = 0, t1 = 0, s0 = part;
            auto take = [&](auto in_flight, auto all_there) {
                constexpr int N = decltype(in_flight)::value;
                constexpr bool ALL = decltype(all_there)::value;
                unsigned v[N];
#pragma unroll
                for (int k = 0; k < N; k++)
                    v[k] = (unsigned)hist[(size_t)(ALL ? s0 + k * share : min(s0 + k * share, n_seg - 1)) * words + col];
#pragma unroll
                for (int k = 0; k < N; k++) {
                    const unsigned w = ALL || s0 + k * share < n_seg ? v[k] : 0u;
                    const int c0 = w & 0xffffu, c1 = w >> 16;
                    t0 += c0;
                    t1 += c1;
                    if (s0 + k * share < seg) {
                        b0 += c0;
                        b1 += c1;
                    }
                }
                s0 += N * share;
            };
            if constexpr (U > R)
                while (s0 + (U - 1) * share < n_seg) take(in_flight, std::true_type());
            while (s0 < n_seg) take(rest, std::false_type());
            atomicAdd(&start[2 * col], t0);
            atomicAdd(&start[2 * col + 1], t1);
            atomicAdd(&before[2 * col], b0);
            atomicAdd(&before[2 * col + 1], b1);
        }
    };
    // One round where eight segments a thread will do, with no more loads than there are segments to the next power of two; more
    // rounds are bound by their loads, so none is made in vain before the last four.  Twelve at a time, those past the end loaded
    // twice, also took 70 registers, which leave no room for a second workgroup per compute unit; inputs of more than 256 segments
    // run two.  MI355X, us in a graph of such calls, so / as it is: 40 960 slots, 512 experts (10 segments a thread) 9.6 / 9.4;
    // 300 000 slots, 257 experts (42) 21.9 / 19.5, 1024 (147) 43.5 / 36.1, 4096 (293) 132 / 106; 2 Mi slots, 4096 experts (512)
    // 248 / 208.  Sixteen and then four took as long, twelve and then four 0 - 15 % longer.
    const std::integral_constant<int, 2> two;
    const std::integral_constant<int, 4> four;
    const std::integral_constant<int, 8> eight;
    if (n_seg <= 2 * share)
        add_up(two, two);
    else if (n_seg <= 4 * share)
        add_up(four, four);
    else if (n_seg <= 8 * share)
        add_up(eight, eight);
    else
        add_up(eight, four);
    count_run<FEW>(ids, lo, hi, E, id_bits, masks, cursors, wave, n_waves, c);
    lds_barrier();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        prefix_over_waves(cursors, e, n_waves);
        start[e] = pad_to(start[e], block_size);
    }
    lds_barrier();
    const int total = block_exclusive_scan(start, E, wave_sums);
    place_run<FEW>(ids, lo, hi, E, id_bits, masks, [&](int e) { return start[e] + before[e]; }, cursors, wave, n_waves, c,
                   sorted_ids);
    write_blocks(start, E, block_size, total, expert_ids, n_blocks, ntpp, seg * blockDim.x + threadIdx.x, n_seg * blockDim.x);
}

constexpr size_t kDefaultLds = 64 << 10;   // dynamic LDS a kernel may have without a word

// The placement kernel's limit is raised once per device, not on every launch.
hipError_t allow_place_lds()
{
    static std::mutex mu;
    static bool done[64];
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    std::lock_guard<std::mutex> lock(mu);
    if (dev >= 0 && dev < 64 && done[dev]) return hipSuccess;
    err = hipFuncSetAttribute(reinterpret_cast<const void *>(align_place_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              80 << 10);
    if (err == hipSuccess && dev >= 0 && dev < 64) done[dev] = true;
    return err;
}

// What is quantised beside an alignment (x == nullptr: nothing).
struct Quant {
    const void *x;
    int is_f32;
    uint8_t *q;
    float *scale;
    int M, K;
};

int check_quant(const Quant &z)
{
    if (!z.x || !z.q || !z.scale) return ALPHA_MOE_ERR_NULL_POINTER;
    if (z.M <= 0 || z.K <= 0 || z.K % 128 != 0) return ALPHA_MOE_ERR_SHAPE;
    return ALPHA_MOE_OK;
}

// workgroups of `threads` threads for the groups of z
unsigned quant_grid(const Quant &z, int threads)
{
    const long long per = threads / 16, want = ((long long)z.M * (z.K / 128) + per - 1) / per, most = 8192 * 256 / threads;
    return (unsigned)(want < most ? want : most);
}

// Where same_expert() has to expect one expert on many lanes of a chunk.  MI355X, us in a graph of such calls, without / with
// FEW, and in brackets without the table of lane masks (a ballot per bit for any number of experts): 4096 slots of 1 expert
// 7.9 / 4.8 (6.2), of 2 evenly 6.7 / 5.1 (6.5), of 8 5.9 / 5.9 (7.4), all of 16 on one 8.2 / 5.6 (7.6), of 64 8.3 / 5.6 (8.5);
// 4 Mi slots of 1 expert 57 / 39 (41), all of 64 on one 53 / 40 (46), half 44 / 41 (44), evenly 43 / 43 (45), all of 128 on one
// 53 / 43 (50); from there on the table alone is ahead of ballots on any input (257 experts, all on one 57 / 54 (61)), and
// below 1024 slots as well (300 of 1 expert 3.6 / 3.5 (4.3), 30 of 16 3.6 / 3.8 (4.6)).
bool few_experts(int numel, int id_bits) { return id_bits <= 7 && numel >= 1024; }

int align(const int32_t *topk_ids, int numel, int num_experts, int block_size, int32_t *sorted_token_ids, int sorted_num,
          int32_t *expert_ids, int n_blocks, int32_t *num_tokens_post_padded, void *workspace, size_t workspace_bytes,
          const Quant &z, hipStream_t hs)
{
    if (!topk_ids || !sorted_token_ids || !expert_ids || !num_tokens_post_padded) return ALPHA_MOE_ERR_NULL_POINTER;
    if (numel <= 0 || num_experts <= 0 || num_experts > kAlignMaxExperts || block_size <= 0) return ALPHA_MOE_ERR_SHAPE;
    if ((long long)sorted_num != (long long)numel + (long long)num_experts * (block_size - 1) ||
        (long long)n_blocks != ((long long)sorted_num + block_size - 1) / block_size)
        return ALPHA_MOE_ERR_SHAPE;
    const int E = num_experts;
    const long long n_groups = z.x ? (long long)z.M * (z.K / 128) : 0;
    int id_bits = 0;
    while ((1 << id_bits) < E) id_bits++;
    if (numel <= kAlignSmall) {
        // a power of two of wavefronts, as many as there are chunks of 64 slots, and no more than have room for their tables
        // and cursors in 64 KiB of LDS
        int n_waves = 2;
        while (n_waves < 16 && n_waves * 64 < numel) n_waves *= 2;
        auto lds_of = [&](int waves) {
            return waves * kMasks * sizeof(lanes_t) + cursor_bytes(waves, E) + (16 + E) * sizeof(int);
        };
        while (lds_of(n_waves) > kDefaultLds) n_waves /= 2;
        const int run = ((numel + n_waves - 1) / n_waves + 63) / 64 * 64;
        const size_t lds = lds_of(n_waves);
        const AlignSmall a = {topk_ids, numel, E, id_bits, block_size, sorted_token_ids, sorted_num, expert_ids, n_blocks,
                              num_tokens_post_padded, n_waves, run};
        auto launch = [&](auto few) {
            constexpr bool FEW = decltype(few)::value;
            if (!z.x)
                hipLaunchKernelGGL(align_small_kernel<FEW>, dim3(1), dim3(1024), lds, hs, a);
            else if (z.is_f32)
                hipLaunchKernelGGL((prepare_small_kernel<float, FEW>), dim3(1 + quant_grid(z, 1024)), dim3(1024), lds, hs, a,
                                   static_cast<const float *>(z.x), z.q, z.scale, n_groups);
            else
                hipLaunchKernelGGL((prepare_small_kernel<uint16_t, FEW>), dim3(1 + quant_grid(z, 1024)), dim3(1024), lds, hs, a,
                                   static_cast<const uint16_t *>(z.x), z.q, z.scale, n_groups);
        };
        if (few_experts(numel, id_bits))
            launch(std::true_type());
        else
            launch(std::false_type());
        return hipGetLastError() == hipSuccess ? ALPHA_MOE_OK : ALPHA_MOE_ERR_LAUNCH;
    }
    if (!workspace || workspace_bytes < alpha_moe_align_workspace_bytes(numel, E)) return ALPHA_MOE_ERR_WORKSPACE;
    int seg = kAlignSeg;   // (counts and cursors of a segment are 16 bits wide)
    while (seg < (32 << 10) && (numel - 1) / seg >= kAlignMaxSeg) seg *= 2;
    const int n_seg = (numel - 1) / seg + 1, words = (E + 1) / 2;
    int *hist = static_cast<int *>(workspace);
    if (!z.x)
        hipLaunchKernelGGL(align_hist_kernel, dim3(n_seg), dim3(256), words * sizeof(int), hs, topk_ids, numel, E, hist,
                           words, sorted_token_ids, sorted_num, seg);
    else if (z.is_f32)
        hipLaunchKernelGGL(prepare_hist_kernel<float>, dim3(n_seg + quant_grid(z, 256)), dim3(256), words * sizeof(int), hs,
                           topk_ids, numel, E, hist, words, sorted_token_ids, sorted_num, n_seg, seg,
                           static_cast<const float *>(z.x), z.q, z.scale, n_groups);
    else
        hipLaunchKernelGGL(prepare_hist_kernel<uint16_t>, dim3(n_seg + quant_grid(z, 256)), dim3(256), words * sizeof(int),
                           hs, topk_ids, numel, E, hist, words, sorted_token_ids, sorted_num, n_seg, seg,
                           static_cast<const uint16_t *>(z.x), z.q, z.scale, n_groups);
    // as many wavefronts, sixteen at most, as have room for their tables and cursors in 64 KiB of LDS, but at least four (up to
    // 72.1 KiB, from 3581 experts on; two workgroups per compute unit all the same): a segment is placed chunk by chunk, and two
    // wavefronts take twice the chunks each.  MI355X, us in a graph of such calls, two / four wavefronts, 4096 experts: 8192 slots
    // 15.1 / 11.8, 73 728 25.6 / 23.6, 600 000 119.5 / 115.4, 2 Mi 208 / 197.
    int n_waves = 16;
    auto lds_of = [&](int waves) {
        return waves * kMasks * sizeof(lanes_t) + cursor_bytes(waves, E) + (4 * words + 16) * sizeof(int);
    };
    while (n_waves > 4 && lds_of(n_waves) > kDefaultLds) n_waves /= 2;
    const size_t lds = lds_of(n_waves);
    if (lds > kDefaultLds && allow_place_lds() != hipSuccess) return ALPHA_MOE_ERR_LAUNCH;
    const auto place = few_experts(numel, id_bits) ? align_place_kernel<true> : align_place_kernel<false>;
    hipLaunchKernelGGL(place, dim3(n_seg), dim3(1024), lds, hs, topk_ids, numel, E, id_bits, block_size, hist,
                       words, sorted_token_ids, expert_ids, n_blocks, num_tokens_post_padded, n_waves, seg);
    return hipGetLastError() == hipSuccess ? ALPHA_MOE_OK : ALPHA_MOE_ERR_LAUNCH;
}

}  // namespace
}  // namespace alpha_moe

using namespace alpha_moe;

extern "C" int alpha_moe_per_token_group_quant_fp8(const void *x, int x_is_f32, uint8_t *q, float *scale, int M, int K,
                                                   void *stream)
{
    const Quant z = {x, x_is_f32, q, scale, M, K};
    const int rc = check_quant(z);
    if (rc != ALPHA_MOE_OK) return rc;
    const dim3 grid(quant_grid(z, 256));
    const long long n_groups = (long long)M * (K / 128);
    hipStream_t hs = static_cast<hipStream_t>(stream);
    if (x_is_f32)
        hipLaunchKernelGGL(quant_group128_kernel<float>, grid, dim3(256), 0, hs, static_cast<const float *>(x), q, scale,
                           n_groups);
    else
        hipLaunchKernelGGL(quant_group128_kernel<uint16_t>, grid, dim3(256), 0, hs, static_cast<const uint16_t *>(x), q,
                           scale, n_groups);
    return hipGetLastError() == hipSuccess ? ALPHA_MOE_OK : ALPHA_MOE_ERR_LAUNCH;
}

extern "C" size_t alpha_moe_align_workspace_bytes(int numel, int num_experts)
{
    if (numel <= 0 || num_experts <= 0) return 0;
    const size_t n_seg = ((size_t)numel + kAlignSeg - 1) / kAlignSeg;
    return n_seg * (size_t)num_experts * sizeof(int);
}

extern "C" int alpha_moe_moe_align_block_size(const int32_t *topk_ids, int numel, int num_experts, int block_size,
                                              int32_t *sorted_token_ids, int sorted_num, int32_t *expert_ids,
                                              int n_blocks, int32_t *num_tokens_post_padded, void *workspace,
                                              size_t workspace_bytes, void *stream)
{
    return align(topk_ids, numel, num_experts, block_size, sorted_token_ids, sorted_num, expert_ids, n_blocks,
                 num_tokens_post_padded, workspace, workspace_bytes, Quant{}, static_cast<hipStream_t>(stream));
}

extern "C" int alpha_moe_prepare_inputs(const void *x, int x_is_f32, uint8_t *q, float *scale, int M, int K,
                                        const int32_t *topk_ids, int numel, int num_experts, int block_size,
                                        int32_t *sorted_token_ids, int sorted_num, int32_t *expert_ids, int n_blocks,
                                        int32_t *num_tokens_post_padded, void *workspace, size_t workspace_bytes,
                                        void *stream)
{
    const Quant z = {x, x_is_f32, q, scale, M, K};
    const int rc = check_quant(z);
    if (rc != ALPHA_MOE_OK) return rc;
    return align(topk_ids, numel, num_experts, block_size, sorted_token_ids, sorted_num, expert_ids, n_blocks,
                 num_tokens_post_padded, workspace, workspace_bytes, z, static_cast<hipStream_t>(stream));
}
