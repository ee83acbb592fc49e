// Fused W8A8 MoE for the smallest batches (at most 16 tokens): two launches, nothing handed over inside either.
//
// At these sizes a call is a chain of dependent memory round trips, each 1 - 2 us, around a stream of weights that takes
// a few microseconds (DeepSeek-V3 shard, one token: 49.6 MB, 8 us).  What shortens the chain:
//
//   * All tokens fit ONE 16-token operand tile, so every expert is multiplied with all of them: the activations are the
//     same operand for every piece of work, loaded into registers once, before anything is known about the routing.
//     A column of the product whose token did not choose the expert is dropped (the matrix unit is idle otherwise).
//   * UP (first launch) is split over w1 ROWS, not over K: a workgroup owns a range of intermediate columns (gate row + up
//     row each) over all of K, its eight wavefronts an eighth of K each, and adds the eight partial sums up in LDS: no
//     partial sums in memory, no arrival counter, no last arrival.  The ranges are equal to within a column, so every
//     compute unit streams the same bytes.
//   * DOWN (second launch) is split over OUTPUT columns: a workgroup owns K / 256 columns of `out` (28 on the DeepSeek-V3
//     shard) for all experts and all tokens, sums over the experts in registers and writes `out` itself: no result rows,
//     no closing pass.  It quantises the SwiGLU rows (a few KiB) for itself: the 128 columns of a quantisation group come
//     from many workgroups of the first launch, and a hand-over to whoever arrives last would be one more round trip.
//   * The two kinds are two launches: one persistent launch in which DOWN parts wait for a count of finished columns was
//     built first and was slower (M = 1: 35 us against 28 of the streaming kernel): 256 workgroups that add to, and poll,
//     one address queue up at ~10 ns each, 5 us for the first ticket and 10 - 15 us for the wait.  A kernel boundary
//     costs about 3 us and no ticket is needed.
//
// Weights go HBM -> LDS by direct-to-LDS loads into a ring of each wavefront's own (no barrier, counted waits), tiles
// swizzled as in moe_stream.hip.
//
// Measured on MI355X, us a call, weights cold, streaming kernel / this one: DeepSeek-V3 shard M = 1 28.5 / 18.9, 4 48.5 /
// 35.8, 8 77.4 / 60.5, 16 116.8 / 98.1; Qwen3-Next shard M = 1 23.4 / 12.8, 3 27.7 / 18.9, 16 61.5 / 51.1; Qwen3-30B shard
// M = 1 27.1 / 17.9, 8 45.0 / 39.9, 16 61.0 / 58.1 (this one is 1.0 - 2.5 us faster since: see the DOWN kernel).  What bounds
// it: from M = 4 on the DeepSeek-V3 shard HBM (5.9 TB/s over the first launch and 5.5 over the second at M = 16, launch and
// prologue included); below, the chain - at M = 1 2.5 us to the first weight load, 6.5 us until 33 MB have landed, 2 us between
// the launches, then the second one's prologue and 4.5 us for its 16.5 MB.
#include <mutex>
#include <type_traits>

#include "moe_common.hpp"

namespace alpha_moe {
namespace {

constexpr int kMaxTokens = 16;
constexpr int kMaxRows = 160;        // most (token, slot) rows, and so most experts
constexpr int kMaxSlices = 8;        // most 128-column slices of the intermediate (I <= 1024)
constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kPassRows = kThreads / 16, kPasses = kMaxRows / kPassRows;   // quantisation: 16 lanes per row
constexpr int kRingBytes = 12 << 10;   // per wavefront
constexpr int kBigRing = 16 << 10;     // DOWN launch, where there is room, and
constexpr int kLowRing = 5 << 10;      // where that lets all slices of the rows in (parts of eight columns)
constexpr int kUpDepth = 5;            // UP tiles of 2 KiB in flight per wavefront (the ring holds one more)
constexpr int kMaxLds = 158 << 10;

// What the first launch finds out about the routing and the second one reads.
struct Active {
    int n;                                  // active experts
    int poison;                             // results on this workspace are not to be trusted: answer NaN
    int repeats;                            // a token names an expert more than once: `same` has entries
    int pad;
    int expert[kMaxRows];
    uint8_t row[kMaxRows][kMaxTokens];      // [expert][token] -> (token, slot) row, 255: not routed
    uint8_t same[kMaxRows];                 // row -> the row that stands for the same (expert, token), 255: itself
};

struct SmallParams {
    MoeParams p;
    StreamCtl *ctl;
    Active *active;
    uint16_t *act;     // [rows][I] bf16 SwiGLU output of each (token, slot) row
    const uint16_t *x16;       // LAYER: the activations before quantisation [M][K] bf16, and
    const int32_t *topk_ids;   // the experts of each (token, slot) row
    int n_ib, nkb, n_mb_max, rows;
    unsigned ib_magic; // x / n_ib == x * ib_magic >> 16 for x <= kMaxRows * kMaxSlices
    int dcols;         // output columns per DOWN part
    int gi;            // slices whose quantised rows are in LDS at a time
    int off_sa, off_w2s;   // byte offsets behind the rings: [rows][n_ib] activation scales, [experts][n_ib][2] w2 scales
};

// UP tiles that are summed between two barriers
constexpr int batch_of(int nkw) { return nkw <= 2 ? 2 : 1; }

constexpr int kLayerExperts = 4096;    // LAYER: most experts (as many as the aligner takes)

// *at = min(*at, v) in LDS; complete behind the next lds_barrier().  (Not atomicMin: the compiler lets it wait for every
// direct-to-LDS load in flight, here the weights' first tiles: 0.3 - 0.8 us a call.)
__device__ __forceinline__ void lds_min(int *at, int v)
{
    const unsigned addr = (unsigned)(size_t)(__attribute__((address_space(3))) int *)at;
    asm volatile("ds_min_i32 %0, %1" ::"v"(addr), "v"(v) : "memory");
}
__device__ __forceinline__ void lds_or(unsigned *at, unsigned v)
{
    const unsigned addr = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned *)at;
    asm volatile("ds_or_b32 %0, %1" ::"v"(addr), "v"(v) : "memory");
}

// A store to LDS; complete behind the next lds_barrier(), and for what the same wavefront reads from LDS after it.  (Not a plain
// store, for the same reason.)
__device__ __forceinline__ void lds_store(void *at, uint2 v)
{
    const unsigned addr = (unsigned)(size_t)(__attribute__((address_space(3))) void *)at;
    asm volatile("ds_write_b64 %0, %1" ::"v"(addr), "v"(v) : "memory");
}
__device__ __forceinline__ void lds_store(float *at, float v)
{
    const unsigned addr = (unsigned)(size_t)(__attribute__((address_space(3))) float *)at;
    asm volatile("ds_write_b32 %0, %1" ::"v"(addr), "v"(v) : "memory");
}

// the largest of the values (not negative, not NaN) of the 16 lanes of a row (lanes 16 k .. 16 k + 15), in all of them: rotations
// within the row.  As integers, which such values compare as: a step is one instruction, where a float maximum is four.
__device__ __forceinline__ float max_of_16_lanes(float v)
{
    unsigned m = __builtin_bit_cast(unsigned, v);
    auto turned = [&](auto by) { return (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x120 + decltype(by)::value, 0xf, 0xf, true); };
    auto step = [&](auto by) {
        const unsigned o = turned(by);
        m = m > o ? m : o;
    };
    step(std::integral_constant<int, 8>());
    step(std::integral_constant<int, 4>());
    step(std::integral_constant<int, 2>());
    step(std::integral_constant<int, 1>());
    return __builtin_bit_cast(float, m);
}

// 128 columns of a row on 16 lanes, 8 each: FP8 codes and the row's scale (in all 16 lanes)
__device__ __forceinline__ uint2 quantise_row(const v4i raw, float *scale)
{
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[2 * i] = __builtin_bit_cast(float, (uint32_t)raw[i] << 16);
        v[2 * i + 1] = __builtin_bit_cast(float, (uint32_t)raw[i] & 0xffff0000u);
    }
    float m = kAmaxFloor;
#pragma unroll
    for (int i = 0; i < 8; i++) m = fmaxf(m, fabsf(v[i]));
    m = max_of_16_lanes(m);
    const RowScale rs(m);
    uint2 o;
    o.x = pack_fp8x4(rs.code(v[0]), rs.code(v[1]), rs.code(v[2]), rs.code(v[3]));
    o.y = pack_fp8x4(rs.code(v[4]), rs.code(v[5]), rs.code(v[6]), rs.code(v[7]));
    *scale = rs.scale;
    return o;
}

// NKW: 128-byte K blocks per wavefront.  LAYER: what a layer call starts from - bf16 activations and the router's output -
// is prepared here, by every workgroup for itself: the active experts come from a bit map of the rows' experts (ascending, as
// the aligner sorts them), and a wavefront quantises its K range of all tokens while its first weights are on their way.  That
// saves the preparation's launch (a chain of a few dependent steps on one workgroup, and the gap behind it: 3.3 - 4 us of a graph
// of layer calls); layer_pays() has both sides.
template <int NKW, bool LAYER>
__global__ __launch_bounds__(kThreads) void moe_small_up_kernel(const SmallParams s)
{
    constexpr int TB = batch_of(NKW);
    constexpr int S = kUpDepth, R = S + 1;
    static_assert(R * 2048 <= kRingBytes && 2 * S < 64, "ring depth");

    __shared__ __attribute__((aligned(1024))) uint8_t s_ring[kWaves * kRingBytes];
    __shared__ v4f s_red[2][TB][kWaves][64];   // partial sums
    __shared__ Active s_act;
    __shared__ __attribute__((aligned(16))) int s_row[kMaxRows][kMaxTokens];   // Active::row, a word each
    __shared__ short s_of_mb[kMaxRows];        // row block -> its expert's place in the list
    __shared__ __attribute__((aligned(16))) float s_ws[kWaves][2][16];   // [128-column block & 1][gate | up][K block]
    __shared__ int s_cnt[3];
    // LAYER: the experts that have a row; the scales of a wavefront's quantised K block
    __shared__ unsigned s_bits[LAYER ? kLayerExperts / 32 : 1];
    __shared__ float s_xs[LAYER ? kWaves : 1][kMaxTokens];

    const MoeParams &p = s.p;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int q = lane >> 4;
    const int K = p.K, I = p.N >> 1;
    const int n_ib = s.n_ib, nkb = s.nkb;
    uint8_t *ring = s_ring + wave * kRingBytes;

    const int kb0 = wave * NKW;
    const int ld_row = lane >> 3;   // loader side: row l / 8 (+ 8), chunk slot l % 8
    const int chunk0 = 16 * ((lane & 7) ^ (ld_row >> 1)), chunk1 = chunk0 ^ 64;

    // operand read offsets inside a 16x128 tile: chunk c of row m sits at c ^ ((m >> 1) & 7)
    const int f_n = (n >> 1) & 7;
    const int frag_lo = n * 128 + 16 * (q ^ f_n);
    const int frag_hi = n * 128 + 16 * ((q ^ f_n) ^ 4);
    v8i x_frag[NKW];   // (columns of tokens behind the last are dropped, K blocks behind the last are zero)
    float x_sc[NKW];
    int n_ids = 0, id0 = -1, n_mb = 0, n_act;
    // LAYER: a wavefront's 4 tokens x 128 columns of a K block, 16 lanes x 8 columns per token
    constexpr int TG = kMaxTokens / 4;
    v4i x_raw[LAYER ? NKW : 1][TG];
    int place = -1;   // LAYER: the place of row tid's expert in the list
    for (int i = tid; i < kMaxRows * kMaxTokens / 4; i += kThreads) reinterpret_cast<v4i *>(s_row)[i] = (v4i){255, 255, 255, 255};
    for (int i = tid; i < kMaxRows; i += kThreads) s_act.same[i] = 255;
    if (tid == 0) s_act.repeats = 0;
    // (loaded here: behind the weights' first tiles it would hold up the first workgroup's)
    unsigned error = 0;
    if (blockIdx.x == 0 && tid == 0) error = s.ctl->error;
    if constexpr (LAYER) {
        // one round trip: the rows' experts, then the activations
        const int e = tid < s.rows ? s.topk_ids[tid] : -1;
#pragma unroll
        for (int i = 0; i < NKW; i++)
#pragma unroll
            for (int j = 0; j < TG; j++) {
                const int t = 4 * j + (lane >> 4);
                if (4 * j < p.M)
                    x_raw[i][j] = *reinterpret_cast<const v4i *>(s.x16 + (size_t)(t < p.M ? t : p.M - 1) * K +
                                                                 (size_t)(kb0 + i < nkb ? kb0 + i : nkb - 1) * 128 + 8 * (lane & 15));
            }
        const bool ok = e >= 0 && e < p.E;
        for (int i = tid; i < kLayerExperts / 32; i += kThreads) s_bits[i] = 0;
        lds_barrier();
        if (ok) lds_or(&s_bits[e >> 5], 1u << (e & 31));
        lds_barrier();
        if (wave < 3) {   // rows are on the first three wavefronts
            // experts in the words before this lane's: two words per lane cover the map
            const unsigned w0 = s_bits[2 * lane], w1 = s_bits[2 * lane + 1];
            const int own = __builtin_popcount(w0) + __builtin_popcount(w1);
            int incl = own;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(incl, d);
                if (lane >= d) incl += o;
            }
            const int word = ok ? e >> 5 : 0;
            int before = __shfl(incl - own, word >> 1);
            if (word & 1) before += __builtin_popcount(s_bits[word - 1]);
            before += __builtin_popcount(s_bits[word] & ((1u << (e & 31)) - 1u));
            if (ok) {
                place = before;
                s_act.expert[place] = e;   // (equal rows write the same)
            }
            if (tid == 63) s_cnt[0] = incl;
        }
        lds_barrier();
        n_act = __builtin_amdgcn_readfirstlane(s_cnt[0]);
        asm volatile("" ::"v"(error));
        // (the activations have arrived: what is loaded from here on is not waited for by their quantisation)
#pragma unroll
        for (int i = 0; i < NKW; i++)
#pragma unroll
            for (int j = 0; j < TG; j++)
                if (4 * j < p.M) asm volatile("" ::"v"(x_raw[i][j]));
    } else {
        // one round trip: this wavefront's K range of all tokens, as operand tiles in the ring (and, where it holds one tile
        // less, where the partial sums go later), and the routing arrays.  (Operand loads straight into registers are 16 rows
        // x 64 bytes each: 3 us of them for 16 tokens.)
        auto x_tile = [&](int i) { return i < R ? ring + i * 2048 : reinterpret_cast<uint8_t *>(s_red) + wave * 2048; };
        static_assert(NKW <= R + 1 && sizeof(s_red) >= kWaves * 2048, "room for the token tiles");
#pragma unroll
        for (int i = 0; i < NKW; i++) {
            const uint8_t *src = p.x + (size_t)(kb0 + i < nkb ? kb0 + i : nkb - 1) * 128;
            dma16<0>(src + (size_t)(ld_row < p.M ? ld_row : p.M - 1) * K + chunk0, x_tile(i));
            dma16<0>(src + (size_t)(8 + ld_row < p.M ? 8 + ld_row : p.M - 1) * K + chunk1, x_tile(i) + 1024);
        }
        int e_mb = -1, e_before = -1;
        if (tid < s.n_mb_max) {
            e_mb = p.expert_ids[tid];
            if (tid > 0) e_before = p.expert_ids[tid - 1];
        }
        n_ids = s.n_mb_max * p.block_m < p.sorted_num ? s.n_mb_max * p.block_m : p.sorted_num;
        id0 = tid < n_ids ? p.sorted_ids[tid] : -1;
        const int ntpp = p.ntpp[0];
#pragma unroll
        for (int i = 0; i < NKW; i++) {
            x_sc[i] = 0.f;
            if (n < p.M && kb0 + i < nkb) x_sc[i] = p.x_scale[(size_t)n * nkb + kb0 + i];
        }

        // the active experts: row blocks whose expert is not the one of the block before
        n_mb = (__builtin_amdgcn_readfirstlane(ntpp) + p.block_m - 1) / p.block_m;
        n_mb = n_mb < s.n_mb_max ? n_mb : s.n_mb_max;
        drain_vmem();
        asm volatile("" ::"v"(error));
#pragma unroll
        for (int i = 0; i < NKW; i++) {
            x_frag[i] = cat(*reinterpret_cast<const v4i *>(x_tile(i) + frag_lo), *reinterpret_cast<const v4i *>(x_tile(i) + frag_hi));
            if (kb0 + i >= nkb) x_frag[i] = (v8i){0, 0, 0, 0, 0, 0, 0, 0};
        }
        const bool live = tid < n_mb && e_mb >= 0 && e_mb < p.E;
        const bool first = live && (tid == 0 || e_mb != e_before);
        const unsigned long long fm = __ballot(first);
        if (wave < 3 && lane == 0) s_cnt[wave] = __builtin_popcountll(fm);
        lds_barrier();
        {
            int at = __builtin_popcountll(fm & (~0ull >> (63 - lane)));   // with this lane
            for (int v = 0; v < 3; v++)
                if (v < wave) at += s_cnt[v];
            if (first) s_act.expert[at - 1] = e_mb;
            if (tid < n_mb) s_of_mb[tid] = live ? (short)(at - 1) : (short)-1;
        }
        n_act = __builtin_amdgcn_readfirstlane(s_cnt[0] + s_cnt[1] + s_cnt[2]);
        lds_barrier();
    }

    // ---- this workgroup's part: an equal range of the C = experts x I intermediate columns ------------------------
    const int C = n_act * I, parts = (int)gridDim.x;
    const int c_lo = (int)((unsigned long long)C * blockIdx.x / parts), c_hi = (int)((unsigned long long)C * (blockIdx.x + 1) / parts);
    auto expert_of = [&](int c) { return (int)(((unsigned)(c >> 7) * s.ib_magic) >> 16); };   // place in the list

    // a tile is at most eight columns of one 128-column block: eight gate rows, then their up rows
    auto tile_end = [&](int c) {
        int e = c + 8;
        const int block_end = (c | 127) + 1;
        e = e < block_end ? e : block_end;
        return e < c_hi ? e : c_hi;
    };
    int ci = c_lo;   // tile of the next load
    const uint8_t *src0 = nullptr, *src1 = nullptr;
    const uint8_t *w_kb0 = p.w + (size_t)kb0 * p.w_ks;
    const int sc_up = (lane >> 3) & 1, sc_i = (lane & 7) < NKW ? lane & 7 : NKW - 1;
    const int sc_kb = kb0 + sc_i < nkb ? kb0 + sc_i : nkb - 1;
    int block = -1;
    auto aim = [&]() {
        const int a = expert_of(ci);
        const int e = __builtin_amdgcn_readfirstlane(s_act.expert[a]);
        // the block's weight scales of this wavefront's K range, ahead of its first tile (a tile's wait then covers them;
        // one more load in flight than the waits count makes them stricter, never wrong)
        if ((ci >> 7) != block) {
            block = ci >> 7;
            if (lane < 16)
                dma4(p.w_scale + ((size_t)e * (p.N >> 7) + 2 * (block - a * n_ib) + sc_up) * nkb + sc_kb, s_ws[wave][block & 1]);
        }
        int col = ci + ld_row;
        const int last = tile_end(ci) - 1;
        col = (col < last ? col : last) - a * I;
        const uint8_t *base = w_kb0 + (size_t)e * p.N * K + (size_t)((col >> 3) * 16 + (col & 7)) * p.w_rs;
        src0 = base + chunk0;
        src1 = base + 8 * p.w_rs + chunk1;
    };
    int slot_w = 0, slot_r = 0;
    // one tile of the ring: K block kb0 + i of the tile at ci (a K block past the end is multiplied with zeros)
    auto issue = [&](int i) {
        const size_t at = (size_t)(kb0 + i < nkb ? i : nkb - 1 - kb0) * p.w_ks;
        uint8_t *dst = ring + slot_w * 2048;
        dma16<2>(src0 + at, dst);
        dma16<2>(src1 + at, dst + 1024);
        slot_w = slot_w + 1 == R ? 0 : slot_w + 1;
    };
    if (c_lo < c_hi) {
        aim();
#pragma unroll
        for (int j = 0; j < S; j++) {
            if (j > 0 && j % NKW == 0 && ci < c_hi) {
                ci = tile_end(ci);
                if (ci < c_hi) aim();
            }
            if (ci < c_hi) issue(j % NKW);
        }
    }

    // ---- while the first tiles are on their way: which row holds a token's share of an expert ----------------------
    // A token that names an expert more than once: its lowest row stands for all.  (The choice must not depend on the order
    // of the wavefronts: every workgroup makes it for itself, and the second launch reads what workgroup 0 chose.)
    auto for_rows = [&](auto f) {
        if constexpr (LAYER) {
            if (place >= 0) f(tid, s_row[place][tid / p.top_k]);
            return;
        }
        for (int idx = tid; idx < n_ids && idx < n_mb * p.block_m; idx += kThreads) {
            const int id = idx == tid ? id0 : p.sorted_ids[idx];
            const int a = s_of_mb[idx / p.block_m];
            if (id >= 0 && id < s.rows && a >= 0) f(id, s_row[a][id / p.top_k]);
        }
    };
    for_rows([&](int id, int &row) { lds_min(&row, id); });
    lds_barrier();
    if (blockIdx.x == 0) {   // for the second launch
        for_rows([&](int id, int &row) {
            if (row != id) {
                s_act.same[id] = (uint8_t)row;
                s_act.repeats = 1;
            }
        });
        if (tid == 0) {
            // a wait that ran out in an earlier launch on this workspace (sticky): the output says so itself, NaN in every element
            s_act.n = n_act;
            s_act.poison = error != 0;
        }
        lds_barrier();
        constexpr int kRow0 = offsetof(Active, row) / 4, kRow1 = kRow0 + kMaxRows * kMaxTokens / 4;
        for (int i = tid; i < (int)sizeof(Active) / 4; i += kThreads) {
            int word = reinterpret_cast<const int *>(&s_act)[i];
            if (i >= kRow0 && i < kRow1) {
                const v4i r = reinterpret_cast<const v4i *>(s_row)[i - kRow0];
                word = r.x | r.y << 8 | r.z << 16 | r.w << 24;
            }
            reinterpret_cast<int *>(s.active)[i] = word;
        }
    }

    if constexpr (LAYER) {
        // this wavefront's K range of the activations: quantised row by row (16 lanes a row), through LDS into the operand
        // layout - where its own partial sums go later, 8 tokens in each buffer.  One wavefront's LDS accesses complete in
        // order: no barrier.
        static_assert(kMaxTokens == 16 && sizeof(s_red[0][0][0]) == 8 * 128, "a buffer holds 8 tokens' K block");
        const int t = lane >> 4, sub = lane & 15;
        auto at = [&](int row) { return reinterpret_cast<uint8_t *>(s_red[row >> 3][0][wave]) + (row & 7) * 128; };
#pragma unroll
        for (int i = 0; i < NKW; i++) {
#pragma unroll
            for (int j = 0; j < TG; j++)
                if (4 * j < p.M) {
                    float sa;
                    const uint2 o = quantise_row(x_raw[i][j], &sa);
                    const int row = 4 * j + t;
                    lds_store(at(row) + 16 * ((sub >> 1) ^ ((row >> 1) & 7)) + 8 * (sub & 1), o);
                    if (sub == 0) lds_store(&s_xs[wave][row], sa);
                }
            // (columns of tokens behind the last are dropped)
            x_frag[i] = cat(*reinterpret_cast<const v4i *>(at(n) + 16 * (q ^ f_n)),
                            *reinterpret_cast<const v4i *>(at(n) + 16 * ((q ^ f_n) ^ 4)));
            x_sc[i] = n < p.M && kb0 + i < nkb ? s_xs[wave][n] : 0.f;
            if (kb0 + i >= nkb) x_frag[i] = (v8i){0, 0, 0, 0, 0, 0, 0, 0};
        }
    }

    int buf = 0;    // partial-sum buffer of the next batch
    int turn = 0;   // wavefront that finishes the next tile
    for (int c = c_lo; c < c_hi;) {
        v4f acc[TB];
        int tile_c[TB + 1];
        tile_c[0] = c;
#pragma unroll
        for (int tb = 0; tb < TB; tb++) {
            acc[tb] = (v4f){0.f, 0.f, 0.f, 0.f};
            const int ct = tile_c[tb];
            if (ct < c_hi) {
                float f[8];
#pragma unroll
                for (int i = 0; i < NKW; i++) {
                    wait_lds_reads();   // the slot loaded next has been read
                    if ((i + S) % NKW == 0 && ci < c_hi) {
                        ci = tile_end(ci);
                        if (ci < c_hi) aim();
                    }
                    if (ci < c_hi) {
                        issue((i + S) % NKW);
                        wait_vmcnt<2 * S>();
                    } else {
                        drain_vmem();   // nothing left to issue: what is in flight lands together
                    }
                    if (i == 0) {
                        const float *ws = &s_ws[wave][(ct >> 7) & 1][8 * (q >> 1)];
                        const v4f w_lo = *reinterpret_cast<const v4f *>(ws), w_hi = *reinterpret_cast<const v4f *>(ws + 4);
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            f[k] = w_lo[k];
                            f[4 + k] = w_hi[k];
                        }
                        if (kb0 + NKW > nkb) {   // past the end: nothing, also where the last block's scale is infinite
#pragma unroll
                            for (int k = 0; k < NKW; k++)
                                if (kb0 + k >= nkb) f[k] = 0.f;
                        }
                    }
                    const uint8_t *tile = ring + slot_r * 2048;
                    slot_r = slot_r + 1 == R ? 0 : slot_r + 1;
                    const v8i w_frag = cat(*reinterpret_cast<const v4i *>(tile + frag_lo), *reinterpret_cast<const v4i *>(tile + frag_hi));
                    acc[tb] += mfma_fp8(w_frag, x_frag[i]) * (f[i] * x_sc[i]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            tile_c[tb + 1] = ct < c_hi ? tile_end(ct) : c_hi;
        }
        c = tile_c[TB];
#pragma unroll
        for (int tb = 0; tb < TB; tb++) s_red[buf][tb][wave][lane] = acc[tb];
        lds_barrier();
#pragma unroll
        for (int tb = 0; tb < TB; tb++) {
            if (wave == ((turn + tb) & (kWaves - 1)) && tile_c[tb] < c_hi) {
                v4f v = s_red[buf][tb][0][lane];
#pragma unroll
                for (int w = 1; w < kWaves; w++) v += s_red[buf][tb][w][lane];
                // lanes q < 2 hold the gate sums of columns 4 q .. 4 q + 3, lanes q + 2 the up sums
                const int a = expert_of(tile_c[tb]);
                const int row = s_row[a][n];
                const int col = tile_c[tb] + 4 * (q & 1);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float up = __shfl_xor(v[j], 32);
                    const float r = swiglu_bf16(v[j], up);
                    if (q < 2 && row != 255 && col + j < tile_c[tb + 1])
                        s.act[row * I + col + j - a * I] = (uint16_t)(__builtin_bit_cast(uint32_t, r) >> 16);
                }
            }
        }
        turn += TB;
        buf ^= 1;
    }
}

// H: groups of 8 output columns per part.  RING: bytes of a wavefront's ring.
// Until its first product a part is a chain of round trips: what the first launch has left, then the weights.  Nothing may wait
// in between - a load that is multiplied where it is loaded, a use of a register that might have been loaded behind the ring, a
// plain store to LDS cost 1.0 - 1.6 us a call together (MI355X, us an operator call: DeepSeek shard 1 token 22.6 -> 21.3, 7 tokens
// 57.8 -> 56.3; Qwen3-Next shard 14.7 -> 14.1, 32.2 -> 30.8; Qwen3-MoE shard 21.8 -> 19.4, 38.8 -> 37.7).
template <int H, int RING>
__global__ __launch_bounds__(kThreads) void moe_small_down_kernel(const SmallParams s)
{
    constexpr int NTD = (H + 1) / 2;                 // 16-column operand tiles
    constexpr int RD = RING / (H * 1024);      // ring: units of H KiB
    constexpr int SD = RD - 1;
    static_assert(H * SD < 64, "ring depth");

    // [8 rings] | quantised rows [rows][gi][128], later partial sums [NTD][8][1 KiB] | tables
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds_dyn[];
    __shared__ Active s_act;
    __shared__ float s_tw[kMaxRows];

    const MoeParams &p = s.p;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int q = lane >> 4;
    const int K = p.K, I = p.N >> 1;
    const int n_ib = s.n_ib;
    uint8_t *ring = lds_dyn + wave * RING;
    uint8_t *area = lds_dyn + kWaves * RING;
    float *s_sa = reinterpret_cast<float *>(area + s.off_sa);
    float *s_w2s = reinterpret_cast<float *>(area + s.off_w2s);
    const int ld_row = lane >> 3;   // loader side: row l / 8 of a group of eight, chunk slot l % 8
    const int chunk0 = 16 * ((lane & 7) ^ (ld_row >> 1)), chunk1 = chunk0 ^ 64;

    // this part's columns
    const int d0 = blockIdx.x * s.dcols;
    const int n_col = s.dcols < K - d0 ? s.dcols : K - d0;

    // ---- everything the first launch has left, the routing weights, what `out` holds: one round trip ----------------
    // wavefront t finishes operand tile t: its lanes' four columns of token n
    const int o_col = 16 * wave + 4 * q;
    const bool o_mine = wave < NTD && n < p.M && o_col < n_col;
    uint2 *op = reinterpret_cast<uint2 *>(p.out + (size_t)(o_mine ? n : 0) * K + d0 + (o_mine ? o_col : 0));
    uint2 prior = make_uint2(0u, 0u);
    if (o_mine && !p.overwrite) prior = *op;

    constexpr int kActWords = (int)sizeof(Active) / 4, kActLoads = (kActWords + kThreads - 1) / kThreads;
    int act_reg[kActLoads];
#pragma unroll
    for (int k = 0; k < kActLoads; k++) {
        const int i = tid + k * kThreads;
        act_reg[k] = i < kActWords ? reinterpret_cast<const int *>(s.active)[i] : 0;
    }
    float tw_reg = 0.f;
    if (tid < s.rows) tw_reg = p.topk_w[tid];
    // Rows to quantise: 16 lanes x 8 columns per row, 32 rows a pass; two slices in flight (what is loaded behind the ring's
    // first tiles arrives behind them, too).
    const int sub = tid & 15;
    v4i raw[2][kPasses];
    auto load_slice = [&](int ib, v4i (&to)[kPasses]) {
#pragma unroll
        for (int u = 0; u < kPasses; u++) {
            const int row = u * kPassRows + (tid >> 4);
            to[u] = (v4i){0, 0, 0, 0};
            if (row < s.rows) to[u] = *reinterpret_cast<const v4i *>(s.act + (size_t)row * I + ib * 128 + sub * 8);
        }
    };
    load_slice(0, raw[0]);
    load_slice(n_ib > 1 ? 1 : 0, raw[1]);
    auto slices_of = [&](int g) { return n_ib - g * s.gi < s.gi ? n_ib - g * s.gi : s.gi; };
#pragma unroll
    for (int k = 0; k < kActLoads; k++) {
        const int i = tid + k * kThreads;
        if (i < kActWords) reinterpret_cast<int *>(&s_act)[i] = act_reg[k];
    }
    tw_reg *= p.scaling;
    if (tid < s.rows) s_tw[tid] = tw_reg;
    // (all of this has arrived, whatever is loaded from here on)
    asm volatile("" ::"v"(prior.x), "v"(prior.y));
#pragma unroll
    for (int u = 0; u < kPasses; u++) asm volatile("" ::"v"(raw[0][u]), "v"(raw[1][u]));
    lds_barrier();
    const int n_act = __builtin_amdgcn_readfirstlane(s_act.n);
    const bool poisoned = s_act.poison != 0;
    const int repeats = __builtin_amdgcn_readfirstlane(s_act.repeats);

    // ---- the weights; units of a wavefront's ring: slice group, then experts wave, wave + 8,
    // ..., then the group's slices
    const int mine = n_act > wave ? (n_act - wave + kWaves - 1) / kWaves : 0;
    int ig = 0, ia = wave, is = 0;   // group, expert, slice in the group of the next load
    const int n_groups = (n_ib + s.gi - 1) / s.gi;
    int slot_w = 0, slot_r = 0;
    const uint8_t *src[H];
#pragma unroll
    for (int h = 0; h < H; h++) {
        const int r = 8 * h + ld_row;
        src[h] = p.w2 + (size_t)(d0 + (r < n_col ? r : n_col - 1)) * p.w2_rs + ((h & 1) ? chunk1 : chunk0);
    }
    auto issue = [&]() {
        const size_t at = (size_t)__builtin_amdgcn_readfirstlane(s_act.expert[ia]) * K * I + (ig * s.gi + is) * p.w2_ks;
#pragma unroll
        for (int h = 0; h < H; h++) dma16<2>(src[h] + at, ring + slot_w * (H * 1024) + h * 1024);
        slot_w = slot_w + 1 == RD ? 0 : slot_w + 1;
        if (++is == slices_of(ig)) {
            is = 0;
            ia += kWaves;
            if (ia >= n_act) {
                ia = wave;
                ig++;
            }
        }
    };
    // the w2 scales of the part's one or two 128-column blocks, ahead of the ring's loads
    const int blk0 = d0 >> 7;
    for (int i0 = wave * 64; i0 < n_act * n_ib * 2; i0 += kThreads) {
        const int i = i0 + lane;
        if (i < n_act * n_ib * 2) {
            const int ai = i >> 1, a = (int)(((unsigned)ai * s.ib_magic) >> 16);
            int blk = blk0 + (i & 1);
            blk = blk < (K >> 7) ? blk : (K >> 7) - 1;
            dma4(p.w2_scale + ((size_t)s_act.expert[a] * (K >> 7) + blk) * n_ib + (ai - a * n_ib), s_w2s + i0);
        }
    }
    int left = mine * n_ib;   // units not yet issued
    for (int j = 0; j < SD; j++)
        if (left > 0) {
            issue();
            left--;
        }
    v4f acc[NTD];
#pragma unroll
    for (int t = 0; t < NTD; t++) acc[t] = (v4f){0.f, 0.f, 0.f, 0.f};
    for (int g = 0; g < n_groups; g++) {
        const int ns = slices_of(g);
        // row r's slice sl of the group at (r * gi + sl) * 128, its 16-byte chunk c at c ^ (r & 7)
        for (int s0 = 0; s0 < ns; s0 += 2) {
            if (g > 0 || s0 > 0) {
#pragma unroll
                for (int h = 0; h < 2; h++)
                    if (s0 + h < ns) load_slice(g * s.gi + s0 + h, raw[h]);
                // (waited for here: the first two slices' quantisation does not wait for the ring)
#pragma unroll
                for (int u = 0; u < kPasses; u++) asm volatile("" ::"v"(raw[0][u]), "v"(raw[1][u]));
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int sl = s0 + h, ib = g * s.gi + sl;
                if (sl >= ns) break;
#pragma unroll
                for (int u = 0; u < kPasses; u++) {
                    if (u * kPassRows >= s.rows) break;
                    const int row = u * kPassRows + (tid >> 4);
                    float sa;
                    const uint2 o = quantise_row(raw[h][u], &sa);
                    if (row < s.rows) {
                        lds_store(area + (row * s.gi + sl) * 128 + 16 * ((sub >> 1) ^ (row & 7)) + 8 * (sub & 1), o);
                        if (sub == 0) lds_store(&s_sa[row * n_ib + ib], sa);
                    }
                }
            }
        }
        if (g == 0) {
            // the w2 scales have arrived, the ring's loads may be outstanding
            if (mine * n_ib >= SD)
                wait_vmcnt<H * SD>();
            else
                drain_vmem();
            // a row that stands for others of its token takes their weights over, in ascending order (a fixed one: the result
            // does not depend on which wavefront comes first)
            if (repeats && tid < s.rows && s_act.same[tid] == 255) {
                float tw = tw_reg;
                for (int r = tid + 1, end = (tid / p.top_k + 1) * p.top_k; r < end; r++)
                    if (s_act.same[r] == tid) tw += s_tw[r];
                s_tw[tid] = tw;
            }
        }
        lds_barrier();
        for (int a = wave; a < n_act; a += kWaves) {
            const int row_n = s_act.row[a][n];
            const bool routed = row_n != 255;
            const int row = routed ? row_n : 0;
            v4f d[NTD];
#pragma unroll
            for (int t = 0; t < NTD; t++) d[t] = (v4f){0.f, 0.f, 0.f, 0.f};
            for (int sl = 0; sl < ns; sl++) {
                wait_lds_reads();
                if (left > 0) {
                    issue();
                    left--;
                    wait_vmcnt<H * SD>();
                } else {
                    drain_vmem();
                }
                const uint8_t *b_row = area + (row * s.gi + sl) * 128;
                const v8i b = cat(*reinterpret_cast<const v4i *>(b_row + 16 * (q ^ (row & 7))),
                                  *reinterpret_cast<const v4i *>(b_row + 16 * ((q + 4) ^ (row & 7))));
                const float sa = s_sa[row * n_ib + g * s.gi + sl];
                const uint8_t *tiles = ring + slot_r * (H * 1024);
                slot_r = slot_r + 1 == RD ? 0 : slot_r + 1;
#pragma unroll
                for (int t = 0; t < NTD; t++) {
                    // (one group of eight columns: rows 8 .. 15 of the tile repeat rows 0 .. 7 and are not stored)
                    const int m = (2 * t + 1 < H) ? n : (n & 7), f_m = (m >> 1) & 7;
                    const uint8_t *tile = tiles + t * 2048 + m * 128;
                    const v8i w_frag = cat(*reinterpret_cast<const v4i *>(tile + 16 * (q ^ f_m)),
                                           *reinterpret_cast<const v4i *>(tile + 16 * ((q ^ f_m) ^ 4)));
                    const int blk = ((d0 + 16 * t + 4 * q) >> 7) - blk0;
                    d[t] += mfma_fp8(w_frag, b) * (sa * s_w2s[(a * n_ib + g * s.gi + sl) * 2 + (blk > 0 ? 1 : 0)]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (routed) {
                const float tw = s_tw[row];
#pragma unroll
                for (int t = 0; t < NTD; t++) acc[t] += d[t] * tw;
            }
        }
        lds_barrier();   // the rows of this group have been read
    }
    v4f *red = reinterpret_cast<v4f *>(area);
#pragma unroll
    for (int t = 0; t < NTD; t++) red[(t * kWaves + wave) * 64 + lane] = acc[t];
    lds_barrier();
    if (o_mine) {
        v4f v = red[wave * kWaves * 64 + lane];
#pragma unroll
        for (int w = 1; w < kWaves; w++) v += red[(wave * kWaves + w) * 64 + lane];
        const float o0 = __builtin_bit_cast(float, prior.x << 16), o1 = __builtin_bit_cast(float, prior.x & 0xffff0000u);
        const float o2 = __builtin_bit_cast(float, prior.y << 16), o3 = __builtin_bit_cast(float, prior.y & 0xffff0000u);
        uint2 r;
        r.x = poisoned ? 0x7fc07fc0u : pack_bf16x2(o0 + v[0], o1 + v[1]);
        r.y = poisoned ? 0x7fc07fc0u : pack_bf16x2(o2 + v[2], o3 + v[3]);
        *op = r;
    }
}

size_t align_up(size_t v) { return (v + 255) & ~(size_t)255; }

int compute_units()
{
    static const int n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            return 256;
        return cus;
    }();
    return n;
}

struct SmallPlan {
    bool ok;
    int nkw, up_parts, h, dcols, n_down, gi, ring, off_sa, off_w2s, lds_bytes;
};

// K blocks of a wavefront of the first launch: the variants there are
int blocks_per_wave(int K)
{
    const int per_wave = (K / 128 + kWaves - 1) / kWaves;
    return per_wave <= 1 ? 1 : per_wave <= 2 ? 2 : per_wave <= 4 ? 4 : 7;
}

SmallPlan make_plan(int top_k, int M, int K, int N, int block_m)
{
    SmallPlan h = {};
    const int n_ib = N / 256, rows = M * top_k;
    if (M > kMaxTokens || rows > kMaxRows || n_ib > kMaxSlices || K > 128 * kWaves * 7 || block_m > 32) return h;
    h.nkw = blocks_per_wave(K);
    const int cus = compute_units();
    h.up_parts = cus;
    // DOWN: one part per compute unit, whole groups of four columns (a lane's), at most 32
    h.dcols = ((K + cus - 1) / cus + 3) / 4 * 4;
    if (h.dcols > 32) h.dcols = 32;
    h.n_down = (K + h.dcols - 1) / h.dcols;
    h.h = h.dcols <= 8 ? 1 : h.dcols <= 16 ? 2 : 4;
    // quantised rows: all slices at once if they fit, else as many as do
    const int partial = (h.h + 1) / 2 * kWaves * 1024;
    const int tables = rows * n_ib * 4 + rows * n_ib * 8;
    const int fixed = tables + (int)sizeof(Active) + kMaxRows * 4 + 1024;
    auto area_of = [&](int gi) {
        const int rows_bytes = rows * gi * 128;
        return ((rows_bytes > partial ? rows_bytes : partial) + 15) & ~15;
    };
    auto fits = [&](int ring, int gi) { return kWaves * ring + area_of(gi) + fixed <= kMaxLds; };
    h.gi = n_ib;
    h.ring = fits(kBigRing, n_ib) ? kBigRing : !fits(kRingBytes, n_ib) && h.h == 1 && fits(kLowRing, n_ib) ? kLowRing : kRingBytes;
    while (h.gi > 1 && !fits(h.ring, h.gi)) h.gi--;
    const int area = area_of(h.gi);
    h.off_sa = area;
    h.off_w2s = area + rows * n_ib * 4;
    h.lds_bytes = kWaves * h.ring + area + tables;
    h.ok = fits(h.ring, h.gi);
    return h;
}

typedef void (*SmallFn)(const SmallParams);

template <bool LAYER>
SmallFn pick_up(int nkw)
{
    switch (nkw) {
    case 1: return moe_small_up_kernel<1, LAYER>;
    case 2: return moe_small_up_kernel<2, LAYER>;
    case 4: return moe_small_up_kernel<4, LAYER>;
    default: return moe_small_up_kernel<7, LAYER>;
    }
}

template <int RING>
SmallFn pick_down(int h)
{
    return h == 1 ? moe_small_down_kernel<1, RING> : h == 2 ? moe_small_down_kernel<2, RING> : moe_small_down_kernel<4, RING>;
}

SmallFn pick_down(int h, int ring)
{
    if (ring == kLowRing) return moe_small_down_kernel<1, kLowRing>;
    return ring == kBigRing ? pick_down<kBigRing>(h) : pick_down<kRingBytes>(h);
}

// The variant's dynamic LDS limit is raised once per (variant, device), not on every launch.
hipError_t allow_dynamic_lds(int h, int ring, SmallFn fn)
{
    static std::mutex mu;
    static bool done[5][kBigRing / 1024 + 1][64];
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    std::lock_guard<std::mutex> lock(mu);
    if (dev >= 0 && dev < 64 && done[h][ring / 1024][dev]) return hipSuccess;
    err = hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kMaxLds - (int)sizeof(Active) - kMaxRows * 4);
    if (err == hipSuccess && dev >= 0 && dev < 64) done[h][ring / 1024][dev] = true;
    return err;
}

}  // namespace

bool small_supported(int top_k, int M, int K, int N, int block_m) { return make_plan(top_k, M, K, N, block_m).ok; }

// Every part of the second launch quantises all rows and walks all experts' slices, whatever K is: on narrow layers with many
// rows that chain takes longer than the streaming kernel's whole call; on wide ones the weights' bytes hide it.  With
// u = (4 min(E, rows) + rows) I / 5, a measure of that chain, the small kernels are ahead while u (1 - K / 2496) is at most
// 19 Ki.  MI355X, cold weights, small / streaming us a call, experts drawn evenly: K = 512, I = 512: 32 rows (u 16 Ki) 21.8 /
// 23.1, 64 (32 Ki) 28.3 / 24.9, 160 (80 Ki) 57.3 / 36.5; K = 1024, I = 256: 96 rows (24 Ki) 28.2 / 34.7, 128 (32 Ki) 31.8 / 31.5,
// 160 (40 Ki) 39.9 / 34.4; K = 1536, I = 768: 64 rows (48 Ki) 47.6 / 51.2, 96 (72 Ki) 58.8 / 55.3; K = 2048, I = 768: 64 rows
// (48 Ki) 54.1 / 58.1, 128 (96 Ki) 77.4 / 76.5 (with Zipf popularity 60.0 / 58.9, 112 rows 53.9 / 54.9); from K = 3072 on the
// small kernels take at most 1.06 of the streaming kernel's time, mostly 0.65 - 0.95 (K = 5120 and 6144, 128 rows of I = 256:
// 68 / 73 and 74 / 82).
bool small_pays(int top_k, int M, int K, int N, int E)
{
    const long long rows = (long long)M * top_k, u5 = (4 * (rows < E ? rows : E) + rows) * (N / 2);
    return K >= 2496 || u5 * (2496 - K) <= 5ll * 19456 * 2496;
}

size_t small_workspace_bytes(int top_k, int M, int N)
{
    return align_up(kPrefixBytes) + align_up(sizeof(Active)) + align_up((size_t)M * top_k * (N / 2) * sizeof(uint16_t));
}

bool layer_supported(int E) { return E <= kLayerExperts; }

// The preparation's launch saved against what every workgroup of the first launch does instead: its eight wavefronts read and
// quantise four tokens at a time, `nkw` K blocks each, so it grows with their product, and the more weights follow the more of
// it they hide.  MI355X, graphs of cold calls, us a layer call, three launches / two:
//   1 group x 7 blocks    DeepSeek shard, 4 tokens 43.4 / 41.1; K = 7168, I = 128, top 1 15.4 / 14.3
//   2 x 7                 DeepSeek shard, 8 tokens 68.2 / 66.7; K = 7168, I = 1024, top 4 66.3 / 65.4; I = 128, top 1 17.1 / 18.0
//   4 x 2                 Qwen3-Next shard, 16 tokens 55.3 / 51.3; K = 2048, I = 128, top 1 14.6 / 13.4
//   4 x 4                 K = 4096, 16 tokens: I = 256, top 8 58.5 / 57.6; I = 128, top 1 17.5 / 18.5
//   3 x 7                 DeepSeek shard, 12 tokens 88.7 / 89.3; K = 7168, I = 256, top 2, 9 tokens 29.3 / 30.1; K = 4224, I = 256,
//                         top 2, 12 tokens 27.8 / 30.3, I = 128, top 1, 9 tokens 17.0 / 20.5
//   4 x 7                 DeepSeek shard, 16 tokens 107.2 / 107.8; K = 6144, I = 256, top 8 75.8 / 78.7; K = 7168, I = 128, top 1
//                         22.8 / 27.5
// Outside a graph the third launch and the five tensors of the preparation cost a caller that waits for each call 1 - 2 us more:
// at 3 x 7 DeepSeek shard, 12 tokens 108.2 / 106.3, K = 7168, I = 256, top 2, 9 tokens 46.0 / 44.3 (99 MB of weights), but
// K = 4224, I = 256, top 2, 12 tokens 45.2 / 45.2 (78 MB), I = 128, top 1, 9 tokens 34.7 / 36.0; at 4 x 7 DeepSeek shard
// 128.3 / 127.7, K = 5120, I = 256, top 8 87.5 / 88.4.
bool layer_pays(int top_k, int M, int K, int N, int E)
{
    const int steps = (M + 3) / 4 * blocks_per_wave(K);
    const long long experts = (long long)M * top_k < E ? (long long)M * top_k : E;
    return steps <= 16 || (steps <= 21 && experts * (N / 2) * 3 * K >= (80ll << 20));
}

hipError_t launch_small(const MoeParams &p, const uint16_t *x16, const int32_t *topk_ids, void *workspace, hipStream_t stream)
{
    const SmallPlan h = make_plan(p.top_k, p.M, p.K, p.N, p.block_m);
    if (!h.ok) return hipErrorInvalidValue;
    uint8_t *ws = static_cast<uint8_t *>(workspace);
    SmallParams s;
    s.p = p;
    s.ctl = reinterpret_cast<StreamCtl *>(ws);
    s.active = reinterpret_cast<Active *>(ws + align_up(kPrefixBytes));
    s.act = reinterpret_cast<uint16_t *>(ws + align_up(kPrefixBytes) + align_up(sizeof(Active)));
    s.x16 = x16;
    s.topk_ids = topk_ids;
    s.n_ib = p.N / 256;
    s.nkb = p.K / 128;
    s.rows = p.M * p.top_k;
    s.n_mb_max = (p.sorted_num + p.block_m - 1) / p.block_m;   // a live row block holds at least one row
    if (s.n_mb_max > s.rows) s.n_mb_max = s.rows;
    s.ib_magic = 65536u / (unsigned)s.n_ib + 1u;
    s.dcols = h.dcols;
    s.gi = h.gi;
    s.off_sa = h.off_sa;
    s.off_w2s = h.off_w2s;
    const SmallFn down = pick_down(h.h, h.ring);
    hipError_t err = allow_dynamic_lds(h.h, h.ring, down);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(x16 ? pick_up<true>(h.nkw) : pick_up<false>(h.nkw), dim3((unsigned)h.up_parts), dim3(kThreads), 0, stream, s);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(down, dim3((unsigned)h.n_down), dim3(kThreads), h.lds_bytes, stream, s);
    return hipGetLastError();
}

}  // namespace alpha_moe
