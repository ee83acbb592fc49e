// Fused W8A8 MoE for row blocks above 32 rows (prefill and large decode batches), and for smaller ones that are too many for the
// streaming kernel: one launch of short-lived workgroups of four
// wavefronts, two to a compute unit (three for blocks of at most 64 rows), each with one work item, then the row sums
// (moe_rows_reduce_kernel).
//
// What bounds it: the weights and result rows at sizes where an expert has few rows (HBM), the path into a compute unit and the
// matrix cores above.  Why independent workgroups: an item has phases that use nothing of what the others wait for - a chain of
// round trips before its first load, the K loop, SwiGLU and requantisation, the acknowledgement of its stores - and a
// workgroup that shares its compute unit with another one in a different phase hides them without any scheduling of ours.  The
// persistent kernels of eight wavefronts that were here before (one row block, or 256 rows, to a workgroup that had the compute
// unit to itself) spent a third of their time in those phases.  MI355X, layer
// calls back to back, before and with this kernel (every launch of the call): Qwen3-30B M = 1024 200 -> 154 us, M = 8192 589 -> 486;
// Qwen3-Next M = 4096 284 -> 236; DeepSeek shard M = 2048 421 -> 387, M = 8192 1040 -> 976.
//
// UP item: a row block x one 128-column slice of the intermediate (256 rows of w1).  Wavefront w multiplies slab rows
// 64 w .. 64 w + 63 with all token tiles.  Nobody else reads its weights, so they go through a small ring of its own: a step's four
// tiles are read into registers at its start and their places refilled at once, which makes the registers one more stage
// and leaves LDS for two stages of token tiles and for the second workgroup.  One barrier a step.  All loads are direct to LDS
// and cover whole 128-byte lines (the register layout of the matrix operands - 16 rows x 64 bytes an instruction - is loaded at a
// quarter of the rate).  A step's loads go out in a burst in front of its matrix work; handed out between the token tiles they
// cost 2 %: the matrix instructions then wait for the memory path, which the other workgroup's matrix work would fill.
// Then SwiGLU, the row maxima of the slice and the FP8 requantisation in registers; the operand tiles are put together in LDS
// (4-byte stores to memory: 3 us an item more), stored, and the unit's flag is raised
// (fused_moe_w8a8_up_down_acc.cu:863-994 of the reference).
//
// DOWN item: a row block x a slab of output columns, all slices; 64 columns to a wavefront and step, w2 through the same ring.
// Up to two slices' tiles stay in LDS for the whole item (then no barrier either), more are streamed like tokens.  Each valid (token, slot)
// row is written once, bf16, to y[slot] (fused_moe_w8a8_up_down_acc.cu:1007-1096 adds top_k * I/128 partial rows per token into the
// output instead).
//
// Which item: eight queues, one per XCD (workgroups are dealt to the XCDs in turn), so that row blocks of one expert meet in one
// L2; a workgroup draws a ticket from its queue's counter.  A queue holds the UP items of all its blocks, then the DOWN items, which
// wait for flags of UP items EARLIER in the same queue: whoever drew those is running and waits for nothing, so every queue drains
// with any number of resident workgroups.  (By workgroup index instead of a ticket: at most 1 % faster, but it needs workgroups to
// start in order.  Workgroups that stay and take item after item: 5 - 15 % slower.)
#include <mutex>
#include <type_traits>

#include "moe_common.hpp"

namespace alpha_moe {
namespace {

// Dynamic LDS: a ring of weight tiles for each wavefront and, behind them, a ring of the steps' token tiles.  Where K is short, what
// token tiles a row block does not have is room for more of both in flight (Qwen3-30B shard, 128-row blocks of which most have
// one to four tiles: M = 512 147 -> 144 us, 1024 165 -> 159.5; Qwen3-Next M = 1500 186 -> 184).  Where K is long, a few-row block that
// runs ahead takes its neighbours' lines out of L2: DeepSeek shard M = 2048 408 -> 412 us, 8192 939 -> 955.  Between the two (128 experts,
// six to a token, I = 512, 128-row blocks, us without -> with, M = 250 / 1000 / 6000): K = 3072 108 -> 106, 125 -> 126, 331 -> 327;
// K = 4096 176 -> 166, 196 -> 191, 420 -> 423; K = 5120 174 -> 170, 201 -> 198, 526 -> 534; K = 6144 205 -> 203, 232 -> 231, 610 -> 616.
constexpr int dyn_lds(int nt) { return nt <= 4 ? 48 * 1024 : 72 * 1024; }   // three workgroups to a compute unit, or two
constexpr int x_stages(int nt, int t, bool deep)   // K steps of token tiles
{
    return deep && (dyn_lds(nt) - 3 * t * 2048) / 8192 >= 5 ? 3 : 2;
}
constexpr int w_tiles(int nt, int t, int stages, bool deep)   // weight tiles of a wavefront (four to a step)
{
    const int r = (dyn_lds(nt) - stages * t * 2048) / 8192;
    return !deep ? 4 : r < 7 ? r : 7;
}
constexpr int kGMaxExpertW2s = 1024;       // most w2 block scales of an expert, (K / 128) * (I / 128)
// Most w2 block scales of a DOWN item; group_plan picks variant and slab so that they fit.  The variant with three workgroups to a compute
// unit has no LDS for more than 512, the others' table holds all that an expert can have.
constexpr int max_w2s(int nt) { return nt <= 4 ? 512 : kGMaxExpertW2s; }
constexpr int kGMaxKb = 128;               // most 128-byte K blocks (K <= 16384)
constexpr int kGChunk = 8;                 // consecutive row blocks of a queue
constexpr int kGHeadStride = 128;          // words between the queues' counters (lines of their own); behind one: the queue's arrivals
constexpr int kGMaxRound = 96;             // most workgroups of a queue counted as running at a time
constexpr int kGDeepKb = 32;               // most K blocks with deep rings
constexpr int kGPiecesKb = 32;             // fewest K blocks whose contraction may be taken in parts
constexpr int kGResidentIb = 2;            // slices whose requantised tiles fit the token ring for a whole DOWN item

struct GroupParams {
    MoeParams p;
    StreamCtl *ctl;
    int *head;        // next item of queue q at [q * kGHeadStride]
    int *flag;        // [row block][n_ib] == epoch once the slice's tiles are in scratch
    int *live;        // [slots] == epoch once y[slot] is written this launch
    uint16_t *y;      // [slots][K] bf16
    uint8_t *aqs;     // [row block][n_ib][tpb] requantised operand tiles of 2 KiB
    float *sas;       // [row block][n_ib][tpb * 16] their per-token scales
    int n_ib, nkb, n_mb_max;
    int tpb;          // 16-row tile slots per row block in scratch
    int gps, n_cs;    // 64-column groups per DOWN item (a multiple of 4), column slabs
    int round;        // workgroups of a queue that run at a time
    int max_pieces;   // most parts of an UP item's contraction
    int xs_chunk;     // 1: a token's activation scales are fetched four K steps at a time (K / 128 a multiple of 4, x_scale
                      // 16-byte aligned), 0: one step at a time
    int w_nt;         // weights with non-temporal loads: 1 always, 0 never, -1 for experts with one row block
};

__device__ __forceinline__ int rfl(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Direct-to-LDS loads of 16 and 4 bytes per lane from (wavefront-uniform base) + (per-lane offset) + (uniform offset): one scalar
// addition a load, where the flat forms take a 64-bit address each.
template <int AUX>
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t base, unsigned voff, unsigned soff, void *lds)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(base, (lptr_t)(uint32_t)(uintptr_t)lds, 16, (int)voff, (int)soff, 0, AUX);
}
template <int AUX>
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t base, unsigned voff, unsigned soff, void *lds)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(base, (lptr_t)(uint32_t)(uintptr_t)lds, 4, (int)voff, (int)soff, 0, AUX);
}

// A step's four weight tiles as matrix operands in registers; their places in the ring may be refilled afterwards.
__device__ __forceinline__ void read_weights(v8i (&a)[4], const uint8_t *const (&tile)[4], int frag_lo, int frag_hi)
{
#pragma unroll
    for (int k = 0; k < 4; k++)
        a[k] = cat(*reinterpret_cast<const v4i *>(tile[k] + frag_lo), *reinterpret_cast<const v4i *>(tile[k] + frag_hi));
    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
    wait_lds_reads();
}

typedef const v4i __attribute__((address_space(3))) * lds_v4i;
typedef const float __attribute__((address_space(3))) * lds_f32;

// 4 weight tiles in registers x T token tiles in LDS: acc[k][t] += (a_k x b_t) * f_t * (k odd ? sc1 : sc0).  A product is scaled
// into its accumulator two matrix instructions after its own, so no wait states stand between the two.  A tile's operands are read while
// the tile before it is multiplied; LDS reads complete in order and the compiler waits for them by count, so none waits for reads
// behind its own - as long as they keep this order, which the scheduling barriers are for.
template <int T, int NT>
__device__ __forceinline__ void multiply(const v8i (&a)[4], const uint8_t *b_tiles, const float *row, int row_stride, float sc0,
                                         float sc1, v4f (&acc)[4][NT], int frag_lo, int frag_hi)
{
    const lds_v4i at_lo = (lds_v4i)(uint32_t)(uintptr_t)(b_tiles + frag_lo), at_hi = (lds_v4i)(uint32_t)(uintptr_t)(b_tiles + frag_hi);
    const lds_f32 at_f = (lds_f32)(uint32_t)(uintptr_t)row;
    v4i b_lo = *at_lo, b_hi = *at_hi;
    float f = *at_f;
    v4f prod[2];
    float fac[2];
    auto tile = [&](auto tc) {
        constexpr int t = decltype(tc)::value;
        v4i n_lo = b_lo, n_hi = b_hi;
        float n_f = f;
        if constexpr (t + 1 < T) {
            n_lo = at_lo[(t + 1) * 128];
            n_hi = at_hi[(t + 1) * 128];
            n_f = at_f[(t + 1) * row_stride];
        }
        __builtin_amdgcn_sched_barrier(0);
        const v8i b = cat(b_lo, b_hi);
        const float p0 = f * sc0, p1 = f * sc1;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const v4f cur = mfma_fp8(a[k], b);
            __builtin_amdgcn_sched_barrier(0);
            if (t > 0 || k >= 2) {
                v4f &dst = k >= 2 ? acc[k - 2][t] : acc[2 + k][t > 0 ? t - 1 : 0];
                dst += prod[0] * fac[0];
                asm volatile("" : "+v"(dst));
            }
            prod[0] = prod[1];
            fac[0] = fac[1];
            prod[1] = cur;
            fac[1] = (k & 1) ? p1 : p0;
            __builtin_amdgcn_sched_barrier(0);
        }
        b_lo = n_lo;
        b_hi = n_hi;
        f = n_f;
    };
    tile(std::integral_constant<int, 0>{});
    if constexpr (T > 1) tile(std::integral_constant<int, 1>{});
    if constexpr (T > 2) tile(std::integral_constant<int, 2>{});
    if constexpr (T > 3) tile(std::integral_constant<int, 3>{});
    if constexpr (T > 4) tile(std::integral_constant<int, 4>{});
    if constexpr (T > 5) tile(std::integral_constant<int, 5>{});
    if constexpr (T > 6) tile(std::integral_constant<int, 6>{});
    if constexpr (T > 7) tile(std::integral_constant<int, 7>{});
    acc[2][T - 1] += prod[0] * fac[0];
    acc[3][T - 1] += prod[1] * fac[1];
}

template <int NT>
__global__ __launch_bounds__(256, NT <= 4 ? 3 : 2) void moe_group_kernel(const GroupParams s)
{
    using std::integral_constant;
    extern __shared__ __attribute__((aligned(128))) uint8_t lds[];   // [weight tile of the ring][wavefront][2048], [stage][token tile][2048]
    union Tables {
        struct {
            union {
                float xc[2 * NT * 64];   // chunked: [chunk & 1][token][step & 3]; else [step & 3][token]
                float amax[4][NT * 16];  // behind the last step
            };
            float ws[2][kGMaxKb];
        } up;
        struct {
            float sa[2][NT * 16];    // [slice or step & 1][token]
            float w2s[max_w2s(NT)];
            float tw[NT * 16];
        } down;
    };
    __shared__ __attribute__((aligned(16))) Tables tab;
    __shared__ int s_row[NT * 16];   // UP: token of each row (0 for none); DOWN: slot of each row (-1: none)
    __shared__ int s_slot[NT * 16];  // UP in pieces: slot of each row (-1: none)
    __shared__ int s_last[2];
    __shared__ int s_item;
    static_assert((NT <= 4 ? 3 : 2) * ((dyn_lds(NT) + (int)sizeof(Tables) + 2 * NT * 64 + 12 + 1279) / 1280 * 1280) <= 160 * 1024,
                  "the workgroups of a compute unit share 160 KiB of LDS, handed out 1280 bytes at a time");

    const MoeParams &p = s.p;
    const int tid = threadIdx.x, lane = tid & 63, w = rfl(tid >> 6);
    const int n = lane & 15, q = lane >> 4;
    const int K = p.K, I = p.N >> 1, nkb = s.nkb, n_ib = s.n_ib;
    const int epoch = next_epoch(rfl(s.ctl->epoch));
    int n_live = (rfl(p.ntpp[0]) + p.block_m - 1) / p.block_m;
    n_live = n_live < s.n_mb_max ? n_live : s.n_mb_max;

    const int f_n = (n >> 1) & 7;
    const int frag_lo = n * 128 + 16 * (q ^ f_n);
    const int frag_hi = n * 128 + 16 * ((q ^ f_n) ^ 4);
    // direct-to-LDS load h of a tile: lane l fills position l & 7 of row 8h + l / 8
    const int ld_row = lane >> 3;
    unsigned ld_chunk[2];
#pragma unroll
    for (int h = 0; h < 2; h++) ld_chunk[h] = 16u * ((lane & 7) ^ (((8 * h + ld_row) >> 1) & 7));
    uint8_t *my_tiles = lds + w * 2048;   // place i of the wavefront's weight ring: + i * 8192

    // the only row block of its expert: nobody else will ask for the weights it streams
    auto alone = [&](int mb, int e) {
        if (s.w_nt >= 0) return s.w_nt != 0;
        bool a = true;
        if (mb > 0) a = rfl(p.expert_ids[mb - 1]) != e;
        if (mb + 1 < n_live) a &= rfl(p.expert_ids[mb + 1]) != e;
        return a;
    };
    auto tiles_of = [&]() {
        int last = s_last[0];
        if (NT > 4) last = s_last[1] > last ? s_last[1] : last;
        return rfl((last >> 4) + 1);   // 0 when no row is valid
    };
    // run(T, non-temporal, deep rings) with the smallest even T that holds the live tiles
    const bool short_k = nkb <= kGDeepKb;
    auto pick = [&](int n_tiles, bool nt, auto run) {
        auto sized = [&](auto ntc) {
            auto few = [&](auto tc) {
                if (short_k) run(tc, ntc, std::true_type{});
                else run(tc, ntc, std::false_type{});
            };
            if (NT >= 8 && n_tiles > 6) run(integral_constant<int, NT >= 8 ? 8 : NT>{}, ntc, std::false_type{});
            else if (NT >= 6 && n_tiles > 4) run(integral_constant<int, NT >= 6 ? 6 : NT>{}, ntc, std::false_type{});
            else if (n_tiles > 2) few(integral_constant<int, 4>{});
            else few(integral_constant<int, 2>{});
        };
        if (nt) sized(std::true_type{});
        else sized(std::false_type{});
    };

    // K steps [k0, k1); pieces > 1: the piece-th of that many parts of the contraction, `arrived` counts the finished ones
    auto up_item = [&](int mb, int ib, int k0, int k1, int piece, int pieces, int *arrived) {
        const int e = rfl(p.expert_ids[mb]);
        if (e < 0 || e >= p.E) return;
        const int row0 = mb * p.block_m;
        const int n_rows = p.block_m < p.sorted_num - row0 ? p.block_m : p.sorted_num - row0;
        if (tid < NT * 16) {
            int id = -1;
            if (tid < n_rows) id = p.sorted_ids[row0 + tid];
            const int tk = id / p.top_k;
            const bool ok = id >= 0 && tk < p.M;
            s_row[tid] = ok ? tk : 0;
            if (pieces > 1) s_slot[tid] = ok ? id : -1;
            const unsigned long long okm = __ballot(ok);
            if (lane == 0) s_last[w] = okm ? w * 64 + 63 - __builtin_clzll(okm) : -1;
        }
        const bool nt = alone(mb, e);
        // Weights: matrix row r of tile i = (32-row group i / 2, gate | up i % 2) is slab row group * 32 + (r / 8) * 16 + r % 8 (+ 8
        // for up)
        const __amdgpu_buffer_rsrc_t wbuf = agent_buffer(p.w + (size_t)e * p.N * K + (size_t)(ib * 256 + w * 64) * p.w_rs);
        unsigned w_voff[2];
#pragma unroll
        for (int h = 0; h < 2; h++) w_voff[h] = (unsigned)(ld_row * p.w_rs) + ld_chunk[h];
        auto issue_w = [&](int place, int k, int i, auto aux) {   // tile i of step k
#pragma unroll
            for (int h = 0; h < 2; h++)
                dma16<decltype(aux)::value>(wbuf, w_voff[h], (unsigned)(k * p.w_ks + ((i >> 1) * 32 + (i & 1) * 8 + h * 16) * p.w_rs),
                                            my_tiles + place * 8192 + h * 1024);
        };
        auto issue_rows = [&](int k, int j, auto aux) {   // the j-th eight rows of the slab, into a ring of four places
            dma16<decltype(aux)::value>(wbuf, w_voff[(j >> 1) & 1], (unsigned)(k * p.w_ks + 8 * j * p.w_rs),
                                        my_tiles + (2 * (j >> 2) + (j & 1)) * 8192 + ((j >> 1) & 1) * 1024);
        };
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (nt) issue_w(i, k0, i, integral_constant<int, 2>{});
            else issue_w(i, k0, i, integral_constant<int, 0>{});
        }
        if (w < 2) {   // this slice's gate (row 2*ib) and up (row 2*ib+1) scales
            const __amdgpu_buffer_rsrc_t wsbuf = agent_buffer(p.w_scale + ((size_t)e * (p.N >> 7) + 2 * ib + w) * nkb);
            for (int c = 0; c < nkb; c += 64)
                if (lane < nkb - c) dma4<0>(wsbuf, 4u * lane, 4u * c, &tab.up.ws[w][c]);
        }
        lds_barrier();
        const int n_tiles = tiles_of();
        if (n_tiles > 0) {
            const __amdgpu_buffer_rsrc_t xsbuf = agent_buffer(p.x_scale);
            const bool xs_chunk = s.xs_chunk != 0;
            v4f acc[4][NT];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int t = 0; t < NT; t++) acc[k][t] = (v4f){0.f, 0.f, 0.f, 0.f};
            pick(n_tiles, nt, [&](auto tc, auto ntc, auto deepc) {
                constexpr int T = decltype(tc)::value;   // token tiles multiplied, even
                constexpr integral_constant<int, decltype(ntc)::value ? 2 : 0> ntc_aux{};
                constexpr int DM = T / 2;                // direct-to-LDS loads of a wavefront and step: 1 KiB halves of tiles
                constexpr int XL = T * 4;                // tokens whose scales a wavefront fetches
                constexpr bool DEEP = decltype(deepc)::value;
                constexpr int S = x_stages(NT, T, DEEP), R = w_tiles(NT, T, S, DEEP);
                uint8_t *ring = lds + R * 8192;
                unsigned x_off[DM];
#pragma unroll
                for (int j = 0; j < DM; j++) {
                    const int hh = w * DM + j;
                    x_off[j] = (unsigned)s_row[hh * 8 + ld_row] * (unsigned)K + ld_chunk[0];
                    if (hh & 1) x_off[j] = x_off[j] - ld_chunk[0] + ld_chunk[1];
                }
                const unsigned xs_off = 4u * (unsigned)s_row[w * XL + (lane < XL ? lane : 0)] * (unsigned)nkb;
                auto issue_xs = [&](int k) {
                    if (!xs_chunk || (k & 3) == 0) {
                        if (lane < XL) {
                            if (xs_chunk) dma16<0>(xsbuf, xs_off, 4u * k, &tab.up.xc[(((k >> 2) & 1) * NT * 16 + w * XL) * 4]);
                            else dma4<0>(xsbuf, xs_off, 4u * k, &tab.up.xc[(k & 3) * NT * 16 + w * XL]);
                        }
                    }
                };
                // (A step's columns are in the base and not in an offset: with 2^32 bytes of activations, the most there can be, the
                // last row's last bytes would be past what a buffer's 32-bit size covers.)
                const uint8_t *x_next = p.x + (size_t)(k0 * 128);   // columns of the next step to be asked for
                auto issue_x = [&](int stage) {
                    const __amdgpu_buffer_rsrc_t xbuf = agent_buffer(x_next);
#pragma unroll
                    for (int j = 0; j < DM; j++) dma16<0>(xbuf, x_off[j], 0u, ring + stage * (T * 2048) + w * (DM * 1024) + j * 1024);
                };
                const int row_stride = xs_chunk ? 64 : 16;
                // A step's loads are issued in this order: the scales and - with two stages - the token tiles of the step that is
                // S - 1 ahead; weight tiles of the next step, into the places this step's have left; with three stages
                // the token tiles here; weight tiles of the step after the next.  Loads complete in order, so at the start of a
                // step what was issued behind its own last weight tile may still be on its way.
                constexpr int BEHIND = 2 * (R - 4) + (S == 3 ? DM : 0);
                issue_xs(k0);
                issue_x(0);
                x_next += 128;
                if (k0 + 1 < k1) {
                    if (S == 3) issue_xs(k0 + 1);
#pragma unroll
                    for (int g = 4; g < R; g++) issue_w(g, k0 + 1, g & 3, ntc_aux);
                    if (S == 3) {
                        issue_x(1);
                        x_next += 128;
                    }
                }
                int first = 0, stage = 0;   // the step's first weight tile, and its token tiles, in their rings
                for (int k = k0; k < k1; k++) {
                    if (k + 1 < k1) wait_vmcnt<BEHIND>();   // this wavefront's loads of step k have landed
                    else wait_vmcnt<0>();
                    lds_barrier();     // everybody's have, and step k - 1 is done with
                    v8i a[4];
                    int place[4];
                    const uint8_t *tile[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        place[i] = first + i < R ? first + i : first + i - R;
                        tile[i] = my_tiles + place[i] * 8192;
                    }
                    first = first + 4 < R ? first + 4 : first + 4 - R;
                    float sc0 = tab.up.ws[0][k], sc1 = tab.up.ws[1][k];
                    asm volatile("" : "+v"(sc0), "+v"(sc1));
                    read_weights(a, tile, frag_lo, frag_hi);
                    const int ahead = stage + S - 1 < S ? stage + S - 1 : stage - 1;
                    if (k + S - 1 < k1) issue_xs(k + S - 1);
                    if constexpr (R == 4) {
                        // (all of a step's weights at once: in the order of their rows and in front of the tokens, which is 1 - 3 %
                        // of a call of the DeepSeek shard at M = 8192, where row blocks of one expert share them in L2)
                        if (k + 1 < k1) {
#pragma unroll
                            for (int j = 0; j < 8; j++) issue_rows(k + 1, j, ntc_aux);
                            issue_x(ahead);
                        }
                    } else if (k + 1 < k1) {
                        if (S == 2) issue_x(ahead);
#pragma unroll
                        for (int i = 0; i < 8 - R; i++) issue_w(place[i], k + 1, (R + i) & 3, ntc_aux);
                    }
                    if (S == 3 && k + 2 < k1) issue_x(ahead);
                    if (R > 4 && k + 2 < k1) {
#pragma unroll
                        for (int i = 8 - R; i < 4; i++) issue_w(place[i], k + 2, (R + i) & 3, ntc_aux);
                    }
                    const float *row = xs_chunk ? &tab.up.xc[(((k >> 2) & 1) * NT * 16 + n) * 4 + (k & 3)]
                                                : &tab.up.xc[(k & 3) * NT * 16 + n];
                    multiply<T>(a, ring + stage * (T * 2048), row, row_stride, sc0, sc1, acc, frag_lo, frag_hi);
                    x_next += 128;
                    stage = stage + 1 < S ? stage + 1 : 0;
                }
            });

            if (pieces > 1) {
                // Partial sums go where the rows' results will be (nobody writes those before this unit's flag is up): 1 KiB
                // of row y[slot] for each (slice, piece).  The last piece to arrive adds them up, in order.
                const unsigned at = (unsigned)((ib * pieces) * 1024 + w * 256 + q * 16);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int id = s_slot[t * 16 + n];
                    if (id >= 0) {
#pragma unroll
                        for (int k = 0; k < 4; k++) stg128_agent(s.y, (unsigned)id * 2u * K + at + piece * 1024 + k * 64, acc[k][t]);
                    }
                }
                wait_vmcnt<0>();
                __syncthreads();
                if (tid == 0) {
                    const int before = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (before == pieces - 1) store_agent(arrived, 0);
                    s_item = before;
                }
                __syncthreads();
                if (rfl(s_item) != pieces - 1) return;
                acquire_fence();
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int id = s_slot[t * 16 + n];
                    v4f sum[4] = {};
                    if (id >= 0) {
                        for (int o = 0; o < pieces; o++) {
                            v4f v[4];
#pragma unroll
                            for (int k = 0; k < 4; k++) v[k] = __builtin_bit_cast(v4f, ldg128_agent(s.y, (unsigned)id * 2u * K + at + o * 1024 + k * 64));
#pragma unroll
                            for (int k = 0; k < 4; k++) sum[k] += v[k];
                        }
                    }
#pragma unroll
                    for (int k = 0; k < 4; k++) acc[k][t] = sum[k];
                }
            }
            __syncthreads();   // the scales' place is the row maxima's from here on
            // SwiGLU, per-token amax over the slice's 128 columns, FP8 requant into operand tiles
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if (t < n_tiles) {
                    float mx = 0.f;
#pragma unroll
                    for (int pr = 0; pr < 2; pr++)
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const float v = swiglu_bf16(acc[2 * pr][t][j], acc[2 * pr + 1][t][j]);
                            acc[2 * pr][t][j] = v;
                            mx = fmaxf(mx, fabsf(v));
                        }
                    mx = fmaxf(mx, __shfl_xor(mx, 16));
                    mx = fmaxf(mx, __shfl_xor(mx, 32));
                    if (q == 0) tab.up.amax[w][t * 16 + n] = mx;
                }
            }
            __syncthreads();
            // the tiles are put together where the weights were, then stored 16 bytes a lane
            const size_t tile0 = ((size_t)mb * n_ib + ib) * s.tpb;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if (t < n_tiles) {
                    float mx = kAmaxFloor;
#pragma unroll
                    for (int wv = 0; wv < 4; wv++) mx = fmaxf(mx, tab.up.amax[wv][t * 16 + n]);
                    const RowScale rs(mx);
#pragma unroll
                    for (int pr = 0; pr < 2; pr++) {
                        const uint32_t packed =
                            pack_fp8x4(rs.code(acc[2 * pr][t][0]), rs.code(acc[2 * pr][t][1]), rs.code(acc[2 * pr][t][2]),
                                       rs.code(acc[2 * pr][t][3]));
                        // columns w*32 + pr*16 + 4q .. +3 of token n: chunk w*2 + pr of the row, bytes 4q .. 4q+3 in it
                        *reinterpret_cast<uint32_t *>(lds + t * 2048 + n * 128 + 16 * ((w * 2 + pr) ^ f_n) + 4 * q) = packed;
                    }
                    if (w == 0 && q == 0) stg32_agent(s.sas + (tile0 + t) * 16, 4u * n, __builtin_bit_cast(uint32_t, rs.scale));
                }
            }
            lds_barrier();
            for (int i = tid; i < n_tiles * 128; i += 256)
                stg128_agent(s.aqs + tile0 * 2048, 16u * i, *reinterpret_cast<const v4f *>(lds + 16 * i));
            wait_vmcnt<0>();
        }
        __syncthreads();
        if (tid == 0) store_agent(&s.flag[mb * n_ib + ib], epoch);
    };

    auto down_item = [&](int mb, int cs, auto resident_c) {
        constexpr bool RESIDENT = decltype(resident_c)::value;
        const int e = rfl(p.expert_ids[mb]);
        if (e < 0 || e >= p.E) return;
        const int row0 = mb * p.block_m;
        const int n_rows = p.block_m < p.sorted_num - row0 ? p.block_m : p.sorted_num - row0;
        float tw = 0.f;
        if (tid < NT * 16) {
            int id = -1;
            if (tid < n_rows) id = p.sorted_ids[row0 + tid];
            const bool ok = id >= 0 && id / p.top_k < p.M;
            s_row[tid] = ok ? id : -1;
            if (ok) {
                tw = p.topk_w[id];
                if (cs == 0) s.live[id] = epoch;
            }
            const unsigned long long okm = __ballot(ok);
            if (lane == 0) s_last[w] = okm ? w * 64 + 63 - __builtin_clzll(okm) : -1;
        }
        const int n_groups = K >> 6;
        const int g0 = cs * s.gps;
        const int g1 = g0 + s.gps < n_groups ? g0 + s.gps : n_groups;
        const bool nt = alone(mb, e);
        lds_barrier();
        const int n_tiles = tiles_of();
        if (n_tiles == 0) return;
        const int rounds = (g1 - g0 + 3) >> 2;   // the slab's groups w, w + 4, ... of wavefront w; past the end: computed, not stored
        const int n_steps = rounds * n_ib;
        const __amdgpu_buffer_rsrc_t wbuf = agent_buffer(p.w2 + (size_t)e * K * I);
        const __amdgpu_buffer_rsrc_t abuf = agent_buffer(s.aqs + (size_t)mb * n_ib * s.tpb * 2048);
        const __amdgpu_buffer_rsrc_t sbuf = agent_buffer(s.sas + (size_t)mb * n_ib * s.tpb * 16);
        // matrix row r of tile k is output column c0 + 16 (r / 4) + 4 k + r % 4: lane (n, q) collects 16 adjacent columns
        unsigned w_voff[2];
#pragma unroll
        for (int h = 0; h < 2; h++) w_voff[h] = (unsigned)((16 * (lane >> 5) + (ld_row & 3)) * p.w2_rs) + ld_chunk[h];
        pick(n_tiles, nt, [&](auto tc, auto ntc, auto deepc) {
            constexpr int T = decltype(tc)::value;
            constexpr int AUX = decltype(ntc)::value ? 2 : 0;
            constexpr int DM = T / 2;
            constexpr int XL = T * 4;
            constexpr int R = w_tiles(NT, T, 2, decltype(deepc)::value);
            uint8_t *ring = lds + R * 8192;
            v4f acc[4][T];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int t = 0; t < T; t++) acc[k][t] = (v4f){0.f, 0.f, 0.f, 0.f};
            // the step that is two ahead of the one multiplied: its slice and column group, and where its weights are
            int lib = 0, lg = g0 + w;
            auto aim = [&]() {
                const int grp = lg < g1 ? lg : g1 - 1;
                return (unsigned)((grp << 6) * p.w2_rs + lib * p.w2_ks);
            };
            auto advance = [&]() {
                if (++lib == n_ib) {
                    lib = 0;
                    lg += 4;
                }
            };
            auto issue_w = [&](int place, unsigned at, int i) {
#pragma unroll
                for (int h = 0; h < 2; h++)
                    dma16<AUX>(wbuf, w_voff[h], at + (unsigned)((4 * i + 32 * h) * p.w2_rs), my_tiles + place * 8192 + h * 1024);
            };
            // slice ib's tiles (past the last one: that one again) and their scales
            auto issue_x = [&](int ib, int stage, int j) {
                {
                    const int hh = w * DM + j, tt = hh >> 1;
                    dma16<kAuxAgent>(abuf, (unsigned)(lane * 16),
                                     (unsigned)((ib * s.tpb + (tt < n_tiles ? tt : n_tiles - 1)) * 2048 + (hh & 1) * 1024),
                                     ring + stage * (T * 2048) + hh * 1024);
                }
            };
            auto issue_xs = [&](int ib, int stage) {
                if (lane < XL) {
                    const int r = w * XL + lane;
                    dma4<kAuxAgent>(sbuf, 4u * (r < n_tiles * 16 ? r : 0), (unsigned)(ib * s.tpb * 64), &tab.down.sa[stage][w * XL]);
                }
            };
            // the weights do not depend on the UP items
            unsigned at1, at2;   // weights of the next step and of the one after it
            {
                const unsigned at0 = aim();
#pragma unroll
                for (int i = 0; i < 4; i++) issue_w(i, at0, i);
                advance();
                at1 = aim();
                if (n_steps > 1) {
#pragma unroll
                    for (int g = 4; g < R; g++) issue_w(g, at1, g & 3);
                }
                advance();
                at2 = aim();
            }
            if (w == 1) {
                const __amdgpu_buffer_rsrc_t w2sbuf = agent_buffer(p.w2_scale + ((size_t)e * (K >> 7) + (g0 >> 1)) * n_ib);
                const int count = ((g1 - g0 + 1) >> 1) * n_ib;
                for (int c = 0; c < count; c += 64)
                    if (lane < count - c) dma4<0>(w2sbuf, 4u * lane, 4u * c, &tab.down.w2s[c]);
            }
            if (tid < NT * 16) tab.down.tw[tid] = tw * p.scaling;
            if (w == 0) spin_all_eq(&s.flag[mb * n_ib], n_ib, epoch, s.ctl);
            lds_barrier();
            if constexpr (RESIDENT) {
                for (int ib = 0; ib < n_ib; ib++) {
                    issue_xs(ib, ib);
#pragma unroll
                    for (int j = 0; j < DM; j++) issue_x(ib, ib, j);
                }
            } else {
                issue_xs(0, 0);
#pragma unroll
                for (int j = 0; j < DM; j++) issue_x(0, 0, j);
            }
            wait_vmcnt<0>();
            __syncthreads();
            int cg = g0 + w, cib = 0, first = 0;
            for (int i = 0; i < n_steps; i++) {
                if (!RESIDENT && i > 0) lds_barrier();   // everybody's loads of the step have landed, the step before is done with
                v8i a[4];
                int place[4];
                const uint8_t *tile[4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    place[t] = first + t < R ? first + t : first + t - R;
                    tile[t] = my_tiles + place[t] * 8192;
                }
                first = first + 4 < R ? first + 4 : first + 4 - R;
                read_weights(a, tile, frag_lo, frag_hi);
                if (i + 1 < n_steps) {   // the next step's loads, as in the UP items
                    if constexpr (!RESIDENT) {
                        const int ib = cib + 1 < n_ib ? cib + 1 : 0;
                        issue_xs(ib, (i + 1) & 1);
#pragma unroll
                        for (int j = 0; j < DM; j++) issue_x(ib, (i + 1) & 1, j);
                    }
                    if constexpr (R == 4) {
#pragma unroll
                        for (int o = 0; o < 8; o++)
                            dma16<AUX>(wbuf, w_voff[o >> 2], at1 + (unsigned)((4 * (o & 3) + 32 * (o >> 2)) * p.w2_rs),
                                       my_tiles + (o & 3) * 8192 + (o >> 2) * 1024);
                    } else {
#pragma unroll
                        for (int t = 0; t < 8 - R; t++) issue_w(place[t], at1, (R + t) & 3);
                    }
                }
                if (R > 4 && i + 2 < n_steps) {
#pragma unroll
                    for (int t = 8 - R; t < 4; t++) issue_w(place[t], at2, (R + t) & 3);
                }
                at1 = at2;
                advance();
                at2 = aim();
                const int st = RESIDENT ? cib : (i & 1);
                const float ws2 = tab.down.w2s[(((cg < g1 ? cg : g1 - 1) - g0) >> 1) * n_ib + cib];
                multiply<T>(a, ring + st * (T * 2048), &tab.down.sa[st][n], 16, ws2, ws2, acc, frag_lo, frag_hi);
                // the next step's loads have landed before any result store is queued behind them
                if (i + 2 < n_steps) wait_vmcnt<2 * (R - 4)>();
                else wait_vmcnt<0>();
                if (++cib == n_ib) {
#pragma unroll
                    for (int t = 0; t < T; t++) {
                        const int slot_id = s_row[t * 16 + n];
                        if (slot_id >= 0 && cg < g1) {
                            const float tw = tab.down.tw[t * 16 + n];
                            uint16_t *yp = s.y + (size_t)slot_id * K + (cg << 6) + 16 * q;
#pragma unroll
                            for (int half = 0; half < 2; half++) {
                                const v4f lo = acc[2 * half][t] * tw, hi = acc[2 * half + 1][t] * tw;
                                v4i o;
                                o.x = (int)pack_bf16x2(lo[0], lo[1]);
                                o.y = (int)pack_bf16x2(lo[2], lo[3]);
                                o.z = (int)pack_bf16x2(hi[0], hi[1]);
                                o.w = (int)pack_bf16x2(hi[2], hi[3]);
                                *reinterpret_cast<v4i *>(yp + 8 * half) = o;
                            }
                        }
#pragma unroll
                        for (int k = 0; k < 4; k++) acc[k][t] = (v4f){0.f, 0.f, 0.f, 0.f};
                    }
                    cib = 0;
                    cg += 4;
                }
            }
        });
    };

    // ---- which item ---------------------------------------------------------------------------------------------------
    const int q_id = blockIdx.x & 7;
    if (blockIdx.x == 0 && tid == 0) s.ctl->stamp = epoch;   // for the reduce kernel, which closes the launch
    if (tid == 0) s_item = __hip_atomic_fetch_add(s.head + q_id * kGHeadStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int item = rfl(s_item);
    // This queue's live row blocks: whole rounds of chunks of kGChunk, what is left in chunks of an eighth of it
    const int whole_chunks = n_live / (8 * kGChunk), left = n_live % (8 * kGChunk), chunk = (left + 7) >> 3;
    const int rest = left - chunk * q_id;
    const int nb = whole_chunks * kGChunk + (rest < 0 ? 0 : rest < chunk ? rest : chunk);
    const int ups = nb * n_ib;
    // Where half a round of workgroups holds all UP items and K is long, each is taken in two parts, so that more loads are in flight.
    // MI355X, 64-row blocks, by UP items of a queue's 96 workgroups, us whole -> two parts: K = 7168 47 items 196 -> 175, 66 271 -> 278,
    // 68 304 -> 314; K = 6144 10 items 99 -> 73, 23 92 -> 85; K = 4096 24 items 87 -> 77, 33 110 -> 113.  More parts change nothing (three
    // to eight at K = 6144, 10 items: 72 - 73).  Shorter K loses as often as it gains: K = 3072 74 -> 67 and, with 128-row blocks,
    // 83 -> 92; K = 2560 65 -> 64 and 60 -> 70.
    const int pieces = nkb >= kGPiecesKb && ups * s.max_pieces <= s.round ? s.max_pieces : 1;
    const int up_items = ups * pieces;
    const bool is_up = item < up_items;
    const int unit_id = item / pieces, piece = item - unit_id * pieces;
    const int k0 = is_up ? (nkb >> 2) * piece / pieces * 4 : 0;   // parts start at multiples of four K steps (the scales' chunks)
    const int k1 = is_up && piece + 1 < pieces ? (nkb >> 2) * (piece + 1) / pieces * 4 : nkb;
    const int i = is_up ? unit_id : item - up_items, per = is_up ? n_ib : s.n_cs;
    const int j = i / per, off = i - j * per;
    if (j >= nb) return;
    const int mb = rfl(j < whole_chunks * kGChunk ? ((j / kGChunk) * 8 + q_id) * kGChunk + j % kGChunk
                                                  : whole_chunks * 8 * kGChunk + chunk * q_id + j - whole_chunks * kGChunk);
    if (is_up)
        up_item(mb, rfl(off), rfl(k0), rfl(k1), rfl(piece), rfl(pieces), s.head + q_id * kGHeadStride + 1 + rfl(unit_id));
    else if (n_ib <= kGResidentIb) down_item(mb, rfl(off), std::true_type());
    else down_item(mb, rfl(off), std::false_type());
}

size_t align_up(size_t v) { return (v + 255) & ~(size_t)255; }

typedef void (*GroupFn)(const GroupParams);

hipError_t allow_dynamic_lds()
{
    static std::mutex mu;
    static bool done[64];
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    std::lock_guard<std::mutex> lock(mu);
    if (dev >= 0 && dev < 64 && done[dev]) return hipSuccess;
    const GroupFn fn[] = {moe_group_kernel<4>, moe_group_kernel<6>, moe_group_kernel<8>};
    for (int i = 0; i < 3 && err == hipSuccess; i++)
        err = hipFuncSetAttribute(reinterpret_cast<const void *>(fn[i]), hipFuncAttributeMaxDynamicSharedMemorySize, dyn_lds(4 + 2 * i));
    if (err == hipSuccess && dev >= 0 && dev < 64) done[dev] = true;
    return err;
}

}  // namespace

// The variant that serves a call and the output columns of its DOWN items.  A row block has up to nt 16-row tiles.  A slab has at least
// four column groups, or all there are; where the scales of so few of them exceed the smallest variant's table (K >= 256: above 256
// slices, K = 128: above 512), the next variant takes the call.
struct GroupPlan {
    int nt;          // template argument of the kernel
    int gps, n_cs;   // 64-column groups per DOWN item (a multiple of 4), column slabs
};

static GroupPlan group_plan(int K, int N, int block_m, int stages)
{
    GroupPlan g;
    const int n_ib = N / 256, tiles = (block_m + 15) / 16, groups = K >> 6;
    const int fewest = (groups < 4 ? groups : 4) / 2 * n_ib;   // scales of the smallest slab
    g.nt = tiles <= 4 && fewest <= max_w2s(4) ? 4 : tiles <= 6 ? 6 : 8;
    const int e_gps = tunable(kTunTileGps, 0);
    g.gps = e_gps > 0 ? ((e_gps < groups ? e_gps : groups) + 3) / 4 * 4 : 4 * ((5 * stages + n_ib - 1) / n_ib);
    while (g.gps > 4 && g.gps / 2 * n_ib > max_w2s(g.nt)) g.gps -= 4;
    g.n_cs = (groups + g.gps - 1) / g.gps;
    return g;
}

// Row blocks of at most 32 rows are the streaming kernel's; the few calls of them it does not take (more than 1 GiB of its fp32 rows,
// more than 64 experts to a token) come here up to eight slices and 512 scales, beyond which the fallback kernel has them: its sums
// are fp32 throughout, those of the rows here are not.  MI355X, DeepSeek shard, 16- and 32-row blocks, here / in the fallback
// kernel: M = 4200 1.12 and 0.77 ms / 7.3 and 7.3 ms, M = 8192 2.00 and 1.35 / 14.2 and 14.1.
bool group_supported(int top_k, int M, int K, int N, int sorted_num, int block_m, bool streams)
{
    const int n_ib = N / 256;
    if (block_m <= 32 && (streams || n_ib > 8 || (K / 128) * n_ib > 512)) return false;
    const int64_t n_mb = ((int64_t)sorted_num + block_m - 1) / block_m;
    return K <= 128 * kGMaxKb && (K / 128) * n_ib <= kGMaxExpertW2s && (int64_t)M * top_k <= kMaxSlots &&
           n_mb * n_ib <= kMaxUnits;
}

size_t group_workspace_bytes(int top_k, int M, int K, int N, int E, int sorted_num, int block_m)
{
    (void)E;
    const size_t n_mb = ((size_t)sorted_num + block_m - 1) / block_m;
    const size_t tiles = n_mb * (N / 256) * ((block_m + 15) / 16);
    return align_up(kPrefixBytes) + align_up((size_t)M * top_k * K * sizeof(uint16_t)) + align_up(tiles * 2048) +
           align_up(tiles * 16 * sizeof(float));
}

void group_plan_numbers(int K, int N, int block_m, int stages, int plan[4])
{
    const GroupPlan g = group_plan(K, N, block_m, stages);
    plan[0] = g.nt;
    plan[1] = g.gps;
    plan[2] = g.n_cs;
    plan[3] = max_w2s(g.nt);
}

hipError_t launch_group(const MoeParams &p, int stages, void *workspace, hipStream_t stream)
{
    uint8_t *ws = static_cast<uint8_t *>(workspace);
    GroupParams s;
    s.p = p;
    s.n_ib = p.N / 256;
    s.nkb = p.K / 128;
    s.n_mb_max = (p.sorted_num + p.block_m - 1) / p.block_m;
    s.tpb = (p.block_m + 15) / 16;
    size_t off = align_up(kPrefixBytes);
    s.ctl = reinterpret_cast<StreamCtl *>(ws);
    s.head = reinterpret_cast<int *>(ws + kOffArrive);
    s.flag = reinterpret_cast<int *>(ws + kOffFlag);
    s.live = reinterpret_cast<int *>(ws + kOffLive);
    s.y = reinterpret_cast<uint16_t *>(ws + off);
    off += align_up((size_t)p.M * p.top_k * p.K * sizeof(uint16_t));
    s.aqs = ws + off;
    off += align_up((size_t)s.n_mb_max * s.n_ib * s.tpb * 2048);
    s.sas = reinterpret_cast<float *>(ws + off);
    const GroupPlan plan = group_plan(p.K, p.N, p.block_m, stages);
    const int nt = plan.nt;
    s.gps = plan.gps;
    s.n_cs = plan.n_cs;
    s.xs_chunk = (s.nkb % 4 == 0 && reinterpret_cast<uintptr_t>(p.x_scale) % 16 == 0) ? 1 : 0;
    s.w_nt = tunable(kTunTileNt, -1);
    hipError_t err = allow_dynamic_lds();
    if (err != hipSuccess) return err;
    const unsigned chunk_rounds = (unsigned)((s.n_mb_max + 8 * kGChunk - 1) / (8 * kGChunk));
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            return 256;
        return n;
    }();
    s.round = (cus >= 8 ? cus / 8 : 1) * (nt <= 4 ? 3 : 2);
    if (s.round > kGMaxRound) s.round = kGMaxRound;
    // The partial sums (1 KiB a row, slice and part) take the rows' places in y.
    s.max_pieces = tunable(kTunGroupPieces, 2);
    const int room = p.K * 2 / (1024 * s.n_ib);
    if (s.max_pieces > room) s.max_pieces = room;
    if ((int64_t)p.M * p.top_k * p.K * 2 > 0xffffffffll) s.max_pieces = 1;   // (their offsets are 32-bit)
    if (s.max_pieces < 1) s.max_pieces = 1;
    if (s.max_pieces > 8) s.max_pieces = 8;
    const unsigned grid = 8 * (chunk_rounds * kGChunk * (s.n_ib + s.n_cs) + s.round * (s.max_pieces - 1));
    const GroupFn fn = nt == 4 ? moe_group_kernel<4> : nt == 6 ? moe_group_kernel<6> : moe_group_kernel<8>;
    // (Each launch's own status: hipGetLastError() also reports what other calls of the thread left behind, and to stop here, with the
    // tickets drawn, would leave the workspace's queues empty for the calls that follow.)
    void *args[] = {&s};
    err = hipLaunchKernel(reinterpret_cast<const void *>(fn), dim3(grid), dim3(256), args, dyn_lds(nt), stream);
    if (err != hipSuccess) return err;
    RowsReduce r;
    r.p = p;
    r.ctl = s.ctl;
    r.live = s.live;
    r.y = s.y;
    r.y_is_f32 = 0;
    r.heads = s.head;
    r.head_stride = kGHeadStride;
    return launch_rows_reduce(r, stream);
}

}  // namespace alpha_moe
