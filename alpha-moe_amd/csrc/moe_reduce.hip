// The sums over a token's result rows, behind the streaming and group kernels.
#include "moe_common.hpp"

namespace alpha_moe {
namespace {

// out[t] = bf16(out[t] + sum over the token's live slots of y[slot]).
// Row is the type of y: bf16 (prefill kernels) or fp32 (streaming kernel).  A thread loads 16 bytes of each row - 8 or 4
// columns -, a workgroup covers 256 threads' columns of one token, and all rows of a token with up to 12 slots are in flight
// at once.  Bound by HBM: the rows are read once.  Nothing else is waited for.  Behind the streaming kernel, which closed the launch
// epoch itself, that is all.  Behind the group kernel this launch ends the call: workgroup 0 sets the eight ticket counters back and
// closes the epoch, so it has to follow every launch of that kernel on the workspace - the next one would find its queues
// drawn empty.  (The last of this kernel's workgroups used to close it: arrivals at one counter are served one by one, ~10 ns each, so 4096
// workgroups took 41 us whatever they had to read.)
// MI355X, kernel trace, before and after: Qwen3-Next M=4096 60 -> 38 us, Qwen3-30B M=1024 18 -> 9.7 and M=8192 78 -> 46,
// DeepSeek shard M=2048 76 -> 61 and M=8192 204 -> 198 (1.18 GB, 6.0 TB/s).  Workgroups that stride over tokens are slower
// (M=8192 with 1024 of them: 220 us).
constexpr int kReduceInFlight = 12;
template <typename Row>
__global__ __launch_bounds__(256) void moe_rows_reduce_kernel(const RowsReduce s, int chunks_per_token)
{
    constexpr bool F32 = sizeof(Row) == 4;
    constexpr int COLS = 16 / (int)sizeof(Row);
    const MoeParams &p = s.p;
    const int epoch = s.heads ? s.ctl->stamp : s.ctl->epoch;   // of the kernel before this one
    if (s.heads && blockIdx.x == 0 && threadIdx.x < 8) {   // (no other workgroup reads these here)
        s.heads[threadIdx.x * s.head_stride] = 0;
        if (threadIdx.x == 0) s.ctl->epoch = epoch;
    }
    // a bounded wait that ran out (in this call's first kernel or in any earlier launch on this workspace: the word is
    // sticky) means result rows may be missing: the output then says so itself, NaN in every element
    // (an ordinary load: this kernel starts after the other has ended, and every wavefront asking the memory side
    // for the same word with an agent-scope load cost ~100 us per call)
    const bool poisoned = s.ctl->error != 0;
    const int t = blockIdx.x / chunks_per_token;
    const int c = (((int)blockIdx.x - t * chunks_per_token) * 256 + (int)threadIdx.x) * COLS;
    if (c >= p.K) return;
    float sum[COLS];
#pragma unroll
    for (int i = 0; i < COLS; i++) sum[i] = 0.f;
    auto add = [&](const v4i v) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (F32) {
                sum[i] += __builtin_bit_cast(v4f, v)[i];
            } else {
                sum[2 * i] += __builtin_bit_cast(float, (uint32_t)v[i] << 16);
                sum[2 * i + 1] += __builtin_bit_cast(float, (uint32_t)v[i] & 0xffff0000u);
            }
        }
    };
    typedef uint32_t OutWords __attribute__((ext_vector_type(COLS / 2)));
    OutWords *op = reinterpret_cast<OutWords *>(p.out + (size_t)t * p.K + c);
    OutWords o = {};
    if (!p.overwrite) o = *op;
    const int *live = s.live + t * p.top_k;
    const Row *yrow = static_cast<const Row *>(s.y) + (size_t)t * p.top_k * p.K + c;
    for (int s0 = 0; s0 < p.top_k; s0 += kReduceInFlight) {   // slot order: the sum depends on nothing but the inputs
        bool on[kReduceInFlight];
        v4i v[kReduceInFlight];
#pragma unroll
        for (int j = 0; j < kReduceInFlight; j++) on[j] = s0 + j < p.top_k && live[s0 + j] == epoch;
#pragma unroll
        for (int j = 0; j < kReduceInFlight; j++)
            if (on[j]) v[j] = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(yrow + (size_t)(s0 + j) * p.K));
#pragma unroll
        for (int j = 0; j < kReduceInFlight; j++)
            if (on[j]) add(v[j]);
    }
#pragma unroll
    for (int i = 0; i < COLS / 2; i++) {
        const float lo = sum[2 * i] + __builtin_bit_cast(float, o[i] << 16);
        const float hi = sum[2 * i + 1] + __builtin_bit_cast(float, o[i] & 0xffff0000u);
        o[i] = poisoned ? 0x7fc07fc0u : pack_bf16x2(lo, hi);
    }
    *op = o;
}

}  // namespace

hipError_t launch_rows_reduce(const RowsReduce &r, hipStream_t stream)
{
    const int cols = r.y_is_f32 ? 1024 : 2048;   // of a workgroup
    const int chunks = (r.p.K + cols - 1) / cols;
    const dim3 grid((unsigned)(r.p.M * chunks));
    typedef void (*Fn)(const RowsReduce, int);
    const Fn fn = r.y_is_f32 ? moe_rows_reduce_kernel<float> : moe_rows_reduce_kernel<uint16_t>;
    void *args[] = {const_cast<RowsReduce *>(&r), const_cast<int *>(&chunks)};
    return hipLaunchKernel(reinterpret_cast<const void *>(fn), grid, dim3(256), args, 0, stream);   // (this launch's own status)
}

}  // namespace alpha_moe
