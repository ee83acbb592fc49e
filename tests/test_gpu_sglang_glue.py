"""The SGLang wiring of extra/sglang_rocm.patch, replayed without SGLang: the weight loader hands gate and up shards of
every expert to W13Interleaver the way FusedMoE.weight_loader does, fused_experts runs the forward path of
fused_experts_impl (tuning table from ALPHA_MOE_CONFIG, HIP quantiser, HIP aligner, storing operator), and the result is
checked against the CPU oracle fed with the ORIGINAL (not interleaved) checkpoint tensors."""
import json
import os

import pytest
import torch

from alpha_moe_python.prep import block_quant_fp8
from alpha_moe_python.sglang_glue import W13Interleaver, fused_experts
from alpha_moe_python.utils import get_best_config, interleave_tensor
from gpu_util import MAX_ABS_OVER_MAX_REF, MIN_COSINE
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M", [3, 40, 300])
def test_fused_experts_matches_the_oracle_on_the_checkpoint_tensors(M, tmp_path):
    E, top_k, K, I = 10, 4, 512, 256
    g = torch.Generator().manual_seed(11 + M)
    # the checkpoint: per expert a gate matrix (w1), an up matrix (w3) and a down matrix (w2), block-quantised FP8
    w13_f = torch.randn((E, 2 * I, K), generator=g) * 0.05
    w2_f = torch.randn((E, K, I), generator=g) * 0.05
    w13_q, w13_s = block_quant_fp8(w13_f)            # [E, 2I, K] fp8 (gate rows first, up rows second), [E, 2I/128, K/128]
    w2_q, w2_s = block_quant_fp8(w2_f)
    # FusedMoE's parameters, filled shard by shard
    w13 = torch.zeros((E, 2 * I, K), dtype=torch.float8_e4m3fn, device=DEV)
    w13_scale = torch.zeros((E, 2 * I // 128, K // 128), dtype=torch.float32, device=DEV)
    il_w, il_s = W13Interleaver(E, 8), W13Interleaver(E, 1)
    for e in range(E):
        for shard in (("w3", "w1") if e % 2 else ("w1", "w3")):
            rows = slice(0, I) if shard == "w1" else slice(I, 2 * I)
            srows = slice(0, I // 128) if shard == "w1" else slice(I // 128, 2 * I // 128)
            w13[e, rows] = w13_q[e, rows].to(DEV)
            il_w.shard_loaded(w13[e], e, shard)
            w13_scale[e, srows] = w13_s[e, srows].to(DEV)
            il_s.shard_loaded(w13_scale[e], e, shard)
    assert torch.equal(w13.cpu().view(torch.uint8), interleave_tensor(w13_q, 8).view(torch.uint8))
    assert torch.equal(w13_scale.cpu(), interleave_tensor(w13_s, 1))
    # the forward call of one layer
    cfg_path = os.path.join(tmp_path, "table.json")
    with open(cfg_path, "w") as fh:
        json.dump({"1": {"block_m": 16, "block_n": 32, "warp_n": 8, "stages": 4},
                   "64": {"block_m": 16, "block_n": 64, "warp_n": 4, "stages": 3},
                   "512": {"block_m": 64, "block_n": 64, "warp_n": 4, "stages": 3}}, fh)
    hidden = (torch.randn((M, K), generator=g)).to(torch.bfloat16)
    probs = torch.softmax(torch.randn((M, E), generator=g), dim=-1)
    topk_weights, topk_ids = probs.topk(top_k, dim=-1)
    os.environ["ALPHA_MOE_CONFIG"] = cfg_path
    try:
        h = hidden.to(DEV).clone()
        print(f"case sglang glue M={M} knobs {get_best_config(cfg_path, M)}", flush=True)
        got = fused_experts(h, w13, w2_q.to(DEV), topk_weights.to(DEV), topk_ids.to(DEV), w13_scale, w2_s.to(DEV),
                            routed_scaling_factor=2.5)
        torch.cuda.synchronize()
    finally:
        del os.environ["ALPHA_MOE_CONFIG"]
    assert got.data_ptr() == h.data_ptr()   # hidden_states is reused as the output, as the reference's patch does
    # oracle: quantise the activations the same way, route, and run the maths on the interleaved tensors' originals
    xq, xs = O.quant_group_reference(hidden)
    ids = O.align_reference(topk_ids.to(torch.int32), 16, E)
    ref = O.fused_moe_oracle(xq.view(torch.float8_e4m3fn), xs, interleave_tensor(w13_q, 8), interleave_tensor(w13_s, 1), w2_q,
                             w2_s, *ids, topk_weights.float().contiguous(), torch.zeros((M, K), dtype=torch.bfloat16),
                             top_k, 16, 2.5)
    m = O.error_metrics(got, ref)
    assert m["max_abs_over_max_ref"] <= MAX_ABS_OVER_MAX_REF and m["cosine"] >= MIN_COSINE, m


@pytest.mark.parametrize("M,top_k,K,I,E,block_m", [
    (1, 1, 128, 128, 1, 8), (1, 9, 7168, 256, 257, 16),             # one row of one block; the widest K of a wavefront
    (2, 20, 1024, 128, 4096, 8), (3, 4, 1152, 256, 33, 16),         # the most experts; K blocks that do not fill the wavefronts
    (4, 5, 2176, 128, 40, 24), (5, 8, 4096, 384, 64, 32), (7, 9, 4224, 256, 257, 16),
    (8, 20, 2560, 128, 64, 8), (8, 8, 640, 256, 31, 64),
    (9, 4, 1152, 256, 33, 16), (16, 10, 3072, 128, 512, 8),         # the second eight tokens; the most tokens and rows
    (12, 9, 7168, 256, 257, 16), (13, 8, 4224, 256, 64, 16), (16, 9, 7168, 256, 257, 16),   # ... with the widest K of a wavefront
    (17, 4, 1152, 256, 33, 16)])                                    # one token too many; blocks of 64: the three steps as well
def test_layer_call_equals_its_three_steps_bit_for_bit(M, top_k, K, I, E, block_m):
    """The smallest batches are quantised and aligned inside the operator's first launch; quantiser, aligner and storing
    operator called one by one are the general path.  Rows with an expert twice, slots without an expert, an infinity, a
    NaN and an all-zero group among them; a base that is not 16-byte aligned, replays of a graph; the C entry, which takes
    every supported size, also where the binding calls the three steps because they are faster."""
    import alpha_moe
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(M * 131 + K)
    gd = torch.Generator(device=DEV).manual_seed(M * 131 + K)
    w13 = (torch.randn((E, 2 * I, K), generator=gd, device=DEV) * 0.5).to(torch.float8_e4m3fn)
    w2 = (torch.randn((E, K, I), generator=gd, device=DEV) * 0.5).to(torch.float8_e4m3fn)
    w13_s = torch.rand((E, 2 * I // 128, K // 128), generator=gd, device=DEV) * 0.1
    w2_s = torch.rand((E, K // 128, I // 128), generator=gd, device=DEV) * 0.1
    taken = alpha_moe.c_abi.alpha_moe_layer_call_supported(top_k, M, K, 2 * I, E, block_m, 32, 8, 4)
    assert taken == (M <= 16 and block_m <= 32)
    for kind in ("plain", "odd", "wild"):
        x = (torch.randn((M, K), generator=g) * 2).to(torch.bfloat16)
        ids = torch.randint(0, E, (M, top_k), generator=g).to(torch.int32)
        if kind != "plain":
            ids.view(-1)[::3] = torch.tensor([-1, E, E - 1], dtype=torch.int32)[torch.arange(0, M * top_k, 3) // 3 % 3]
            x[0, :128] = 0
        if kind == "wild":
            x[M - 1, K - 1], x[M // 2, K // 2] = float("inf"), float("nan")
            x[0, 0] = torch.finfo(torch.bfloat16).max
        x, ids, weights = x.to(DEV), ids.to(DEV), torch.rand((M, top_k), generator=g).to(DEV)
        ids_were, weights_were = ids.clone(), weights.clone()
        print(f"case layer call M={M} top_k={top_k} K={K} I={I} E={E} block_m={block_m} {kind}", flush=True)
        q, q_s, *routing = prep_hip.prepare_inputs(x, ids, 128, block_m, E)
        want = torch.empty_like(x)
        torch.ops.alpha_moe.fused_moe_w8a8_up_down_store(q, q_s, w13, w13_s, w2, w2_s, *routing, weights, want, top_k,
                                                         block_m, 32, 8, 4, 2.5)

        def call(h):
            torch.ops.alpha_moe.fused_experts(h, ids, w13, w13_s, w2, w2_s, weights, 128, block_m, 32, 8, 4, 2.5)

        def same(h, want):
            torch.cuda.synchronize()
            assert torch.equal(h.view(torch.int16), want.view(torch.int16)), kind

        h = x.clone()
        call(h)
        same(h, want)
        odd = torch.empty(M * K + 4, dtype=torch.bfloat16, device=DEV)[4:].view(M, K)
        odd.copy_(x)
        call(odd)
        same(odd, want)
        if taken:
            sizes = (top_k, M, K, 2 * I, E)
            ws = torch.zeros(alpha_moe.c_abi.alpha_moe_workspace_bytes(*sizes, M * top_k + E * (block_m - 1), block_m),
                             dtype=torch.uint8, device=DEV)
            out = torch.empty_like(x)
            assert alpha_moe.c_abi.alpha_moe_layer_call(
                x.data_ptr(), ids.data_ptr(), w13.data_ptr(), w13_s.data_ptr(), w2.data_ptr(), w2_s.data_ptr(),
                weights.data_ptr(), out.data_ptr(), *sizes, block_m, 32, 8, 4, 2.5, ws.data_ptr(), ws.numel(),
                torch.cuda.current_stream().cuda_stream) == 0
            same(out, want)
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.stream(stream):
            call(h)   # scratch memory is per stream and is not allocated under capture
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            call(h)
        for _ in range(3):
            h.copy_(x)
            graph.replay()
            same(h, want)
        assert torch.equal(ids, ids_were) and torch.equal(weights, weights_were)   # nothing but hidden_states is written


@pytest.mark.parametrize("M", [3, 40])
@pytest.mark.parametrize("knob", ["block_m", "block_n", "warp_n", "stages"])
def test_layer_call_refuses_knobs_that_only_their_low_32_bits_make_legal(knob, M):
    """With and without the two-launch form: a legal value plus or minus 2**32 is no legal value."""
    import alpha_moe  # noqa: F401
    E, top_k, K, I = 4, 2, 256, 128
    w13 = torch.zeros((E, 2 * I, K), device=DEV).to(torch.float8_e4m3fn)
    w2 = torch.zeros((E, K, I), device=DEV).to(torch.float8_e4m3fn)
    w13_s, w2_s = torch.ones((E, 2 * I // 128, K // 128), device=DEV), torch.ones((E, K // 128, I // 128), device=DEV)
    ids = torch.arange(M * top_k, dtype=torch.int32, device=DEV).view(M, top_k) % E
    legal = {"block_m": 16, "block_n": 32, "warp_n": 8, "stages": 4}
    for value in (legal[knob] - 2 ** 32, legal[knob] + 2 ** 32, 0, -legal[knob]):
        h = torch.ones((M, K), dtype=torch.bfloat16, device=DEV)
        print(f"case layer call M={M} {knob}={value}", flush=True)
        with pytest.raises(RuntimeError):
            torch.ops.alpha_moe.fused_experts(h, ids, w13, w13_s, w2, w2_s, torch.ones((M, top_k), device=DEV), 128,
                                              *{**legal, knob: value}.values(), 1.0)
        assert bool((h == 1).all())


@pytest.mark.parametrize("M,K,E,whole", [(1, 4224, 8, True), (8, 4224, 8, True), (9, 4224, 8, False), (8, 7168, 8, True),
                                         (9, 7168, 8, False), (9, 7168, 64, True), (9, 4224, 64, False), (16, 4096, 8, True),
                                         (16, 7168, 64, False)])
def test_layer_call_takes_two_launches_only_where_they_are_faster(M, K, E, whole):
    """The two-launch form allocates nothing; the preparation returns five tensors."""
    import alpha_moe  # noqa: F401
    top_k, I = 2, 256
    g = torch.Generator(device=DEV).manual_seed(M + K)
    w13 = torch.randn((E, 2 * I, K), generator=g, device=DEV).to(torch.float8_e4m3fn)
    w2 = torch.randn((E, K, I), generator=g, device=DEV).to(torch.float8_e4m3fn)
    w13_s, w2_s = torch.ones((E, 2 * I // 128, K // 128), device=DEV), torch.ones((E, K // 128, I // 128), device=DEV)
    ids = torch.arange(M * top_k, dtype=torch.int32, device=DEV).view(M, top_k) % E
    h, weights = torch.randn((M, K), generator=g, device=DEV).to(torch.bfloat16), torch.ones((M, top_k), device=DEV)

    def call():
        torch.ops.alpha_moe.fused_experts(h, ids, w13, w13_s, w2, w2_s, weights, 128, 16, 32, 8, 4, 1.0)

    print(f"case route of a layer call M={M} K={K} E={E}", flush=True)
    call()   # takes the scratch memory
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    call()
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == (0 if whole else 5)
