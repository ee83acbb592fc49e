"""GPU input preparation (per-token-group FP8 quantisation, expert alignment) against the CPU oracle: bit-exact."""
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,K,dtype", [(1, 128, torch.bfloat16), (7, 512, torch.bfloat16), (64, 7168, torch.bfloat16),
                                       (33, 2048, torch.float32), (4096, 2048, torch.bfloat16)])
def test_quant_matches_oracle_bit_for_bit(M, K, dtype):
    from alpha_moe_python import prep, prep_hip
    g = torch.Generator().manual_seed(M * 31 + K)
    x = (torch.randn((M, K), generator=g) * torch.rand((M, 1), generator=g) * 4).to(dtype)
    x[0, :128] = 0                      # an all-zero group: scale = 1e-10 / 448, q = 0
    if M > 1:
        x[1, 5] = 3.0e4                 # a large outlier
    print(f"case quant M={M} K={K} {dtype}", flush=True)
    q, s = prep_hip.per_token_group_quant_fp8(x.to(DEV))
    torch.cuda.synchronize()
    q_ref, s_ref = O.quant_group_reference(x)
    assert q.dtype == torch.float8_e4m3fn and s.dtype == torch.float32
    assert torch.equal(s.cpu(), s_ref)
    assert torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8))
    # and the torch restatement the package ships agrees as well
    q_t, s_t = prep.per_token_group_quant_fp8(x)
    assert torch.equal(q_t.view(torch.uint8), q_ref.view(torch.uint8)) and torch.equal(s_t, s_ref)


@pytest.mark.parametrize("M,top_k,E,block", [(1, 9, 257, 16), (4, 2, 8, 8), (64, 9, 257, 16), (300, 8, 128, 64),
                                              (455, 9, 257, 128), (456, 9, 257, 16), (8192, 9, 257, 128),
                                              (4096, 10, 512, 24)])
def test_align_matches_oracle_bit_for_bit(M, top_k, E, block):
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(M + 7 * E)
    # skewed routing: some experts empty, some hot
    probs = torch.rand(E, generator=g) ** 4
    ids = torch.multinomial(probs.expand(M, E), top_k, replacement=False, generator=g).to(torch.int32)
    print(f"case align M={M} top_k={top_k} E={E} block={block}", flush=True)
    s_ids, e_ids, total = prep_hip.moe_align_block_size(ids.to(DEV), block, E)
    torch.cuda.synchronize()
    r_ids, r_e, r_total = O.align_reference(ids, block, E)
    assert torch.equal(total.cpu(), r_total)
    assert torch.equal(e_ids.cpu(), r_e)
    assert torch.equal(s_ids.cpu(), r_ids)


@pytest.mark.parametrize("numel,E,block", [(1, 1, 8), (63, 2, 8), (65, 3, 128), (1025, 1, 16), (4096, 512, 56),
                                            (4096, 4096, 8), (4097, 4096, 8), (4097, 1, 128), (5120, 257, 64),
                                            (40000, 3, 8), (81920, 512, 96),
                                            (524288, 3, 8), (524289, 40, 16), (1048577, 301, 64)])
def test_align_at_the_edges_of_its_runs_and_segments(numel, E, block):
    """one chunk, one segment and their remainders; one workgroup (up to 4096 slots) and several; segments of 1024,
    2048 and 4096 slots (beyond 512 segments); an even and an odd number
    of experts, one, and the most there can be; slots without an expert among them"""
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(numel + E)
    ids = torch.randint(-1, E + 1, (numel, 1), generator=g).to(torch.int32)
    ids[: numel // 3] = E // 2          # a hot expert over several chunks
    print(f"case align numel={numel} E={E} block={block}", flush=True)
    s_ids, e_ids, total = prep_hip.moe_align_block_size(ids.to(DEV), block, E)
    torch.cuda.synchronize()
    flat = ids.flatten().long()
    keep = torch.nonzero((flat >= 0) & (flat < E)).flatten()
    r_ids, r_e = torch.full_like(s_ids.cpu(), numel), torch.full_like(e_ids.cpu(), -1)
    at = 0
    for e in torch.unique(flat[keep]).tolist():
        slots = keep[flat[keep] == e]
        r_ids[at:at + len(slots)] = slots.to(torch.int32)
        padded = (len(slots) + block - 1) // block * block
        r_e[at // block:(at + padded) // block] = e
        at += padded
    assert total.item() == at
    assert torch.equal(e_ids.cpu(), r_e)
    assert torch.equal(s_ids.cpu(), r_ids)


@pytest.mark.parametrize("E", [1024, 1025, 2045, 2046, 2048, 2049])
def test_align_where_the_wavefronts_of_a_segment_change(E):
    """16, 8 and 4 wavefronts place a segment; columns of the histogram are shared by threads up to 1023 of them"""
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(E)
    ids = torch.randint(0, E, (4500, 1), generator=g, dtype=torch.int32)
    print(f"case align E={E}", flush=True)
    got = prep_hip.moe_align_block_size(ids.to(DEV), 8, E)
    for a, b in zip(got, O.align_reference(ids, 8, E)):
        assert torch.equal(a.cpu(), b)


@pytest.mark.parametrize("numel", [4096, 4500, 70000])
@pytest.mark.parametrize("E", [256, 817, 818, 2045, 2046, 3580, 3581])
def test_align_where_tables_and_cursors_fill_the_memory(E, numel):
    """16, 8 and 4 wavefronts place a segment, the last with more slots each than they keep in registers; 3581 experts and more of
    them have more than 64 KiB of tables and cursors"""
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(E)
    ids = torch.randint(-1, E, (numel, 1), generator=g, dtype=torch.int32)
    ids[100:1500] = E - 1
    print(f"case align E={E} numel={numel}", flush=True)
    got = prep_hip.moe_align_block_size(ids.to(DEV), 8, E)
    for a, b in zip(got, O.align_reference(ids, 8, E)):
        assert torch.equal(a.cpu(), b)


@pytest.mark.parametrize("E", [1100, 2100])
@pytest.mark.parametrize("segments", [5, 8, 9, 11, 12, 13, 16, 17, 20])
def test_align_adds_up_the_segments_of_a_thread(segments, E):
    """one thread per column (two columns a thread from 2049 experts on): up to eight segments in one round, then rounds of eight
    and of four, the last one part-filled"""
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(E + segments)
    ids = torch.randint(-1, E + 1, (1024 * segments - 7, 1), generator=g, dtype=torch.int32)
    print(f"case align segments={segments} E={E}", flush=True)
    got = prep_hip.moe_align_block_size(ids.to(DEV), 8, E)
    ids[(ids < 0) | (ids >= E)] = E   # (an expert of its own behind the last, cut off below)
    s_ids, e_ids, total = O.align_reference(ids, 8, E + 1)
    n = total.item() - -(-int((ids == E).sum()) // 8) * 8
    assert got[2].item() == n
    assert got[0][:n].tolist() == s_ids[:n].tolist() and bool((got[0][n:] == ids.numel()).all())
    assert got[1][:n // 8].tolist() == e_ids[:n // 8].tolist() and bool((got[1][n // 8:] == -1).all())


@pytest.mark.parametrize("kind", ["even", "one", "half", "none"])
@pytest.mark.parametrize("numel", [1023, 1024, 4159])
@pytest.mark.parametrize("E", [1, 8, 9, 128, 129])
def test_align_of_few_experts(E, numel, kind):
    """1024 slots and more of up to 128 experts are ranked without the lane masks (up to 8 experts), or with them behind the
    first lane's expert; all slots on one expert, half of them, none valid, first lanes without an expert among them"""
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(E * 7 + numel)
    ids = torch.randint(-1, E + 1, (numel, 1), generator=g, dtype=torch.int32)
    if kind == "one":
        ids[:] = E - 1
    elif kind == "half":
        ids[torch.rand(numel, generator=g) < 0.5] = E // 2
    elif kind == "none":
        ids[:] = torch.where(torch.rand((numel, 1), generator=g) < 0.5, -1, E).to(torch.int32)
    print(f"case align numel={numel} E={E} {kind}", flush=True)
    got = prep_hip.moe_align_block_size(ids.to(DEV), 16, E)
    flat = ids.flatten()
    want, experts = [], []
    for e in range(E):
        slots = torch.nonzero(flat == e).flatten().tolist()
        slots += [numel] * (-len(slots) % 16)
        want += slots
        experts += [e] * (len(slots) // 16)
    assert got[2].item() == len(want)
    assert got[0].tolist() == want + [numel] * (got[0].numel() - len(want))
    assert got[1].tolist() == experts + [-1] * (got[1].numel() - len(experts))


@pytest.mark.parametrize("M,K,top_k,E,block,dtype", [
    (1, 128, 1, 3, 16, torch.bfloat16),        # one group, one slot
    (7, 7168, 9, 257, 8, torch.bfloat16),
    (65, 2048, 10, 512, 16, torch.float32),    # an odd number of groups per thread
    (512, 256, 8, 128, 64, torch.bfloat16),    # 4096 slots: the last size with one workgroup for the alignment
    (513, 384, 8, 128, 64, torch.float32),     # two launches
    (3000, 7168, 9, 257, 96, torch.bfloat16)])
def test_prepare_inputs_equals_the_two_separate_calls(M, K, top_k, E, block, dtype):
    from alpha_moe_python import prep_hip
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn((M, K), generator=g).to(dtype).to(DEV)
    ids = torch.randint(0, E, (M, top_k), generator=g, dtype=torch.int32).to(DEV)
    print(f"case prepare M={M} K={K} top_k={top_k} E={E} {dtype}", flush=True)
    got = prep_hip.prepare_inputs(x, ids, 128, block, E)
    torch.cuda.synchronize()
    q_ref, s_ref = O.quant_group_reference(x.cpu())
    assert torch.equal(got[0].cpu().view(torch.uint8), q_ref.view(torch.uint8)) and torch.equal(got[1].cpu(), s_ref)
    for a, b in zip(got[2:], O.align_reference(ids.cpu(), block, E)):
        assert torch.equal(a.cpu(), b)


def test_align_drops_slots_with_an_expert_out_of_range():
    from alpha_moe_python import prep_hip
    ids = torch.tensor([[0, 3], [7, -1], [9, 3]], dtype=torch.int32)
    s_ids, e_ids, total = prep_hip.moe_align_block_size(ids.to(DEV), 4, 8)
    torch.cuda.synchronize()
    assert total.item() == 12
    assert s_ids.cpu()[:12].tolist() == [0, 6, 6, 6, 1, 5, 6, 6, 2, 6, 6, 6]
    assert e_ids.cpu()[:3].tolist() == [0, 3, 7] and (e_ids.cpu()[3:] == -1).all()


def test_prepared_inputs_drive_the_fused_operator():
    """quantise + align on the GPU, then the fused call: same result as with the torch-prepared inputs."""
    from alpha_moe_python import prep, prep_hip
    from alpha_moe_python.workloads import SHAPES, make_weights
    import alpha_moe  # noqa: F401
    shape = SHAPES["c1"]
    W = make_weights(shape, device=DEV, seed=0)
    g = torch.Generator().manual_seed(5)
    M = 40
    x = torch.randn((M, shape.K), generator=g).to(torch.bfloat16).to(DEV)
    ids = torch.multinomial(torch.ones(M, shape.E), shape.top_k, generator=g).to(torch.int32).to(DEV)
    tw = torch.rand((M, shape.top_k), generator=g).to(DEV)
    outs = []
    for mod in (prep_hip, prep):
        if mod is prep_hip:
            xq, xs = mod.per_token_group_quant_fp8(x)
            s_ids, e_ids, total = mod.moe_align_block_size(ids, 16, shape.E)
        else:   # the torch restatement on the CPU (IEEE division), then copied over
            xq, xs = (t.to(DEV) for t in mod.per_token_group_quant_fp8(x.cpu()))
            s_ids, e_ids, total = (t.to(DEV) for t in mod.moe_align_block_size(ids.cpu(), 16, shape.E))
        out = torch.zeros((M, shape.K), dtype=torch.bfloat16, device=DEV)
        torch.ops.alpha_moe.fused_moe_w8a8_up_down(xq, xs, W.w1, W.w1_scale, W.w2, W.w2_scale, s_ids, e_ids, total, tw,
                                                   out, shape.top_k, 16, 64, 4, 3, 1.0)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
