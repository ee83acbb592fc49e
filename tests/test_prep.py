"""Input preparation (quantisers, moe_align_block_size) against brute force and invariants."""
import numpy as np
import pytest
import torch
from hypothesis import given, settings, strategies as st

from alpha_moe_python.prep import block_quant_fp8, moe_align_block_size, per_token_group_quant_fp8
from oracle import moe_oracle as O


@settings(max_examples=60, deadline=None)
@given(st.integers(1, 40), st.integers(1, 6), st.integers(1, 12), st.sampled_from([1, 4, 8, 16, 24]), st.integers(0, 10 ** 6))
def test_align_matches_brute_force(M, top_k, E, block, seed):
    g = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, E, (M, top_k), generator=g, dtype=torch.int32)   # duplicates within a token allowed
    got = moe_align_block_size(ids, block, E)
    ref = O.align_reference(ids, block, E)
    for a, b in zip(got, ref):
        assert a.dtype == torch.int32
        assert torch.equal(a, b)


def test_align_invariants():
    g = torch.Generator().manual_seed(3)
    M, top_k, E, block = 64, 9, 257, 16
    ids = torch.randint(0, E, (M, top_k), generator=g, dtype=torch.int32)
    sorted_ids, expert_ids, total = moe_align_block_size(ids, block, E)
    numel = M * top_k
    assert sorted_ids.numel() == numel + E * (block - 1)
    assert expert_ids.numel() == -(-sorted_ids.numel() // block)
    counts = torch.bincount(ids.flatten().long(), minlength=E)
    assert int(total) == int(((counts + block - 1) // block * block).sum())
    live = sorted_ids[sorted_ids < numel]
    assert sorted(live.tolist()) == list(range(numel))            # every slot exactly once
    assert (sorted_ids[int(total):] == numel).all()
    flat = ids.flatten()
    prev_e = -1
    for b in range(int(total) // block):
        e = int(expert_ids[b])
        assert e >= prev_e                                        # ascending experts
        prev_e = e
        seg = sorted_ids[b * block:(b + 1) * block]
        real = seg[seg < numel]
        assert (flat[real.long()] == e).all()
        assert (real[1:] > real[:-1]).all()                       # stable inside a block
    assert (expert_ids[int(total) // block:] == -1).all()


def test_align_empty_experts_and_single_token():
    ids = torch.tensor([[5, 5]], dtype=torch.int32)               # duplicate expert in one token
    s, e, t = moe_align_block_size(ids, 8, 7)
    assert int(t) == 8 and e[0] == 5 and (e[1:] == -1).all()
    assert s[:2].tolist() == [0, 1] and (s[2:] == 2).all()


def test_group_quant_matches_own_encoder_and_bound():
    g = torch.Generator().manual_seed(0)
    x = (torch.randn((17, 384), generator=g) * 3).to(torch.bfloat16)
    q, s = per_token_group_quant_fp8(x)
    codes, s_ref = O.quant_group_reference(x)
    assert torch.equal(s, s_ref)
    assert torch.equal(q.view(torch.uint8), codes)
    assert torch.equal(s, x.float().reshape(17, 3, 128).abs().amax(-1) / 448.0)
    deq = O.fp8_to_float(q).reshape(17, 3, 128) * s.unsqueeze(-1)
    err = (deq - x.float().reshape(17, 3, 128)).abs()
    # half an ulp of a 3-bit mantissa relative to the value, plus half a subnormal step (2^-10) in scaled units
    assert (err <= deq.abs() * 2.0 ** -4 + s.unsqueeze(-1) * 2.0 ** -10 + 1e-12).all()


def test_group_quant_exact_and_zero_rows():
    x = torch.zeros((2, 128))
    x[0, :5] = torch.tensor([448.0, -224.0, 1.0, 0.5, -0.015625])
    q, s = per_token_group_quant_fp8(x)
    assert float(s[0, 0]) == 1.0
    assert torch.equal(O.fp8_to_float(q)[0, :5], x[0, :5])      # exactly representable values survive
    assert float(s[1, 0]) == pytest.approx(1e-10 / 448.0)
    assert (q.view(torch.uint8)[1] == 0).all()


def test_block_quant():
    g = torch.Generator().manual_seed(1)
    w = torch.randn((3, 256, 384), generator=g) * 0.02
    q, s = block_quant_fp8(w)
    assert q.shape == w.shape and s.shape == (3, 2, 3)
    for e in range(3):
        for i in range(2):
            for j in range(3):
                blk = w[e, 128 * i:128 * i + 128, 128 * j:128 * j + 128]
                assert float(s[e, i, j]) == pytest.approx(float(blk.abs().max()) / 448.0, rel=1e-6)
                ref = torch.from_numpy(O.fp8_e4m3fn_encode((blk / s[e, i, j]).clamp(-448, 448).numpy()))
                assert torch.equal(q[e, 128 * i:128 * i + 128, 128 * j:128 * j + 128].view(torch.uint8), ref)
    assert int((O.fp8_to_float(q).abs() == 448.0).sum()) >= 3 * 2 * 3   # each block's amax maps to +-448


def _fma32(a, b, c):
    """a * b + c of float32 arrays, rounded once: the product is exact in float64, the sum is rounded to odd there."""
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)
    even = (s.view(np.int64) & 1) == 0
    return np.where((err != 0) & even, np.nextafter(s, np.copysign(np.inf, err)), s).astype(np.float32)


def _divide32(a, s, r):
    """What the small kernels take for a / s: one residual correction of a * r (r about 1 / s)."""
    t = a * r
    return _fma32(_fma32(-t, s, a), r, t)


def _bf16_values(exponents):
    return np.concatenate([np.float32(2.0) ** np.float32(e) * (1 + np.arange(128, dtype=np.float32) / 128) for e in exponents])


def test_requantisation_without_a_division_gives_the_codes_of_the_division():
    """Scale m / 448 and codes a / scale as moe_small.hip computes them, against the exact float32 division: every bf16 row
    maximum (scale), and every mantissa of maximum and value with the value up to 2^20 below the maximum (smaller ones are 0
    either way) at eleven of the maximum's exponents, the ends of its range among them; the reciprocal estimate right to one
    unit in the last place, either way."""
    f448 = np.float32(448.0)
    every = np.concatenate([np.array([1e-10], np.float32), _bf16_values(range(-33, 128))])
    every = every[every >= np.float32(1e-10)]
    assert np.array_equal(_divide32(every, f448, np.full_like(every, np.float32(1.0) / f448)), every / f448)
    checked = 0
    for e_m in (-33, -32, -31, -20, -1, 0, 1, 40, 125, 126, 127):
        for m in np.concatenate([_bf16_values([e_m]), np.array([1e-10], np.float32) if e_m == -33 else np.array([], np.float32)]):
            if m < np.float32(1e-10):
                continue
            a = _bf16_values(range(max(e_m - 20, -126), e_m + 1))
            a = a[a <= m]
            s = np.full_like(a, m / f448)
            want = torch.from_numpy(np.minimum(a / s, f448)).to(torch.float8_e4m3fn).view(torch.uint8)
            for ulps in (-1, 0, 1):
                r = (np.float32(1.0) / s).view(np.int32) + np.int32(ulps)
                r = r.view(np.float32)
                r = _fma32(_fma32(-s, r, np.ones_like(s)), r, r)
                got = torch.from_numpy(np.minimum(_divide32(a, s, r), f448)).to(torch.float8_e4m3fn).view(torch.uint8)
                assert torch.equal(got, want), (float(m), ulps)
                checked += got.numel()
    assert checked > 10_000_000


def test_swiglu_quotient_without_a_division():
    """g / (1 + exp(-g)) as swiglu_bf16 of moe_common.hpp takes it - (g / 4) / ((1 + exp(-g)) / 4), the reciprocal of the divisor right to
    one unit in the last place either way, one residual correction - for every finite bf16 gate whose quotient is not 0: at
    most one unit in the last place from the float32 division, no further from the float64 quotient than three quarters
    of one, and the same bf16 value with any `up` but where the product is on a rounding boundary."""
    g = np.concatenate([_bf16_values(range(-100, 7)), -_bf16_values(range(-100, 7))])
    g = g[(g > -88.5) & (g < 1e30)]
    e = np.exp(-g.astype(np.float64)).astype(np.float32)
    one_plus = (np.float32(1) + e).astype(np.float32)
    den = _fma32(e, np.full_like(e, 0.25), np.full_like(e, 0.25))
    assert np.array_equal(den * np.float32(4), one_plus)
    num = g * np.float32(0.25)
    want, exact = g / one_plus, g.astype(np.float64) / one_plus.astype(np.float64)
    for ulps in (-1, 0, 1):
        r = ((np.float32(1) / den).view(np.int32) + np.int32(ulps)).view(np.float32)
        assert np.all(np.abs(r) >= np.finfo(np.float32).tiny)
        got = _divide32(num, den, r)
        assert np.abs(got.view(np.int32) - want.view(np.int32)).max() <= 1, ulps
        assert np.all(np.abs(got - exact) <= 0.75 * np.spacing(np.abs(want))), ulps
        same = torch.from_numpy(got).bfloat16() == torch.from_numpy(want).bfloat16()
        assert float((~same).float().mean()) < 1e-3, ulps
