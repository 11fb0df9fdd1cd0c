"""GPU: the general map kernel at the edges of its tiles and dispatch.

Tiles hold 64 or 128 tokens, column tiles 16; waves own 16 output pairs and
chunks 32 input pairs, so the head dims here leave every kind of remainder
(half sizes 3, 40, 48, 64, 80, 128, 160, 256). The split operands keep 22
to 24 bits (fp16 keys below 2^-16 fewer: an absolute 2^-38), so the
mapped rows are held to 2^-18 of their summands' magnitude where rounding to
the pool's type does not decide.
"""

from __future__ import annotations

import pytest
import torch

from cachebridge_amd.mapper import HeadwiseMapper
from cachebridge_amd.plan import rows_from_layers, rows_from_page
from oracle import install as oi
from oracle import tolerance as ot

pytestmark = pytest.mark.gpu


def _mapper(dim, dtype, support, seed=5, ls=5, hs=2, lt=3, ht=2):
    g = torch.Generator().manual_seed(seed + dim)
    layers = torch.stack([torch.randperm(ls, generator=g)[:support] for _ in range(lt * ht)])
    std = (support * dim) ** -0.5
    spec = {"assign_layer": layers.view(lt, ht, support),
            "assign_head": torch.randint(0, hs, (lt, ht, support), generator=g),
            "k_weight": torch.randn(lt, ht, support * dim, dim, generator=g) * std,
            "v_weight": torch.randn(lt, ht, support * dim, dim, generator=g) * std,
            "k_bias": torch.randn(lt, ht, dim, generator=g) * 0.1,
            "v_bias": torch.randn(lt, ht, dim, generator=g) * 0.1}
    mapper = HeadwiseMapper.from_assignment(**spec, source_rope_theta=1e4, target_rope_theta=1e6, dtype=dtype,
                                            device="cuda", max_positions=1024)
    return g, spec, mapper


def _reference(spec, page, position):
    virtual = oi.virtual_source_page(page, spec["assign_layer"], spec["assign_head"])
    return oi.assignment_mapper(spec, source_rope_theta=1e4, target_rope_theta=1e6).map_page(
        virtual, position_start=position)


@pytest.mark.parametrize("dim,dtype,support", [
    (256, torch.bfloat16, 1), (256, torch.bfloat16, 3), (96, torch.bfloat16, 2), (6, torch.bfloat16, 2),
    (320, torch.bfloat16, 1), (512, torch.float16, 1), (128, torch.float16, 1), (64, torch.float16, 4),
    (80, torch.float16, 1), (160, torch.float16, 2), (256, torch.float32, 1), (128, torch.float32, 2),
    (96, torch.float32, 1),
])
@pytest.mark.parametrize("tokens", [1, 16, 17, 63, 64, 129, 300])
def test_tiles_and_remainders_match_oracle(dim, dtype, support, tokens):
    print(f"any kernel D={dim} {dtype} s={support} T={tokens}", flush=True)
    g, spec, mapper = _mapper(dim, dtype, support)
    page = torch.randn(2, 5, tokens, 2, dim, generator=g).to(dtype)
    out = mapper.map_page(page.cuda(), position_start=11, output_device="cuda")
    bound = ot.magnitude_bound(page, spec, position_start=11, source_theta=1e4, target_thetas=1e6)
    # (A page of one token is too small a sample for the share within 1 ulp.)
    ot.check_mapped(out, _reference(spec, page, 11), bound, abs_factor=2.0 ** -18,
                    min_within_ulp=0.999 if tokens > 16 else 0.99)


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("scale,mixed", [(1.0, False), (1e-2, False), (1e-3, False), (1e-4, False), (1.0, True),
                                         (1e-2, True)])
def test_small_half_precision_keys_keep_their_bits(dim, scale, mixed):
    """fp16 keys far below 1, mapped up by large weights, alone or as quiet
    channels (down to 2^-8 of the loudest, with weights to match).

    fp32 multiply-adds leave a relative error of 2e-7, an ulp is 2^-11 to
    2^-10: at most about 0.01% of the elements (those near a cancellation) may
    lie two ulps apart, and no summand more than 2^-20 of the bound (32-bit
    sums of up to 256 terms: 256 2^-24 at worst, their root for random signs).
    """
    print(f"small fp16 keys D={dim} scale={scale} mixed={mixed}", flush=True)
    g, spec, _ = _mapper(dim, torch.float16, 1)
    channel = torch.full((dim // 2,), scale)
    if mixed:
        channel = channel * 2.0 ** torch.randint(-8, 1, (dim // 2,), generator=g)
    channel = channel.repeat(2)  # RoPE partners share their scale
    spec["k_weight"] = spec["k_weight"] / channel[:, None] * (100 * scale if scale < 1 else 1)
    mapper = HeadwiseMapper.from_assignment(**spec, source_rope_theta=1e4, target_rope_theta=1e6, dtype=torch.float16,
                                            device="cuda", max_positions=1024)
    page = (torch.randn(2, 5, 160, 2, dim, generator=g) * channel).to(torch.float16)
    out = mapper.map_page(page.cuda(), position_start=11, output_device="cuda")
    ref = _reference(spec, page, 11)
    bound = ot.magnitude_bound(page, spec, position_start=11, source_theta=1e4, target_thetas=1e6)
    ot.check_mapped(out[:1], ref[:1], bound[:1], abs_factor=2.0 ** -20, min_within_ulp=0.9995)


@pytest.mark.parametrize("dim,dtype", [(256, torch.bfloat16), (128, torch.float16), (128, torch.float32)])
def test_layers_at_odd_addresses_map_to_the_same_rows(dim, dtype):
    """Per-layer pointers that are only element-aligned take the element-wise
    accesses: the same bits as the 16-byte ones."""
    print(f"odd addresses D={dim} {dtype}", flush=True)
    g, _, mapper = _mapper(dim, dtype, 1)
    page = torch.randn(2, 5, 70, 2, dim, generator=g).to(dtype).cuda()
    want = mapper.map_page(page, position_start=3, output_device="cuda")

    def odd(t):
        flat = torch.zeros(t.numel() + 1, dtype=dtype, device="cuda")
        flat[1:] = t.reshape(-1)
        return flat[1:].view(t.shape)

    source = rows_from_layers([odd(t) for t in page[0]], [odd(t) for t in page[1]])
    tk, tv = ([odd(torch.zeros_like(want[0, 0])) for _ in range(3)] for _ in range(2))
    mapper.map_install(source, rows_from_layers(tk, tv), num_tokens=70, position_start=3)
    torch.cuda.synchronize()
    assert torch.equal(torch.stack(tk), want[0]) and torch.equal(torch.stack(tv), want[1])
    # One odd side is enough to need them.
    out = torch.zeros_like(want)
    mapper.map_install(source, rows_from_page(out), num_tokens=70, position_start=3)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("dim,dtype", [(256, torch.bfloat16), (96, torch.bfloat16), (128, torch.float16),
                                       (128, torch.float32)])
def test_infinities_and_nans_come_out_as_in_fp32(dim, dtype):
    print(f"not finite D={dim} {dtype}", flush=True)
    g, spec, mapper = _mapper(dim, dtype, 2)
    page = torch.randn(2, 5, 40, 2, dim, generator=g).to(dtype)
    page[:, :, 3, :, 5] = float("inf")
    page[:, :, 17, :, dim - 1] = float("-inf")
    page[:, :, 30, :, 0] = float("nan")
    if dtype == torch.float16:
        page[:, :, 35] = 65504.0  # the largest finite input must stay finite inside
    out = mapper.map_page(page.cuda(), position_start=0, output_device="cuda").cpu()
    ref = _reference(spec, page, 0)
    # Values: one infinite input per member, so every sum keeps its sign; keys
    # mix two infinities, whose sum's kind depends on the order of summation.
    assert torch.equal(torch.isnan(out[1]), torch.isnan(ref[1]))
    assert torch.equal(out[1][torch.isinf(ref[1])], ref[1][torch.isinf(ref[1])])
    assert torch.equal(torch.isfinite(out), torch.isfinite(ref))


@pytest.mark.parametrize("dim,support", [(128, 1), (80, 2), (256, 1)])
def test_recomputed_tiles_match_oracle(dim, support):
    """fp16 keys of 2^14 and more (finite, but not as scaled terms) take the
    recompute beside tokens that do not; outputs stay in range by small maps."""
    print(f"large fp16 keys D={dim} s={support}", flush=True)
    g, spec, _ = _mapper(dim, torch.float16, support)
    spec["k_weight"] = spec["k_weight"] * 0.1
    mapper = HeadwiseMapper.from_assignment(**spec, source_rope_theta=1e4, target_rope_theta=1e6, dtype=torch.float16,
                                            device="cuda", max_positions=1024)
    page = torch.randn(2, 5, 150, 2, dim, generator=g)
    page[0, :, [0, 5, 40, 41, 77, 149]] *= 15000
    page = page.clamp(-65504, 65504).to(torch.float16)
    assert bool((page[0].abs() > 2 ** 14).any())
    out = mapper.map_page(page.cuda(), position_start=11, output_device="cuda")
    bound = ot.magnitude_bound(page, spec, position_start=11, source_theta=1e4, target_thetas=1e6)
    ot.check_mapped(out, _reference(spec, page, 11), bound, abs_factor=2.0 ** -18, min_within_ulp=0.999)


@pytest.mark.parametrize("dim,dtype", [(256, torch.bfloat16), (128, torch.float16)])
def test_rows_that_are_not_finite_cost_a_few_passes(dim, dtype):
    """A page of NaN rows against a finite one: one fp32 pass beside the split
    one (3 to 4.5 times the time here), not the 25 to 110 times that a
    term-by-term recompute per lane took."""
    print(f"time of NaN rows D={dim} {dtype}", flush=True)
    g, _, mapper = _mapper(dim, dtype, 1, lt=24, ht=8)
    page = torch.randn(2, 5, 1024, 2, dim, generator=g).to(dtype).cuda()
    nans = torch.full_like(page, float("nan"))
    out = torch.empty(2, 24, 1024, 8, dim, dtype=dtype, device="cuda")
    times = {}
    for name, rows in (("finite", page), ("nan", nans), ("finite", page), ("nan", nans)):  # the first pair warms up
        start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(5):
            mapper.map_page(rows, position_start=0, output_device="cuda", output=out)
        stop.record()
        torch.cuda.synchronize()
        times[name] = start.elapsed_time(stop)
    assert bool(torch.isnan(out).all())
    assert times["nan"] <= 10 * times["finite"], times
