"""The prompt products of more than 64 rows: each form of the ring kernel, and what serves the
shapes beside them, at the edges of its tiles: ragged row tiles, one row past a tile, odd group counts (a last step
without a partner) and group counts its k slices do not divide.

Reference: float64 on the device over the exactly dequantised weights
(``ops.dequantize``, itself checked bit for bit against the oracle).  Bars as the
prompt-row tests': one bf16 rounding of the true value plus 1e-4 of the largest output
(fp32 sums of values up to about 144 times the weights' own).
"""

import pytest
import torch

from oracle import w4a16 as ow
from torch2iron_amd import _lib
from torch2iron_amd import model as gm
from torch2iron_amd import ops
from torch2iron_amd.formats import W4A16Weight, interleave_gate_up

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

# what plan_prompt (csrc/prompt_plan.h) gives the product with its own row sums, rows, K, N;
# test_prompt_plan holds the plan to these names
SHAPES = [
    ("decode tiles", 500, 3200, 1024), ("decode tiles", 470, 3072, 1024),
    ("64x128, 2 slices", 520, 2176, 128), ("64x128, 2 slices", 577, 2048, 384), ("64x128, 2 slices", 300, 1024, 6144),
    ("64x128 kernel", 2050, 2176, 1024), ("64x128, pairs", 577, 1920, 6144), ("64x128, pairs", 1100, 2176, 3072),
    ("64x128, pairs", 197, 2048, 12288),
    ("128x256", 390, 1920, 12288), ("128x256", 321, 2176, 12288), ("128x256", 3969, 3072, 2048),
    # few steps, two to five: the prologue's loads reach past the last one, and every load that is
    # off is then waited beside one that is on
    ("64x128, pairs", 500, 256, 8192), ("64x128, pairs", 257, 384, 12288), ("64x128, pairs", 321, 512, 8192),
    ("128x256", 321, 256, 20480), ("128x256", 450, 384, 10752), ("128x256", 257, 512, 16384),
    ("64x128, pairs", 500, 384, 4096), ("64x128, 2 slices", 197, 512, 8192), ("64x128, 2 slices", 390, 640, 4096),
    ("64x128, 2 slices", 321, 896, 4096), ("decode tiles", 116, 1920, 4096), ("decode tiles", 113, 2176, 3968),
]
# the same with given row sums
SUMS_SHAPES = [
    ("64x128, 2 slices", 520, 2176, 128), ("64x128, 2 slices", 577, 2048, 384), ("64x128, 2 slices", 833, 2304, 1024),
    ("64x128 kernel", 2050, 2176, 1024), ("64x128 kernel", 1100, 2176, 3072),
    ("128x256", 3969, 3072, 2048), ("128x256", 520, 1920, 12288), ("128x256", 1153, 1024, 6144),
]


def _ids(shapes):
    return [f"M{m}-K{k}-N{n}" for _, m, k, n in shapes]


def _bound(ref):
    return 2.0 ** -8 * 1.01 * ref.abs() + 1e-4 * ref.abs().max()


def _ref(x, w):
    return x.double() @ ops.dequantize(w).double().T


def _weight(k, n, seed, dev):
    return W4A16Weight.from_numpy(*ow.synthetic_tensors(k, n, seed=seed), device=dev)


def _x(m, k, seed, dev):
    return torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).to(BF16).to(dev)


@pytest.mark.parametrize("form,m,k,n", SHAPES, ids=_ids(SHAPES))
def test_linear_and_residual(gpu, form, m, k, n):
    w, x = _weight(k, n, m + k, gpu), _x(m, k, m + n, gpu)
    ref = _ref(x, w)
    y = ops.linear(x, w)
    assert ((y.double() - ref).abs() <= _bound(ref)).all(), form
    assert torch.equal(y, ops.linear(x, w)), "repeat call differs"
    res = _x(m, n, 5, gpu)
    out = res.clone()
    ops.linear(x, w, residual=out, out=out)
    assert torch.equal(out, (y.float() + res.float()).to(BF16))


@pytest.mark.parametrize("form,m,k,n", SHAPES, ids=_ids(SHAPES))
def test_paired_and_swiglu(gpu, form, m, k, n):
    gate, up = ow.synthetic_tensors(k, n // 2, seed=m), ow.synthetic_tensors(k, n // 2, seed=m + 1)
    w, x = W4A16Weight.from_numpy(*interleave_gate_up(gate, up), device=gpu), _x(m, k, m + n, gpu)
    ref = _ref(x, w)
    g, u = ops.gate_up(x, w, swiglu=False)
    assert ((g.double() - ref[:, 0::2]).abs() <= _bound(ref)[:, 0::2]).all(), form
    assert ((u.double() - ref[:, 1::2]).abs() <= _bound(ref)[:, 1::2]).all(), form
    # the epilogue on this form's own gate and up: where the fast SiLU rounds the other way, one
    # bf16 step of it (2^-7 of the value at most), and the two products' roundings (2^-9 each)
    h = ops.gate_up(x, w).float()
    chain = (torch.nn.functional.silu(g.float()).to(BF16).float() * u.float()).to(BF16).float()
    assert ((h - chain).abs() <= (2.0 ** -7 + 2.0 ** -8) * chain.abs() + 1e-30).all()
    # |g| up to 2^7 here: the exponential's fp32 argument is off by 2^-17, a relative 1e-5 of silu,
    # which crosses a bf16 boundary (2^-8 apart) in some 0.3 % of the values
    assert (h == chain).float().mean() > 0.99


@pytest.mark.parametrize("form,m,k,n", SHAPES, ids=_ids(SHAPES))
def test_equal_rows_give_equal_bits(gpu, form, m, k, n):
    """A row's result does not depend on its place in the call."""
    w, x = _weight(k, n, m + k, gpu), _x(1, k, m + n, gpu).expand(m, k).contiguous()
    y = ops.linear(x, w)
    assert torch.equal(y, y[:1].expand(m, n)), form


@pytest.mark.parametrize("form,m,k,n", SUMS_SHAPES, ids=_ids(SUMS_SHAPES))
@pytest.mark.parametrize("parts", [1, 2])
def test_given_row_sums(gpu, form, m, k, n, parts):
    w, x = _weight(k, n, m + k, gpu), _x(m, k, m + n, gpu)
    sums = x.float().view(m, -1, 128 // parts).sum(-1).t().contiguous()
    ref = _ref(x, w)
    y = ops.linear(x, w, x_sums=sums, sum_parts=parts)
    assert ((y.double() - ref).abs() <= _bound(ref)).all(), form
    x = x[:1].expand(m, k).contiguous()     # equal rows: equal bits
    y = ops.linear(x, w, x_sums=x.float().view(m, -1, 128 // parts).sum(-1).t().contiguous(), sum_parts=parts)
    assert torch.equal(y, y[:1].expand(m, n)), form


@pytest.mark.parametrize("m,k,n", [(577, 2048, 384), (2050, 2176, 1024), (520, 2048, 12288), (577, 1920, 6144)])
def test_swiglu_output_sums(gpu, m, k, n):
    """The half-group sums of h, within 1e-5 of the sum of the magnitudes (fp32, 64 terms)."""
    gate, up = ow.synthetic_tensors(k, n // 2, seed=m), ow.synthetic_tensors(k, n // 2, seed=m + 1)
    w, x = W4A16Weight.from_numpy(*interleave_gate_up(gate, up), device=gpu), _x(m, k, m + n, gpu)
    hs = torch.full((n // 128, m), float("nan"), device=gpu)
    h = ops.gate_up(x, w, out_sums=hs)
    assert torch.equal(h, ops.gate_up(x, w))
    hd = h.double().view(m, -1, 64)
    assert ((hs.double().t() - hd.sum(-1)).abs() <= 1e-5 * hd.abs().sum(-1) + 1e-30).all()


@pytest.mark.parametrize("form,m,k,n", [s for s in SHAPES if s[1] < ops.PROMPT_GEMM_ROWS and s[2] >= 1024],
                         ids=_ids([s for s in SHAPES if s[1] < ops.PROMPT_GEMM_ROWS and s[2] >= 1024]))
def test_tiles_without_the_words(gpu, form, m, k, n):
    """65 to 511 rows over the tiles alone (qweight NULL) run the decode kernel whatever the plan names:
    the reference's value within the same bar, and the same bits as a call with both where the plan is
    the decode tiles too."""
    w, x = ops.tile_weight(_weight(k, n, m + k, gpu)), _x(m, k, m + n, gpu)
    y = torch.empty(m, n, dtype=BF16, device=gpu)
    rc = _lib.load().t2i_w4a16_linear_tiles(x.data_ptr(), m, None, 0.0, None, w.tiles.data_ptr(), w.qzeros.data_ptr(),
                                            w.scales.data_ptr(), k, n, 128, _lib.T2I_TILES_STORE, None, y.data_ptr(),
                                            None, _lib.stream_handle(gpu))
    _lib.check(rc, "t2i_w4a16_linear_tiles")
    ref = _ref(x, w)
    assert ((y.double() - ref).abs() <= _bound(ref)).all()
    both = ops.linear(x, w)
    assert ((both.double() - ref).abs() <= _bound(ref)).all()
    assert form != "decode tiles" or torch.equal(y, both)


@pytest.mark.parametrize("style", [0, 1])
@pytest.mark.parametrize("b,t,p0,hq,hkv,k", [(4, 509, 3, 16, 8, 1024), (1, 520, 0, 1, 1, 2176), (5, 133, 1, 16, 8, 2048),
                                             (3, 1333, 1, 16, 8, 1024)])
def test_fused_projection_matches_two_launches(gpu, b, t, p0, hq, hkv, k, style):
    d, cap = 128, t + p0 + 5
    w, x = _weight(k, (hq + 2 * hkv) * d, t, gpu), _x(b * t, k, t + 1, gpu)
    g = torch.Generator().manual_seed(9)
    qn, kn = ((torch.rand(d, generator=g) * 0.2 + 0.9).to(BF16).to(gpu) for _ in range(2))
    rope = gm.rope_table(d, cap, 1e6, gpu)
    kc, vc, kc1, vc1 = (torch.zeros(b, hkv, cap, d, dtype=BF16, device=gpu) for _ in range(4))
    q = ops.prefill_qkv_rope_kv(x, w, b, p0, hq, hkv, qn, kn, 1e-6, rope, kc, vc, rope_style=style)
    q1 = ops.prefill_qk_rope_kv(ops.linear(x, w), b, p0, hq, hkv, qn, kn, 1e-6, rope, kc1, vc1, rope_style=style)
    assert torch.equal(q, q1) and torch.equal(kc, kc1) and torch.equal(vc, vc1)
