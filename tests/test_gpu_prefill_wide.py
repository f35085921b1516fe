"""Prompt attention with two row sets a wave (blocks of 128 rows) and, beside it, with one: one
row, ragged last blocks, one key block and many, every q-head count a kv head, against float64
attention on the device.  Which of the two a case runs is checked on the host
(test_prefill_plan).

Tolerance: bf16 keeps 8 significant bits, so one rounding is up to 2^-8 of the value.  The
weights are rounded and divided by the sum of the rounded ones: 2^-8 (sum p |v| + |o|); the
output is rounded once more: 2^-8 |o|; 1e-5 of the largest output for fp32 scores,
exponentials and sums."""

import math

import pytest
import torch

from torch2iron_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

# two row sets a wave or one (csrc/prefill_plan.h), B, rows, first position, kv heads, q heads a kv head
CASES = [(False, 100, 1, 0, 8, 1), (False, 99, 1, 0, 8, 1), (False, 20, 600, 0, 8, 1), (False, 13, 500, 0, 8, 2),
         (False, 51, 3, 500, 8, 4), (False, 9, 129, 3001, 8, 4), (True, 26, 61, 1500, 4, 8), (False, 60, 65, 63, 8, 2),
         (True, 52, 255, 100, 8, 1), (True, 64, 97, 100, 8, 2), (True, 64, 127, 63, 8, 2), (True, 16, 512, 0, 8, 2),
         (True, 63, 33, 500, 8, 4), (True, 256, 15, 500, 4, 8), (False, 100, 8, 200, 4, 8)]


@pytest.mark.parametrize("b,t,p0,hkv,q_per", [c[1:] for c in CASES],
                         ids=["B%d-T%d-p%d-H%dx%d" % c[1:] for c in CASES])
def test_prompt_attention(gpu, b, t, p0, hkv, q_per):
    d, hq, n = 128, hkv * q_per, p0 + t
    g = torch.Generator(device=gpu).manual_seed(b * 1000 + t)
    q = torch.randn(b, hq, t, d, generator=g, device=gpu).to(BF16)
    kc, vc = (torch.randn(b, hkv, n + 3, d, generator=g, device=gpu).to(BF16) for _ in range(2))
    kc[:, :, n:], vc[:, :, n:] = float("nan"), float("nan")      # slots past the prompt carry nothing
    kc[:, :, n // 2] *= 4.0                                      # a new maximum after the first blocks
    sums = torch.empty(hq, b * t, dtype=torch.float32, device=gpu)
    out = ops.prefill_attention(q, p0, hkv, kc, vc, out_sums=sums)
    assert torch.equal(out, ops.prefill_attention(q, p0, hkv, kc, vc)), "repeat calls differ"
    got = out.view(b, t, hq, d).double()
    mask = torch.arange(n, device=gpu)[None, :] > p0 + torch.arange(t, device=gpu)[:, None]
    for i in range(0, b, max(1, b // 5)):
        for h in range(hq):
            sc = (q[i, h].double() @ kc[i, h // q_per, :n].double().T.contiguous()) / math.sqrt(d)
            p = torch.softmax(sc.masked_fill(mask, -math.inf), 1)
            v = vc[i, h // q_per, :n].double()
            ref, mag = p @ v, p @ v.abs()
            err = (got[i, :, h] - ref).abs()
            assert (err <= 2.0 ** -8 * (mag + 2 * ref.abs()) + 1e-5 * ref.abs().max()).all(), \
                f"sequence {i} head {h}: worst {err.max():.3e}"
    want = got.sum(-1).permute(2, 0, 1).reshape(hq, b * t)
    assert (sums.double() - want).abs().max() <= 128 * 2.0 ** -24 * got.abs().sum(-1).max()
