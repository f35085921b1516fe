"""Decode attention over more splits than one merge chain takes (the parallel merge):
one split past the bound, a ragged last slice of states, empty splits (short positions in
a long cache), every q-head count a kv head, against float64 attention on the device.

Tolerance: one bf16 rounding of the true value (2^-9 relative, doubled for a value at a
rounding boundary) plus 1e-5 of the largest output (fp32 scores, exponentials and sums)."""

import math

import pytest
import torch

from torch2iron_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

# chunks of 128 slots (1 and 2 q heads a kv head), 64 (4) and 32 (8)
CASES = [(1, 2, 2, 128 * 33, [128 * 33 - 1]), (2, 4, 2, 128 * 37 + 5, [4000, 128 * 37 + 4]),
         (1, 4, 1, 64 * 70 + 1, [64 * 70]), (3, 8, 2, 64 * 33, [7, 2000, 64 * 33 - 1]),
         (2, 8, 1, 32 * 50 + 3, [0, 32 * 50 + 2]), (1, 8, 2, 64 * 200, [-1])]


@pytest.mark.parametrize("b,hq,hkv,cap,positions", CASES, ids=[f"B{c[0]}-H{c[1]}-{c[2]}-cap{c[3]}" for c in CASES])
def test_many_splits(gpu, b, hq, hkv, cap, positions):
    d, q_per = 128, hq // hkv
    g = torch.Generator().manual_seed(cap + hq)
    q, k, v = (torch.randn(b, n * d, generator=g).to(BF16).to(gpu) for n in (hq, hkv, hkv))
    kc, vc = (torch.randn(b, hkv, cap, d, generator=g).to(BF16).to(gpu) for _ in range(2))
    pos = torch.tensor(positions, dtype=torch.int32, device=gpu)
    ws = ops.Workspace()
    outs = [ops.decode_attention_prepared(q, k, v, pos, hq, hkv, kc, vc, workspace=ws).clone() for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), "repeat calls differ"
    for buf in ws._bufs.values():
        assert torch.count_nonzero(buf[:b * hkv * 4]).item() == 0, "arrival counters not reset"
    ref = torch.zeros(b, hq, d, dtype=torch.float64, device=gpu)
    for i, p in enumerate(positions):
        if p < 0:
            continue   # outside the cache: a zero row
        for h in range(hq):
            sc = kc[i, h // q_per, :p + 1].double() @ q.view(b, hq, d)[i, h].double() / math.sqrt(d)
            ref[i, h] = torch.softmax(sc, 0) @ vc[i, h // q_per, :p + 1].double()
    err = (outs[0].view(b, hq, d).double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 1e-5 * ref.abs().max()).all(), f"worst {err.max():.3e}"
