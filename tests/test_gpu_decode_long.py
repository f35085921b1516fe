"""Decode attention over more splits than one merge chain takes (the parallel merge) and on the
other side of that line: one split past the bound, a ragged last slice of states, empty splits
(short positions in a long cache), every q-head count a kv head, against float64 attention on
the device; the entry points of the same attention give the same bits.

Tolerance: one bf16 rounding of the true value (2^-9 relative, doubled for a value at a
rounding boundary) plus 1e-5 of the largest output (fp32 scores, exponentials and sums)."""

import math

import pytest
import torch

from torch2iron_amd import _lib
from torch2iron_amd import model as gm
from torch2iron_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

# chunks of 128 slots (1 and 2 q heads a kv head), 64 (4) and 32 (8); more than 256 (sequence, kv
# head) pairs keep the chain up to 63 splits
CASES = [(1, 2, 2, 128 * 33, [128 * 33 - 1]), (2, 4, 2, 128 * 37 + 5, [4000, 128 * 37 + 4]),
         (1, 4, 1, 64 * 70 + 1, [64 * 70]), (3, 8, 2, 64 * 33, [7, 2000, 64 * 33 - 1]),
         (2, 8, 1, 32 * 50 + 3, [0, 32 * 50 + 2]), (1, 8, 2, 64 * 200, [-1]),
         (130, 4, 2, 128 * 33, [128 * 33 - 1 - 32 * i for i in range(130)]),
         (257, 8, 1, 32 * 62 + 3, [5 + 7 * i for i in range(257)]),
         (257, 8, 1, 32 * 63 + 3, [32 * 63 + 2 - 7 * i for i in range(257)])]
IDS = [f"B{c[0]}-H{c[1]}-{c[2]}-cap{c[3]}" for c in CASES]


def _reference(q, kc, vc, positions, hq, hkv, rows):
    d, q_per = 128, hq // hkv
    ref = torch.zeros(len(rows), hq, d, dtype=torch.float64, device=q.device)
    for n, i in enumerate(rows):
        p = positions[i]
        if p < 0:
            continue   # outside the cache: a zero row
        for h in range(hq):
            sc = kc[i, h // q_per, :p + 1].double() @ q.view(-1, hq, d)[i, h].double() / math.sqrt(d)
            ref[n, h] = torch.softmax(sc, 0) @ vc[i, h // q_per, :p + 1].double()
    return ref


def _check(out, ref, rows, hq):
    err = (out.view(-1, hq, 128)[rows].double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 1e-5 * ref.abs().max()).all(), f"worst {err.max():.3e}"


def _inputs(b, hq, hkv, cap, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    q, k, v = (torch.randn(b, n * 128, generator=g, device=dev).to(BF16) for n in (hq, hkv, hkv))
    kc, vc = (torch.randn(b, hkv, cap, 128, generator=g, device=dev).to(BF16) for _ in range(2))
    return q, k, v, kc, vc


@pytest.mark.parametrize("b,hq,hkv,cap,positions", CASES, ids=IDS)
def test_many_splits(gpu, b, hq, hkv, cap, positions):
    q, k, v, kc, vc = _inputs(b, hq, hkv, cap, gpu, cap + hq)
    pos = torch.tensor(positions, dtype=torch.int32, device=gpu)
    ws = ops.Workspace()
    outs = [ops.decode_attention_prepared(q, k, v, pos, hq, hkv, kc, vc, workspace=ws).clone() for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), "repeat calls differ"
    rows = list(range(0, b, max(1, b // 5)))
    _check(outs[0], _reference(q, kc, vc, positions, hq, hkv, rows), rows, hq)


def test_one_workspace_for_both_merges(gpu):
    """Long and short caches in turn on one workspace: each call finds it as the calls before left it."""
    b, hq, hkv = 3, 8, 2
    lib = _lib.load()
    calls = []
    for cap in (64 * 70 + 1, 64 * 20, 64 * 33):
        q, k, v, kc, vc = _inputs(b, hq, hkv, cap, gpu, cap)
        positions = [cap - 1, cap // 2, 3]
        pos = torch.tensor(positions, dtype=torch.int32, device=gpu)
        calls.append((q, k, v, pos, kc, vc, cap, positions, lib.t2i_decode_attention_workspace_bytes(b, hq, hkv, cap)))
    ws = torch.zeros(max(c[-1] for c in calls), dtype=torch.uint8, device=gpu)
    for _ in range(2):
        for q, k, v, pos, kc, vc, cap, positions, nbytes in calls:
            out = torch.full((b, hq * 128), 7.0, dtype=BF16, device=gpu)
            _lib.check(lib.t2i_decode_attention_prepared(q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), b, hq,
                                                         hkv, 128, kc.data_ptr(), vc.data_ptr(), cap, out.data_ptr(),
                                                         ws.data_ptr(), nbytes, _lib.stream_handle(gpu)), "attention")
            _check(out, _reference(q, kc, vc, positions, hq, hkv, [0, 1, 2]), [0, 1, 2], hq)


@pytest.mark.parametrize("b,hq,hkv,cap,positions", CASES[1:5], ids=IDS[1:5])
def test_entry_points_agree(gpu, b, hq, hkv, cap, positions):
    """t2i_decode_attention on its workspace and on the library's scratch, and the prepared entry point
    on the q and k that they norm and rotate."""
    q, k, v, kc, vc = _inputs(b, hq, hkv, cap, gpu, cap + 1)
    pos = torch.tensor(positions, dtype=torch.int32, device=gpu)
    qn, kn = (torch.rand(128, device=gpu).mul(0.2).add(0.9).to(BF16) for _ in range(2))
    rope = gm.rope_table(128, cap, 1e6, gpu)
    qkv = torch.cat((q, k, v), 1).contiguous()
    caches = [(kc.clone(), vc.clone()) for _ in range(3)]
    out = ops.decode_attention(qkv, pos, hq, hkv, qn, kn, 1e-6, rope, *caches[0], workspace=ops.Workspace())
    lib = _lib.load()
    out1 = torch.full_like(out, 7.0)
    _lib.check(lib.t2i_decode_attention_noalloc(qkv.data_ptr(), pos.data_ptr(), b, hq, hkv, 128, qn.data_ptr(),
                                                kn.data_ptr(), 1e-6, rope.data_ptr(), 0, caches[1][0].data_ptr(),
                                                caches[1][1].data_ptr(), cap, out1.data_ptr(), _lib.stream_handle(gpu)),
               "noalloc")
    ang = rope[pos.long()].contiguous()
    qr = ops.rmsnorm_rope(q.view(b * hq, 128), qn, ang, 1e-6).view(b, -1)
    kr = ops.rmsnorm_rope(k.view(b * hkv, 128), kn, ang, 1e-6).view(b, -1)
    out2 = ops.decode_attention_prepared(qr, kr, v, pos, hq, hkv, *caches[2], workspace=ops.Workspace())
    rows = list(range(b))
    for o, (kc1, vc1) in ((out, caches[0]), (out1, caches[1]), (out2, caches[2])):
        assert torch.equal(o, out) and torch.equal(kc1, caches[0][0]) and torch.equal(vc1, caches[0][1])
    _check(out, _reference(qr, *caches[0], positions, hq, hkv, rows), rows, hq)
