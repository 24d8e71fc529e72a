"""Causal walks cut by length where equal parts left them whole (``causal_splits`` in dispatch.cpp),
and decode at the edges of its automatic split counts, on the GPU (marker ``gpu``).

Causal grids: tiles of 32 and 64 rows, forced heights, GQA, a last query tile and a last key tile
that are not full, more than one batch, contiguous operands and views of a packed projection. Every
head is compared with plain fp32 attention at the op's tolerance, O and LSE.

Decode: the last cache that stays one split and the first that does not at each head dim and where
half the CUs are busy, single-tile splits, the count where a split keeps four tiles, both sides of
two workgroups per CU at D = 64 and of two rounds; each against the fp64 decode oracle.
"""

from __future__ import annotations

import math

import pytest
import torch

import fused_attn
from _checks import LSE_ATOL, O_TOL, assert_close_tol, assert_every_head_close
from fused_attn import capi
from oracle.oracle import decode_reference

pytestmark = pytest.mark.gpu


def _randn(gen, dtype, *shape):
    return torch.randn(*shape, generator=gen).to("cuda", dtype)


@pytest.mark.parametrize("b,h,hkv,n,d,dtype", [
    (1, 5, 5, 2048, 128, torch.float16),
    (2, 3, 1, 1568, 128, torch.bfloat16),   # 49 tiles of 32 rows, GQA, ragged last key tile
    (1, 6, 2, 3008, 128, torch.float16),    # 47 tiles of 64 rows
    (1, 3, 3, 4128, 64, torch.bfloat16),
], ids=lambda x: str(x).replace("torch.", ""))
def test_causal_walks_cut_by_length(b, h, hkv, n, d, dtype, monkeypatch):
    monkeypatch.delenv("FA_FORCE_SPLITS", raising=False)
    gen = torch.Generator().manual_seed(n + h)
    packed = _randn(gen, dtype, b, n, (h + 2 * hkv) * d)
    views = tuple(x.view(b, n, -1, d).transpose(1, 2)
                  for x in packed.split((h * d, hkv * d, hkv * d), dim=-1))
    q, k, v = (x.contiguous() for x in views)
    scale = 1.0 / math.sqrt(d)
    assert capi.workspace_bytes(5, q, k, True, scale) > 0, "the walks should be cut here"
    o, lse = fused_attn.forward_stage(q, k, v, 5, is_causal=True)
    assert_every_head_close(o, lse, q, k, v, True, scale)
    assert torch.equal(fused_attn.forward_strided(*views, is_causal=True), o)


@pytest.mark.parametrize("br", [32, 64, 128])
@pytest.mark.parametrize("n", [2048, 2080])
def test_causal_parts_at_forced_heights(br, n, monkeypatch):
    """The parts of a forced height, in the workspace of the chosen one."""
    monkeypatch.delenv("FA_FORCE_SPLITS", raising=False)
    gen = torch.Generator().manual_seed(br + n)
    q, k, v = (_randn(gen, torch.bfloat16, 1, 5, n, 128) for _ in range(3))
    scale = 1.0 / math.sqrt(128)
    assert capi.workspace_bytes(5, q, k, True, scale) > 0, "the walks should be cut here"
    fused_attn.set_debug_overrides(br, 0)
    try:
        o, lse = fused_attn.forward_stage(q, k, v, 5, is_causal=True)
    finally:
        fused_attn.set_debug_overrides(0, 0)
    assert_every_head_close(o, lse, q, k, v, True, scale)


@pytest.mark.parametrize("b,hkv,group,nq,nkv,d", [
    (1, 8, 4, 1, 768, 128), (1, 8, 4, 1, 769, 128),     # one split, seven of a tile each
    (4, 32, 1, 2, 896, 128), (4, 32, 1, 2, 897, 128),   # 128 groups: one
    (4, 32, 1, 2, 1152, 128), (4, 32, 1, 2, 1153, 128), # and here one, two
    (3, 12, 2, 5, 896, 64), (3, 12, 2, 5, 897, 64),     # D = 64: one
    (3, 12, 2, 5, 1024, 64), (3, 12, 2, 5, 1025, 64),   # and here one, five
    (1, 1, 8, 1, 17000, 128),                           # 33 splits of four tiles and one more
    (8, 8, 4, 2, 8192, 64),                             # eight, two workgroups per CU
    (3, 12, 2, 1, 4096, 64), (3, 12, 2, 1, 4632, 64),   # seven
    (4, 10, 2, 1, 8064, 64), (4, 10, 2, 1, 8065, 64),   # 63 tiles: six, 64: twelve, two per CU
    (10, 13, 1, 1, 6016, 128), (10, 13, 1, 1, 6017, 128),  # 130 groups: one, three in two rounds
    (10, 17, 33, 1, 6017, 64),                          # 170, 8-wave workgroups: three
    (9, 8, 6, 8, 7680, 64),                             # three, 8-wave workgroups
    (15, 17, 1, 1, 1100, 128),                          # 255 groups: one
], ids=lambda x: str(x))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
def test_decode_automatic_splits(b, hkv, group, nq, nkv, d, dtype):
    gen = torch.Generator().manual_seed(nkv)
    q = _randn(gen, dtype, b, hkv * group, nq, d)
    k, v = (_randn(gen, dtype, b, hkv, nkv, d) for _ in range(2))
    o, lse = fused_attn.decode(q, k, v, is_causal=True)
    atol, rtol = O_TOL[dtype]
    ref, lse64 = decode_reference(q, k, v, is_causal=True)
    assert_close_tol(o, ref, atol, rtol)
    assert_close_tol(lse.double().cpu().numpy(), lse64, LSE_ATOL, 0.0, what="LSE")
