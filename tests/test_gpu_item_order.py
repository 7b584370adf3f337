"""GPU parity of the single pass and its short form where their work items are
dealt over the XCDs (item_of in gqa_fwd_parts.hpp) against the CPU oracle:
batch * kv heads 16, 24 and 32 (two to four pairs per XCD), beside 8 and 12
(pair after pair), one to several query blocks, split blocks, LSE, and ragged
paged batches; and at sizes on both sides of the lines of set_item_order,
against the same sequences alone."""
from __future__ import annotations

import pytest
import torch

from helpers import BASELINE_TOL, assert_close, make_inputs, oracle
from test_gpu_paged import _check, _paged_inputs

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


@pytest.mark.parametrize("B,Hkv", [(1, 8), (2, 8), (3, 8), (4, 8), (3, 4), (8, 2), (5, 8)])
@pytest.mark.parametrize("sq", [64, 129, 333])
def test_single_pass_order(B, Hkv, sq):
    from gqa_kernels.dispatch import single_pass_forward
    q, k, v = make_inputs(B, 4 * Hkv, Hkv, sq, sq + 70, 64, torch.bfloat16, seed=B * 7 + sq, device=DEV)
    ref = oracle(q, k, v)
    for n_split in sorted({0, 1, -(-sq // 64)}):
        print(f"single B={B} Hkv={Hkv} sq={sq} n_split={n_split}", flush=True)
        o, _ = single_pass_forward(q, k, v, torch.empty_like(q), True, n_split, True)
        torch.cuda.synchronize()
        assert_close(o, ref, BASELINE_TOL[torch.bfloat16], f"B={B} Hkv={Hkv} sq={sq} split={n_split}")


@pytest.mark.parametrize("route,splits", [("single", 0), ("single", 3), ("chunks", 4), ("short", None)])
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("lens", [[700, 130], [180, 640, 0], [333, 131, 200, 500], [140, 1, 260, 600, 133]])
def test_ragged_paged_order(lens, D, route, splits):
    from gqa_kernels.paged import paged_attention
    q, kc, vc, table, seq_lens = _paged_inputs(len(lens), 32, 8, 131, lens, D, 16, torch.bfloat16, seed=len(lens))
    args = [t.to(DEV) for t in (q, kc, vc, table, seq_lens)]
    print(f"paged {lens} D={D} {route} {splits}", flush=True)
    o, lse = paged_attention(*args, True, max_seq_len=max(lens), return_lse=True, route=route, splits=splits)
    torch.cuda.synchronize()
    _check(o, lse, q, kc, vc, table, seq_lens, True, torch.bfloat16)


@pytest.mark.parametrize("B,D,sq", [(3, 64, 800), (2, 64, 2100), (24, 64, 200), (25, 64, 200), (32, 64, 200),
                                    (33, 64, 200), (3, 128, 900), (12, 128, 333), (13, 128, 333),
                                    (24, 128, 333), (25, 128, 333)])
@pytest.mark.parametrize("causal,n_split", [(True, 0), (True, 2), (False, 0), (False, 2)])
def test_order_does_not_change_results(B, D, sq, causal, n_split):
    """More items than CUs, on both sides of the line where pairs are dealt: each
    sequence of the batch has the bits that it has alone (eight pairs, pair after
    pair)."""
    from gqa_kernels.dispatch import single_pass_forward
    print(f"order B={B} D={D} sq={sq} causal={causal} n_split={n_split}", flush=True)
    q, k, v = make_inputs(B, 32, 8, sq, sq + 70, D, torch.bfloat16, seed=B + sq, device=DEV)
    o, lse = single_pass_forward(q, k, v, torch.empty_like(q), causal, n_split, True)
    for b in range(0, B, 1 if B < 4 else 5):
        one = [t[b:b + 1] for t in (q, k, v)]
        ob, lb = single_pass_forward(*one, torch.empty_like(one[0]), causal, n_split, True)
        torch.cuda.synchronize()
        assert torch.equal(o[b:b + 1], ob) and torch.equal(lse[b:b + 1], lb), b
