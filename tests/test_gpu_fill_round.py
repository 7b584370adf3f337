"""GPU parity of the single pass without a mask where the last round's query
blocks run as two key halves, placed after the whole blocks (gqa_fwd.hip
decode, dispatch._fill_last_round): against the CPU oracle, with pairs dealt
to the XCDs (batch * kv heads a multiple of 8) and not, one key tile to
several, ragged rows, and every block split."""
from __future__ import annotations

import pytest
import torch

from helpers import BASELINE_TOL, assert_close, make_inputs, oracle, to_np
from oracle.gqa_oracle import gqa_lse

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("B,Hkv", [(1, 8), (2, 8), (3, 8), (3, 4)])
@pytest.mark.parametrize("sq,skv", [(1, 1), (64, 64), (65, 129), (257, 200), (385, 700)])
def test_split_blocks_without_a_mask(B, Hkv, sq, skv, D):
    from gqa_kernels.dispatch import single_pass_forward
    q, k, v = make_inputs(B, 4 * Hkv, Hkv, sq, skv, D, torch.float16, seed=B + sq, device=DEV)
    ref = oracle(q, k, v, False)
    ref_lse = gqa_lse(to_np(q), to_np(k), to_np(v), False)
    n = -(-sq // 64)
    for ns in sorted({0, 1, n // 2, n}):
        print(f"B={B} Hkv={Hkv} {sq}x{skv} D={D} split={ns}", flush=True)
        o, lse = single_pass_forward(q, k, v, torch.empty_like(q), False, ns, True)
        torch.cuda.synchronize()
        assert_close(o, ref, BASELINE_TOL[torch.float16], f"split={ns}")
        # (fp32 sums of at most 700 terms and the device's log2 / exp2)
        assert abs(to_np(lse) - ref_lse).max() < 2e-3


@pytest.mark.parametrize("B,S,D", [(4, 1025, 128), (4, 1025, 64), (1, 2304, 128)])
def test_default_route_fills_the_last_round(B, S, D):
    from gqa_kernels import gqa_flash_attn
    from gqa_kernels.dispatch import _cu_count, choose_plan
    plan = choose_plan(B, 32, 8, S, S, _cu_count(0), False, D)
    q, k, v = make_inputs(B, 32, 8, S, S, D, torch.float16, seed=S, device=DEV)
    print(f"B={B} S={S} D={D} {plan}", flush=True)
    assert plan.kind == "single" and (plan.fwd_split > 0 or _cu_count(0) != 256)
    outs = [gqa_flash_attn(q, k, v, causal=False) for _ in range(4)]
    torch.cuda.synchronize()
    rows = sorted({0, 63, 64, S // 2, S - 65, S - 2, S - 1})
    ref = oracle(q[:, :, rows].contiguous(), k, v, False)
    assert_close(outs[0][:, :, rows], ref, BASELINE_TOL[torch.float16], f"{plan}")
    for o in outs[1:]:
        assert torch.equal(o, outs[0])


@pytest.mark.parametrize("B,Hkv", [(2, 8), (3, 8), (8, 2), (3, 4)])
@pytest.mark.parametrize("sq,skv", [(64, 64), (129, 200), (333, 333), (900, 900)])
def test_dealt_fixed_lists(B, Hkv, sq, skv):
    """Causal, head_dim 128: pairs dealt to the XCDs in the persistent
    kernel's fixed lists (16 and 24 pairs; 12 not), with split blocks."""
    from gqa_kernels.dispatch import single_pass_forward
    q, k, v = make_inputs(B, 4 * Hkv, Hkv, sq, skv, 128, torch.bfloat16, seed=B * 5 + sq, device=DEV)
    ref = oracle(q, k, v)
    n = -(-sq // 64)
    for ns in sorted({0, 1, n // 2, n}):
        print(f"dealt B={B} Hkv={Hkv} {sq}x{skv} split={ns}", flush=True)
        o, _ = single_pass_forward(q, k, v, torch.empty_like(q), True, ns, True)
        torch.cuda.synchronize()
        assert_close(o, ref, BASELINE_TOL[torch.bfloat16], f"split={ns}")


@pytest.mark.parametrize("B,S", [(1, 2500), (2, 1700)])
def test_head_dim_64_heaviest_blocks_split(B, S):
    from gqa_kernels import gqa_flash_attn
    from gqa_kernels.dispatch import _cu_count, choose_plan
    plan = choose_plan(B, 32, 8, S, S, _cu_count(0), True, 64)
    assert plan.kind == "single" and (plan.fwd_split > 0 or _cu_count(0) != 256)
    q, k, v = make_inputs(B, 32, 8, S, S, 64, torch.float16, seed=S, device=DEV)
    print(f"B={B} S={S} {plan}", flush=True)
    o = gqa_flash_attn(q, k, v)
    torch.cuda.synchronize()
    assert_close(o, oracle(q, k, v), BASELINE_TOL[torch.float16], f"{plan}")
