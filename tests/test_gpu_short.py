"""GPU parity of the short form of the single pass (gqa_fwd_short_launch,
gqa_paged_fwd_short_launch: 128 packed rows per workgroup, two wave groups
that split the keys) against the CPU oracle, where it can go wrong: tile
counts 0 to 5 (one group without a tile, an odd last step, both parities of
the stage ring), blocks of one row, groups that do not divide 128, more
queries than keys, scores that force the rescale, every page form, variable
query lengths; and against the single pass over the layouts and types a call
may come in."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import BASELINE_TOL, assert_close, make_inputs, oracle, to_np
from test_gpu_paged import LSE_TOL, _check, _paged_inputs

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


def _short(q, k, v, causal=True):
    from gqa_kernels.dispatch import short_forward
    return short_forward(q, k, v, torch.empty_like(q), causal, True)


def _compare(q, k, v, causal, o, lse):
    from oracle.gqa_oracle import gqa_lse
    ref, got = oracle(q, k, v, causal), to_np(o)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert_close(got[~nan], ref[~nan], BASELINE_TOL[q.dtype], "short")
    want, l = gqa_lse(to_np(q), to_np(k), to_np(v), causal), to_np(lse)
    fin = np.isfinite(want)
    assert np.array_equal(np.isneginf(l), ~fin)
    assert np.abs(l[fin] - want[fin]).max(initial=0.0) <= LSE_TOL


@pytest.mark.parametrize("sq,skv", [(1, 1), (5, 64), (64, 65), (33, 128), (31, 129), (200, 200), (32, 257), (100, 320),
                                    (7, 3), (65, 40)])
@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (24, 8), (5, 5), (128, 1)])
@pytest.mark.parametrize("D", [128, 64])
def test_short_shapes(sq, skv, Hq, Hkv, D):
    q, k, v = make_inputs(1, Hq, Hkv, sq, skv, D, torch.bfloat16, seed=sq + skv, device=DEV)
    for causal in (True, False):
        _compare(q, k, v, causal, *_short(q, k, v, causal))


def test_short_no_keys():
    q, k, v = make_inputs(2, 8, 2, 40, 0, 128, torch.bfloat16, device=DEV)
    o, lse = _short(q, k, v)
    assert (o == 0).all() and torch.isneginf(lse).all()


def test_short_rescale():
    """Scores that grow along the keys move every row's reference in both
    groups."""
    q, k, v = make_inputs(1, 8, 2, 150, 400, 128, torch.bfloat16, seed=9)
    k = (k.float() * torch.linspace(0.1, 4.0, 400)[:, None]).to(torch.bfloat16)
    q, k, v = q.to(DEV), k.to(DEV), v.to(DEV)
    _compare(q, k, v, True, *_short(q, k, v))


@pytest.mark.parametrize("layout", ["bhsd", "bshd", "cache"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_short_matches_single_pass(layout, dtype, causal):
    """The routed call against the 256-row single pass, over the layouts q, k
    and v come in."""
    from gqa_kernels import gqa_flash_attn
    from gqa_kernels.dispatch import _cu_count, choose_plan, single_pass_forward
    q, k, v = make_inputs(2, 32, 8, 203, 203, 128, dtype, seed=4, device=DEV)
    assert choose_plan(2, 32, 8, 203, 203, _cu_count(0), causal).kind == "short"
    if layout == "bshd":
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    elif layout == "cache":  # views of longer caches
        k, v = (torch.cat([t, torch.full_like(t, float("nan"))], 2)[:, :, :203] for t in (k, v))
    o, lse = gqa_flash_attn(q, k, v, causal, return_lse=True)
    so, slse = single_pass_forward(q, k, v, torch.empty_like(q), causal, 0, True)
    # Both round P and o once: two results differ by at most the parity gate.
    assert_close(o, so, BASELINE_TOL[dtype], "short against single")
    assert (lse - slse).abs().max().item() <= LSE_TOL
    assert o.stride() == so.stride()


@pytest.mark.parametrize("bs,hnd", [(128, True), (64, False), (32, False), (16, True), (8, False)])
@pytest.mark.parametrize("D", [128, 64])
def test_short_paged(bs, hnd, D):
    from gqa_kernels.paged import paged_attention
    L = [130, 77, 500, 64, 0, 1]
    q, kc, vc, table, seq_lens = _paged_inputs(len(L), 32, 8, 70, L, D, bs, torch.bfloat16, seed=bs, hnd=hnd)
    args = [t.to(DEV) for t in (q, kc, vc, table, seq_lens)]
    for causal in (True, False):
        o, lse = paged_attention(*args, causal, max_seq_len=max(L), return_lse=True, route="short")
        _check(o, lse, q, kc, vc, table, seq_lens, causal, torch.bfloat16)


def test_short_paged_varlen():
    from gqa_kernels.dispatch import _cu_count
    from gqa_kernels.paged import paged_attention, paged_short
    L, ql = [300, 90, 200, 333], [100, 1, 0, 77]
    q, kc, vc, table, seq_lens = _paged_inputs(len(L), 32, 8, 100, L, 128, 16, torch.bfloat16, seed=5)
    start = np.concatenate([[0], np.cumsum(ql)[:-1]]).tolist()
    q3 = torch.cat([q[b, :, :n].transpose(0, 1) for b, n in enumerate(ql)])
    assert paged_short(len(L), 32, 8, 100, max(L), _cu_count(0), True, 16)
    o, lse = paged_attention(q3.to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), seq_lens.to(DEV), True,
                             max_seq_len=max(L), return_lse=True,
                             query_start=torch.tensor(start, dtype=torch.int32, device=DEV),
                             query_lens=torch.tensor(ql, dtype=torch.int32, device=DEV), max_query_len=100)
    for b, n in enumerate(ql):
        if n:
            one = slice(b, b + 1)
            _check(o[start[b]:start[b] + n].transpose(0, 1)[None], lse[start[b]:start[b] + n].t()[None], q[one, :, :n],
                   kc, vc, table[one], seq_lens[one], True, torch.bfloat16)


def test_short_rows_far_apart():
    """K rows too far apart for 32-bit offsets take the route by shape alone
    (here the split-KV pass), as they always have."""
    from gqa_kernels import gqa_flash_attn
    from gqa_kernels.dispatch import _cu_count, choose_plan
    assert choose_plan(16, 32, 8, 16, 1100, _cu_count(0)).kind == "short"
    q, k, v = make_inputs(16, 32, 8, 16, 1100, 128, torch.bfloat16, seed=2, device=DEV)
    big = torch.empty(1100 * 900_000 + 16 * 8 * 128, dtype=torch.bfloat16, device=DEV)
    far = big.as_strided((16, 8, 1100, 128), (8 * 128, 128, 900_000, 1))
    far.copy_(k)
    assert_close(gqa_flash_attn(q, far, v), gqa_flash_attn(q, k, v), BASELINE_TOL[torch.bfloat16], "far rows")


def test_short_calls_hold_no_workspace():
    from gqa_kernels import gqa_flash_attn, gqa_split
    from gqa_kernels.dispatch import _cu_count, choose_plan
    assert choose_plan(1, 32, 8, 1024, 1024, _cu_count(0)).kind == "short"
    q, k, v = make_inputs(1, 32, 8, 1024, 1024, 128, torch.bfloat16, device=DEV)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        first, again = gqa_flash_attn(q, k, v), gqa_flash_attn(q, k, v)
    torch.cuda.synchronize()
    assert torch.equal(first, again)
    assert (torch.cuda.current_device(), s.cuda_stream) not in gqa_split._workspaces
