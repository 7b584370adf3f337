"""GPU parity of the flat split (gqa_split_flat_launch,
gqa_paged_split_flat_launch: all sequences' keys cut into equal ranges that
may cross sequences) against the CPU oracle, where its partition can go wrong:
more sequences than the 64 lanes that scan the lengths, empty sequences at
every end, lengths around one 64-key step, fewer steps than slots, one slot
for everything, one slot per sequence (the first pass writes the output),
odd groups, several tokens, head_dim 64, and variable query lengths; and
against the fixed split over the layouts and types a call may come in."""
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


def _flat(q, k, v, causal, slots, return_lse=True):
    from gqa_kernels.gqa_split import flat_forward
    return flat_forward(q, k, v, causal, slots, return_lse, torch.cuda.current_device())


@pytest.mark.parametrize("B,Hq,Hkv,sq,skv,D,slots", [
    (5, 32, 8, 1, 700, 128, 32),    # pieces cross sequences
    (5, 32, 8, 1, 700, 128, 1),     # one slot for all
    (5, 32, 8, 1, 700, 128, 5),     # one per sequence: written directly
    (5, 32, 8, 1, 700, 128, 1000),  # 55 steps, more slots than steps
    (1, 24, 8, 1, 1, 128, 1),       # one key, odd group, direct
    (3, 64, 8, 4, 65, 128, 7),      # 32 rows, two steps per sequence
    (3, 64, 8, 4, 65, 128, 3),      # ... direct
    (2, 24, 8, 5, 1500, 128, 9),    # 15 rows
    (2, 40, 8, 5, 300, 128, 5),     # 25 rows (32-row kernel), odd group
    (7, 32, 8, 1, 300, 64, 10),     # 128-key steps
    (7, 32, 8, 3, 129, 64, 7),
    (2, 8, 2, 4, 2, 128, 3),        # more queries than keys: rows without a key
])
@pytest.mark.parametrize("causal", [True, False])
def test_flat_contiguous(B, Hq, Hkv, sq, skv, D, slots, causal):
    from oracle.gqa_oracle import gqa_lse
    q, k, v = make_inputs(B, Hq, Hkv, sq, skv, D, torch.bfloat16, seed=B + skv, device=DEV)
    o, lse = _flat(q, k, v, causal, slots)
    ref, got = oracle(q, k, v, causal), to_np(o)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert_close(got[~nan], ref[~nan], BASELINE_TOL[torch.bfloat16], "flat")
    want = gqa_lse(to_np(q), to_np(k), to_np(v), causal)
    fin = np.isfinite(want)
    assert np.array_equal(np.isneginf(to_np(lse)), ~fin)
    assert np.abs(to_np(lse)[fin] - want[fin]).max() <= LSE_TOL


@pytest.mark.parametrize("layout", ["bhsd", "bshd", "cache"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sq", [1, 7])
def test_flat_matches_fixed_split(layout, dtype, sq):
    """The routed call (B = 5 takes the flat split) against the fixed split,
    over the layouts q, k and v come in."""
    from gqa_kernels import gqa_flash_attn
    from gqa_kernels.dispatch import _cu_count, choose_plan
    from gqa_kernels.gqa_split import split_kv_forward
    assert choose_plan(5, 32, 8, sq, 4000, _cu_count(0)).kind == "flat"
    q, k, v = make_inputs(5, 32, 8, sq, 4000, 128, dtype, seed=sq, device=DEV)
    if layout == "bshd":
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    elif layout == "cache":  # views of longer caches
        k, v = (torch.cat([t, torch.full_like(t, float("nan"))], 2)[:, :, :4000] for t in (k, v))
    o, lse = gqa_flash_attn(q, k, v, True, return_lse=True)
    fo, flse = split_kv_forward(q, k, v, True, 4, return_lse=True)
    # Both round P and o once: two results differ by at most the parity gate.
    assert_close(o, fo, BASELINE_TOL[dtype], "flat against fixed")
    assert (lse - flse).abs().max().item() <= LSE_TOL
    assert o.stride() == fo.stride()


def _force_flat(monkeypatch):
    """Split-KV calls take the flat split, whatever the rule says of their
    sizes; returns the slots chosen, in order."""
    from gqa_kernels import paged
    chosen = []

    def slots(batch, num_heads, num_kv_heads, seq_q, max_seq_len, cu_count, *rest):
        chosen.append(cu_count // num_kv_heads)
        return chosen[-1]

    monkeypatch.setattr(paged, "paged_flat_slots", slots)
    return chosen


LENS = {
    "crossing": [300, 1, 64, 65, 63, 2000, 128, 7],
    "empty ends": [0, 0, 500, 0, 90, 0],
    "all empty": [0, 0, 0],
    "two": [3000, 5],
    "70 sequences": [(37 * i) % 400 for i in range(70)],
    "130 sequences": [(91 * i) % 150 for i in range(130)],
}


@pytest.mark.parametrize("lens", list(LENS))
@pytest.mark.parametrize("Hq,Hkv,sq,D,bs", [(32, 8, 1, 128, 16), (64, 8, 4, 128, 64), (24, 8, 1, 64, 8),
                                          (4, 1, 2, 128, 4)])
def test_flat_paged(lens, Hq, Hkv, sq, D, bs, monkeypatch):
    from gqa_kernels.paged import paged_attention
    chosen = _force_flat(monkeypatch)
    L = LENS[lens]
    q, kc, vc, table, seq_lens = _paged_inputs(len(L), Hq, Hkv, sq, L, D, bs, torch.bfloat16, seed=len(L), hnd=bs == 64)
    mx = max(1, max(L))
    o, lse = paged_attention(*(t.to(DEV) for t in (q, kc, vc, table, seq_lens)), True, max_seq_len=mx, return_lse=True,
                             route="split")
    assert chosen and chosen[0] > 0
    if not any(L):  # (the check below takes a maximum over the finite LSEs)
        assert torch.isneginf(lse).all()
        lse = None
    _check(o, lse, q, kc, vc, table, seq_lens, True, torch.bfloat16)


def test_flat_paged_varlen(monkeypatch):
    """Variable query lengths through the flat split: sequences without query
    rows take no part, each has its own causal alignment."""
    from gqa_kernels.paged import paged_attention
    chosen = _force_flat(monkeypatch)
    L, ql = [500, 40, 0, 333, 1000, 3], [1, 4, 2, 0, 3, 3]
    B, H, Hkv, D = len(L), 32, 8, 128
    q, kc, vc, table, seq_lens = _paged_inputs(B, H, Hkv, 4, L, D, 16, torch.bfloat16, seed=3)
    start = np.concatenate([[0], np.cumsum(ql)[:-1]]).tolist()
    q3 = torch.cat([q[b, :, :n].transpose(0, 1) for b, n in enumerate(ql)])
    o, lse = paged_attention(q3.to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), seq_lens.to(DEV), True,
                             max_seq_len=max(L), return_lse=True, route="split",
                             query_start=torch.tensor(start, dtype=torch.int32, device=DEV),
                             query_lens=torch.tensor(ql, dtype=torch.int32, device=DEV), max_query_len=4)
    assert chosen and chosen[0] > 0
    for b, n in enumerate(ql):
        if n:
            one = slice(b, b + 1)
            got_o, got_l = o[start[b]:start[b] + n].transpose(0, 1)[None], lse[start[b]:start[b] + n].t()[None]
            assert L[b] or torch.isneginf(got_l).all()
            _check(got_o, got_l if L[b] else None, q[one, :, :n], kc, vc, table[one], seq_lens[one], True,
                   torch.bfloat16)


def test_flat_launch_validation():
    """Calls the flat split does not take are refused before any launch."""
    from gqa_kernels import _lib
    from gqa_kernels.gqa_split import flat_forward
    q, k, v = make_inputs(2, 32, 8, 9, 100, 128, torch.bfloat16, device=DEV)  # 36 packed rows
    assert flat_forward(q, k, v, True, 4, False, 0) is None
    q, k, v = make_inputs(2, 32, 8, 1, 100, 128, torch.bfloat16, device=DEV)
    assert flat_forward(q, k, v, True, _lib.GQA_MAX_SPLITS + 1, False, 0) is None
