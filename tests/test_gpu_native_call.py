"""The native whole calls (gqa_host.cpp flash_attn, paged_attn, write_kv)
against the Python path they stand in for: the first call of a shape runs in
Python and registers its route, later ones run natively and give the same
bits on every route, also on another stream and under graph capture; calls
they do not take (unaligned rows, tensor subclasses) fall to Python, and
wrong arguments raise as before once the shape is planned."""
from __future__ import annotations

import pytest
import torch

from helpers import make_inputs
from test_gpu_paged import _paged_inputs

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from gqa_kernels import _lib
    _lib.load_host()


def _python_only(monkeypatch):
    """Calls take the Python path (the launches still go through the bindings)."""
    from gqa_kernels import _lib

    class Bindings:
        def __init__(self, host):
            self._host = host

        def flash_attn(self, *a):
            return None

        paged_attn = flash_attn

        def write_kv(self, *a):
            return False

        def __getattr__(self, name):
            return getattr(self._host, name)

    monkeypatch.setattr(_lib, "_host", Bindings(_lib._host))


# split, flat, flat with one slot per sequence, short, chunks, single with and
# without split blocks
SHAPES = [(1, 32, 8, 1, 3000, 128), (5, 32, 8, 1, 4000, 128), (64, 32, 8, 1, 300, 64), (2, 32, 8, 150, 150, 128),
          (1, 32, 8, 64, 5000, 128), (2, 8, 2, 3000, 3000, 64), (2, 32, 8, 1100, 1100, 128)]


def test_shapes_cover_the_kinds():
    from gqa_kernels.dispatch import _KIND_IDS, _cu_count, choose_plan
    plans = [choose_plan(*s[:5], _cu_count(0), True, s[5]) for s in SHAPES]
    assert {p.kind for p in plans} == set(_KIND_IDS)
    assert {p.fwd_split > 0 for p in plans if p.kind == "single"} == {True, False}
    assert {p.splits == s[0] for p, s in zip(plans, SHAPES) if p.kind == "flat"} == {True, False}


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("lse", [False, True])
def test_same_bits(shape, lse, monkeypatch):
    from gqa_kernels import _lib, gqa_flash_attn
    from gqa_kernels import gqa_split
    q, k, v = make_inputs(*shape, torch.bfloat16, seed=1, device=DEV)
    gqa_flash_attn(q, k, v)  # planned from here on
    native = _lib._host.flash_attn(q, k, v, True, lse, gqa_split._workspaces, gqa_split._counters)
    assert native is not None
    with monkeypatch.context() as m:
        _python_only(m)
        ref = gqa_flash_attn(q, k, v, return_lse=lse)
    for a, b in zip(native if lse else (native,), ref if lse else (ref,)):
        assert torch.equal(a, b) and a.stride() == b.stride() and a.dtype == b.dtype


def test_other_stream_and_capture():
    """A stream without buffers falls to Python, which makes them; a captured
    call replays to the eager bits."""
    from gqa_kernels import gqa_flash_attn
    for shape in SHAPES:
        q, k, v = make_inputs(*shape, torch.bfloat16, seed=2, device=DEV)
        want = gqa_flash_attn(q, k, v)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for _ in range(2):
                assert torch.equal(gqa_flash_attn(q, k, v), want)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = gqa_flash_attn(q, k, v)
        for _ in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            gqa_flash_attn(q, k, v)


def test_refused_and_python_calls():
    from gqa_kernels import gqa_flash_attn
    q, k, v = make_inputs(2, 32, 8, 150, 150, 128, torch.bfloat16, seed=3, device=DEV)
    want = gqa_flash_attn(q, k, v)
    # rows off 16 bytes: copied
    odd = torch.empty(k.numel() + 1, dtype=k.dtype, device=DEV)[1:].view_as(k)
    odd.copy_(k)
    assert torch.equal(gqa_flash_attn(q, odd, v), want)
    # a tensor subclass

    class Sub(torch.Tensor):
        pass

    assert torch.equal(gqa_flash_attn(q.as_subclass(Sub), k, v).as_subclass(torch.Tensor), want)
    for args in ((q, k, v[:, :4]), (q, k.half(), v), (q.float(), k.float(), v.float()), (q, k.cpu(), v.cpu()),
                 (q[:, :31], k, v)):
        with pytest.raises(AssertionError):
            gqa_flash_attn(*args)


# (lengths, query tokens, keyword arguments, kind): the flat split, the fixed
# count, the short form, key chunks, the single pass without and with split
# blocks.
PAGED = [([6000, 40, 2000, 1000, 700, 2500], 1, "flat"), ([2000], 1, "split"), ([300, 200], 150, "short"),
         ([3000, 3000], 40, "chunks"), ([700, 650, 600, 500], 400, "single"), ([2000, 1500, 1999, 30] * 2, 300, "halves")]


def _paged_kind(lens, sq):
    from gqa_kernels.dispatch import _cu_count
    from gqa_kernels.paged import paged_flat_slots, paged_route, paged_short, paged_single_plan
    args = (len(lens), 32, 8, sq, max(lens), _cu_count(0))
    if paged_short(*args, True, 16):
        return "short"
    if paged_route(32, 8, sq, 16) == "split":
        return "flat" if paged_flat_slots(*args, 16, 128, True) else "split"
    chunks, halves = paged_single_plan(*args)
    return "chunks" if chunks else "halves" if halves else "single"


def _native_paged(q, kc, vc, table, seq_lens, max_seq_len, lse, out=None, qs=None, ql=None, max_query_len=-1):
    from gqa_kernels import _lib, gqa_split
    return _lib._host.paged_attn(q, kc, vc, table, seq_lens, True, max_seq_len, 128 ** -0.5 * gqa_split.LOG2E, lse, out,
                                 qs, ql, max_query_len, gqa_split._workspaces, gqa_split._counters)


@pytest.mark.parametrize("lse", [False, True])
@pytest.mark.parametrize("varlen", [False, True])
@pytest.mark.parametrize("lens,sq,kind", PAGED)
def test_paged_same_bits(lens, sq, kind, varlen, lse, monkeypatch):
    """The native call of a planned shape, asked for directly, gives the bits and
    the layout of the Python path; token-major queries of unequal counts too."""
    from gqa_kernels.paged import paged_attention
    assert _paged_kind(lens, sq) == kind
    q, kc, vc, table, seq_lens = (t.to(DEV) for t in _paged_inputs(len(lens), 32, 8, sq, lens, 128, 16, torch.bfloat16,
                                                                   seed=4))
    kw, native_kw = {}, {}
    if varlen:
        n = [max(0, sq - 3 * b) if b != 1 else sq for b in range(len(lens))]
        ql = torch.tensor(n, dtype=torch.int32, device=DEV)
        qs = torch.tensor([sum(n[:b]) for b in range(len(n))], dtype=torch.int32, device=DEV)
        q = torch.cat([q[b, :, :m].transpose(0, 1) for b, m in enumerate(n)]).contiguous()
        kw = dict(query_start=qs, query_lens=ql, max_query_len=sq)
        native_kw = dict(qs=qs, ql=ql, max_query_len=sq)
    mx = max(lens)
    with monkeypatch.context() as m:
        _python_only(m)
        ref = paged_attention(q, kc, vc, table, seq_lens, max_seq_len=mx, return_lse=lse, **kw)
    out = torch.empty_like(q)
    for o in (None, out):
        native = _native_paged(q, kc, vc, table, seq_lens, mx, lse, o, **native_kw)
        assert native is not None, "the native call did not take a planned shape"
        for a, b in zip(native if lse else (native,), ref if lse else (ref,)):
            assert torch.equal(torch.nan_to_num(a.float()), torch.nan_to_num(b.float()))
            assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype
    assert (native[0] if lse else native).data_ptr() == out.data_ptr()


def test_write_kv_same_bytes_and_refused_paged_calls(monkeypatch):
    from gqa_kernels import _lib
    from gqa_kernels.paged import paged_attention, write_kv
    lens = [300, 40, 1000]
    q, kc, vc, table, seq_lens = (t.to(DEV) for t in _paged_inputs(3, 32, 8, 1, lens, 128, 16, torch.bfloat16, seed=4))
    new = torch.randn(3, 8, 128, device=DEV).to(torch.bfloat16)
    slots = torch.tensor([int(table[0, 0]) * 16 + 5, -1, int(table[0, 0]) * 16 + 6], device=DEV)
    k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    with monkeypatch.context() as m:
        _python_only(m)
        write_kv(new, new, k1, v1, slots)
    assert _lib._host.write_kv(new, new, k2, v2, slots) is True
    for a, b in ((k1, k2), (v1, v2)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    paged_attention(q, kc, vc, table, seq_lens, max_seq_len=1000)
    for bad in (dict(max_seq_len=10 ** 6), dict(out=torch.empty(1, device=DEV))):
        with pytest.raises(AssertionError):
            paged_attention(q, kc, vc, table, seq_lens, **bad)
    with pytest.raises(AssertionError):
        paged_attention(q, kc, vc, table.long(), seq_lens, max_seq_len=1000)


def test_strides_of_one_call_do_not_plan_the_shape():
    """A cache whose slots lie too far apart for the short form: the shape is
    planned by the next ordinary cache, not by the route that this one takes."""
    from gqa_kernels.dispatch import _cu_count
    from gqa_kernels.paged import paged_attention, paged_short
    lens, sq, bs = [301, 250, 90], 45, 4
    q, kc, vc, table, seq_lens = (t.to(DEV) for t in _paged_inputs(3, 32, 8, sq, lens, 128, bs, torch.bfloat16, seed=8))
    assert paged_short(3, 32, 8, sq, 301, _cu_count(0), True, bs)
    n, far = kc.shape[0], 1 << 24

    def spread(c):
        buf = torch.empty(far * (bs - 1) + n * 8 * 128, dtype=c.dtype, device=DEV)
        v = buf.as_strided(c.shape, (8 * 128, far, 128, 1))
        return v.copy_(c)

    call = lambda k, v, **kw: paged_attention(q, k, v, table, seq_lens, max_seq_len=301, **kw)
    apart = call(spread(kc), spread(vc))
    near = [call(kc, vc) for _ in range(2)]
    short = call(kc, vc, route="short")
    assert not torch.equal(apart, short), "the far cache took the short form too"
    for o in near:
        assert torch.equal(o, short)


def test_threads_on_their_own_streams():
    """Native calls of every kind from three threads, each on a stream of its own
    (the single launches let the other threads run): every result has the bits
    of the call alone."""
    import threading
    from gqa_kernels import gqa_flash_attn
    cases = []
    for i, shape in enumerate(SHAPES):
        q, k, v = make_inputs(*shape, torch.bfloat16, seed=20 + i, device=DEV)
        cases.append((q, k, v, gqa_flash_attn(q, k, v)))
    torch.cuda.synchronize()
    bad = []

    def work(seed):
        with torch.cuda.stream(torch.cuda.Stream()):
            for n in range(30):
                q, k, v, want = cases[(n * (seed + 1) + seed) % len(cases)]
                if not torch.equal(gqa_flash_attn(q, k, v), want):
                    bad.append((seed, n))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
