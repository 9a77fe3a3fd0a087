"""The native form of the Python entry points (csrc/pycalls.cpp) against their Python form: over the
operand forms that a call may take the two give the same bits, or refuse with the same exception."""
import threading

import pytest
import torch

from helpers import bits, flat, say
from tileinfer_amd import _lib
from tileinfer_amd.kernels import (gqa_decode_paged_fn, gqa_prefill_paged_fn, qknorm_rope_append,
                                   store_kvcache)
from tileinfer_amd.workloads import make_step, prefill_step


class _Declines:
    """As calls(), with every call left to the Python form."""

    def __getattr__(self, name):
        return lambda *a: None


class _Watched:
    """As calls(), and notes in `taken` whether each call was taken (True) or declined (False)."""

    def __init__(self, taken):
        self.calls, self.taken = _lib.calls(), taken

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self.calls, name)(*a)
            self.taken.append(r is not None)
            return r
        return call


def both(monkeypatch, call, taken=None):
    """call()'s tensors from either form (or the exception), and compares them. `taken`: whether the
    native form has to have taken the call (True) or declined it (False)."""
    got, seen = [], []
    for native in (True, False):
        with monkeypatch.context() as m:
            c = _Watched(seen) if native else _Declines()
            m.setattr(_lib, "calls", lambda: c)
            try:
                got.append(call())
            except Exception as e:  # noqa: BLE001 (compared by type)
                got.append(type(e))
    a, b = got
    assert taken is None or seen in ([[True]] if taken else [[], [False]]), seen
    if isinstance(a, type) or isinstance(b, type):
        assert a is b
        return a
    for x, y in zip(a, b, strict=True):
        assert x.shape == y.shape and x.stride() == y.stride() and torch.equal(bits(x), bits(y))
    return None


def test_declines_what_is_not_its_form():
    """CPU tensors, None and numbers are left to the Python form; a wrong argument count is an error."""
    c, t = _lib.calls(), torch.zeros(1, 1, 256)
    for f, n in ((c.decode, 11), (c.prefill, 12), (c.append, 6), (c.qknorm_append, 12)):
        for x in (t, None, 3):
            assert f(*[x] * n) is None
        with pytest.raises(TypeError):
            f(t)


@pytest.mark.parametrize("case", ["missing", "not a module", "other torch"])
def test_without_the_native_form(case, tmp_path, monkeypatch):
    """Not built here, broken, or built for another torch: one warning, and every call is left to the
    Python form; the library itself stays required."""
    path = tmp_path / "_pycalls.so"
    if case == "not a module":
        path.write_bytes(b"not a shared object")
    if case == "other torch":
        path = _lib.CALLS_PATH
        monkeypatch.setattr(torch, "__version__", "1.0.0")
    monkeypatch.setattr(_lib, "CALLS_PATH", path)
    monkeypatch.setattr(_lib, "_calls", None)
    with pytest.warns(RuntimeWarning, match="host time"):
        c = _lib.calls()
    assert _lib.calls() is c and c.decode(*range(11)) is None and _lib.result(c.append(1)) is None


def _strided(t):
    """t's values as every second row of a larger tensor (rows stay 16-byte aligned)."""
    out = torch.empty(t.shape[0], 2, *t.shape[1:], dtype=t.dtype, device=t.device)[:, 0]
    return out.copy_(t)


def _odd(t):
    """t's values two elements past a 16-byte boundary."""
    f = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    return f[2:2 + t.numel()].view(t.shape).copy_(t)


def _transposed(t):
    """t's values with the last two axes swapped in memory."""
    return t.transpose(-1, -2).contiguous().transpose(-1, -2)


_FORMS = {"plain": lambda t: t, "strided": _strided, "odd": _odd, "transposed": _transposed,
          "parameter": lambda t: torch.nn.Parameter(t, requires_grad=False),
          "short": lambda t: t[:-1], "wide": lambda t: t.double()}


def _expect(refused, form, wrong=False):
    """Wrong sizes and types are refused. A contiguous operand off its alignment is copied by neither
    form, so that it may be refused too; every other form is taken."""
    if wrong or form in ("short", "wide"):
        assert refused is not None
    elif form != "odd":
        assert refused is None


def _taken(which, form, qknorm=False, append=False):
    """Whether the native form takes the call: the plain form always; a parameter, but for the operand
    whose type the entry point looks at; operands a stride apart where the kernels take strides (not
    the gate, nor the vectors of one number per sequence or token); addresses off 16 bytes where they
    take 4 or 2 (table, vectors, the input side)."""
    if form == "parameter":
        return which != ("k" if append else "q")
    if form == "strided":
        return which not in ("gate", "lens", "slots")
    if form == "odd":
        return which in ("table", "lens", "slots") or qknorm or append
    return form == "plain"


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(_FORMS))
@pytest.mark.parametrize("which", ["q", "table", "lens", "gate", "key", "slots", "page"])
def test_decode(which, form, dev, monkeypatch):
    say(f"native decode {which} {form}")
    s = make_step([1, 17, 300], 64, seed=3)
    f = lambda name, t: _FORMS[form](t) if which == name else t  # noqa: E731
    if form == "transposed" and which in ("lens", "slots") or which == "page" and form != "plain":
        pytest.skip("no such form")
    g = torch.Generator(device=dev).manual_seed(1)
    gate = torch.randn(3, 1, s.q.shape[1] * s.q.shape[2], generator=g, device=dev).to(s.q.dtype)
    d = {n: getattr(s, n).to(dev) for n in ("q", "k_cache", "v_cache", "block_table", "seqlen",
                                            "k_new", "v_new", "slot_mapping")}

    def call():
        k, v = d["k_cache"].clone(), d["v_cache"].clone()
        page = 7 if which == "page" else s.page_size
        more = {}
        if which == "gate":
            more["gate"] = f("gate", gate)
        if which in ("key", "slots"):
            more["append"] = (f("key", d["k_new"]), d["v_new"], f("slots", d["slot_mapping"]))
        out = gqa_decode_paged_fn(f("q", d["q"]), k, v, f("table", d["block_table"]),
                                  f("lens", d["seqlen"]), page, **more)
        return out, k, v
    # (The gate's last two axes, one of them of size one, swapped are the same gate.)
    refused = both(monkeypatch, call, which != "page" and (
        _taken(which, form) or (which, form) == ("gate", "transposed")))
    _expect(refused, form, which == "page")


@pytest.mark.gpu
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("missing", [(0,), (1,), (2,), (0, 1, 2)])
def test_append_without_an_operand_is_refused(missing, gated, dev, monkeypatch):
    """An append= with None in it is no call without an append: it raises, and no cache row changes."""
    say(f"native decode append without {missing} gated={gated}")
    s = make_step([1, 17, 300], 64, seed=3)
    q, k, v, table, lens, slots = (t.to(dev) for t in (s.q, s.k_cache, s.v_cache, s.block_table,
                                                       s.seqlen, s.slot_mapping))
    append = tuple(None if i in missing else t
                   for i, t in enumerate((s.k_new.to(dev), s.v_new.to(dev), slots)))
    gate = torch.zeros_like(q) if gated else None
    before = k.clone(), v.clone()
    assert both(monkeypatch, lambda: (gqa_decode_paged_fn(q, k, v, table, lens, s.page_size,
                                                          gate=gate, append=append),)) is ValueError
    assert torch.equal(bits(k), bits(before[0])) and torch.equal(bits(v), bits(before[1]))


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(_FORMS))
@pytest.mark.parametrize("which", ["q", "table", "lens", "gate"])
@pytest.mark.parametrize("schedule", ["auto", "balanced"])
def test_prefill(schedule, which, form, dev, monkeypatch):
    if form == "transposed" and which == "lens":
        pytest.skip("no such form")
    say(f"native prefill {schedule} {which} {form}")
    s = prefill_step([5, 40], [70, 40], seed=4)
    f = lambda name, t: _FORMS[form](t) if which == name else t  # noqa: E731
    d = {n: getattr(s, n).to(dev) for n in ("q", "k_cache", "v_cache", "block_table", "cu_seqlens_q",
                                            "seqlen_k")}
    gate = torch.randn_like(d["q"]) if which == "gate" else None

    def call():
        return (gqa_prefill_paged_fn(
            f("q", d["q"]), d["k_cache"], d["v_cache"], f("table", d["block_table"]),
            d["cu_seqlens_q"], f("lens", d["seqlen_k"]), s.max_seqlen_q, s.page_size,
            schedule=schedule, gate=f("gate", gate) if gate is not None else None),)
    # A shorter q is fewer tokens than cu_seqlens_q states, which only the device sees.
    if form == "short" and which == "q":
        pytest.skip("not a form to refuse on the host")
    refused = both(monkeypatch, call, _taken(which, form))
    _expect(refused, form)


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(_FORMS))
@pytest.mark.parametrize("which", ["q", "k", "v", "cos", "slots"])
def test_append_and_qknorm(which, form, dev, monkeypatch):
    if form == "transposed" and which == "slots":
        pytest.skip("no such form")
    say(f"native append {which} {form}")
    g = torch.Generator(device=dev).manual_seed(2)
    rnd = lambda *z: torch.randn(*z, generator=g, device=dev).to(torch.bfloat16)  # noqa: E731
    q, k, v, w, cos, sin = rnd(6, 8, 256), rnd(6, 2, 256), rnd(6, 2, 256), rnd(256), rnd(6, 64), rnd(6, 64)
    slots = torch.tensor([3, 1, -1, 7, 0, 5], dtype=torch.int32, device=dev)
    f = lambda name, t: _FORMS[form](t) if which == name else t  # noqa: E731

    def qknorm():
        kc, vc = torch.zeros(8, 512, dtype=q.dtype, device=dev), torch.zeros(8, 512, dtype=q.dtype, device=dev)
        out = qknorm_rope_append(f("q", q), f("k", k), f("v", v), w, w, f("cos", cos), f("cos", sin),
                                 kc, vc, f("slots", slots))
        return out, kc, vc

    def append():
        kc, vc = torch.zeros(8, 512, dtype=q.dtype, device=dev), torch.zeros(8, 512, dtype=q.dtype, device=dev)
        store_kvcache(f("k", k), f("v", v), kc, vc, f("slots", slots))
        return kc, vc
    refused = both(monkeypatch, qknorm, _taken(which, form, qknorm=True))
    if form == "wide" and which != "cos" or form == "short":
        assert refused is not None
    both(monkeypatch, append, None if which in ("q", "cos") else _taken(which, form, append=True))


@pytest.mark.gpu
def test_threads_and_streams(dev):
    """Four threads, each on its own stream: every result is the one of a call alone."""
    say("native calls from four threads")
    s = make_step([900, 40, 2000, 1], 256, seed=5)
    q, kc, vc, table, lens = (t.to(dev) for t in (s.q, s.k_cache, s.v_cache, s.block_table, s.seqlen))
    want = gqa_decode_paged_fn(q, kc, vc, table, lens, s.page_size)
    torch.cuda.synchronize()
    outs = [None] * 4

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            outs[i] = [gqa_decode_paged_fn(q, kc, vc, table, lens, s.page_size) for _ in range(20)]
            torch.cuda.current_stream().synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(bits(o), bits(want)) for got in outs for o in got)
