"""The compiled host path of the table entries (``csrc/host_adapters.cpp``) against the Python adapters it stands in for."""

from __future__ import annotations

import pytest
import torch

from coffin_amd import backend, synth
from coffin_amd.weights import QWeight, W4A8Weight
from tests import gpu_util as G

pytestmark = pytest.mark.gpu

K, N = 2560, 1536


def _q8(n=N, k=K, seed=1):
    q = synth.int8_weight(n, k, synth.generator(seed))
    return QWeight(q.wq.to(G.DEV), q.scale.to(G.DEV))


def _w4(n=N, k=K, seed=1):
    w = synth.int4_weight(n, k, synth.generator(seed))
    return W4A8Weight(w.packed.to(G.DEV), w.scale.to(G.DEV), k=k)


def _x(rows, k=K, seed=7):
    return synth.activations(rows, k, synth.generator(seed)).to(G.DEV)


def _adapters(monkeypatch):
    """From here on the Python adapters answer every call."""
    for name in backend._HOST_CALLS:
        monkeypatch.setattr(backend, "_host_" + name, lambda *args: None)


def _same(a, b):
    return a.shape == b.shape and bool((a.view(torch.int16) == b.view(torch.int16)).all())


def test_tensors_replaced_under_the_same_weight_object():
    """An entry is good while the weight object holds the tensors it was made from."""
    x = _x(4)
    w, other = _q8(seed=1), _q8(seed=2)
    want, want_other = backend.linear(_q8(seed=1), x), backend.linear(_q8(seed=2), x)
    for _ in range(3):
        assert _same(backend.linear(w, x), want)
    w.wq, w.scale = other.wq, other.scale
    for _ in range(3):
        assert _same(backend.linear(w, x), want_other)
    w.scale = torch.ones_like(w.scale)                             # one of the two
    ones = QWeight(other.wq, torch.ones_like(w.scale))
    for _ in range(2):
        assert _same(backend.linear(w, x), backend.linear(ones, x))


@pytest.mark.parametrize("make", [_q8, _w4])
def test_a_released_weight_is_refused(make):
    """One whose tensors are gone, which both its entry's dead references and its attributes then say as None."""
    w, x = make(), _x(4)
    for _ in range(2):
        backend.linear(w, x)
    torch.cuda.synchronize()
    for name in ("wq", "packed", "scale"):
        if hasattr(w, name):
            setattr(w, name, None)
    with pytest.raises(AttributeError):
        backend.linear(w, x)


class _Swaps:
    """A weight whose ``wq`` is a property that, when told to, replaces the tensors and projects with itself: the
    outer call's table entry goes while its attributes are being read."""

    def __init__(self, q):
        self._wq, self.scale, self.k, self.n = q.wq, q.scale, q.k, q.n
        self.swap = None

    @property
    def wq(self):
        if self.swap is not None:
            swap, self.swap = self.swap, None
            self._wq, self.scale = swap.wq, swap.scale
            for _ in range(3):
                self.inner = backend.linear(self, _x(1)[0])
            others = [_q8(64, 256, seed) for seed in range(40)]    # and the table grows
            for o in others:
                for _ in range(2):
                    backend.linear(o, _x(1, 256)[0])
        return self._wq


def test_an_entry_that_goes_while_the_weight_is_being_read():
    first, second = _q8(seed=3), _q8(seed=4)
    x = _x(1)[0]
    want = backend.linear(second, x)
    w = _Swaps(first)
    for _ in range(3):
        assert _same(backend.linear(w, x), backend.linear(first, x))
    for _ in range(4):
        w.swap = second
        assert _same(backend.linear(w, x), want) and _same(w.inner, want)
        first, second = second, first
        want = backend.linear(second, x)


def test_row_thresholds_are_read_on_every_call(monkeypatch):
    """A changed threshold moves the compiled calls and the adapters alike, to the bits of the other route."""
    w, x = _q8(), _x(70)
    weight_only, quantised = backend.linear_prefill(w, x[:63]), backend.linear_prefill(w, x)
    dot, mfma = backend.linear(w, x[:4]), backend.linear_m_verify(w, x[:4])
    assert not _same(weight_only, quantised[:63]) and not _same(dot, mfma)
    monkeypatch.setattr(backend, "PREFILL_MIN_ROWS", 63)
    monkeypatch.setattr(backend, "MFMA_MIN_ROWS", 5)
    for _ in range(2):
        assert _same(backend.linear_prefill(w, x[:63]), quantised[:63])
        assert _same(backend.linear_m_verify(w, x[:4]), dot)
        _adapters(monkeypatch)


@pytest.mark.parametrize("make", [_q8, _w4])
def test_a_new_weight_is_resolved_once_and_by_the_compiled_call(monkeypatch, make):
    """Also one that lives where a dead one did, whose record is still under the same id."""
    x = _x(3)
    want = backend.linear(make(seed=12), x)                        # the host path is bound
    made, real = [], backend._make_record
    monkeypatch.setattr(backend, "_make_record", lambda w: made.append(id(w)) or real(w))

    def unexpected(*args, **kwargs):
        raise AssertionError("a weight that the kernels take went to the Python adapter")

    monkeypatch.setattr(backend, "_project", unexpected)
    for n in range(1, 9):
        w = make(seed=12 if n % 2 else 13)
        for _ in range(2):
            assert _same(backend.linear(w, x), want) == bool(n % 2) and len(made) == n
        del w


class _Views:
    """An int8 weight that hands out new tensor objects each time it is read."""

    def __init__(self, q):
        self.q, self.k, self.n = q, q.k, q.n

    wq = property(lambda self: self.q.wq[:])
    scale = property(lambda self: self.q.scale[:])


def test_weights_that_cannot_be_remembered_or_taken_end_as_before(monkeypatch):
    q, x = _q8(seed=21), _x(3)
    want = backend.linear(q, x)
    views = _Views(q)
    for _ in range(3):
        assert _same(backend.linear(views, x), want)
    with pytest.raises(ValueError):                                # the width is looked at before the weight is resolved
        backend.linear(_q8(seed=22), _x(3, K - 128))
    with pytest.raises(ValueError):
        backend.linear(QWeight(q.wq.cpu(), q.scale.cpu()), x)
    wide = _w4(seed=23)
    wide.scale = wide.scale[:-1]                                   # buffers that do not hold the weight
    with pytest.raises(ValueError):
        backend.linear(wide, x)
    fresh, graph = _q8(seed=24), torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="first use"):
        with torch.cuda.graph(graph):
            backend.linear(fresh, x)
    torch.cuda.synchronize()
    assert _same(backend.linear(fresh, x), backend.linear(_q8(seed=24), x))


@pytest.mark.parametrize("mode", ["grad", "no_grad", "inference"])
@pytest.mark.parametrize("rows", [0, 1, 5, 70])                    # 0: a [K] activation
def test_parts_of_a_fused_projection_are_those_of_split(monkeypatch, mode, rows):
    """Values, sizes, pitch, offset, shared version counter, view relation and what autograd allows on them."""
    x = _x(rows) if rows else _x(1)[0]
    sizes = [1024, 128, 384]
    switch = {"grad": torch.enable_grad, "no_grad": torch.no_grad, "inference": torch.inference_mode}[mode]
    for make in (_q8, _w4):
        w = make()
        for entry in ("linear", "linear_m", "linear_m_verify", "linear_prefill") if rows else ("linear",):
            with switch():
                backend.linear_parts(entry, w, x, sizes)           # the weight is known
                got = backend.linear_parts(entry, w, x, sizes)
                whole = getattr(backend, entry)(w, x)
                want = whole.split(sizes, dim=-1)
            assert type(got) is tuple and len(got) == 3
            base = None
            for a, b in zip(got, want):
                assert _same(a, b) and a.stride() == b.stride() and a.storage_offset() == b.storage_offset()
                assert a._is_view() == b._is_view() and a.is_inference() == b.is_inference()
                assert a.untyped_storage().data_ptr() == got[0].untyped_storage().data_ptr()
                if mode != "inference":
                    base = a._base
                    assert base is got[0]._base and _same(base, whole)
            if mode == "inference":
                continue
            got[1].add_(1)
            assert got[0]._version == got[2]._version == base._version == 1
            assert torch.equal(base[..., 1024:1152], got[1]) and torch.equal(base[..., 1152:], want[2])
            leaf = torch.ones(1024, dtype=torch.bfloat16, device=G.DEV, requires_grad=True)
            for part in (got[0], want[0]):                         # a write that would need the other parts' history
                with pytest.raises(RuntimeError):
                    part.mul_(leaf)
    with pytest.raises(RuntimeError):
        backend.linear_parts("linear", w, x, [1024, 128])
    with pytest.raises(RuntimeError):
        backend.linear_parts("linear", w, x, [1024, 128, 385])


class _Rows(torch.Tensor):
    """A tensor subclass: the compiled calls leave it to the adapters."""


def _odd_rows(kind, rows, k):
    x = _x(rows, k)
    if kind == "cpu":
        return x.cpu()
    if kind in ("float32", "float16"):
        return x.to(getattr(torch, kind))
    if kind == "columns":
        return x.t().contiguous().t()
    if kind == "pitch":
        return torch.cat([x, x], dim=1)[:, :k]
    if kind == "offset":                                           # rows that start 2 bytes past a 16-byte boundary
        flat = torch.empty(rows * k + 1, dtype=x.dtype, device=x.device)
        flat[1:] = x.reshape(-1)
        return flat[1:].view(rows, k)
    if kind == "subclass":
        return x.as_subclass(_Rows)
    if kind == "empty":
        return x[:0]
    if kind == "3-D":
        return x.view(1, rows, k)
    if kind == "narrow":
        return x[:, :k - 16].contiguous()
    assert kind == "plain"
    return x


def _outcome(call):
    try:
        return None, call()
    except Exception as exc:                                       # noqa: BLE001 - the two paths must raise alike
        return type(exc), None


@pytest.mark.parametrize("mode", ["grad", "inference"])
@pytest.mark.parametrize("kind", ["plain", "cpu", "float32", "float16", "columns", "pitch", "offset", "subclass", "empty", "3-D",
                                  "narrow"])
def test_calls_that_are_not_the_common_case_end_as_the_adapters_end_them(monkeypatch, kind, mode):
    """Other devices, types, layouts, subclasses, shapes and inference tensors: values, shape, type and kind of error of
    every entry with the compiled calls and without them."""
    rows = 5
    weights = {"int8": _q8(), "int4": _w4()}
    gain = _x(1, seed=9)[0].contiguous()
    calls = {}
    for name, w in weights.items():
        for entry in ("linear", "linear_m", "linear_m_verify", "linear_prefill"):
            calls[name, entry] = lambda x, w=w, entry=entry: getattr(backend, entry)(w, x)
            calls[name, entry, "parts"] = lambda x, w=w, entry=entry: backend.linear_parts(entry, w, x, [1024, 512])

    def zeros(x, shape, dtype):
        return torch.zeros(shape, dtype=dtype, device=x.device)

    def gain_for(x):
        return gain.to(x.device, x.dtype)[:x.shape[-1]]

    def silu_mul(x):
        out = zeros(x, x.shape, x.dtype)
        return backend.silu_mul(x, x, out), out

    def kv_quant(x):
        q, s = zeros(x, x.shape, torch.int8), zeros(x, x.shape[:-1], torch.float32)
        return backend.kv_quant(x, q, s), q, s

    def add_rms_norm(x):
        total, out = x.clone(), zeros(x, x.shape, x.dtype)
        return backend.add_rms_norm(total, x, gain_for(x), out), total, out

    calls["rms_norm"] = lambda x: backend.rms_norm(x, gain_for(x))
    calls["silu_mul"], calls["kv_quant"], calls["add_rms_norm"] = silu_mul, kv_quant, add_rms_norm
    calls["embed_rows"] = lambda x: backend.embed_rows(weights["int8"], torch.arange(3, device=x.device))
    calls["embed_rows", "int32"] = lambda x: backend.embed_rows(weights["int4"], torch.arange(3, dtype=torch.int32, device=x.device))
    switch = {"grad": torch.enable_grad, "inference": torch.inference_mode}[mode]

    def outcomes():
        with switch():
            x = _odd_rows(kind, rows, K)
            return {name: _outcome(lambda: call(x)) for name, call in calls.items()}

    for call in calls.values():                                    # the weights are known
        _outcome(lambda: call(_x(rows)))
    got = outcomes()
    _adapters(monkeypatch)
    want = outcomes()

    def flat(v):
        return [t for e in v for t in flat(e)] if isinstance(v, (tuple, list)) else [v]

    for name in calls:
        assert got[name][0] == want[name][0], (name, got[name][0], want[name][0])
        for a, b in zip(flat(got[name][1]), flat(want[name][1]), strict=True):
            if b is None:
                continue
            assert type(a) is type(b) and a.dtype == b.dtype and a.device == b.device and a.shape == b.shape, name
            assert a.is_inference() == b.is_inference() and a.requires_grad == b.requires_grad, name
            assert torch.equal(a.float().cpu(), b.float().cpu()), name
