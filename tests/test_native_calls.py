"""The native call marshalling against the Python path it stands in for.

On the CPU: what is not the plain case is handed back (None) before any work,
and so is every call where the extension is not built for this torch.
On the GPU: every form a caller may pass gives the same bits whether the native
path takes it or not, and mistakes raise the same exception either way; the
native path takes exactly the forms it is for.
"""
import sys
import types
import warnings

import pytest
import torch

import tilelang_fa_v100 as fa
from tilelang_fa_v100 import _native
from tilelang_fa_v100._cache_write import reshape_and_cache

DEV = "cuda:0"
NAMES = ("dense_forward", "decode", "paged_forward", "cache_write")


def test_cpu_tensors_and_foreign_objects_are_handed_back():
    m = _native.load()
    t = torch.zeros(2, 16, 2, 64, dtype=torch.float16)
    assert m.dense_forward(t, t, t, 0.1, True, -1, -1, True, 0, 0) is None
    assert m.dense_forward(1, t, t, 0.1, True, -1, -1, True, 0, 0) is None
    assert m.decode(t[0], t, t, t, t, 16, None, None, 0, 0) is None
    assert m.paged_forward(t, t, t, t, t, t, t, 16, None, None, True, -1, -1, 0, 0) is None
    assert m.cache_write(t, t, t, t, t, 0, 0) is None
    for name in NAMES:
        assert getattr(m, name)() is None
    assert _native.dense_forward(t, t, t, 0.1, True, (-1, -1), True) is None
    with pytest.raises(TypeError):
        m.bind(1)


@pytest.mark.parametrize("found", [None, types.ModuleType("stale"),
                                   types.SimpleNamespace(torch_version="1.0")],
                         ids=["none", "no version", "another torch"])
def test_without_the_extension_python_takes_the_calls(found, monkeypatch):
    """One warning, then every call is handed back; load() itself still says what is missing."""
    monkeypatch.setattr(_native, "_module", None)
    monkeypatch.setattr(_native, "_missing", False)
    monkeypatch.setitem(sys.modules, "tilelang_fa_v100._fa_torch", found)
    monkeypatch.delattr(fa, "_fa_torch", raising=False)
    if found is not None:
        monkeypatch.setattr(fa, "_fa_torch", found, raising=False)
    with pytest.raises(RuntimeError, match="not built for this torch"):
        _native.load()
    device = types.SimpleNamespace(is_cuda=True)
    monkeypatch.setattr(_native, "torch", types.SimpleNamespace(
        Tensor=types.SimpleNamespace, __version__=torch.__version__))
    with pytest.warns(RuntimeWarning, match="marshalled in Python"):
        assert _native.decode(device) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _native.dense_forward(device, device, device, 0.1, True, (-1, -1), True) is None
        assert _native.cache_write(device) is None


def _dense(**over):
    g = torch.Generator(device=DEV).manual_seed(3)
    mk = lambda h, s=70: torch.randn(2, s, h, 64, generator=g, device=DEV, dtype=torch.float16)  # noqa: E731
    a = dict(q=mk(4), k=mk(2, 90), v=mk(2, 90))
    a.update({k: f(a) for k, f in over.items()})
    return a


def _paged(decode=False):
    g = torch.Generator(device=DEV).manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV, dtype=torch.bfloat16)  # noqa: E731
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    a = dict(q=mk(2 if decode else 9, 8, 128), k_cache=mk(6, 16, 2, 128), v_cache=mk(6, 16, 2, 128),
             block_table=i32([3, 0, 5], [1, 2, -1]), seq_lens=i32(41, 20))
    if not decode:
        a.update(query_start_loc=i32(0, 5, 9), prefix_kv_lens=i32(36, 16))
    return a


def _cache():
    g = torch.Generator(device=DEV).manual_seed(7)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV, dtype=torch.float16)  # noqa: E731
    return dict(key=mk(3, 2, 64), value=mk(3, 2, 64), key_cache=mk(4, 8, 2, 64),
                value_cache=mk(4, 8, 2, 64),
                slot_mapping=torch.tensor([31, -1, 4], device=DEV))


def _attend(a):
    return fa.tilelang_flash_attn_func(**a)


def _run_cache(a):
    reshape_and_cache(**a)
    return a["key_cache"], a["value_cache"]


def _with(make, **change):
    def build():
        a = make()
        a.update({k: f(a) if callable(f) else f for k, f in change.items()})
        return a
    return build


def _wide(name):  # a strided view: every other head of a wider tensor
    return lambda a: torch.cat([a[name], a[name]], -2)[..., ::2, :]


def _off(name):  # misaligned base: copied by the Python path
    return lambda a: torch.cat([a[name].flatten(), a[name].flatten()[:1]])[1:].view(a[name].shape)


FORMS = {
    "dense plain": (_attend, _dense),
    "dense causal int": (_attend, _with(_dense, causal=1)),
    "dense window": (_attend, _with(_dense, causal=True, window_size=(20, 0))),
    "dense window list": (_attend, _with(_dense, window_size=[20, 5])),
    "dense scale int": (_attend, _with(_dense, softmax_scale=1)),
    "dense lse": (_attend, _with(_dense, return_attn_probs=True)),
    "dense strided": (_attend, _with(_dense, q=_wide("q"), v=_wide("v"))),
    "dense [B, H, S, D] storage": (_attend, _with(
        _dense, k=lambda a: a["k"].transpose(1, 2).contiguous().transpose(1, 2))),
    "dense expanded": (_attend, _with(_dense, k=lambda a: a["k"][:1].expand(2, -1, -1, -1))),
    "dense misaligned": (_attend, _with(_dense, q=_off("q"))),
    "dense one row": (_attend, _with(_dense, q=lambda a: a["q"][:, :1])),
    "dense no rows": (_attend, _with(_dense, q=lambda a: a["q"][:, :0])),
    "dense parameter": (_attend, _with(_dense, q=lambda a: torch.nn.Parameter(a["q"]))),
    "decode plain": (lambda a: fa.tilelang_decode_forward(**a), lambda: _paged(True)),
    "decode int64": (lambda a: fa.tilelang_decode_forward(**a), _with(
        lambda: _paged(True), seq_lens=lambda a: a["seq_lens"].long())),
    "decode table view": (lambda a: fa.tilelang_decode_forward(**a), _with(
        lambda: _paged(True), block_table=lambda a: torch.cat([a["block_table"]] * 2, 1)[:, :3])),
    "decode heads given": (lambda a: fa.tilelang_decode_forward(**a), _with(
        lambda: _paged(True), num_kv_heads=2, softmax_scale=0.3)),
    "paged plain": (lambda a: fa.tilelang_paged_forward(**a), _paged),
    "paged not causal": (lambda a: fa.tilelang_paged_forward(**a), _with(_paged, causal=False)),
    "paged windows": (lambda a: fa.tilelang_paged_forward(**a), _with(
        _paged, sliding_window_q=30, sliding_window_k=40)),
    "paged strided q": (lambda a: fa.tilelang_paged_forward(**a), _with(_paged, q=_wide("q"))),
    "paged out": (lambda a: fa.tilelang_paged_forward(**a), _with(
        _paged, out=lambda a: torch.empty_like(a["q"]))),
    "cache plain": (_run_cache, _cache),
    "cache int32 slots": (_run_cache, _with(
        _cache, slot_mapping=lambda a: a["slot_mapping"].int())),
    "cache strided": (_run_cache, _with(_cache, key=_wide("key"))),
    # mistakes
    "dense dtype": (_attend, _with(_dense, v=lambda a: a["v"].bfloat16())),
    "dense float": (_attend, _with(_dense, q=lambda a: a["q"].float())),
    "dense heads": (_attend, _with(_dense, q=lambda a: a["q"][:, :, :3])),
    "dense device": (_attend, _with(_dense, k=lambda a: a["k"].cpu())),
    "dense bad window": (_attend, _with(_dense, window_size=(-2, 0))),
    "decode block size": (lambda a: fa.tilelang_decode_forward(**a), _with(
        lambda: _paged(True), block_size=8)),
    "decode batch": (lambda a: fa.tilelang_decode_forward(**a), _with(
        lambda: _paged(True), seq_lens=lambda a: a["seq_lens"][:1])),
    "decode kv heads": (lambda a: fa.tilelang_decode_forward(**a), _with(
        lambda: _paged(True), num_kv_heads=4)),
    "paged starts": (lambda a: fa.tilelang_paged_forward(**a), _with(
        _paged, query_start_loc=lambda a: a["query_start_loc"][:2])),
    "cache rows": (_run_cache, _with(_cache, key=lambda a: a["key"][:, :1])),
    "cache slots": (_run_cache, _with(_cache, slot_mapping=lambda a: a["slot_mapping"][:2])),
}


# Forms the native path takes; it hands back all others, and an `out` argument
# is not put to it.
TAKEN = {"dense plain", "dense causal int", "dense window", "dense scale int", "dense lse",
         "dense strided", "dense [B, H, S, D] storage", "dense expanded", "dense one row",
         "dense parameter", "decode plain", "decode heads given", "paged plain",
         "paged not causal", "paged windows", "cache plain", "cache strided"}


def _outcome(call, make):
    try:
        r = call(make())
        torch.cuda.synchronize()
        return r if isinstance(r, tuple) else (r,)
    except Exception as e:  # noqa: BLE001 - compared by type and text
        return type(e), str(e)


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(FORMS))
def test_native_and_python_paths_agree(form, monkeypatch):
    call, make = FORMS[form]
    print(f"form {form}", flush=True)
    taken = []

    def recorded(f):
        def g(*a, **k):
            r = f(*a, **k)
            taken.append(r is not None)
            return r
        return g

    for name in NAMES:
        monkeypatch.setattr(_native, name, recorded(getattr(_native, name)))
    native = _outcome(call, make)
    assert taken == ([] if form == "paged out" else [form in TAKEN])
    for name in NAMES:
        monkeypatch.setattr(_native, name, lambda *a, **k: None)
    python = _outcome(call, make)
    assert len(native) == len(python)
    for x, y in zip(native, python):
        if isinstance(y, torch.Tensor):
            assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride()
            assert torch.equal(x, y)
        else:
            assert x == y
