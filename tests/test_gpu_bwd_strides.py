"""GPU: the dense backward on strided tensors, all eight of them with strides of their own.

Every path of fa_bwd (pieces, dS tiles of window bands, recompute, each
head_dim) is run on packed tensors and on views of the same values: columns of
wider rows, [B, H, S, D] storage, every other token, heads of a wider tensor.
The operations and their order do not depend on strides, so the gradients must
have the same bits; the packed ones are checked against the oracle elsewhere.
The memory around the views is NaN, which a read outside a view would carry
into the result, and must still be NaN after the call.
"""
import ctypes

import pytest
import torch

from helpers import randn
from tilelang_fa_v100 import _dense, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F16, BF16 = torch.float16, torch.bfloat16

CASES = [
    # (B, Sq, Sk, H, Hk, D, causal, window, dtype)
    (2, 600, 1000, 6, 2, 64, True, (-1, -1), BF16),
    (1, 1111, 90, 4, 4, 64, False, (-1, -1), F16),
    (2, 333, 333, 4, 2, 64, True, (100, 0), F16),
    (2, 300, 500, 8, 2, 128, True, (-1, -1), BF16),
    (2, 257, 600, 6, 3, 128, False, (-1, -1), F16),
    (2, 333, 333, 4, 2, 128, False, (40, 30), F16),
    (1, 300, 500, 2, 1, 128, False, (-1, 33), BF16),
    (2, 700, 700, 4, 1, 256, True, (-1, -1), F16),
    (2, 300, 450, 2, 1, 256, False, (10, 90), BF16),
]


def _ids(c):
    B, Sq, Sk, H, Hk, D, causal, w, dt = c
    return f"B{B}-{Sq}x{Sk}-H{H}/{Hk}-D{D}-{'c' if causal else 'nc'}-w{w[0]},{w[1]}-{str(dt)[6:]}"


def spread(shape, dtype, kind):
    """(view of `shape`, the NaN tensor it lies in)."""
    B, S, H, D = shape
    nan = lambda *s: torch.full(s, float("nan"), dtype=dtype, device=DEV)  # noqa: E731
    if kind == 0:
        base = nan(B, S, H, D + 24)
        return base[..., 16:16 + D], base
    if kind == 1:
        base = nan(B, H + 1, S, D)
        return base[:, 1:].transpose(1, 2), base
    if kind == 2:
        base = nan(B, 2 * S, H, D)
        return base[:, 1::2], base
    base = nan(B, S, 3 * H, D + 8)
    return base[:, :, H:2 * H, :D], base


def untouched(view, base):
    outside = torch.ones_like(base, dtype=torch.bool)
    outside.as_strided(view.shape, view.stride(), view.storage_offset()).fill_(False)
    return bool(base[outside].isnan().all())


@pytest.mark.parametrize("case", CASES, ids=[_ids(c) for c in CASES])
def test_strided_backward_has_the_packed_bits(case):
    B, Sq, Sk, H, Hk, D, causal, window, dt = case
    g = torch.Generator().manual_seed(59)
    q, do = (randn(g, B, Sq, H, D, dtype=dt).to(DEV) for _ in range(2))
    k, v = (randn(g, B, Sk, Hk, D, dtype=dt).to(DEV) for _ in range(2))
    out, lse = _dense.forward(q, k, v, D ** -0.5, causal, window)
    lib = _lib.load()

    def run(ins, grads, size):
        qi, ki, vi, oi, doi = ins
        a = _dense.bwd_args(qi, ki, vi, oi, doi, lse, *grads, D ** -0.5, causal, False, window)
        n = size(ctypes.byref(a))
        ws = torch.full((n,), 0xFF, dtype=torch.uint8, device=DEV)
        _lib.check(lib.fa_bwd(ctypes.byref(a), ws.data_ptr(), n, _lib.stream_handle(q.device)),
                   "fa_bwd")
        torch.cuda.synchronize()

    packed = (q, k, v, out, do)
    for size in (lib.fa_bwd_preferred_workspace_bytes, lib.fa_bwd_min_workspace_bytes):
        print(f"case {_ids(case)}", flush=True)
        want = [torch.empty_like(t) for t in (q, k, v)]
        run(packed, want, size)
        for turn in range(2):
            views = []
            for i, t in enumerate(packed):
                view, _ = spread(t.shape, dt, (i + turn) % 4)
                views.append(view.copy_(t))
            outs = [spread(t.shape, dt, (i + 2 + turn) % 4) for i, t in enumerate(want)]
            run(views, [o[0] for o in outs], size)
            for name, (got, base), ref in zip(("dq", "dk", "dv"), outs, want):
                assert got.stride() != ref.stride()
                assert torch.isfinite(ref.float()).all() and torch.equal(got, ref), name
                assert untouched(got, base), f"{name}: written outside"
