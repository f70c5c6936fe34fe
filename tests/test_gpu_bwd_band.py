"""GPU parity: the dS-store backward of window bands (head_dim 128 and 256).

With fa_bwd_preferred_workspace_bytes a band's dS tiles are stored too, each
query tile with room for the widest row of key blocks, and dq is formed from
them; with the minimal workspace S and dP are recomputed.  dk and dv come from
the same products on both paths and must agree exactly; everything is checked
against the fp32 CPU oracle (fp16: atol 2e-3 / rtol 1e-2; both types: relative
L2 < 1e-2, as for the other window gradients) and repeats bit for bit.  The
workspace is filled with NaN bytes first: a tile that is read but not written
shows up as NaN.
"""
import ctypes

import pytest
import torch

from helpers import assert_close, randn, rel_l2
from oracle import attention_ref as ref
from tilelang_fa_v100 import _dense, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F16, BF16 = torch.float16, torch.bfloat16
BIG = 2 ** 31 - 1

CASES = [
    # (B, Sq, Sk, H, Hk, D, causal, window, dtype)
    (1, 700, 700, 2, 2, 128, True, (100, 0), F16),
    (2, 333, 333, 4, 2, 128, False, (40, 30), F16),       # both sides, GQA
    (1, 500, 300, 2, 2, 128, True, (31, 0), F16),         # rows that see no key, one block wide
    (1, 300, 500, 2, 1, 128, False, (-1, 33), BF16),      # left open
    (1, 290, 610, 2, 2, 128, False, (64, -1), F16),       # right open
    (1, 400, 400, 2, 2, 128, True, (0, 0), F16),          # the diagonal alone
    (1, 70, 70, 2, 2, 128, True, (5000, 0), F16),         # a band wider than the keys
    (1, 90, 2000, 1, 1, 128, False, (700, 200), F16),
    (1, 2100, 2100, 2, 2, 128, True, (512, 0), BF16),     # several query blocks
    (1, 700, 700, 2, 2, 256, True, (129, 0), F16),
    (1, 300, 450, 2, 1, 256, False, (10, 90), F16),
    # Bounds at the end of 32 bits, as "unbounded" is often written.
    (1, 400, 400, 2, 2, 128, True, (BIG, 0), F16),
    (1, 300, 500, 2, 1, 128, False, (-1, BIG), F16),
    (1, 500, 300, 2, 2, 128, False, (BIG, BIG), F16),
    (1, 500, 300, 2, 2, 128, True, (BIG - 100, 0), BF16),
    (1, 290, 610, 2, 2, 256, False, (BIG, 3), F16),
]


def _ids(c):
    B, Sq, Sk, H, Hk, D, causal, w, dt = c
    return f"B{B}-{Sq}x{Sk}-H{H}/{Hk}-D{D}-w{w[0]},{w[1]}-{str(dt)[6:]}"


@pytest.mark.parametrize("case", CASES, ids=[_ids(c) for c in CASES])
def test_band_dq_paths_match_oracle_and_each_other(case):
    B, Sq, Sk, H, Hk, D, causal, window, dt = case
    g = torch.Generator().manual_seed(53)
    q, do = randn(g, B, Sq, H, D, dtype=dt), randn(g, B, Sq, H, D, dtype=dt)
    k, v = randn(g, B, Sk, Hk, D, dtype=dt), randn(g, B, Sk, Hk, D, dtype=dt)
    qd, kd, vd, dod = (t.to(DEV) for t in (q, k, v, do))
    out, lse = _dense.forward(qd, kd, vd, D ** -0.5, causal, window)
    lib = _lib.load()

    def run(size):
        dq, dk, dv = (torch.empty_like(t) for t in (qd, kd, vd))
        a = _dense.bwd_args(qd, kd, vd, out, dod, lse, dq, dk, dv, D ** -0.5, causal, False,
                            window)
        assert lib.fa_bwd_preferred_workspace_bytes(ctypes.byref(a)) > \
            lib.fa_bwd_min_workspace_bytes(ctypes.byref(a)), "the dS path applies"
        n = size(ctypes.byref(a))
        ws = torch.full((n,), 0xFF, dtype=torch.uint8, device=DEV)
        print(f"case {_ids(case)}", flush=True)
        _lib.check(lib.fa_bwd(ctypes.byref(a), ws.data_ptr(), n, _lib.stream_handle(qd.device)),
                   "fa_bwd")
        torch.cuda.synchronize()
        return dq, dk, dv

    got, again = run(lib.fa_bwd_preferred_workspace_bytes), run(lib.fa_bwd_preferred_workspace_bytes)
    recomputed = run(lib.fa_bwd_min_workspace_bytes)
    want = ref.dense_attention_backward(q, k, v, do, causal=causal, window=window)
    assert rel_l2(out, ref.dense_attention(q, k, v, causal=causal, window=window)[0]) < 1e-2, "out"
    for i, name in enumerate(("dq", "dk", "dv")):
        assert torch.equal(got[i], again[i]), f"{name}: two runs differ"
        if name != "dq":
            assert torch.equal(got[i], recomputed[i]), f"{name}: paths differ"
        for x in (got[i], recomputed[i]):
            assert torch.isfinite(x.float()).all(), name
            if dt == F16:
                assert_close(x, want[i], what=name)
            if want[i].abs().max() > 1e-4:
                assert rel_l2(x, want[i]) < 1e-2, name
