"""GPU parity: the dK / dV kernel cut into pieces over its query tiles.

With fa_bwd_preferred_workspace_bytes, small grids run several workgroups per
(key tile, KV head), each writing fp32 partials that a reduction adds in their
order.  Checked against the fp32 CPU oracle (fp16: atol 2e-3 / rtol 1e-2; both
types: relative L2 < 1e-2) and for bit-for-bit repeats; against the unsplit kernel only the
order of fp32 sums differs, so at most one step of the 16-bit result.  The
workspace is filled with NaN bytes first: a partial that is read but not
written shows up as NaN.
"""
import ctypes

import pytest
import torch

from helpers import assert_close, randn, rel_l2
from oracle import attention_ref as ref
from tilelang_fa_v100 import _dense, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # (B, Sq, Sk, H, Hk, D, causal, dtype)
    (1, 1030, 1030, 2, 2, 128, True, torch.float16),    # pieces start inside a head's tiles
    (1, 300, 500, 8, 2, 128, True, torch.bfloat16),     # GQA, pieces cross query heads
    (2, 257, 600, 12, 3, 128, False, torch.float16),    # full attention, ragged tiles
    (1, 1200, 500, 8, 4, 128, True, torch.float16),     # Sq > Sk: rows that see no key
    (1, 600, 1000, 7, 1, 64, True, torch.bfloat16),     # MQA, seven heads
    (1, 1111, 90, 4, 4, 64, False, torch.float16),      # one partial key tile
    (1, 700, 700, 4, 1, 256, True, torch.float16),
    (2, 1040, 130, 2, 2, 256, False, torch.bfloat16),    # a key tile of two rows
]


def _ids(c):
    B, Sq, Sk, H, Hk, D, causal, dt = c
    return f"B{B}-{Sq}x{Sk}-H{H}/{Hk}-D{D}-{'c' if causal else 'nc'}-{str(dt)[6:]}"


@pytest.mark.parametrize("case", CASES, ids=[_ids(c) for c in CASES])
def test_pieces_match_oracle_and_whole(case):
    B, Sq, Sk, H, Hk, D, causal, dt = case
    g = torch.Generator().manual_seed(47)
    q, do = randn(g, B, Sq, H, D, dtype=dt), randn(g, B, Sq, H, D, dtype=dt)
    k, v = randn(g, B, Sk, Hk, D, dtype=dt), randn(g, B, Sk, Hk, D, dtype=dt)
    qd, kd, vd, dod = (t.to(DEV) for t in (q, k, v, do))
    out, lse = _dense.forward(qd, kd, vd, D ** -0.5, causal)
    lib = _lib.load()

    def run(size):
        dq, dk, dv = (torch.empty_like(t) for t in (qd, kd, vd))
        a = _dense.bwd_args(qd, kd, vd, out, dod, lse, dq, dk, dv, D ** -0.5, causal, False)
        n = size(ctypes.byref(a))
        assert lib.fa_bwd_preferred_workspace_bytes(ctypes.byref(a)) > \
            lib.fa_bwd_workspace_bytes(ctypes.byref(a)), "the split applies"
        ws = torch.full((n,), 0xFF, dtype=torch.uint8, device=DEV)
        print(f"case {_ids(case)}", flush=True)
        _lib.check(lib.fa_bwd(ctypes.byref(a), ws.data_ptr(), n, _lib.stream_handle(qd.device)),
                   "fa_bwd")
        torch.cuda.synchronize()
        return dq, dk, dv

    got, again = run(lib.fa_bwd_preferred_workspace_bytes), run(lib.fa_bwd_preferred_workspace_bytes)
    whole = run(lib.fa_bwd_workspace_bytes)
    want = ref.dense_attention_backward(q, k, v, do, causal=causal)
    step = 2.0 ** (-10 if dt == torch.float16 else -7)
    assert torch.equal(got[0], whole[0]), "dq does not depend on the pieces"
    for i, name in ((1, "dk"), (2, "dv")):
        assert torch.equal(got[i], again[i]), f"{name}: two runs differ"
        # bf16 rounds P and dS to 8 bits before the products: a gradient that
        # sums n terms of size t is off by up to about 4 sqrt(n) 2^-9 t element
        # by element (n = 2000, t = 0.05: 1.7e-2), so only fp16 meets the
        # elementwise bar; its relative L2 error stays near 2^-9.
        if dt == torch.float16:
            assert_close(got[i], want[i], what=name)
        assert rel_l2(got[i], want[i]) < 1e-2, name
        # fp32 sums of up to ~4000 terms in another order: far below one step
        # of the result's type (2^-10 or 2^-7 relative), which rounding can
        # cross, plus an absolute 1e-5 of the largest gradient.
        x, y = got[i].float(), whole[i].float()
        assert ((x - y).abs() <= step * y.abs() + 1e-5 * y.abs().max()).all(), name
