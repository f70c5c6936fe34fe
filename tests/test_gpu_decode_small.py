"""GPU parity: decode batches too small to fill the GPU.

The split (keys per work item) goes down to 64 for them, chosen on the host
from the block table's width and halved on the device from the actual lengths
as far as the workspace's partials allow: lengths at the edges of 64-, 128- and
256-key items, tables as wide as the longest sequence, many times wider, and
just wide enough that halving has to stop; up to 128 partials to merge.
"""
import pytest
import torch

from test_gpu_decode import check, make_case

pytestmark = pytest.mark.gpu

CASES = [
    # (lens, Hq, Hkv, D, page, dtype, table keys: 0 = the longest sequence's)
    ([63, 64, 65, 1], 8, 2, 128, 16, torch.float16, 0),
    ([127, 128, 129, 0], 16, 4, 128, 16, torch.bfloat16, 32768),
    ([8192], 4, 1, 128, 16, torch.float16, 0),            # 128 partials of 64 keys
    ([8191, 60], 4, 1, 128, 16, torch.float16, 8192),
    ([4097, 100, 700], 32, 8, 128, 64, torch.float16, 4160),
    ([4500, 30, 30, 30], 32, 8, 128, 16, torch.float16, 32768),
    ([300, 65], 8, 8, 64, 16, torch.bfloat16, 16384),
    ([257, 1000], 12, 2, 64, 8, torch.float16, 0),
    ([2000, 66], 16, 2, 256, 32, torch.float16, 8192),
    ([900, 64], 4, 1, 512, 16, torch.bfloat16, 4096),
]


@pytest.mark.parametrize("case", CASES,
                         ids=[f"D{c[3]}-B{len(c[0])}-max{max(c[0])}-t{c[6]}" for c in CASES])
def test_small_batches(case):
    lens, Hq, Hkv, D, page, dt, table = case
    q, kc, vc, bt, sl, page = make_case(51, lens, Hq, Hkv, D, page=page, dtype=dt)
    width = max(bt.shape[1], table // page)
    bt = torch.cat([bt, bt.new_full((bt.shape[0], width - bt.shape[1]), -1)], 1)
    print(f"case {case}", flush=True)
    check((q, kc, vc, bt, sl, page))


@pytest.mark.parametrize("batch,Hq,Hkv,D,table", [(72, 32, 8, 128, 0), (72, 32, 8, 128, 32768),
                                                  (130, 16, 2, 512, 0), (64, 32, 32, 64, 0),
                                                  (63, 32, 4, 256, 8192)])
def test_many_rows(batch, Hq, Hkv, D, table):
    """Eight (sequence, head) rows a CU on either side: the one-wave merge, with one partial, many
    and none; batches of more than 64 lengths."""
    lens = [(37 * i) % 700 for i in range(batch - 2)] + [3000, 1025]
    q, kc, vc, bt, sl, page = make_case(53, lens, Hq, Hkv, D, page=16, dtype=torch.float16)
    width = max(bt.shape[1], table // page)
    bt = torch.cat([bt, bt.new_full((bt.shape[0], width - bt.shape[1]), -1)], 1)
    print(f"case {batch} {Hq}/{Hkv} D{D}", flush=True)
    check((q, kc, vc, bt, sl, page))
