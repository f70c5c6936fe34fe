"""GPU parity: paged tiles of at most 32 rows (keys split over the waves).

A tile's row count is (new tokens x query heads per KV head) minus the rows of
the tiles before it; 32 takes the key-split core and 33 the row-tile one, at
the same shapes, in one batch with sequences that do the other.  Key counts
sit at the edges of the 32-key tiles, of the 16-key halves that one page base
serves, and of the ranges of 4 and 8 waves; caches hold NaN past every
sequence's end.  Oracle bar as for the other paged paths (outputs atol 2e-3 /
rtol 1e-2, LSE within 1e-3, relative L2 < 1e-2).
"""
import pytest
import torch

from test_gpu_paged import make_case
from test_gpu_paged_split import run_split

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16
CASES = [
    # (q_lens, seq_lens, Hq, Hkv, D, page, dtype, causal, wq, wk, splits); prefix = seq - q
    ([1, 8, 9, 1, 1], [1, 31, 33, 257, 513], 16, 4, 128, 16, F16, True, -1, -1, 1),
    ([1, 8, 9, 1, 200], [16, 255, 300, 2049, 260], 16, 4, 128, 64, BF16, True, -1, -1, 3),
    ([4, 5, 0, 1], [1000, 1001, 40, 15], 64, 8, 128, 32, F16, False, -1, -1, 2),
    ([1, 7, 32], [700, 333, 47], 8, 8, 128, 16, F16, True, 100, 30, 1),
    ([1, 8, 9, 1], [1, 129, 140, 1025], 8, 2, 64, 16, F16, True, -1, -1, 1),
    ([2, 33, 1], [100, 99, 4000], 7, 1, 64, 8, BF16, True, -1, -1, 4),   # pages of 8: no key split
    ([1, 32, 1], [33, 77, 2000], 8, 8, 64, 64, F16, True, 50, -1, 2),
    ([1, 4, 5, 1], [1, 127, 131, 1500], 16, 2, 256, 16, F16, True, -1, -1, 1),
    ([1, 3, 140], [2000, 31, 170], 16, 2, 256, 32, BF16, True, -1, -1, 3),
    # Around the least count that is split, 384 keys (of a range), and the
    # edges of tiles and of the waves' ranges above it.
    ([1, 8, 9, 1, 1, 1], [383, 384, 385, 415, 513, 767], 16, 4, 128, 16, F16, True, -1, -1, 1),
    ([1, 1, 8, 2, 1], [1151, 1152, 1154, 1249, 1700], 16, 4, 128, 32, BF16, True, -1, -1, 3),
    ([1, 1, 8, 1], [383, 384, 417, 2051], 8, 2, 64, 16, F16, True, -1, -1, 1),
    ([1, 3, 1, 1], [384, 497, 777, 128], 16, 2, 256, 16, F16, True, -1, -1, 1),
    ([1] * 20, [384 + 5 * i for i in range(20)], 16, 16, 256, 16, F16, True, -1, -1, 1),  # > CUs
    ([1, 1, 900], [900, 2000, 1000], 64, 8, 128, 16, F16, True, -1, -1, 1),  # mostly full tiles
]


@pytest.mark.parametrize("case", CASES,
                         ids=[f"D{c[4]}-p{c[5]}-{str(c[6])[6:]}-s{c[10]}-{i}"
                              for i, c in enumerate(CASES)])
def test_few_row_tiles_match_oracle(case):
    ql, sl, Hq, Hkv, D, page, dt, causal, wq, wk, ns = case
    c = make_case(29, ql, sl, [s - q for q, s in zip(ql, sl)], Hq, Hkv, D, page=page, dtype=dt)
    print(f"case {case}", flush=True)
    run_split(c, ns, causal=causal, wq=wq, wk=wk)


@pytest.mark.parametrize("Hkv,splits", [(1, 1), (2, 1), (2, 3), (3, 1), (4, 2), (5, 1), (8, 2),
                                        (12, 1), (16, 1)])
def test_workgroup_order_covers_every_tile(Hkv, splits):
    """Every (KV head, key range) count of the workgroup order: more than,
    fewer than and no divisor of the 8 XCDs."""
    c = make_case(31, [300, 1, 0, 40, 257], [300, 77, 9, 640, 300], [0, 76, 9, 600, 43],
                  Hkv, Hkv, 128, page=16)
    run_split(c, splits)


@pytest.mark.parametrize("q_lens,heads", [
    ([1] * 20 + [600] * 9, 32),           # 65 tiles x 32 heads: sequences by history
    ([1, 2, 129, 64, 0, 300] * 10, 4),    # 60 sequences, tiles by reach, many ties
    ([3, 1, 130, 0, 1] * 14, 4),          # 70 sequences: scanned in their own order
], ids=["by-history", "by-reach", "over-64"])
def test_tile_orders_cover_every_tile(q_lens, heads):
    g = torch.Generator().manual_seed(37)
    pf = torch.randint(0, 5, (len(q_lens),), generator=g).mul(50).tolist()
    c = make_case(33, q_lens, [p + q for p, q in zip(pf, q_lens)], pf, heads, heads, 64, page=16)
    run_split(c, 1)


@pytest.mark.parametrize("q_lens,step,heads,dim", [
    ([1] * 20 + [600] * 9, 300, 32, 64),          # 65 tiles x 32 heads: sequences by reach
    ([1, 2, 129, 64, 0, 300] * 10, 300, 4, 64),   # 60 sequences, 320 workgroups: tiles by reach
    ([200, 1, 370, 0, 129, 300] * 2, 0, 50, 64),  # no histories, 700 workgroups: tiles by reach
    ([1100, 300, 0, 700], 0, 32, 128),            # no histories, 320 workgroups: tiles by reach
    ([1100, 300, 0, 700], 0, 60, 128),            # 600, XCDs share heads: tiles by reach
    ([1100, 300, 0, 700], 0, 76, 128),            # 760, as above: just below three rounds
    ([1100, 300, 0, 700], 0, 78, 128),            # 780: sequences in their own order
    ([1100, 300, 0, 700], 0, 32, 256),            # 544, one a CU: sequences in their own order
    ([500, 0, 530], 0, 66, 128),                  # two short prompts: no search
    ([500, 0, 530], 100, 66, 128),                # two histories
], ids=["by-sequence-reach", "by-reach", "two-rounds-d64", "two-rounds-d128", "shared",
        "shared-three", "own-order", "own-order-d256",
        "two", "two-histories"])
def test_tile_orders_by_rounds(q_lens, step, heads, dim):
    """Each order, at one workgroup a CU (D = 128, 256) and two (D = 64)."""
    g = torch.Generator().manual_seed(41)
    pf = torch.randint(0, 5, (len(q_lens),), generator=g).mul(step).tolist()
    c = make_case(35, q_lens, [p + q for p, q in zip(pf, q_lens)], pf, heads, heads, dim, page=16)
    run_split(c, 1)


@pytest.mark.parametrize("Hkv,splits,dim", [(1, 2, 128), (2, 3, 128), (3, 5, 64), (8, 2, 128),
                                            (5, 2, 256)])
def test_ranges_in_turn_cover_every_tile(Hkv, splits, dim):
    """Split prompts of at least 512 new tokens a sequence: one key range after the other."""
    c = make_case(43, [1300, 0, 600], [1700, 5, 640], [400, 5, 40], Hkv, Hkv, dim, page=16)
    run_split(c, splits)
