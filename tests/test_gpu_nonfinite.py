"""NaN and infinity in the inputs come out of the merged forms of the forward
as out of the one-pass tile.

A NaN in a query row, or an infinity, makes every score of the row NaN or
infinite; in a key it does so for every row that scores it above the rest, in
a value for one dim of every row. The parts of a cut tile or of a split launch
must not lose it when they are combined: the merge once took NaN for "sees no
key" and wrote O = 0, lse = -inf. Both merge kernels, behind the cut tiles,
the split 256-row tiles and the few-row kernel, are held to the unsplit
V^T tile: NaN and infinities at the same places, finite values within the
oracle's bounds of each other.
"""

import pytest
import torch

from fa_amd.binding import AttentionConfig, Operator

from test_gpu_parity import ATOL, LSE_ATOL, RTOL, say

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")

# (B, Hq, Hkv, Nq, Nk, kernel, splits): 264 tiles of which the last 8 are cut;
# split 256-row tiles under the row and the workgroup-per-row merge; the
# few-row kernel under both.
SHAPES = {
    "cut": (2, 24, 2, 1400, 3000, 0, None),
    "tiles": (1, 12, 2, 300, 3000, 4, 3),
    "tiles_wide": (1, 12, 2, 40, 4500, 4, 35),
    "rows": (1, 12, 2, 30, 3000, 0, 5),
    "rows_wide": (1, 12, 2, 5, 6000, 0, 47),
}
# What is planted, in (batch 0, KV head 1) of each launch and its last query rows.
PLANTS = {
    "query_nan": lambda q, k, v: q[0, -1, -1, 5].fill_(NAN),
    "query_inf": lambda q, k, v: q[-1, -1, -1, 5].fill_(INF),
    "first_query_nan": lambda q, k, v: q[0, 0, 0].fill_(NAN),
    "key_nan": lambda q, k, v: k[-1, -1, 1234, 7].fill_(NAN),
    "key_inf": lambda q, k, v: k[-1, -1, 1234, 7].fill_(INF),
    "value_nan": lambda q, k, v: v[-1, -1, 1234, 9].fill_(NAN),
    "value_inf": lambda q, k, v: v[-1, -1, 1234, 9].fill_(-INF),
}


def same(got, want, atol, rtol, what):
    assert torch.equal(got.isnan(), want.isnan()), what + ": NaN at other places"
    assert torch.equal(got.isposinf(), want.isposinf()), what + ": infinities"
    assert torch.equal(got.isneginf(), want.isneginf()), what + ": negative infinities"
    ok = want.isfinite()
    g, w = got[ok].float(), want[ok].float()
    assert bool(((g - w).abs() <= atol + rtol * w.abs()).all()), what


@pytest.mark.parametrize("acc", ["fp32", "fp16"])
@pytest.mark.parametrize("plant", PLANTS)
@pytest.mark.parametrize("shape", SHAPES)
def test_nonfinite_inputs_as_in_one_pass(library_path, shape, plant, acc):
    say(f"case nonfinite {shape} {plant} {acc}")
    b, hq, hkv, nq, nk, kernel, splits = SHAPES[shape]
    g = torch.Generator().manual_seed(nq + nk)
    q, k, v = (torch.randn(b, h, n, 128, generator=g).half().cuda()
               for h, n in ((hq, nq), (hkv, nk), (hkv, nk)))
    PLANTS[plant](q, k, v)
    got = Operator(library_path, AttentionConfig(acc=acc, kernel=kernel, splits=splits))(q, k, v, return_lse=True)
    want = Operator(library_path, AttentionConfig(acc=acc, kernel=3))(q, k, v, return_lse=True)
    torch.cuda.synchronize()
    assert not bool(want[0].isfinite().all()), "nothing was planted"
    # Both sides are within the oracle's bounds of the exact value.
    same(got[0], want[0], 2 * ATOL[acc], 2 * RTOL[acc], "O")
    same(got[1], want[1], 2 * LSE_ATOL, 0.0, "lse")
