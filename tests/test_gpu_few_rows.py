"""The few-row split kernel: at most eight 32-row tiles per KV head, each wave
of a workgroup on its own 32-key blocks.

Checked against the float64 oracle where it can go wrong: one row, a full and
a just overfull tile, the most tiles it takes and one row more (which the
256-row tiles take), parts with fewer blocks than waves, parts that see no
key, ragged keys with NaN planted behind the last one, sequence-major views,
heads that do not share a KV head, and rows too far apart for 32-bit offsets.
"""

import numpy as np
import pytest
import torch

from fa_amd.binding import AttentionConfig, Operator
from oracle import attention as orc

from test_gpu_parity import check, check_lse, say

pytestmark = pytest.mark.gpu


def make(b, hq, hkv, nq, nk, seed, sig=1.0):
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(b, hq, nq, 128, generator=g) * sig).half()
    k = (torch.randn(b, hkv, nk, 128, generator=g) * sig).half()
    v = torch.randn(b, hkv, nk, 128, generator=g).half()
    if sig > 1:
        v[:, :, ::23] *= 8
    return q, k, v


# (B, Hq, Hkv, Nq, Nk, causal, splits, few-row kernel): short parts of few rows
# run on the 256-row tile, which is then the faster one. None: the rows see one
# block of 32 keys, where both kernels may give the same bits.
CASES = [
    (1, 12, 1, 1, 129, "none", 2, False),           # two blocks in all, one key in the last
    (1, 12, 1, 8, 129, "none", 2, True),
    (1, 12, 1, 1, 4099, "none", 0, False),
    (1, 12, 1, 1, 4099, "none", 17, True),
    (2, 8, 2, 8, 1000, "none", 3, True),            # 32 packed rows: one full tile
    (2, 8, 2, 8, 1000, "top_left", 3, None),        # only the first 8 keys are seen
    (2, 16, 2, 16, 1000, "top_left", 3, None),      # the first 16, by 128 rows
    (1, 3, 1, 11, 2048, "bottom_right", 5, True),   # 33 rows: a tile of one row
    (1, 1, 1, 31, 777, "bottom_right", 7, False),
    (1, 1, 1, 31, 777, "bottom_right", 3, True),
    (3, 4, 4, 1, 515, "none", 2, True),             # no shared KV heads
    (1, 12, 1, 16, 5001, "bottom_right", 0, True),  # 192 rows, 6 tiles
    (1, 8, 1, 32, 3000, "none", 11, True),          # 256 rows, the most it takes
    (1, 1, 1, 257, 3000, "none", 4, False),         # one more
    (1, 2, 1, 128, 64 * 128, "bottom_right", 64, False),
    (1, 2, 1, 128, 64 * 128, "bottom_right", 30, True),
    (2, 2, 1, 70, 300, "bottom_right", 3, True),
    (1, 2, 2, 200, 130, "bottom_right", 2, True),   # rows 0..69 see no key
]


@pytest.mark.parametrize("layout", ["bhnd", "bnhd"])
@pytest.mark.parametrize("acc", ["fp32", "fp16"])
@pytest.mark.parametrize("b,hq,hkv,nq,nk,causal,splits,few_rows", CASES)
def test_few_rows_vs_f64(library_path, b, hq, hkv, nq, nk, causal, splits, few_rows, acc, layout):
    say(f"case few rows B{b} Hq{hq} Hkv{hkv} nq={nq} nk={nk} causal={causal} splits={splits} "
        f"acc={acc} {layout}")
    q, k, v = make(b, hq, hkv, nq, nk, seed=nq * 31 + nk)
    behind = 128                                # keys behind the last one, all NaN
    dev = [q.cuda()]
    for t in (k, v):
        shape = (b, hkv, nk + behind, 128) if layout == "bhnd" else (b, nk + behind, hkv, 128)
        room = torch.full(shape, float("nan"), dtype=torch.float16, device="cuda")
        room = (room if layout == "bhnd" else room.transpose(1, 2))[:, :, :nk]
        room.copy_(t)
        dev.append(room)
    op = Operator(library_path, AttentionConfig(acc=acc, causal=causal, splits=splits))
    say(f"  parts per tile: {op.split_count(q.shape, k.shape)}")
    out, lse = op(*dev, return_lse=True)
    torch.cuda.synchronize()
    out = out.float().cpu().numpy()
    check(out, orc.attention_f64(q, k, v, causal=causal), acc, "few rows",
          orc.attention_f64(q, k, v.abs(), causal=causal))
    exact_lse = orc.lse_f64(q, k, causal=causal)
    check_lse(lse.cpu().numpy(), exact_lse, "few rows")
    empty = np.isneginf(exact_lse)
    assert bool(np.all(out[empty] == 0)), "rows without keys must be exactly zero"
    # The kernels round P against other running maxima: other bits, another kernel.
    tile = AttentionConfig(acc=acc, causal=causal, splits=op.split_count(q.shape, k.shape), kernel=4)
    same = np.array_equal(out, Operator(library_path, tile)(*dev).float().cpu().numpy())
    assert few_rows is None or same != few_rows


@pytest.mark.parametrize("acc", ["fp32", "fp16"])
def test_few_rows_stress_and_repeat(library_path, acc):
    """Peaked rows: the waves' maxima differ widely when they are combined."""
    say(f"case few rows stress acc={acc}")
    q, k, v = make(2, 6, 2, 9, 6000, seed=5, sig=3.0)
    op = Operator(library_path, AttentionConfig(acc=acc, splits=3))
    out, lse = (t.clone() for t in op(q.cuda(), k.cuda(), v.cuda(), return_lse=True))
    again, lse2 = op(q.cuda(), k.cuda(), v.cuda(), return_lse=True)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and torch.equal(lse, lse2)
    check(out.float().cpu().numpy(), orc.attention_f64(q, k, v), acc, "few rows stress",
          orc.attention_f64(q, k, v.abs()))
    check_lse(lse.cpu().numpy(), orc.lse_f64(q, k), "few rows stress")


@pytest.mark.parametrize("heads", [4, 48])        # the 256-row tile, the few-row kernel
@pytest.mark.parametrize("rows_apart", [(1 << 22) - 8, 1 << 22])
def test_few_rows_far_apart(library_path, rows_apart, heads):
    """130 keys 2^22 elements apart are copied (256 padded rows span 2 GiB),
    8 elements closer they are read in place: the same output bit for bit."""
    nk = 130
    say(f"case few rows far apart n={rows_apart} heads={heads}")
    q, k, v = (t.cuda() for t in make(1, heads, 1, 2, nk, seed=9))
    op = Operator(library_path, AttentionConfig(splits=2))
    want = op(q, k, v).clone()
    far = []
    for t in (k, v):
        buf = torch.empty((nk - 1) * rows_apart + 128, dtype=torch.float16, device="cuda")
        view = buf.as_strided((1, 1, nk, 128), (nk * rows_apart, nk * rows_apart, rows_apart, 1))
        view.copy_(t)
        far.append(view)
    got = op(q, *far)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
