"""Short launches of the automatic tile equal the V^T tile.

Where every tile, or part of one, has a workgroup of its own and the keys are few, the
automatic choice reads V in its natural layout instead of running the prep
kernel first. Both give the same values in the same order, so outputs and lse
must be equal bit for bit on either side of that rule: ragged lengths, masks,
both accumulators, strides of every kind the entry points take, debug modes
and repeated graph replays. The V^T tile is held to the float64 oracle
throughout the suite. Which of the two ran shows in the workspace: V^T starts
at its first byte, and a launch that reads V in place leaves the first 256
bytes alone.
"""

import pytest
import torch

from fa_amd.binding import AttentionConfig, Operator

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

VT = 3


def draw(b, hq, hkv, nq, nk, seed, layout="bhnd"):
    g = torch.Generator().manual_seed(seed)

    def rand(h, n):
        t = torch.randn(b, h, n, 128, generator=g).half().cuda()
        return t if layout == "bhnd" else t.transpose(1, 2).contiguous().transpose(1, 2)

    return rand(hq, nq), rand(hkv, nk), rand(hkv, nk)


def read_in_place(op, *args, **kwargs):
    """Whether a call of op, which has its workspace, leaves the place of V^T alone."""
    op.workspace.fill_(0x5b)
    op(*args, **kwargs)
    torch.cuda.synchronize()
    return bool((op.workspace[:256] == 0x5b).all())


# (B, Hq, Hkv, Nq, Nk, causal, read in place): one key to the 64 key blocks the
# rule reaches, past them, a full round of 256 tiles and more than one (causal:
# without a mask the tiles past the first round are cut into key parts, which
# sum in another order; test_gpu_cut_tiles.py holds those to their bound).
CASES = [
    (1, 12, 1, 256, 1, "none", True), (1, 12, 1, 200, 127, "top_left", True),
    (2, 12, 1, 256, 128, "none", True), (1, 12, 1, 257, 129, "bottom_right", True),
    (1, 12, 1, 1000, 1000, "top_left", True), (1, 12, 1, 2049, 2049, "none", False),
    (1, 16, 16, 3000, 3001, "none", True), (1, 64, 8, 1024, 1024, "top_left", True),
    (1, 64, 8, 1025, 1025, "top_left", False), (1, 64, 8, 1000, 8192, "none", True),
    (1, 64, 8, 1000, 8193, "none", False), (2, 24, 2, 700, 555, "bottom_right", True),
]


@pytest.mark.parametrize("acc", ["fp32", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_equal_to_the_transposed_tile(library_path, case, acc):
    b, hq, hkv, nq, nk, causal, in_place = case
    for layout in ("bhnd", "bnhd"):
        say(f"case short {case} {acc} {layout}")
        q, k, v = draw(b, hq, hkv, nq, nk, nq + nk, layout)
        vt = Operator(library_path, AttentionConfig(acc=acc, causal=causal, kernel=VT))
        want = vt(q, k, v, return_lse=True)
        op = Operator(library_path, AttentionConfig(acc=acc, causal=causal))
        got = op(q, k, v, return_lse=True)
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (case, acc, layout)
        assert read_in_place(op, q, k, v, return_lse=True) == in_place
        assert not read_in_place(vt, q, k, v, return_lse=True)


# Parts of every length up to past the 64 key blocks, items up to past one
# round of 256; above 2048 query rows per KV head.
SPLIT_CASES = [
    (1, 12, 1, 256, 4099, "bottom_right", 33, False), (1, 12, 1, 256, 8192, "none", 21, True),
    (1, 12, 1, 300, 8321, "bottom_right", 2, False), (1, 32, 8, 600, 2500, "none", 2, True),
    (1, 12, 1, 256, 16640, "none", 2, False), (1, 12, 1, 256, 2048, "top_left", 22, True),
]


@pytest.mark.parametrize("case", SPLIT_CASES, ids=str)
def test_split_equal_to_the_transposed_tile(library_path, case):
    b, hq, hkv, nq, nk, causal, splits, in_place = case
    for acc, layout in (("fp32", "bhnd"), ("fp16", "bnhd")):
        say(f"case short split {case} {acc} {layout}")
        q, k, v = draw(b, hq, hkv, nq, nk, nq + nk, layout)
        want = Operator(library_path, AttentionConfig(acc=acc, causal=causal, splits=splits, kernel=VT))(q, k, v, return_lse=True)
        op = Operator(library_path, AttentionConfig(acc=acc, causal=causal, splits=splits))
        got = op(q, k, v, return_lse=True)
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (case, acc, layout)
        assert read_in_place(op, q, k, v) == in_place


def test_far_value_rows_keep_the_transposed_tile(library_path):
    """V rows at the distance from which 32-bit offsets no longer reach: the
    V^T tile reads them through 64-bit addresses, as before."""
    for apart in ((1 << 23) - 8, 1 << 23):
        say(f"case short far rows n={apart}")
        q, k, v = draw(1, 12, 1, 256, 5, 3)
        want = Operator(library_path, AttentionConfig(kernel=VT))(q, k, v).clone()
        buf = torch.zeros(4 * apart + 128, dtype=torch.float16, device="cuda")
        far = buf.as_strided((1, 1, 5, 128), (5 * apart, 5 * apart, apart, 1))
        far.copy_(v)
        op = Operator(library_path, AttentionConfig())
        assert torch.equal(op(q, k, far), want)
        assert read_in_place(op, q, k, far) == (apart < 1 << 23)


def test_debug_modes(library_path):
    say("case short debug modes")
    q, k, v = draw(1, 12, 1, 300, 700, 5)
    want = Operator(library_path, AttentionConfig(kernel=VT))(q, k, v).clone()
    for mode in ("sync", "trace", "capture"):
        op = Operator(library_path, AttentionConfig(**{mode: True}))
        assert torch.equal(op(q, k, v), want), mode
        # Sync mode poisons the workspace itself.
        assert mode == "sync" or read_in_place(op, q, k, v), mode


def test_captured_replays(library_path):
    say("case short graph")
    q, k, v = draw(1, 12, 1, 300, 700, 7)
    op, ref = Operator(library_path, AttentionConfig()), Operator(library_path, AttentionConfig(kernel=VT))
    op(q, k, v)
    assert read_in_place(op, q, k, v)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = op(q, k, v)
    for i in range(3):
        for t in (q, k, v):
            t.copy_(torch.randn_like(t))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref(q, k, v)), i
