"""Graph capture of launches that run more than one attention kernel's worth of
work: cut tiles behind work queues, and the few-row kernel; and of a first call
of a shape, whose kernels must have been set up by the first call of the
selector and variant, whatever that call's shape was.
"""

import shutil

import pytest
import torch

from fa_amd.binding import AttentionConfig, Operator

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

# (B, Hq, Hkv, Nq, Nk, splits): uncut packed and unpacked launches of either V
# layout, cut ones, split 256-row tiles and the few-row kernel.
SHAPES = {
    "natural": (1, 12, 1, 64, 500, None),
    "transposed": (1, 12, 1, 4096, 4096, None),
    "unpacked": (1, 4, 4, 3000, 9000, None),
    "cut": (2, 24, 2, 1400, 3000, None),
    "cut_unpacked": (1, 5, 5, 13400, 2001, None),
    "tiles": (1, 16, 16, 241, 5000, 0),
    "rows": (1, 12, 1, 16, 20000, 0),
    "parts": (1, 12, 1, 300, 8000, 0),
}


def draw(shape):
    b, hq, hkv, nq, nk, _ = SHAPES[shape]
    return [torch.randn(b, h, n, 128, device="cuda").half() for h, n in ((hq, nq), (hkv, nk), (hkv, nk))]


def capture(op, tensors):
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = op(*tensors)
    return graph, out


def replays(library, graph, out, tensors, splits):
    torch.manual_seed(3)
    ref = Operator(library, AttentionConfig(splits=splits))
    for i in range(3):
        for t in tensors:
            t.copy_(torch.randn_like(t))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref(*tensors)), i


@pytest.mark.parametrize("shape", ["cut", "cut_unpacked", "tiles", "rows"])
def test_captured_replays(library_path, shape):
    say(f"case captured {shape}")
    splits = SHAPES[shape][-1]
    tensors = draw(shape)
    op = Operator(library_path, AttentionConfig(splits=splits))
    op(*tensors)
    replays(library_path, *capture(op, tensors), tensors, splits)


@pytest.mark.parametrize("first", ["natural", "transposed"])
def test_set_up_by_the_first_call_of_any_shape(library_path, tmp_path, first):
    """A copy of the library has state of its own, so its first call is here."""
    fresh = str(shutil.copy(library_path, tmp_path / f"libfa_hip_{first}.so"))
    Operator(fresh)(*draw(first))
    for shape in SHAPES:
        say(f"case first call captured: {shape} after {first}")
        tensors = draw(shape)
        splits = SHAPES[shape][-1]
        graph, out = capture(Operator(fresh, AttentionConfig(splits=splits)), tensors)
        replays(library_path, graph, out, tensors, splits)
