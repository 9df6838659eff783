"""One Operator, many call signatures: a call that looks its set-up up by
shapes, strides, scale and outputs returns what a fresh Operator returns, and
refuses what a fresh one refuses."""

import pytest
import torch

from fa_amd.binding import SIGNATURES_KEPT, AttentionConfig, Operator

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [None, 0])
def test_signatures_do_not_mix(library_path, splits):
    say(f"case signatures splits={splits}")
    g = torch.Generator().manual_seed(4)
    draws = {(b, h, n): torch.randn(b, h, n, 128, generator=g).half().cuda()
             for b, h, n in ((1, 4, 33), (1, 4, 300), (1, 2, 300), (1, 2, 517))}
    q, big, k, long = draws[1, 4, 33], draws[1, 4, 300], draws[1, 2, 300], draws[1, 2, 517]

    def bnhd(t):
        return t.transpose(1, 2).contiguous().transpose(1, 2)

    calls = [(q, k, k, {}), (bnhd(q), k, k, {}), (q, bnhd(k), k, {}), (q, long[:, :, :300], k, {}),
             (q, k, k, {"scale": 0.2}), (q, k, k, {"scale": torch.tensor(0.3)}),
             (q, k, k, {"return_lse": True}), (big, long, long, {"return_lse": True}),
             (big[:, :, :33], k, k, {})]
    op = Operator(library_path, AttentionConfig(splits=splits))
    for rep in range(2):
        for i, (a, b, c, kw) in enumerate(calls):
            got = op(a, b, c, **kw)
            want = Operator(library_path, AttentionConfig(splits=splits))(a, b, c, **kw)
            got, want = (got, want) if "return_lse" in kw else ((got,), (want,))
            torch.cuda.synchronize()
            assert all(torch.equal(x, y) for x, y in zip(got, want)), (rep, i)
    # The same signature at an address that is not 16-byte aligned.
    room = torch.zeros(k.numel() + 8, dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError, match="16-byte"):
        op(q, room[4:4 + k.numel()].view(k.shape), k)
    with pytest.raises(ValueError, match="FP16"):
        op(q, k.float(), k)
    with pytest.raises(ValueError, match="finite"):
        op(q, k, k, scale=float("nan"))
    # Another stream: its own order of launches, the same result.
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = op(q, k, k).clone()
    side.synchronize()
    assert torch.equal(got, Operator(library_path, AttentionConfig(splits=splits))(q, k, k))


def test_a_growing_cache_keeps_memory_flat(library_path):
    """A decode loop has a new key length, so a new signature, in every step:
    what an Operator keeps for them is bounded, and an output that the caller
    holds is neither handed out for another length nor replaced."""
    say("case growing cache")
    g = torch.Generator().manual_seed(6)
    q = torch.randn(2, 16, 1, 128, generator=g).half().cuda()
    cache = torch.randn(2, 2, 700, 128, generator=g).half().cuda()
    op = Operator(library_path, AttentionConfig(splits=0))
    held = {}
    op(q, cache, cache)                             # the largest workspace
    for n in (60, 61):
        held[n] = op(q, cache[:, :, :n], cache[:, :, :n])
    torch.cuda.synchronize()
    want = {n: t.clone() for n, t in held.items()}
    used = []
    for step in range(4):
        for n in range(62 + 3 * step * SIGNATURES_KEPT // 4, 62 + 3 * (step + 1) * SIGNATURES_KEPT // 4):
            out = op(q, cache[:, :, :n], cache[:, :, :n], return_lse=n % 2 == 0)
            out = out[0] if n % 2 == 0 else out
            assert all(out.data_ptr() != t.data_ptr() for t in held.values())
        assert len(op.plans) <= SIGNATURES_KEPT
        used.append(torch.cuda.memory_allocated())
    torch.cuda.synchronize()
    # Outputs and lse of at most SIGNATURES_KEPT lengths, in blocks of 512 bytes each.
    assert max(used) - min(used) <= SIGNATURES_KEPT * (2 * 16 * 128 * 2 + 512)
    for n, t in held.items():
        assert torch.equal(t, want[n])
        assert op(q, cache[:, :, :n], cache[:, :, :n]).data_ptr() == t.data_ptr()


def test_captured_calls_outlive_their_signatures(library_path):
    """A graph replays into the buffers of its capture, also after so many
    other signatures that the set-up of its own was dropped."""
    say("case captured signatures")
    g = torch.Generator().manual_seed(8)
    q = torch.randn(1, 16, 1, 128, generator=g).half().cuda()
    cache = torch.randn(1, 2, 3000, 128, generator=g).half().cuda()
    op = Operator(library_path, AttentionConfig(splits=0))
    k = cache[:, :, :1000]
    op(q, k, k)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        kept = op(q, k, k).clone()
    for n in range(2000, 2000 + 2 * SIGNATURES_KEPT):   # larger workspaces too
        op(q, cache[:, :, :n], cache[:, :, :n])
    others = [torch.full((1 << n,), 7, dtype=torch.uint8, device="cuda") for n in range(9, 22) for _ in range(4)]
    for i in range(3):
        q.copy_(torch.randn_like(q))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(kept, Operator(library_path, AttentionConfig(splits=0))(q, k, k)), i
        assert all(bool((t == 7).all()) for t in others)
