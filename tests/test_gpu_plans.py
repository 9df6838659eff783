"""One Operator, many call signatures: a call that looks its set-up up by
shapes, strides, scale and outputs returns what a fresh Operator returns, and
refuses what a fresh one refuses."""

import pytest
import torch

from fa_amd.binding import AttentionConfig, Operator

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
