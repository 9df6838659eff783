"""Ragged key tails read in place.

A key length that is no whole number of key blocks is read where it lies: the
buffer descriptors end at the last real row, and the rows past it arrive as
zeros. Nothing behind the last key may reach the output (NaN is planted
there), and K or V rows too far apart for 32-bit offsets, which still go
through padded copies, give the same output bit for bit.
"""

import pytest
import torch

from fa_amd.binding import AttentionConfig, Operator
from oracle import attention as orc

from test_gpu_parity import check, say

pytestmark = pytest.mark.gpu


def make(hq, hkv, nq, nk, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(1, hq, nq, 128, generator=g).half(),
            torch.randn(1, hkv, nk, 128, generator=g).half(),
            torch.randn(1, hkv, nk, 128, generator=g).half())


@pytest.mark.parametrize("splits", [None, 0, 3])
@pytest.mark.parametrize("kernel", [1, 2, 3, 4])
@pytest.mark.parametrize("nk", [1, 63, 65, 127, 129, 1001])
def test_nothing_behind_the_last_key_is_read(library_path, kernel, nk, splits):
    say(f"case tail kernel={kernel} nk={nk} splits={splits}")
    q, k, v = make(4, 2, 70, nk, seed=nk)
    room = -(-nk // 128) * 128 + 128
    kd, vd = (torch.full((1, 2, room, 128), float("nan"), dtype=torch.float16, device="cuda")
              for _ in range(2))
    kd[:, :, :nk] = k.cuda()
    vd[:, :, :nk] = v.cuda()
    op = Operator(library_path, AttentionConfig(kernel=kernel, splits=splits))
    out = op(q.cuda(), kd[:, :, :nk], vd[:, :, :nk]).float().cpu().numpy()
    check(out, orc.attention_f64(q, k, v), "fp32", "tail", orc.attention_f64(q, k, v.abs()))


@pytest.mark.parametrize("kernel", [3, 4])
@pytest.mark.parametrize("rows_apart", [(1 << 23) - 8, 1 << 23])
def test_far_rows_through_copies_bit_equal(library_path, kernel, rows_apart):
    """128 padded rows of 2^23 elements reach 2^31 bytes: from there on the
    rows are copied (nk = 5, so each tensor spans 84 MB)."""
    nk = 5
    say(f"case far rows kernel={kernel} n={rows_apart}")
    q, k, v = (t.cuda() for t in make(2, 1, 33, nk, seed=9))
    op = Operator(library_path, AttentionConfig(kernel=kernel))
    want = op(q, k, v).clone()
    far = []
    for t in (k, v):
        buf = torch.zeros(4 * rows_apart + 128, dtype=torch.float16, device="cuda")
        view = buf.as_strided((1, 1, nk, 128), (nk * rows_apart, nk * rows_apart, rows_apart, 1))
        view.copy_(t)
        far.append(view)
    got = op(q, *far)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("kernel", [3, 4])
def test_largest_head(library_path, kernel):
    """8388480 keys, one 128-key block short of the 2 GiB a head's rows may
    span: offsets of blocks past the last one must not fall into the buffer or
    wrap. The last key takes half of every row's weight."""
    nk = (1 << 23) - 128
    say(f"case largest head kernel={kernel}")
    g = torch.Generator(device="cuda").manual_seed(kernel)
    q, k, v = (torch.randn(1, h, n, 128, generator=g, device="cuda", dtype=torch.float16)
               for h, n in ((2, 1), (1, nk), (1, nk)))
    q[0, 1] = -q[0, 0]
    scores = (torch.cat([k[0, 0, i:i + (1 << 20)].float() @ q[0, 0, 0].float()
                         for i in range(0, nk, 1 << 20)]) * 128 ** -0.5).double()
    # k_last = a q makes its score a |q|^2 / sqrt(128): as much as all others together.
    want = torch.logsumexp(scores, 0) * 128 ** 0.5 / (q[0, 0, 0].double() ** 2).sum()
    k[0, 0, -1] = (want * q[0, 0, 0].double()).half()
    scores[-1] = (k[0, 0, -1].double() @ q[0, 0, 0].double()) * 128 ** -0.5
    out, lse = Operator(library_path, AttentionConfig(kernel=kernel, splits=64))(q, k, v, return_lse=True)
    for h, sign in ((0, 1.0), (1, -1.0)):
        exact_lse = torch.logsumexp(sign * scores, 0)
        w = torch.exp(sign * scores - exact_lse)
        exact = sum(w[i:i + (1 << 20)].float() @ v[0, 0, i:i + (1 << 20)].float()
                    for i in range(0, nk, 1 << 20))
        check(out[:, h:h + 1].float().cpu().numpy(), exact.cpu().numpy().reshape(1, 1, 1, 128), "fp32", "largest head")
        assert abs(float(lse[0, h, 0]) - float(exact_lse)) < 1e-3
