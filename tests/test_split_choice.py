"""Which kernel and how many parts the key-split forward takes by itself.

Up to 256 rows per KV head two kernels can run a split launch: the few-row
kernel, whose every 32 rows stream the keys for themselves, and the 256-row
tile. With one KV head the first is the faster one, with many the second; the
automatic choice compares both with their own part counts, and an explicit
count takes the kernel that is modelled to be the faster one with it. Both
round P against different running maxima, so that their outputs differ in the
last bits, which tells them apart here.
"""

import ctypes as C
import time

import pytest
import torch

from fa_amd import binding
from fa_amd.binding import AttentionConfig, Operator

CUS = 256


def parts(lib, shape, causal="none", splits=0, kernel=0):
    prob = binding.FaProblem(*shape, 128, 128 ** -0.5, 0, kernel, binding.FA_CAUSAL[causal])
    n = C.c_int32()
    assert lib.fa_fwd_split_count(C.byref(prob), splits, CUS, C.byref(n)) == 0
    return n.value


# (B, Hq, Hkv, Nq, Nk): rows for several KV heads behind enough keys that the
# parts have to fill the CUs; with 2 parts (or none) they took up to twice the
# time of the 256-row tile's own count.
MANY_HEADS = [(4, 32, 8, 57, 62129), (1, 16, 16, 241, 100393), (4, 64, 8, 25, 47916),
              (4, 16, 16, 178, 10937), (1, 96, 8, 14, 85632), (16, 1, 1, 1, 65536),
              (8, 64, 8, 1, 8192), (64, 1, 1, 160, 8192), (64, 1, 1, 256, 16384)]


@pytest.mark.parametrize("shape", MANY_HEADS, ids=lambda s: "x".join(map(str, s)))
def test_parts_fill_the_cus(library_path, shape):
    lib = binding.load_library(library_path)
    kv_heads = shape[0] * shape[2]
    n = parts(lib, shape)
    assert 0.6 * CUS <= kv_heads * n <= 1.1 * CUS, n
    assert parts(lib, shape, splits=n) == n


def test_hidden_keys_are_no_reason_to_split(library_path):
    """Eight rows of a top-left mask see one key block, however many there are."""
    lib = binding.load_library(library_path)
    assert parts(lib, (2, 8, 2, 8, 50000), causal="top_left") == 1
    assert parts(lib, (2, 8, 2, 8, 50000), causal="bottom_right") > 16


# (B, Hq, Hkv, Nq, Nk, splits, few-row kernel)
ROUTES = [
    (1, 12, 1, 1, 131072, 0, True), (1, 12, 1, 16, 20000, 0, True), (1, 8, 1, 32, 5000, 0, True),
    (1, 12, 1, 16, 20000, 9, True), (1, 8, 1, 32, 5000, 11, True),
    (1, 16, 16, 241, 9000, 0, False), (4, 16, 16, 178, 4100, 0, False),
    (4, 16, 16, 178, 4100, 4, False), (1, 257, 1, 1, 3000, 0, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("acc", ["fp32", "fp16"])
@pytest.mark.parametrize("case", ROUTES, ids=str)
def test_kernel_taken(library_path, case, acc):
    b, hq, hkv, nq, nk, splits, few_rows = case
    print(f"case route {case} {acc}", flush=True)
    g = torch.Generator().manual_seed(nk)
    q, k, v = (torch.randn(b, h, n, 128, generator=g).half().cuda()
               for h, n in ((hq, nq), (hkv, nk), (hkv, nk)))
    op = Operator(library_path, AttentionConfig(acc=acc, splits=splits))
    n = op.split_count(q.shape, k.shape)
    assert n > 1
    out, lse = op(q, k, v, return_lse=True)
    tile = Operator(library_path, AttentionConfig(acc=acc, splits=n, kernel=4 if hq // hkv * nq <= 2048 else 3))
    want, _ = tile(q, k, v, return_lse=True)
    again, lse2 = Operator(library_path, AttentionConfig(acc=acc, splits=n))(q, k, v, return_lse=True)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and torch.equal(lse, lse2), "the resolved count takes another way"
    assert torch.equal(out, want) == (not few_rows)


def host_us(fn):
    """Shortest mean of several short runs: other processes only lengthen one."""
    def mean():
        start = time.perf_counter()
        for _ in range(100):
            fn()
        return (time.perf_counter() - start) * 1e4

    return min(mean() for _ in range(20))


def test_causal_search_costs_little_more_than_the_unmasked_one(library_path):
    """300 rows of 12 heads behind 16000 keys: 15 tiles and 125 counts. A walk
    over the tiles for every count made the search six times the unmasked one."""
    lib = binding.load_library(library_path)
    shape = (1, 12, 1, 300, 16000)
    assert parts(lib, shape, "bottom_right") > 1
    masked = host_us(lambda: parts(lib, shape, "bottom_right"))
    unmasked = host_us(lambda: parts(lib, shape))
    print(f"masked {masked:.1f} us, unmasked {unmasked:.1f} us")
    assert masked < 3 * unmasked


@pytest.mark.gpu
def test_operator_resolves_the_count_once(library_path):
    print("case resolved count", flush=True)
    op = Operator(library_path, AttentionConfig(splits=0, causal="bottom_right"))
    q = torch.randn(1, 12, 300, 128, device="cuda").half()
    k = torch.randn(1, 1, 16000, 128, device="cuda").half()
    op(q, k, k)
    (plan,) = op.plans.values()
    assert plan.before[1] == op.split_count(q.shape, k.shape) > 1


# (B, Hq, Hkv, Nq, Nk, mask, most parts): more items than CUs bring back the
# pass over V and the queues; parts that many tiles cannot use only cost a merge.
@pytest.mark.parametrize("shape,causal,most", [
    ((3, 1, 1, 2329, 2329), "top_left", 8), ((1, 1, 1, 3589, 10404), "top_left", 17),
    ((2, 12, 2, 576, 1104), "top_left", 1), ((3, 8, 4, 3544, 5788), "top_left", 1),
    ((1, 64, 64, 1087, 6144), "bottom_right", 1), ((4, 2, 1, 2421, 2862), "bottom_right", 4),
], ids=str)
def test_causal_parts_stay_within_the_cus(library_path, shape, causal, most):
    lib = binding.load_library(library_path)
    assert 1 <= parts(lib, shape, causal) <= most
