"""One-pass launches whose last round of tiles is cut into parts of the keys.

A launch of more than one round of 256 tiles that leaves CUs idle in its last
round cuts those tiles; everything else about it stays. Checked where it can
go wrong: packed and unpacked rows, ragged queries and keys, several KV heads,
strided views, both accumulators, against the float64 oracle on sampled rows
and, over every row, against the same tile without cuts (selector 3); the
debug modes' bit equality; and a workspace without room for the parts.
"""

import ctypes as C

import numpy as np
import pytest
import torch

from fa_amd import binding
from fa_amd.binding import AttentionConfig, Operator
from oracle import attention as orc

from test_gpu_parity import ATOL, LSE_ATOL, LSE_RTOL, P_ROUND, RTOL, say

# (B, Hq, Hkv, Nq, Nk): 264 packed tiles of 24 blocks; 265 unpacked ones with a
# ragged last tile per head; 384 = one and a half rounds; 513, one tile over.
CUT = [(2, 24, 2, 1400, 3000), (1, 5, 5, 13400, 2001), (2, 12, 1, 4096, 4096),
       (1, 9, 3, 14510, 1500)]


def workspace_bytes(lib, shape, kernel=0, causal=0):
    b, hq, hkv, nq, nk = shape
    size = C.c_uint64()
    prob = binding.FaProblem(b, hq, hkv, nq, nk, 128, 128 ** -0.5, 0, kernel, causal)
    assert lib.fa_fwd_workspace_bytes(C.byref(prob), C.byref(size)) == 0
    return size.value


def test_workspace_holds_the_parts_only_where_tiles_are_cut(library_path):
    lib = binding.load_library(library_path)
    for shape in CUT:
        whole = workspace_bytes(lib, shape, kernel=3)
        size = workspace_bytes(lib, shape)
        rows = binding.query_tiles(*shape[:4]) % 256 * 256
        parts = (size - whole) // (rows * 129 * 4)
        assert 2 <= parts <= 16 and size == whole + parts * rows * 129 * 4, (shape, parts)
        assert size <= binding.NOALLOC_SCRATCH_BYTES
        assert workspace_bytes(lib, shape, causal=1) == workspace_bytes(lib, shape, 3, 1)
    # A whole number of rounds, less than one round, no room beside 64 MiB of V^T.
    for shape in ((1, 12, 1, 32768, 4096), (1, 12, 1, 4096, 4096), (2, 12, 1, 4096, 131072)):
        assert workspace_bytes(lib, shape) == workspace_bytes(lib, shape, kernel=3), shape


def make(shape, seed, sig=1.0):
    b, hq, hkv, nq, nk = shape
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(b, h, n, 128, generator=g) * s).half()
            for h, n, s in ((hq, nq, sig), (hkv, nk, sig), (hkv, nk, 1.0))]


@pytest.mark.gpu
@pytest.mark.parametrize("acc", ["fp32", "fp16"])
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("shape", CUT, ids=lambda s: "x".join(map(str, s)))
def test_cut_tiles_vs_f64(library_path, shape, strided, acc):
    say(f"case cut tiles {shape} strided={strided} acc={acc}")
    q, k, v = make(shape, seed=shape[3], sig=2.0 if strided else 1.0)
    dev = [t.cuda() for t in (q, k, v)]
    if strided:
        dev = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in dev]
    out, lse = Operator(library_path, AttentionConfig(acc=acc))(*dev, return_lse=True)
    whole, lse3 = Operator(library_path, AttentionConfig(acc=acc, kernel=3))(*dev, return_lse=True)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    # Both sides are within the oracle's bound, whose relative part is largest for FP16 O.
    diff = (out.float() - whole.float()).abs()
    assert bool((diff <= 2 * ATOL[acc] + 2 * RTOL[acc] * whole.float().abs()).all()), diff.max()
    assert float((lse - lse3).abs().max()) < LSE_ATOL
    assert not torch.equal(out, whole), "no tile was cut"
    rows = orc.sample_rows(q.shape, 48, seed=1)
    rows += [(shape[0] - 1, shape[1] - 1, n) for n in (shape[3] - 1, shape[3] - 200)]   # cut ones
    idx = torch.tensor(rows)
    got = out[idx[:, 0], idx[:, 1], idx[:, 2]].double().cpu().numpy()
    got_lse = lse[idx[:, 0], idx[:, 1], idx[:, 2]].double().cpu().numpy()
    exact = orc.attention_rows_f64(q, k, v, rows)
    wabs = orc.attention_rows_f64(q, k, v.abs(), rows)
    exact_lse = orc.lse_rows_f64(q, k, rows)
    err = np.abs(got - exact)
    assert bool(np.all(err <= ATOL[acc] + RTOL[acc] * np.abs(exact) + P_ROUND * (wabs + np.abs(exact)))), err.max()
    assert bool(np.all(np.abs(got_lse - exact_lse) <= LSE_ATOL + LSE_RTOL * np.abs(exact_lse)))


@pytest.mark.gpu
@pytest.mark.parametrize("acc", ["fp32", "fp16"])
def test_cut_tiles_debug_modes_and_small_workspace(library_path, acc):
    shape = CUT[0]
    say(f"case cut tiles modes {shape} acc={acc}")
    q, k, v = (t.cuda() for t in make(shape, seed=3))
    prod = Operator(library_path, AttentionConfig(acc=acc))
    out, lse = (t.clone() for t in prod(q, k, v, return_lse=True))
    so, sl = Operator(library_path, AttentionConfig(acc=acc, sync=True))(q, k, v, return_lse=True)
    traced = Operator(library_path, AttentionConfig(acc=acc, trace=True))
    to = traced(q, k, v)
    one, lone = Operator(library_path, AttentionConfig(acc=acc, splits=1))(q, k, v, return_lse=True)
    torch.cuda.synchronize()
    assert torch.equal(out, so) and torch.equal(lse, sl)
    assert torch.equal(out, to)
    assert torch.equal(out, one) and torch.equal(lse, lone)
    rec = traced.last["trace"].cpu().numpy()
    tiles = binding.query_tiles(*shape[:4])
    assert np.array_equal(rec[:, 5], np.arange(tiles))
    assert np.all(rec[:256, 6] == 24) and np.all(rec[256:, 6] < 24)
    # Room for V^T and the queues alone, as with selector 3: no tile is cut.
    b, hq, hkv, nq, nk = shape
    lib = binding.load_library(library_path)
    prob = binding.FaProblem(b, hq, hkv, nq, nk, 128, 128 ** -0.5, binding.FA_ACC[acc], 0, 0)
    ws = torch.empty(workspace_bytes(lib, shape, kernel=3), dtype=torch.uint8, device="cuda")
    got = torch.empty_like(q)
    assert lib.fa_fwd(C.byref(prob), q.data_ptr(), k.data_ptr(), v.data_ptr(), got.data_ptr(),
                      ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
    want = Operator(library_path, AttentionConfig(acc=acc, kernel=3))(q, k, v)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
