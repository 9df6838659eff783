"""ctypes binding of ``libfa_hip.so``: public inputs q/k/v, public output O.

Mirrors the reference's operator binding
(``backends/cce_fa_nk_nz_vector_fp32_v5_sumpack/binding.py:6-110``):

  * the library is opened with ``RTLD_LOCAL``;
  * a call is two-phase: ``fa_fwd_workspace_bytes`` sizes the workspace,
    ``fa_fwd`` (or ``fa_fwd_lse`` when the per-row log-sum-exp is asked for)
    enqueues the forward on the current torch stream;
  * geometry, dtype, device and layout errors raise ``ValueError`` before any
    launch (any [B,H,N,128] view whose last dimension is contiguous and whose
    rows are 16-byte aligned is accepted: non-contiguous views, such as the
    sequence-major tensors of FlashAttention-style code, go through
    ``fa_fwd_strided`` without a copy); a nonzero library status raises ``RuntimeError("fa_fwd <where>:
    <status> (<message>)")``;
  * output and workspace tensors are allocated by torch, cached per
    (shapes, device, config), and the same cached output tensor is returned
    on every call; the workspace grows on demand. After ``SIGNATURES_KEPT``
    call signatures the set-up of all of them is dropped, and with it the
    outputs that nobody else holds. Calls of one ``Operator``
    therefore share its output and workspace: forwards that may overlap on
    different streams need an ``Operator`` each.

Nothing here falls back to another implementation: without the built library
construction fails.
"""

import ctypes as C
import math
import struct
import weakref
from dataclasses import dataclass

FA_ACC = {"fp32": 0, "fp16": 1}
# Attention masks (enum fa_causal): full attention, the reference's only mode,
# or a causal mask aligned top-left (key j <= query i, torch's
# scaled_dot_product_attention(is_causal=True)) or bottom-right
# (j <= i + Nk - Nq).
FA_CAUSAL = {"none": 0, "top_left": 1, "bottom_right": 2}
# 64-bit words per query-tile record of trace mode (fa_fwd_trace).
TRACE_WORDS = 8
# Workspace bytes fa_fwd_noalloc's static device array holds (FA_NOALLOC_SCRATCH_BYTES).
NOALLOC_SCRATCH_BYTES = (64 << 20) + (64 << 10)


class FaProblem(C.Structure):
    _fields_ = [
        ("batch", C.c_int64),
        ("heads_q", C.c_int64),
        ("heads_kv", C.c_int64),
        ("seq_q", C.c_int64),
        ("seq_k", C.c_int64),
        ("dim", C.c_int64),
        ("scale", C.c_float),
        ("acc", C.c_int32),
        ("kernel", C.c_int32),
        ("causal", C.c_int32),
    ]


class FaStrides(C.Structure):
    """Element strides of dims B, H, N of q, k, v and o (``fa_strides``)."""
    _fields_ = [("q", C.c_int64 * 3), ("k", C.c_int64 * 3), ("v", C.c_int64 * 3),
                ("o", C.c_int64 * 3)]


# Every symbol include/fa_hip.h declares, with its ctypes signature.
SIGNATURES = {
    "fa_fwd_workspace_bytes": (C.c_int, [C.POINTER(FaProblem), C.POINTER(C.c_uint64)]),
    "fa_fwd": (C.c_int, [C.POINTER(FaProblem), C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                         C.c_void_p, C.c_uint64, C.c_void_p]),
    "fa_fwd_lse": (C.c_int, [C.POINTER(FaProblem), C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                             C.c_void_p, C.c_void_p, C.c_uint64, C.c_void_p]),
    "fa_fwd_strided": (C.c_int, [C.POINTER(FaProblem), C.POINTER(FaStrides), C.c_void_p,
                                 C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                                 C.c_uint64, C.c_void_p]),
    "fa_fwd_capture_count": (C.c_int, [C.POINTER(FaProblem), C.POINTER(C.c_uint64),
                                       C.POINTER(C.c_int32)]),
    "fa_fwd_capture": (C.c_int, [C.POINTER(FaProblem), C.c_void_p, C.c_void_p, C.c_void_p,
                                 C.c_void_p, C.c_void_p, C.c_void_p, C.c_uint64, C.c_void_p,
                                 C.c_uint64, C.c_void_p]),
    "fa_fwd_trace_count": (C.c_int, [C.POINTER(FaProblem), C.POINTER(C.c_uint64)]),
    "fa_fwd_trace": (C.c_int, [C.POINTER(FaProblem), C.c_void_p, C.c_void_p, C.c_void_p,
                               C.c_void_p, C.c_void_p, C.c_uint64, C.c_void_p, C.c_uint64,
                               C.c_void_p]),
    "fa_fwd_sync": (C.c_int, [C.POINTER(FaProblem), C.c_void_p, C.c_void_p, C.c_void_p,
                              C.c_void_p, C.c_void_p, C.c_void_p, C.c_uint64, C.c_void_p]),
    "fa_fwd_noalloc": (C.c_int, [C.POINTER(FaProblem), C.c_void_p, C.c_void_p, C.c_void_p,
                                 C.c_void_p, C.c_void_p]),
    "fa_fwd_split_count": (C.c_int, [C.POINTER(FaProblem), C.c_int32, C.c_int32,
                                     C.POINTER(C.c_int32)]),
    "fa_fwd_split_workspace_bytes": (C.c_int, [C.POINTER(FaProblem), C.c_int32,
                                               C.POINTER(C.c_uint64)]),
    "fa_fwd_split": (C.c_int, [C.POINTER(FaProblem), C.c_int32, C.POINTER(FaStrides), C.c_void_p,
                               C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                               C.c_uint64, C.c_void_p]),
    "fa_fwd_tile": (C.c_int, [C.POINTER(FaProblem), C.POINTER(C.c_int32), C.POINTER(C.c_int32)]),
    "fa_fwd_select": (C.c_int, [C.POINTER(FaProblem), C.POINTER(C.c_int32)]),
    "fa_kernel_count": (C.c_int, []),
    "fa_kernel_name": (C.c_char_p, [C.c_int32]),
    "fa_strerror": (C.c_char_p, [C.c_int]),
}


def load_library(path):
    """Open the shared library and attach the C signatures of every entry point."""
    lib = C.CDLL(str(path), mode=C.RTLD_LOCAL)
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    return lib


@dataclass(frozen=True)
class AttentionConfig:
    """Launch configuration: accumulation variant, tile selector (0 = automatic),
    capture (debug) mode, which records every row's online-softmax
    statistics per key block (the reference config's ``capture`` flag,
    ``backends/cce_fa_nk_nz_vector_fp32_v5_sumpack/backend.py:27``), the
    attention mask (``FA_CAUSAL``; a row that sees no key gets O = 0 and
    lse = -inf), trace mode, which records per 256-row query tile where
    it ran and its clock stamps (the reference kernel's ``trace`` output),
    and the synchronous debug mode (``fa_fwd_sync``: poisoned staging
    buffers, no load/compute overlap; the reference's ``SYNCHRONOUS`` build
    flag), whose output must equal the production kernel's bit for bit.
    ``splits`` selects the key-split forward (``fa_fwd_split``): None (the
    default) runs one work item per query tile, 0 lets the library choose a
    split count, n >= 1 asks for n parts of every tile's key range (1 is the
    unsplit forward)."""
    acc: str = "fp32"
    kernel: int = 0
    capture: bool = False
    causal: str = "none"
    trace: bool = False
    sync: bool = False
    splits: "int | None" = None

    def __post_init__(self):
        if self.acc not in FA_ACC:
            raise ValueError(f"unknown accumulation variant {self.acc!r}")
        if not isinstance(self.kernel, int) or self.kernel < 0:
            raise ValueError("kernel selector must be a non-negative int")
        if not isinstance(self.capture, bool):
            raise ValueError("capture must be a bool")
        if self.causal not in FA_CAUSAL:
            raise ValueError(f"unknown causal mode {self.causal!r}")
        if not isinstance(self.trace, bool):
            raise ValueError("trace must be a bool")
        if not isinstance(self.sync, bool):
            raise ValueError("sync must be a bool")
        if self.trace + self.capture + self.sync > 1:
            raise ValueError("capture, trace and sync are separate kernels; pick one")
        if self.splits is not None:
            if not isinstance(self.splits, int) or isinstance(self.splits, bool) \
                    or not 0 <= self.splits <= 1024:
                raise ValueError("splits must be None or an int in 0..1024")
            if self.capture or self.trace or self.sync:
                raise ValueError("the key-split forward has no capture, trace or sync mode")


LAYOUT_ERROR = ("Q/K/V must be [B,H,N,128] views with a contiguous last dimension and 16-byte "
                "aligned rows")

# Query rows per attention tile.
TILE_ROWS = 256

# Call signatures an Operator keeps set up. A decode loop has a new one (one
# more key) in every step, so there has to be a limit; a program's recurring
# ones are far fewer.
SIGNATURES_KEPT = 64


def query_tiles(batch, heads_q, heads_kv, seq_q):
    """Attention tiles of one launch, as the library lays them out: unpacked,
    ``batch * heads_q`` row sequences of ``seq_q`` query rows; packed, when
    that needs fewer 256-row tiles (grouped-query attention with few query
    rows), ``batch * heads_kv`` sequences of ``seq_q * group`` rows, the
    group's query heads position by position. Every row's result is the same
    either way, but for tiles cut into key parts. (One trace record per tile: ``fa_fwd_trace_count`` / 8.)"""
    def tiles(seqs, rows):
        return seqs * -(-rows // TILE_ROWS)

    plain = tiles(batch * heads_q, seq_q)
    group = heads_q // heads_kv
    if group <= 1 or seq_q * group >= 2 ** 30:
        return plain
    return min(plain, tiles(batch * heads_kv, seq_q * group))


def make_problem(q_shape, k_shape, scale, config):
    b, hq, nq, d = q_shape
    _, hkv, nk, _ = k_shape
    return FaProblem(b, hq, hkv, nq, nk, d, float(scale), FA_ACC[config.acc], config.kernel,
                     FA_CAUSAL[config.causal])


class Plan:
    """What a call derives from its signature alone (shapes, strides, dtypes,
    devices, scale and outputs): the checks of ``Operator.validate`` passed,
    the problem and the library function with the arguments around the
    pointers, the output buffers and the workspace size."""
    __slots__ = ("config", "fn", "before", "after", "size", "out", "lse", "stats", "block", "trace",
                 "outputs", "extra")


class Operator:
    """Callable ``(q, k, v) -> o`` over ``libfa_hip.so``."""

    def __init__(self, library, config=AttentionConfig()):
        self.config = config
        self.lib = load_library(library) if not isinstance(library, C.CDLL) else library
        self.workspace = None
        self.plans = {}          # call signature -> Plan
        # Weak references to the outputs of the plans, and to those of dropped
        # plans that the caller still holds: a signature met again gets the same
        # tensor, and no two live outputs of different shapes share memory.
        self.buffers = {}
        self.captured = {}       # plans and workspaces that captured graphs refer to
        self.streams = {}        # (device index, raw stream) -> torch stream
        self.tiles = {}          # selector -> (rows, keys) granularity
        self.last = None

    def message(self, status):
        text = self.lib.fa_strerror(status)
        return text.decode() if text else "unknown status"

    def check(self, status, where):
        if status:
            raise RuntimeError(f"fa_fwd {where}: {status} ({self.message(status)})")

    def tile(self, q_shape, k_shape):
        """(query rows, keys) granularity of the kernel the library would use.
        Every tile masks ragged tails, so it follows from the selector alone."""
        kernel = self.config.kernel
        if kernel not in self.tiles:
            prob = make_problem(q_shape, k_shape, 1.0, self.config)
            rows, keys = C.c_int32(), C.c_int32()
            self.check(self.lib.fa_fwd_tile(C.byref(prob), C.byref(rows), C.byref(keys)), "tile")
            self.tiles[kernel] = (rows.value, keys.value)
        return self.tiles[kernel]

    def kernel(self, q_shape, k_shape):
        """1-based tile configuration the library would launch (automatic choice resolved)."""
        prob = make_problem(q_shape, k_shape, 1.0, self.config)
        idx = C.c_int32()
        self.check(self.lib.fa_fwd_select(C.byref(prob), C.byref(idx)), "select")
        return idx.value

    def kernel_name(self, q_shape, k_shape):
        return self.lib.fa_kernel_name(self.kernel(q_shape, k_shape)).decode()

    def split_count(self, q_shape, k_shape, cus=0):
        """Key-range parts per query tile the key-split forward would run
        (``config.splits`` resolved; ``cus`` = 0: the current device)."""
        if self.config.splits is None:
            return 1
        return self.problem_splits(make_problem(q_shape, k_shape, 1.0, self.config), cus)

    def problem_splits(self, prob, cus=0):
        n = C.c_int32()
        self.check(self.lib.fa_fwd_split_count(C.byref(prob), self.config.splits, cus,
                                               C.byref(n)), "split")
        return n.value

    def validate(self, q, k, v):
        import torch

        if q.ndim != 4 or k.ndim != 4 or v.shape != k.shape:
            raise ValueError("Q/K/V must be [B,H,N,128]")
        b, h, nq, d = q.shape
        if min(q.shape) <= 0 or min(k.shape) <= 0 or k.shape[0] != b or d != 128 \
                or k.shape[3] != 128 or h % k.shape[1]:
            raise ValueError("invalid attention geometry")
        rows, keys = self.tile(q.shape, k.shape)
        if nq % rows or k.shape[2] % keys or max(nq, k.shape[2]) >= 2 ** 30:
            raise ValueError(f"unsupported query/key tail (Nq % {rows}, Nk % {keys})")
        device = q.device
        if device.type != "cuda" or k.device != device or v.device != device \
                or not q.dtype == k.dtype == v.dtype == torch.float16:
            raise ValueError("Q/K/V must be FP16 on the same GPU")
        for t in (q, k, v):
            b, h, n, d = t.stride()
            if d != 1 or b % 8 or h % 8 or n % 8 or b < 0 or h < 0 or n < 128 or t.data_ptr() % 16:
                raise ValueError(LAYOUT_ERROR)

    def buffer(self, q, k, what, make):
        """The live buffer `what` of these shapes, or a new one from make()."""
        key = (q.shape, k.shape, q.device, self.config, what)
        held = self.buffers.get(key)
        tensor = held() if held is not None else None
        if tensor is None:
            tensor = make()
            self.buffers[key] = weakref.ref(tensor)
        return tensor

    def buffers_for(self, q, k, lse=False):
        import torch

        if lse:
            return self.buffer(q, k, True, lambda: torch.empty(
                q.shape[:3], dtype=torch.float32, device=q.device))
        return self.buffer(q, k, False, lambda: torch.empty(
            q.shape, dtype=torch.float16, device=q.device))

    def drop_plans(self):
        """Forgets the plans, and every buffer that nobody else holds."""
        self.plans.clear()
        for key, held in list(self.buffers.items()):
            if held() is None:
                self.buffers.pop(key, None)

    # Capture buffers are for small debug inputs, as in the reference binding
    # (binding.py:40-42: at most 64 Mi FP32 values).
    CAPTURE_LIMIT = 64 * 1024 * 1024

    def stats_for(self, q, k, prob):
        import torch

        count, block = C.c_uint64(), C.c_int32()
        self.check(self.lib.fa_fwd_capture_count(C.byref(prob), C.byref(count), C.byref(block)),
                   "capture")
        if count.value > self.CAPTURE_LIMIT:
            raise ValueError("debug capture is restricted to small inputs (at most 256 MiB)")
        nblk = count.value // (4 * q.shape[0] * q.shape[1] * q.shape[2])
        stats = self.buffer(q, k, "stats", lambda: torch.empty(
            (4, nblk) + tuple(q.shape[:3]), dtype=torch.float32, device=q.device))
        return stats, block.value

    def trace_for(self, q, k, prob):
        import torch

        count = C.c_uint64()
        self.check(self.lib.fa_fwd_trace_count(C.byref(prob), C.byref(count)), "trace")
        return self.buffer(q, k, "trace", lambda: torch.empty(
            (count.value // TRACE_WORDS, TRACE_WORDS), dtype=torch.int64, device=q.device))

    def __call__(self, q, k, v, scale=None, return_lse=False):
        """O (cached tensor), or (O, lse) with ``return_lse``: lse [B, Hq, Nq] FP32
        natural-log log-sum-exp of the scaled scores of each query row.

        With ``config.capture`` the call also fills ``self.last["stats"]``,
        FP32 [4, nblk, B, Hq, Nq]: per key block of ``self.last["block_keys"]``
        keys, each row's running max m (natural-log units), running sum l
        relative to m, rescale factor alpha and block sum z relative to m.
        With ``config.trace`` it fills ``self.last["trace"]``, int64
        [tiles, 8]: the per-query-tile records of ``fa_fwd_trace``."""
        import torch

        # Everything but the pointers' alignment follows from these values,
        # so one lookup stands for the checks and the set-up of a signature
        # met before. A decode step of 12 heads (two launches, 7 us of the
        # host's time) takes 13.3 us where its signature is met again, and
        # 27.9 where its key length is new, as in a decode loop, both with the
        # slicing of the cache; 25.6 and 34.7 with every check, conversion and
        # allocation made anew each time.
        if scale is not None:
            scale = float(scale)
        key = (q.shape, k.shape, v.shape, q.stride(), k.stride(), v.stride(), q.dtype, k.dtype,
               v.dtype, q.device, k.device, v.device, scale, bool(return_lse))
        plan = self.plans.get(key)
        if plan is None or plan.config is not self.config:
            plan = self.plan(q, k, v, scale, return_lse)
            if len(self.plans) >= SIGNATURES_KEPT:
                self.drop_plans()
            self.plans[key] = plan
        qp, kp, vp = q.data_ptr(), k.data_ptr(), v.data_ptr()
        if (qp | kp | vp) % 16:
            raise ValueError(LAYOUT_ERROR)
        index = q.device.index
        if index == torch.cuda.current_device():
            self.launch(plan, q, k, v, qp, kp, vp, index)
        else:
            with torch.cuda.device(index):
                self.launch(plan, q, k, v, qp, kp, vp, index)
        self.last = {"output": plan.out, "lse": plan.lse, "stats": plan.stats,
                     "block_keys": plan.block, "trace": plan.trace}
        return (plan.out, plan.lse) if return_lse else plan.out

    def plan(self, q, k, v, scale, return_lse):
        """The Plan of a call signature; raises what the call must refuse."""
        import torch

        self.validate(q, k, v)
        scale = q.shape[3] ** -0.5 if scale is None else scale
        if not (scale > 0 and math.isfinite(scale)):
            raise ValueError("scale must be finite and positive")
        config, splits, lib = self.config, self.config.splits, self.lib
        prob = make_problem(q.shape, k.shape, scale, config)
        size = C.c_uint64()
        if splits is None:
            self.check(lib.fa_fwd_workspace_bytes(C.byref(prob), C.byref(size)), "prepare")
        else:
            with torch.cuda.device(q.device):
                # The automatic count is resolved here, once, and not again by every launch.
                if splits == 0:
                    splits = self.problem_splits(prob)
                self.check(lib.fa_fwd_split_workspace_bytes(C.byref(prob), splits,
                                                            C.byref(size)), "prepare")
        p = Plan()
        p.config, p.size = config, max(size.value, 16)
        p.out = self.buffers_for(q, k)
        capture = config.capture
        p.lse = self.buffers_for(q, k, lse=True) if (return_lse or capture) else None
        p.stats, p.block = self.stats_for(q, k, prob) if capture else (None, 0)
        p.trace = self.trace_for(q, k, prob) if config.trace else None
        strided = not all(t.is_contiguous() for t in (q, k, v))
        if strided and (capture or p.trace is not None or config.sync):
            raise ValueError("capture, trace and sync modes need contiguous Q/K/V")
        st = None
        if strided:
            st = C.byref(FaStrides.from_buffer_copy(struct.pack(
                "=12q", *q.stride()[:3], *k.stride()[:3], *v.stride()[:3], *p.out.stride()[:3])))
        # The call is fn(*before, q, k, v, *outputs, *after, workspace, bytes, stream);
        # an output of None is passed as a null pointer.
        p.before, p.outputs, p.after = (C.byref(prob),), (p.out, p.lse), ()
        if splits is not None:
            p.fn, p.before = lib.fa_fwd_split, (C.byref(prob), splits, st)
        elif strided:
            p.fn, p.before = lib.fa_fwd_strided, (C.byref(prob), st)
        elif capture:
            p.fn, p.outputs = lib.fa_fwd_capture, (p.out, p.lse, p.stats)
            p.after = (p.stats.numel(),)
        elif p.trace is not None:
            p.fn, p.outputs, p.after = lib.fa_fwd_trace, (p.out, p.trace), (p.trace.numel(),)
        elif config.sync:
            p.fn = lib.fa_fwd_sync
        elif return_lse:
            p.fn = lib.fa_fwd_lse
        else:
            p.fn, p.outputs = lib.fa_fwd, (p.out,)
        p.extra = tuple(t for t in (p.out, p.lse, p.stats, p.trace) if t is not None)
        return p

    def launch(self, plan, q, k, v, qp, kp, vp, index):
        """Enqueue the planned call on the current stream of device `index`,
        which is the current device."""
        import torch

        ws = self.workspace
        if ws is None or ws.device != q.device or ws.numel() < plan.size:
            ws = self.workspace = torch.empty(plan.size, dtype=torch.uint8, device=q.device)
        raw = torch._C._cuda_getCurrentRawStream(index)
        stream = self.streams.get((index, raw))
        if stream is None:
            if len(self.streams) >= 64:
                self.streams.clear()
            stream = self.streams[index, raw] = torch.cuda.current_stream(index)
        if raw and torch.cuda.is_current_stream_capturing():   # never the default stream
            self.captured[id(plan), ws.data_ptr()] = plan, ws
        outputs = [t.data_ptr() if t is not None else None for t in plan.outputs]
        status = plan.fn(*plan.before, qp, kp, vp, *outputs, *plan.after, ws.data_ptr(), ws.numel(),
                         raw)
        if status:
            self.check(status, "launch")
        for t in (q, k, v, ws) + plan.extra:
            t.record_stream(stream)
