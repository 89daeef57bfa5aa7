"""Host-side mirror of the reference's W4A4 operator interface over the C ABI.

Names follow the reference's backend entry points (patches/llama.cpp-ruquant.patch, rq-w4a4.cuh, lines
2391-2401 of the patch): ``supported`` <-> ggml_cuda_rq_w4a4_supported, ``W4A4Weight.ready`` <->
ggml_cuda_rq_w4a4_ready, ``mul_mat`` <-> ggml_cuda_mul_mat_rq_w4a4, ``mul_mat_fused`` <->
ggml_cuda_mul_mat_rq_w4a4_fused. A ``W4A4Weight`` plays the part of the ggml weight tensor plus the
``rq_tensor_info`` the reference hangs on ``src0->extra`` at first use (patch lines 2027-2043).

torch owns device memory and the stream; every computation happens inside librq_w4a4.so.
"""
import contextlib
import ctypes
import threading

import numpy as np
import torch

from .lib import load_library

TYPE_W4A4, TYPE_W4A4H, TYPE_A4, TYPE_A4H = 44, 45, 46, 47
BLOCK_DTYPE = np.dtype([("d", "<f4"), ("sum", "<i4"), ("pad", "<i4", (2,)), ("qs", "<u4", (32,))])


class RqError(RuntimeError):
    pass


_ERRORS = {-1: "unsupported shape or type", -2: "workspace / prepared buffer too small or misaligned",
           -3: "bad argument"}


def _check(rc, what):
    if rc != 0:
        raise RqError("%s failed: %s" % (what, _ERRORS.get(rc, "hipError_t %d" % rc)))


def _stream_ptr():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


# the current stream's handle as a number (a torch without a GPU backend does not have the call, and runs this package's
# tools for block files all the same)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (
    lambda index: torch.cuda.current_stream(index).cuda_stream)


def _on_device_of(x, fn, *args):
    """fn(*args, stream) with x's device current and its current stream. A decode step's products are a few microseconds
    each, so what the host does per call shows: the device guard is entered only when another device is current, and
    the stream's handle is asked for as the number it is (the guard and a Stream object cost 4.3 us per call)."""
    index = x.get_device()
    if torch.cuda.current_device() == index:
        return fn(*args, _raw_stream(index))
    with torch.cuda.device(index):
        return fn(*args, _raw_stream(index))


def _device_bytes(n, device):
    # torch's caching allocator returns 512-byte aligned blocks; the ABI needs 256
    t = torch.empty(max(int(n), 256), dtype=torch.uint8, device=device)
    assert t.data_ptr() % 256 == 0
    return t


def hadamard_factor(n):
    p, m = ctypes.c_int(0), ctypes.c_int(0)
    ok = load_library().rq_w4a4_hadamard_factor(int(n), ctypes.byref(p), ctypes.byref(m))
    return (p.value, m.value) if ok else None


def supported(type_, K, N, M, ldx_bytes=None, ldy_bytes=None):
    ldx_bytes = 4 * K if ldx_bytes is None else ldx_bytes
    ldy_bytes = 4 * N if ldy_bytes is None else ldy_bytes
    return bool(load_library().rq_w4a4_supported(type_, K, N, M, ldx_bytes, ldy_bytes))


def resolve_clip(block0, type_):
    """block0: the first block of the tensor (numpy, host). Environment > header pad[1] > 1."""
    b = np.ascontiguousarray(block0).view(np.uint8)
    return float(load_library().rq_w4a4_resolve_clip(b.ctypes.data, type_))


def tensor_rot(block0, type_, K):
    b = np.ascontiguousarray(block0).view(np.uint8)
    return int(load_library().rq_w4a4_tensor_rot(b.ctypes.data, type_, K))


class W4A4Weight:
    """A W4A4 / W4A4H weight tensor on the GPU: [N, K/256] blocks as ggml stores them, plus what the first use
    derives (clip, Hadamard length, the prepared streaming form)."""

    def __init__(self, blocks, type_, device="cuda:0", keep_blocks=True, in_place=False):
        blocks = np.ascontiguousarray(blocks)
        assert blocks.dtype == BLOCK_DTYPE and blocks.ndim == 2
        self.type = int(type_)
        self.N, nb = blocks.shape
        self.K = nb * 256
        self.device = torch.device(device)
        L = load_library()
        # first use: header of block 0 (the reference reads it back from the device, patch lines 2030-2040)
        self.clip = resolve_clip(blocks[0, 0], self.type)
        self.n_rot = tensor_rot(blocks[0, 0], self.type, self.K)
        if self.type == TYPE_W4A4H and self.n_rot < 0:
            raise RqError("W4A4H: Hadamard length %d does not divide this row of %d"
                          % (int(blocks[0, 0]["pad"][0]), self.K))
        b0 = np.ascontiguousarray(blocks[0, 0]).view(np.uint8)
        if L.rq_w4a4_weight_group(b0.ctypes.data) == 64 and L.rq_w4a4_act_group() != 64:
            # the reference asserts the same in ggml_vec_dot_w4a4_a4 (patch lines 169-170)
            raise RqError("weight groups of 64 need activation groups of 64 (RQ_ACT_GROUP=%d)" % L.rq_w4a4_act_group())
        raw = torch.from_numpy(blocks.view(np.uint8).reshape(-1).copy()).to(self.device)
        nbytes = L.rq_w4a4_prepared_bytes(self.K, self.N)
        if nbytes == 0:
            raise RqError("unsupported weight shape K=%d N=%d" % (self.K, self.N))
        self.plane6 = None
        if in_place:
            # as the reference repacks (patch lines 2046-2075): the tensor's own buffer becomes the prepared weight
            # (one copy of the codes resident), the fp6 plane of the wide-batch kernel lives beside it
            n6 = L.rq_w4a4_plane6_bytes(self.K, self.N)
            self.plane6 = _device_bytes(n6, self.device) if n6 else None
            staging = _device_bytes(L.rq_w4a4_inplace_staging_bytes(self.K, self.N), self.device)
            with torch.cuda.device(self.device):
                _check(L.rq_w4a4_prepare_inplace(raw.data_ptr(), self.K, self.N,
                                                 self.plane6.data_ptr() if n6 else None, n6, staging.data_ptr(),
                                                 staging.numel(), _stream_ptr()), "rq_w4a4_prepare_inplace")
                torch.cuda.current_stream().synchronize()   # staging is released below
            self.prepared = raw
            self.blocks = None
        else:
            self.prepared = _device_bytes(nbytes, self.device)
            with torch.cuda.device(self.device):
                _check(L.rq_w4a4_prepare(raw.data_ptr(), self.K, self.N, self.prepared.data_ptr(), nbytes,
                                         _stream_ptr()), "rq_w4a4_prepare")
            self.blocks = raw if keep_blocks else None
        self.ready = True

    def workspace(self, M):
        n = load_library().rq_w4a4_workspace_bytes(self.type, self.K, self.N, M)
        return _device_bytes(n, self.device)


def mul_mat(weight, x, out=None, workspace=None, clip=None):
    """y[M, N] = x[M, K] . W^T, bit-identical to the ggml-cpu W4A4 / W4A4H MUL_MAT. The workspace holds nothing for later
    calls afterwards (SharedActivation fills one that does)."""
    # (the single product's own entry point: no argument arrays to build. With the device and stream handled as in
    # _on_device_of the host takes 5 us for a one-token call instead of 11.7: less than the kernel from K = 5120,
    # N = 5120 on (6.3 us), about as long as the smallest ones (K = 4096, N = 1024: 5.3))
    L = load_library()
    assert x.is_cuda and x.dtype == torch.float32 and x.dim() == 2 and x.stride(1) == 1
    M, K = x.shape
    assert K == weight.K
    N = weight.N
    if out is None:
        out = torch.empty((M, N), dtype=torch.float32, device=x.device)
    if workspace is None:
        workspace = _device_bytes(fused_workspace_bytes([weight], M), x.device)
    ldx = x.stride(0) if M > 1 else K
    ldy = out.stride(0) if out.shape[0] > 1 else out.shape[1]
    rc = _on_device_of(x, L.rq_w4a4_mul_mat_once, weight.type, weight.prepared.data_ptr(), K, N, x.data_ptr(), ldx, M,
                       out.data_ptr(), ldy, weight.clip if clip is None else clip, max(weight.n_rot, 0),
                       workspace.data_ptr(), workspace.numel())
    if rc != 0:
        _check(rc, "rq_w4a4_mul_mat")
    return out


def fused_workspace_bytes(weights, M):
    """Workspace for a fused call that serves all its weights from one launch of the streaming kernels: split-K
    cells for the rows of every weight (each padded to 64). With room for the largest weight only
    (rq_w4a4_workspace_bytes of the largest N) the call still works, one product launch per weight up to 64 tokens.
    Above 64 tokens the room per weight does not count, and how many launches there are does not depend on it."""
    w0 = weights[0]
    N = w0.N if len(weights) == 1 else sum((w.N + 63) // 64 * 64 for w in weights)
    return load_library().rq_w4a4_workspace_bytes(w0.type, w0.K, N, M)


def mul_mat_fused(weights, x, outs=None, workspace=None, clip=None):
    """Up to three weights of one type, K, clip and rotation length against the same activations. As after mul_mat, the
    workspace holds nothing for later calls."""
    L = load_library()
    w0 = weights[0]
    assert x.is_cuda and x.dtype == torch.float32 and x.dim() == 2 and x.stride(1) == 1
    M, K = x.shape
    assert K == w0.K
    for w in weights[1:]:
        if (w.type, w.K, w.clip, w.n_rot) != (w0.type, w0.K, w0.clip, w0.n_rot):
            raise RqError("weights cannot be fused: type, K, clip and rotation length must match")
    if outs is None:
        outs = [torch.empty((M, w.N), dtype=torch.float32, device=x.device) for w in weights]
    n = len(weights)
    if workspace is None:
        workspace = _device_bytes(fused_workspace_bytes(weights, M), x.device)
    prepared = (ctypes.c_void_p * n)(*[w.prepared.data_ptr() for w in weights])
    ys = (ctypes.c_void_p * n)(*[o.data_ptr() for o in outs])
    Ns = (ctypes.c_int64 * n)(*[w.N for w in weights])
    ldys = (ctypes.c_int64 * n)(*[o.stride(0) if o.shape[0] > 1 else o.shape[1] for o in outs])
    ldx = x.stride(0) if M > 1 else K
    rc = _on_device_of(x, L.rq_w4a4_mul_mat_fused_once, w0.type, n, prepared, K, Ns, x.data_ptr(), ldx, M, ys, ldys,
                       w0.clip if clip is None else clip, max(w0.n_rot, 0), workspace.data_ptr(), workspace.numel())
    _check(rc, "rq_w4a4_mul_mat")
    return outs


class SharedActivation:
    """The reference's rq_act_cache (patch lines 1996-2023, 2160-2172) for this host: consecutive MUL_MATs of one x
    that were not fused rotate and quantize x once. The cache is the workspace itself; `begin()` plays
    ggml_cuda_rq_graph_begin (x may have changed in place since the last evaluation)."""

    def __init__(self, workspace):
        self.workspace = workspace
        workspace.zero_()            # the split-K cells inside must read zero before stage 2 first uses them
        self.key = None
        self.rows_cleared = 0
        self.hits = self.misses = 0

    def begin(self):
        self.key = None

    def mul_mat(self, weight, x, out):
        L = load_library()
        M, K = x.shape
        key = (x.data_ptr(), x.stride(0), M, K, weight.type, weight.clip, weight.n_rot)
        rows = (weight.N + 63) // 64 * 64
        hit = key == self.key and rows <= self.rows_cleared
        ldx = x.stride(0) if M > 1 else K
        ldy = out.stride(0) if M > 1 else weight.N
        stages = 2 if hit else 3
        rc = _on_device_of(x, lambda *a: L.rq_w4a4_mul_mat_stages(*a, stages), weight.type, weight.prepared.data_ptr(),
                           K, weight.N, x.data_ptr(), ldx, M, out.data_ptr(), ldy, weight.clip, max(weight.n_rot, 0),
                           self.workspace.data_ptr(), self.workspace.numel())
        _check(rc, "rq_w4a4_mul_mat_stages")
        if hit:
            self.hits += 1
        else:
            self.misses += 1
            self.key, self.rows_cleared = key, rows
        return out


def hadamard(x, n_rot=None):
    """x[M, K] -> x diag(H, H, ...) with H of length n_rot (default K), as ggml_rq_hadamard does per block."""
    L = load_library()
    assert x.is_cuda and x.dtype == torch.float32 and x.dim() == 2 and x.stride(1) == 1
    M, K = x.shape
    out = torch.empty((M, K), dtype=torch.float32, device=x.device)
    with torch.cuda.device(x.device):
        rc = L.rq_w4a4_hadamard(x.data_ptr(), x.stride(0) if M > 1 else K, M, K, n_rot or K, out.data_ptr(), K,
                                _stream_ptr())
    _check(rc, "rq_w4a4_hadamard")
    return out


def quantize_act(x, clip, hadamard_=False, n_rot=None):
    """x[M, K] -> [M, K/256] activation blocks in the reference's A4 / A4H layout (numpy, host)."""
    L = load_library()
    assert x.is_cuda and x.dtype == torch.float32 and x.dim() == 2 and x.stride(1) == 1
    M, K = x.shape
    out = torch.zeros(M * (K // 256) * 144, dtype=torch.uint8, device=x.device)
    with torch.cuda.device(x.device):
        rc = L.rq_w4a4_quantize_act(TYPE_A4H if hadamard_ else TYPE_A4, x.data_ptr(), x.stride(0) if M > 1 else K,
                                    M, K, clip, (n_rot or K) if hadamard_ else 0, out.data_ptr(), _stream_ptr())
    _check(rc, "rq_w4a4_quantize_act")
    return out.cpu().numpy().view(BLOCK_DTYPE).reshape(M, K // 256)


# Blocks travel between the host's ordinary memory and the GPU through pinned buffers of this size, a few at a time: a
# copy from or to pageable memory is staged by the runtime on one thread and waits for each stage (17.7 MB from the GPU
# 950 us, of which the link needs 320; 12.5 MB to it 350 + 185 us for a private copy, the link 230), this way the
# link, the host's copy (several threads) and the kernels run side by side. torch's pinned-memory cache hands the
# buffers out and takes them back, so concurrent calls have their own and no call keeps any.
_STAGE_BYTES = 4 << 20
_STAGES = 3
# Blocks that fit one buffer have nothing to run beside: they cross through one buffer on the caller's own stream. (The
# second stream, its events and two more buffers cost 40 us, more than a small tensor's whole conversion.)


def _chunks(n, most):
    """[0, n) in equal runs of at most `most`"""
    k = max(1, -(-n // most))
    return [(n * i // k, n * (i + 1) // k) for i in range(k)]


def _pinned(nbytes):
    # (host memory whatever torch's default device is)
    return torch.empty(nbytes, dtype=torch.uint8, device="cpu", pin_memory=True)


# A stream's first work costs 0.2 ms, and 2.9 ms while it gets a hardware queue of its own (a few per process), so a
# conversion in several runs does not take another of torch's streams each time but keeps the one that its thread used
# beside the same current stream. (Not one for all: its runs wait for the work in front of them on the current stream,
# and would make another stream's conversion wait for it too.)
_copiers = threading.local()
_COPIERS = 8   # per thread, the latest ones


def _second_stream(current):
    kept = _copiers.__dict__.setdefault("streams", {})
    key = (current.device_index, current.cuda_stream)
    stream = kept.pop(key, None)
    if stream is None:
        stream = torch.cuda.Stream(current.device)
        if len(kept) >= _COPIERS:
            del kept[next(iter(kept))]
    kept[key] = stream   # (the latest at the end)
    return stream


def _refuse_capture():
    """A graph replays a copy from the pinned buffer's address, and the buffer is another call's by then."""
    if torch.cuda.is_current_stream_capturing():
        raise RqError("conversions read and write host memory: not under graph capture")


def _copy_bytes(pinned, src):
    """numpy bytes into the head of a pinned tensor (torch's copy uses several threads; it takes writable arrays only)"""
    if src.flags.writeable:
        pinned[:src.size].copy_(torch.from_numpy(src))
    else:
        np.copyto(pinned[:src.size].numpy(), src)


def quantize_weights(w, type_, n_rot=None, wgroup=0):
    """w[N, K] fp32 on the GPU -> [N, K/256] weight blocks (numpy, host): the type's from_float_ref for whole
    tensors (quantize_row_w4a4_ref / quantize_row_w4a4h_ref, patch lines 2681-2710). wgroup 0 / 256 / 64 is the
    reference's RQ_WGROUP switch; n_rot (W4A4H) its K / RQ_ROT_BLOCKS, default K."""
    L = load_library()
    assert w.is_cuda and w.dtype == torch.float32 and w.dim() == 2 and w.stride(1) == 1
    N, K = w.shape
    n_rot = int(n_rot or K)
    # Runs of rows whose blocks fit one buffer, in turn on two streams, the conversion and its copy behind one another: a run is
    # converted while the one before travels, and the link, which is what takes long, starts with the first one's blocks and
    # goes from copy to copy without a pause. (6144 x 5120: rows in runs of 4096, all launched in front of the first copy, left
    # it idle for 130 us at first: 637 us, this way 585.) Up to one and a half buffers' worth is one run: 1500 x 5120 215 us in
    # one, 275 in two.
    row = (K // 256) * 144
    runs = [(0, N)] if 2 * N * row <= 3 * _STAGE_BYTES else _chunks(N, max(1, _STAGE_BYTES // row))
    nbytes = L.rq_w4a4_quantize_weights_workspace_bytes(int(type_), K, max(b - a for a, b in runs), int(wgroup))
    if nbytes == 0:
        raise RqError("unsupported weight shape or group: K=%d N=%d wgroup=%d" % (K, N, wgroup))
    out = torch.empty(N * row, dtype=torch.uint8, device=w.device)
    ldw = w.stride(0) if N > 1 else K

    def convert(a, b, ws):
        rc = L.rq_w4a4_quantize_weights(int(type_), w.data_ptr() + 4 * ldw * a, ldw, b - a, K, n_rot, int(wgroup),
                                        out.data_ptr() + row * a, ws.data_ptr(), ws.numel(), _stream_ptr())
        _check(rc, "rq_w4a4_quantize_weights")

    with torch.cuda.device(w.device):
        _refuse_capture()
        if len(runs) == 1:
            # (what the host can do while the GPU works stands behind the launch: a Stream object in front of it is 3 of 55 us)
            convert(0, N, _device_bytes(nbytes, w.device))
            host = np.empty(N * row, dtype=np.uint8)
            to = torch.from_numpy(host)
            stage = _pinned(N * row)
            stage.copy_(out, non_blocking=True)
            torch.cuda.current_stream().synchronize()
            to.copy_(stage)
            return host.view(BLOCK_DTYPE).reshape(N, K // 256)
        # But the next but one run waits for the copy in front of it on its stream, and rotated rows with a scale per 64 inputs take so
        # long that the link then stands still: those are converted one behind the other on the current stream, the copies on the
        # second. (In turn -> apart, us: 1024 x 48828 966 -> 747, 4096 x 12207 827 to 898 -> 743 to 846, 17408 x 2872 859 -> 770, 5120 x 3000 330 ->
        # 326; not rotated, 17408 x 804 298 -> 328; a scale per row 5120 x 6144 490 -> 513, per 256 5120 x 9765 691 to 720 -> 724.)
        apart = wgroup == 64 and type_ == TYPE_W4A4H
        current = torch.cuda.current_stream()
        other = _second_stream(current)
        ws = [_device_bytes(nbytes, w.device) for _ in range(1 if apart else 2)]
        # (for w, and behind the allocations: their memory may still be in use by work in front of this call, another thread's too)
        if not apart:   # (apart, the second stream waits for what it copies)
            other.wait_stream(current)
        host = np.empty(N * row, dtype=np.uint8)
        to = torch.from_numpy(host)
        stages, done = [], []

        def fetch(i):
            a, b = runs[i]
            stages[i % _STAGES][:row * (b - a)].copy_(out[row * a:row * b], non_blocking=True)
            done.append(torch.cuda.Event())
            done[i].record()

        def land(i):
            a, b = runs[i]
            done[i].synchronize()
            to[row * a:row * b].copy_(stages[i % _STAGES][:row * (b - a)])

        try:
            for i, (a, b) in enumerate(runs):
                with torch.cuda.stream(other) if i & 1 and not apart else contextlib.nullcontext():
                    convert(a, b, ws[0 if apart else i & 1])
                    if apart:
                        ready = torch.cuda.Event()
                        ready.record()
                    if i >= _STAGES:
                        land(i - _STAGES)
                    else:
                        stages.append(_pinned(row * max(d - c for c, d in runs)))
                    if not apart:
                        fetch(i)
                if apart:
                    other.wait_event(ready)
                    with torch.cuda.stream(other):
                        fetch(i)
            for i in range(max(0, len(runs) - _STAGES), len(runs)):
                land(i)
        except BaseException:
            current.wait_stream(other)   # (the memory given back here may still be in use there)
            raise
        return host.view(BLOCK_DTYPE).reshape(N, K // 256)


def _decodes_slowly(K, n_rot):
    """Whether a run of rotated rows takes more than half as long to decode as to travel (4 MiB: 75 us on the link). Long columns of few
    (K = 5376 = 84 x 64 96 us, 9216 = 72 x 128 58, 1280 = 20 x 64 40, 27648 = 108 x 256 45; 11264 = 44 x 256 23, 17408 = 68 x 256 23) and many short
    rows (K = 256 65, 512 39; 1024 25)."""
    factor = hadamard_factor(n_rot) if n_rot > 0 else None
    if factor is None:   # (refused by the library)
        return False
    p = factor[0]
    return K <= 512 or (p > 1 and (p >= 104 or K <= (128 if p >= 60 else 64) * p))


def dequantize(blocks, type_, n_rot=None, device="cuda:0"):
    """[rows, K/256] blocks of any of the four types (numpy, host) -> [rows, K] fp32 on the GPU: the type's to_float
    (dequantize_row_w4a4 / _w4a4h / _a4 / _a4h, patch lines 2738-2773). The rotation length of the rotated types
    comes from block 0 (pad[0] of weights, pad[1] of activations) unless given."""
    L = load_library()
    blocks = np.ascontiguousarray(blocks)
    assert blocks.dtype == BLOCK_DTYPE and blocks.ndim == 2
    rows, nb = blocks.shape
    K = nb * 256
    if n_rot is None:
        n_rot = int(blocks[0, 0]["pad"][0 if type_ in (TYPE_W4A4, TYPE_W4A4H) else 1]) if rows else K
    dev = torch.device(device)
    row = nb * 144
    out = torch.empty((rows, K), dtype=torch.float32, device=dev)
    raw = torch.empty(rows * row, dtype=torch.uint8, device=dev)
    with torch.cuda.device(dev):
        _refuse_capture()
        if rows * row <= _STAGE_BYTES:
            if rows:
                stage = _pinned(rows * row)
                _copy_bytes(stage, blocks.view(np.uint8).reshape(-1))
                raw.copy_(stage, non_blocking=True)
            rc = L.rq_w4a4_dequantize(int(type_), raw.data_ptr(), rows, K, int(n_rot), out.data_ptr(), K, _stream_ptr())
            _check(rc, "rq_w4a4_dequantize")
            return out
        # Runs of rows, in turn on two streams: one is decoded while the next one travels, and the link goes from copy to copy without
        # a pause. But a copy waits for the run that is decoded in front of it on its stream, so where decoding takes long the
        # copies go one behind the other on the current stream, and the runs but the last are decoded on the second. (Call by call /
        # one call behind another in us, in turn -> apart: 5376 x 5000 587 / 611 -> 486 / 449, 9216 x 5582 807 / 843 -> 753 / 708, 256 x 200977
        # 887 / 997 -> 782 / 735, 1280 x 40195 717 / 800 -> 740 / 703; 4096 x 12207 626 / 612 -> 684 / 642, 5120 x 6144 432 / 398 -> 461 / 422.)
        apart = type_ in (TYPE_W4A4H, TYPE_A4H) and _decodes_slowly(K, int(n_rot))
        current = torch.cuda.current_stream()
        other = _second_stream(current)
        # The memory of `raw` and `out` may still be in use by work in front of this call. (Apart, what the second stream does waits for
        # copies on the first one, and an event in front of the first copy delays it: 9216 x 865 212 us without, 262 with one.)
        if not apart:
            other.wait_stream(current)
        runs = _chunks(rows, max(1, _STAGE_BYTES // row))   # (a row too long for the library is refused by it)
        host = blocks.view(np.uint8).reshape(-1)
        stages, sent = [], []

        def decode(a, b):
            rc = L.rq_w4a4_dequantize(int(type_), raw.data_ptr() + row * a, b - a, K, int(n_rot), out.data_ptr() + 4 * K * a, K,
                                      _stream_ptr())
            _check(rc, "rq_w4a4_dequantize")

        try:
            for i, (a, b) in enumerate(runs):
                n, k = row * (b - a), i % _STAGES
                if i < _STAGES:
                    stages.append(_pinned(row * max(d - c for c, d in runs)))
                else:
                    sent[i - _STAGES].synchronize()
                _copy_bytes(stages[k], host[row * a:row * b])
                behind = apart and i + 1 < len(runs)   # (decoded on the second stream, behind the copy on the current one)
                with torch.cuda.stream(other) if i & 1 and not apart else contextlib.nullcontext():
                    raw[row * a:row * b].copy_(stages[k][:n], non_blocking=True)
                    if i + _STAGES < len(runs) or behind:
                        sent.append(torch.cuda.Event())
                        sent[i].record()
                    if not behind:
                        decode(a, b)
                if behind:
                    other.wait_event(sent[i])
                    with torch.cuda.stream(other):
                        decode(a, b)
        finally:
            current.wait_stream(other)   # (what comes behind this call, also on an error the reuse of the memory)
    return out


# ---- on-disk format tools (host memory; the converter side of the reference) ----------------------------------

def pack(codes, scales):
    """int4 codes [N, K] (int8, -8..7) and one scale per row -> blocks [N, K/256] (src/gptq.rs:210-231 `pack`)."""
    codes = np.ascontiguousarray(codes, dtype=np.int8)
    scales = np.ascontiguousarray(scales, dtype=np.float32)
    N, K = codes.shape
    assert scales.shape == (N,)
    out = np.zeros((N, K // 256), dtype=BLOCK_DTYPE)
    _check(load_library().rq_w4a4_pack(codes.ctypes.data, scales.ctypes.data, N, K, out.ctypes.data), "rq_w4a4_pack")
    return out


def pack_groups(codes, units, mults):
    """As pack, with integer weight multipliers: mults [N, K/256] (per block) or [N, K/64] (per 64 inputs)
    (src/gptq.rs:193-207 `pack_groups`)."""
    codes = np.ascontiguousarray(codes, dtype=np.int8)
    units = np.ascontiguousarray(units, dtype=np.float32)
    mults = np.ascontiguousarray(mults, dtype=np.uint8)
    N, K = codes.shape
    per = mults.shape[1] // (K // 256)
    assert mults.shape == (N, per * (K // 256)) and per in (1, 4)
    out = np.zeros((N, K // 256), dtype=BLOCK_DTYPE)
    _check(load_library().rq_w4a4_pack_groups(codes.ctypes.data, units.ctypes.data, mults.ctypes.data, per, N, K,
                                              out.ctypes.data), "rq_w4a4_pack_groups")
    return out


def set_clip(blocks, clip):
    """Activation clip into pad[1] of every block, in place (`ruquant setclip`, src/convert.rs:876-878)."""
    assert blocks.dtype == BLOCK_DTYPE and blocks.flags.c_contiguous
    load_library().rq_w4a4_set_clip(blocks.ctypes.data, blocks.size, float(clip))


def set_rot_len(blocks, n):
    """Hadamard length into pad[0] of every block, in place (src/convert.rs:99-101 `set_rot_len`)."""
    assert blocks.dtype == BLOCK_DTYPE and blocks.flags.c_contiguous
    load_library().rq_w4a4_set_rot_len(blocks.ctypes.data, blocks.size, int(n))


def dequantize_rows(blocks):
    """The type's to_float for W4A4 weights: code * (multiplier * d) (patch lines 2738-2742). Returns [N, K] fp32."""
    assert blocks.dtype == BLOCK_DTYPE and blocks.ndim == 2 and blocks.flags.c_contiguous
    N, nb = blocks.shape
    out = np.empty((N, nb * 256), dtype=np.float32)
    _check(load_library().rq_w4a4_dequantize_rows(blocks.ctypes.data, N, nb * 256, out.ctypes.data),
           "rq_w4a4_dequantize_rows")
    return out
