"""GPU parity of the weight-side quantizer and the dequantizers (the types' from_float_ref / to_float, patch lines
2507-2580, 2681-2710, 2738-2773) against the CPU oracle: every byte of every block, every bit of every float."""
import threading

import numpy as np
import pytest
import torch

import ruquant_amd as rq
from ruquant_amd import w4a4
from tests.gpu_util import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
f32 = np.float32


def tensor(N, K, seed):
    """Rows of several characters: gaussian, heavy-tailed, one outlier, group-scaled, flat +-1, all zero."""
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((N, K)).astype(f32) * f32(0.02)
    for r in range(N):
        kind = r % 6
        if kind == 1:
            w[r] = (rng.standard_t(3, size=K) * 0.02).astype(f32)
        elif kind == 2:
            w[r, rng.integers(K)] = 3.0
        elif kind == 3:
            w[r] = (rng.uniform(-1, 1, size=K) * np.exp2((np.arange(K) // 64 + r) % 5 - 2)).astype(f32)
        elif kind == 4:
            w[r] = np.where(rng.uniform(size=K) < 0.5, -1.0, 1.0)
        elif kind == 5 and r % 12 == 5:
            w[r] = 0.0
    return w


def blocks_equal(got, want):
    return got.shape == want.shape and got.tobytes() == want.tobytes()


def block_diff(got, want):
    for name in ("d", "sum", "pad", "qs"):
        bad = np.argwhere(got[name].view(np.uint32) != want[name].view(np.uint32))
        if bad.size:
            i = tuple(bad[0])
            return "%s differs at %s: got %r want %r (%d places)" % (name, i, got[name][i], want[name][i], len(bad))
    return "equal"


@pytest.mark.parametrize("wgroup", [0, 256, 64])
@pytest.mark.parametrize("K", [256, 1536, 5120])
def test_quantize_w4a4_vs_oracle(oracle, K, wgroup):
    N = 37
    w = tensor(N, K, K + wgroup)
    got = rq.quantize_weights(torch.from_numpy(w).to(DEV), rq.TYPE_W4A4, wgroup=wgroup)
    want = oracle.quantize_rows_w(w, wgroup=wgroup)
    assert blocks_equal(got, want), block_diff(got, want)


@pytest.mark.parametrize("K,n_rot,wgroup", [(256, 256, 0), (1536, 1536, 0), (1536, 768, 64), (4096, 4096, 256),
                                             (5120, 5120, 0), (5120, 2560, 0), (5120, 5120, 64), (6144, 6144, 0),
                                             (17408, 17408, 0), (17408, 4352, 256), (11264, 11264, 0)])
def test_quantize_w4a4h_vs_oracle(oracle, K, n_rot, wgroup):
    N = 19
    w = tensor(N, K, K + n_rot + wgroup)
    got = rq.quantize_weights(torch.from_numpy(w).to(DEV), rq.TYPE_W4A4H, n_rot=n_rot, wgroup=wgroup)
    want = oracle.quantize_rows_w(w, hadamard=True, n_rot=n_rot, wgroup=wgroup)
    assert blocks_equal(got, want), block_diff(got, want)


def test_quantize_strided_rows(oracle):
    N, K = 8, 1024
    full = np.zeros((N, K + 64), dtype=f32)
    full[:, :K] = tensor(N, K, 4)
    wd = torch.from_numpy(full).to(DEV)[:, :K]
    got = rq.quantize_weights(wd, rq.TYPE_W4A4H)
    want = oracle.quantize_rows_w(np.ascontiguousarray(full[:, :K]), hadamard=True)
    assert blocks_equal(got, want), block_diff(got, want)


def test_quantize_rejects_bad_arguments():
    w = torch.zeros((4, 512), dtype=torch.float32, device=DEV)
    with pytest.raises(rq.RqError):
        rq.quantize_weights(w, rq.TYPE_W4A4, wgroup=128)
    with pytest.raises(rq.RqError):
        rq.quantize_weights(w, rq.TYPE_W4A4H, n_rot=96)            # no Hadamard of that length
    with pytest.raises(rq.RqError):
        rq.quantize_weights(torch.zeros((4, 384), dtype=torch.float32, device=DEV), rq.TYPE_W4A4)


@pytest.mark.parametrize("K,n_rot,wgroup", [(512, 512, 0), (1536, 1536, 64), (5120, 5120, 256), (5120, 1280, 0),
                                             (17408, 17408, 0), (6144, 6144, 64)])
def test_dequantize_weights_vs_oracle(oracle, K, n_rot, wgroup):
    N = 11
    w = tensor(N, K, 5 * K + wgroup)
    for had, type_ in ((False, rq.TYPE_W4A4), (True, rq.TYPE_W4A4H)):
        blocks = oracle.quantize_rows_w(w, hadamard=had, n_rot=n_rot, wgroup=wgroup)
        got = rq.dequantize(blocks, type_).cpu().numpy()
        want = np.stack([oracle.dequantize_row_w(blocks[r], hadamard=had) for r in range(N)])
        assert bits_equal(got, want), first_mismatch(got, want)


@pytest.mark.parametrize("G", [64, 128, 256])
@pytest.mark.parametrize("K,n_rot", [(512, 512), (5120, 5120), (5120, 2560), (17408, 17408)])
def test_dequantize_activations_vs_oracle(oracle, K, n_rot, G):
    M = 5
    rng = np.random.default_rng(K + G)
    x = (rng.standard_normal((M, K)) * np.exp2(rng.integers(-3, 4, size=(M, K)))).astype(f32)
    for had, type_ in ((False, rq.TYPE_A4), (True, rq.TYPE_A4H)):
        if had:
            blocks = np.stack([oracle.quantize_row_a4h(x[t], 0.9, n_rot, G) for t in range(M)])
        else:
            blocks = np.stack([oracle.quantize_row_a(x[t], 0.9, G) for t in range(M)])
        got = rq.dequantize(blocks, type_).cpu().numpy()
        want = np.stack([oracle.dequantize_row_a(blocks[t], hadamard=had) for t in range(M)])
        assert bits_equal(got, want), first_mismatch(got, want)


def test_quantized_tensor_feeds_the_op(oracle):
    """from_float_ref on the GPU -> the op: same y as the oracle computes from its own quantizer's blocks."""
    N, K, M = 128, 5120, 9
    w = tensor(N, K, 77)
    blocks = rq.quantize_weights(torch.from_numpy(w).to(DEV), rq.TYPE_W4A4H, wgroup=64)
    rq.set_clip(blocks, 0.9)
    x = np.random.default_rng(5).standard_normal((M, K)).astype(f32)
    weight = rq.W4A4Weight(blocks, rq.TYPE_W4A4H, DEV)
    got = rq.mul_mat(weight, torch.from_numpy(x).to(DEV)).cpu().numpy()
    ref_blocks = oracle.quantize_rows_w(w, hadamard=True, wgroup=64)
    rq.set_clip(ref_blocks, 0.9)
    want = oracle.mul_mat(rq.TYPE_W4A4H, ref_blocks, x, f32(0.9), K)
    assert bits_equal(got, want), first_mismatch(got, want)


def test_full_size_tensor_sampled_rows(oracle):
    """A whole 17408 x 5120 tensor (the `down` projection) through the GPU quantizer; the oracle checks a sample of
    rows, and every block of the tensor must carry its row's header."""
    N, K = 5120, 17408
    g = torch.Generator(device=DEV)
    g.manual_seed(1)
    w = torch.randn((N, K), dtype=torch.float32, device=DEV, generator=g) * 0.02
    torch.cuda.synchronize()
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    L = rq.load_library()
    ws = torch.empty(L.rq_w4a4_quantize_weights_workspace_bytes(rq.TYPE_W4A4H, K, N, 0), dtype=torch.uint8, device=DEV)
    out = torch.zeros(N * (K // 256) * 144, dtype=torch.uint8, device=DEV)
    import ctypes
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    t0.record()
    rc = L.rq_w4a4_quantize_weights(rq.TYPE_W4A4H, w.data_ptr(), K, N, K, K, 0, out.data_ptr(), ws.data_ptr(),
                                    ws.numel(), st)
    t1.record()
    torch.cuda.synchronize()
    assert rc == 0
    print("quantize 5120 x 17408 W4A4H: %.2f ms" % t0.elapsed_time(t1), flush=True)
    blocks = out.cpu().numpy().view(rq.BLOCK_DTYPE).reshape(N, K // 256)
    assert (blocks["pad"][:, :, 0] == K).all() and (blocks["pad"][:, :, 1] == 0).all()
    assert (blocks["d"] == blocks["d"][:, :1]).all() and (blocks["sum"] == blocks["sum"][:, :1]).all()
    sample = [0, 1, 63, 64, 1000, 2559, 2560, 4095, 5118, 5119]
    wn = w[sample].cpu().numpy()
    want = oracle.quantize_rows_w(wn, hadamard=True)
    assert blocks_equal(blocks[sample], want), block_diff(blocks[sample], want)


def repeated(rows, N):
    return np.tile(rows, (-(-N // len(rows)),) + (1,) * (rows.ndim - 1))[:N]


# (groups of 256 and 64, and rows of 256, are searched in element order up to 5 or 3.5 Mi floats and by fp32 sums above that; more
# segments than a multiple of four leave lanes of the last wavefront without one)
@pytest.mark.parametrize("K,wgroup,N", [(256, 0, 12), (1536, 0, 12), (1536, 64, 12), (1280, 256, 12),
                                        (256, 0, 20501), (1536, 64, 2731), (1280, 256, 4101)])
def test_search_at_rounding_boundaries_and_extreme_scales(oracle, K, wgroup, N):
    """The clip search takes the correctly rounded quotient only where x * (1 / s) is near a half-way point or 1 / s is
    no normal number: rows full of exact ties and of values one step beside them, rows of denormals, of the largest
    floats, with an infinity, and ordinary ones."""
    rng = np.random.default_rng(K + wgroup)
    half = rng.integers(-14, 15, size=(12, K)).astype(f32) * f32(0.5)     # k / 2: ties at scale 1
    half[:, ::64] = 7.0                                                    # amax 7: the first ratio's scale is exactly 1
    w = half.copy()
    w[1] = np.nextafter(half[1], f32(np.inf))
    w[2] = np.nextafter(half[2], f32(-np.inf))
    w[3] = half[3] * f32(2.0 ** -140)
    w[4] = half[4] * f32(2.0 ** -124)
    w[5] = half[5] * f32(2.0 ** 124)
    w[6] = half[6] * f32(0.1)
    w[7] = half[7] * f32(1.0 / 3.0)
    w[8] = (rng.standard_normal(K) * 2.0 ** -130).astype(f32)
    w[9] = (rng.standard_normal(K) * 1e37).astype(f32)
    w[10, 5] = np.inf
    w[11] = rng.standard_normal(K).astype(f32)
    got = rq.quantize_weights(torch.from_numpy(repeated(w, N)).to(DEV), rq.TYPE_W4A4, wgroup=wgroup)
    want = repeated(oracle.quantize_rows_w(w, wgroup=wgroup), N)
    assert blocks_equal(got, want), block_diff(got, want)


def grid_rows(kind, N, K, rng):
    """Rows on an int4 grid: `seven` with 7 as the largest code (the first ratio reproduces them), `eight` with -8 (the sixth does),
    `ternary`, and `negative` from {-1, 0} (both do)."""
    c = rng.integers(-7, 8, size=(N, K)).astype(f32)
    if kind == "seven":
        c[:, ::64] = 7.0
    elif kind == "eight":
        c[:, ::64] = -8.0
    elif kind == "ternary":
        c = np.sign(c)
    else:
        c = -(c > 0).astype(f32)
    return c * np.abs(rng.normal(0.02, 0.005, size=(N, 1))).astype(f32)


@pytest.mark.parametrize("K,wgroup,N", [(256, 0, 20501), (1280, 0, 48), (1280, 256, 4101), (1536, 64, 2731)])
def test_tensors_on_the_grid(oracle, K, wgroup, N):
    """Ratios without any error, one or two of them, and such rows where squares underflow in fp32: scaled down, or with an element so
    small that only the reference's sums see it."""
    rng = np.random.default_rng(K + wgroup)
    kinds = [grid_rows(kind, 3, K, rng) for kind in ("seven", "eight", "ternary", "negative")]
    w = np.concatenate(kinds + [k * f32(1e-15) for k in kinds] + [k * f32(1e-25) for k in kinds] + kinds)
    w[36:, 1::64] = f32(1e-24)
    got = rq.quantize_weights(torch.from_numpy(repeated(w, N)).to(DEV), rq.TYPE_W4A4, wgroup=wgroup)
    want = repeated(oracle.quantize_rows_w(w, wgroup=wgroup), N)
    assert blocks_equal(got, want), block_diff(got, want)


@pytest.mark.parametrize("K,N,wgroup", [(256, 32768, 0), (5120, 4096, 0), (5120, 4096, 256), (5120, 4096, 64)])
def test_tensors_on_the_grid_need_no_search_in_order(K, N, wgroup):
    """Converting a dequantized tensor again takes about as long as converting any other one (three to seven times as long where
    every segment goes to the search in element order behind the fp32 sums)."""
    L = rq.load_library()
    ws = torch.empty(L.rq_w4a4_quantize_weights_workspace_bytes(rq.TYPE_W4A4, K, N, wgroup), dtype=torch.uint8, device=DEV)
    out = torch.empty(N * (K // 256) * 144, dtype=torch.uint8, device=DEV)
    rng = np.random.default_rng(3)
    us = []
    for w in (rng.normal(0, 0.02, size=(N, K)).astype(f32), grid_rows("seven", N, K, rng), grid_rows("ternary", N, K, rng)):
        w = torch.from_numpy(w).to(DEV)
        times = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(10):
                assert L.rq_w4a4_quantize_weights(rq.TYPE_W4A4, w.data_ptr(), K, N, K, K, wgroup, out.data_ptr(),
                                                  ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1) * 100)
        us.append(min(times))
    print("K=%d N=%d wgroup=%d: %.0f us, on the grid %.0f, %.0f" % ((K, N, wgroup) + tuple(us)), flush=True)
    assert max(us[1:]) < 2 * us[0]


def test_conversions_in_several_runs(oracle):
    """Blocks on the way to the GPU in more runs of rows than there are pinned buffers, from a read-only array. (Tensors on the way to
    the host in one run here, in several in the tests below.)"""
    w = tensor(4097, 256, 3)
    got = rq.quantize_weights(torch.from_numpy(w).to(DEV), rq.TYPE_W4A4)
    want = oracle.quantize_rows_w(w)
    assert blocks_equal(got, want), block_diff(got, want)
    blocks = np.tile(want, (9, 4))[:30001]            # 17 MB of blocks: five runs
    blocks.flags.writeable = False
    got = rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV).cpu().numpy()
    assert bits_equal(got, rq.dequantize_rows(blocks))


@pytest.mark.parametrize("type_,wgroup", [(rq.TYPE_W4A4H, 0), (rq.TYPE_W4A4, 64), (rq.TYPE_W4A4H, 64)])
def test_blocks_fetched_in_more_runs_than_buffers(type_, wgroup):
    """9000 rows of 4096: five runs of rows (20.7 MB) through three buffers, in turn on two streams or, rotated with a scale per 64
    inputs, converted on the one and copied on the other. The bytes are those of one call of the C entry point."""
    N, K = 9000, 4096
    g = torch.Generator(device=DEV)
    g.manual_seed(4)
    w = torch.randn((N, K), dtype=torch.float32, device=DEV, generator=g) * 0.02
    L = rq.load_library()
    ws = torch.empty(L.rq_w4a4_quantize_weights_workspace_bytes(type_, K, N, wgroup), dtype=torch.uint8, device=DEV)
    out = torch.full((N * (K // 256) * 144,), 0xA5, dtype=torch.uint8, device=DEV)
    assert L.rq_w4a4_quantize_weights(type_, w.data_ptr(), K, N, K, K, wgroup, out.data_ptr(), ws.data_ptr(), ws.numel(),
                                      torch.cuda.current_stream().cuda_stream) == 0
    want = out.cpu().numpy().view(rq.BLOCK_DTYPE).reshape(N, K // 256)
    for _ in range(2):
        got = rq.quantize_weights(w, type_, wgroup=wgroup)
        assert blocks_equal(got, want), block_diff(got, want)


@pytest.mark.parametrize("K,rows,apart", [(256, 100001, True), (5376, 1400, True), (5376, 6001, True), (17408, 1280, False)])
def test_rotated_rows_in_several_runs(K, rows, apart):
    """Rows whose runs are decoded on the second stream alone (four runs, two, five) and in turn on both: the same floats as in pieces
    that go through in one run."""
    assert w4a4._decodes_slowly(K, K) == apart
    g = torch.Generator(device=DEV)
    g.manual_seed(K)
    blocks = rq.quantize_weights(torch.randn((rows, K), dtype=torch.float32, device=DEV, generator=g) * 0.02, rq.TYPE_W4A4H)
    step = w4a4._STAGE_BYTES // (K // 256 * 144)
    want = torch.cat([rq.dequantize(blocks[a:a + step], rq.TYPE_W4A4H, device=DEV) for a in range(0, rows, step)])
    for _ in range(3):
        got = rq.dequantize(blocks, rq.TYPE_W4A4H, device=DEV)
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
        got.fill_(float("nan"))   # (the next call gets this memory)
        del got


@pytest.mark.parametrize("rows", [1, 3639, 3640, 3641, 5461, 5462])
def test_conversions_around_one_buffer(oracle, rows):
    """A tensor whose blocks fit one pinned buffer (3640 rows of 8 blocks, 4 MiB; 5461 on the way to the host) goes through
    without the second stream; the last that fits and the first that does not; a read-only array and a writable one."""
    w = tensor(rows, 2048, 5)
    got = rq.quantize_weights(torch.from_numpy(w).to(DEV), rq.TYPE_W4A4)
    want = oracle.quantize_rows_w(w)
    assert blocks_equal(got, want), block_diff(got, want)
    for writable in (True, False):
        blocks = want.copy()
        blocks.flags.writeable = writable
        out = rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV).cpu().numpy()
        assert bits_equal(out, rq.dequantize_rows(blocks))


@pytest.mark.parametrize("rows", [200, 30001])
def test_conversions_under_a_default_device(oracle, rows):
    """A program may have made the GPU torch's default device: the conversions' host buffers stay on the host (one
    buffer; several)."""
    w = tensor(200, 256, 9)
    want = oracle.quantize_rows_w(w)
    blocks = np.tile(want, (rows // 200 + 1, 4))[:rows]
    with torch.device(DEV):
        got = rq.quantize_weights(torch.from_numpy(np.tile(w, (rows // 200 + 1, 1))[:rows]).to(DEV), rq.TYPE_W4A4)
        out = rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV)
    assert blocks_equal(got, np.tile(want, (rows // 200 + 1, 1))[:rows])
    assert bits_equal(out.cpu().numpy(), rq.dequantize_rows(blocks))


@pytest.mark.parametrize("rows", [200, 9000])
def test_conversions_are_refused_under_capture(rows):
    """A captured conversion would replay a copy of whatever its host buffer holds by then: it is refused (one buffer;
    several), and works again outside."""
    w = torch.randn((rows, 1024), dtype=torch.float32, device=DEV)
    blocks = rq.quantize_weights(w, rq.TYPE_W4A4)
    want = rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV)
    torch.cuda.synchronize()
    for convert in (lambda: rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV), lambda: rq.quantize_weights(w, rq.TYPE_W4A4)):
        with pytest.raises(rq.RqError, match="capture"):
            with torch.cuda.graph(torch.cuda.CUDAGraph()):
                convert()
    assert torch.equal(rq.dequantize(rq.quantize_weights(w, rq.TYPE_W4A4), rq.TYPE_W4A4, device=DEV), want)


def test_conversions_keep_their_second_stream():
    """Conversions in several runs keep the stream that their copies go to (a new one costs milliseconds at its first
    work): one per thread and current stream, a bounded number of them; the blocks are right on all of them."""
    w = torch.randn((9000, 1024), dtype=torch.float32, device=DEV)   # 5.2 MB of blocks
    blocks = rq.quantize_weights(w, rq.TYPE_W4A4)
    want = rq.dequantize_rows(blocks)
    kept = w4a4._copiers.streams
    n = len(kept)
    before = dict(kept)
    for _ in range(3):
        assert blocks_equal(rq.quantize_weights(w, rq.TYPE_W4A4), blocks)
        assert bits_equal(rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV).cpu().numpy(), want)
    assert w4a4._copiers.streams == before and len(kept) == n
    torch.cuda.synchronize()
    for _ in range(2 * w4a4._COPIERS):
        with torch.cuda.stream(torch.cuda.Stream()):
            assert bits_equal(rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV).cpu().numpy(), want)
    assert len(w4a4._copiers.streams) == w4a4._COPIERS

    seen, ok = [], []

    def other():
        for _ in range(5):
            ok.append(blocks_equal(rq.quantize_weights(w, rq.TYPE_W4A4), blocks))
            ok.append(bits_equal(rq.dequantize(blocks, rq.TYPE_W4A4, device=DEV).cpu().numpy(), want))
        seen.append(list(w4a4._copiers.streams.values()))

    threads = [threading.Thread(target=other) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(ok) == 20 and all(ok)
    assert [len(s) for s in seen] == [1, 1] and seen[0][0] is not seen[1][0]


def test_a_small_conversion_launches_first(monkeypatch):
    """In one run the host makes no Stream object in front of the launch but the one that the launch needs: the GPU would wait for it."""
    order = []
    real_stream, real_library = torch.cuda.current_stream, rq.load_library()

    class Library:
        def __getattr__(self, name):
            if name == "rq_w4a4_quantize_weights":
                order.append("launches")
            return getattr(real_library, name)

    def current_stream(*args):
        order.append("stream")
        return real_stream(*args)

    w = torch.randn((97, 1024), dtype=torch.float32, device=DEV)
    want = rq.quantize_weights(w, rq.TYPE_W4A4, wgroup=256)
    monkeypatch.setattr(w4a4, "load_library", Library)
    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    got = rq.quantize_weights(w, rq.TYPE_W4A4, wgroup=256)
    assert order == ["launches", "stream", "stream"]   # (the call's name is looked up, then its arguments are made)
    assert blocks_equal(got, want)


def test_second_stream_waits_behind_the_allocations(monkeypatch):
    """Device memory that a conversion takes may still be in use by work that another thread queued on the same stream meanwhile:
    the second stream waits for the first behind the last allocation."""
    order = []
    real_bytes, real_wait = w4a4._device_bytes, torch.cuda.Stream.wait_stream

    def device_bytes(*args):
        order.append("allocates")
        return real_bytes(*args)

    def wait_stream(self, other):
        order.append("waits")
        return real_wait(self, other)

    w = torch.randn((9000, 4096), dtype=torch.float32, device=DEV)
    monkeypatch.setattr(w4a4, "_device_bytes", device_bytes)
    monkeypatch.setattr(torch.cuda.Stream, "wait_stream", wait_stream)
    rq.quantize_weights(w, rq.TYPE_W4A4)
    assert order == ["allocates", "allocates", "waits"]


@pytest.mark.parametrize("wgroup", [0, 256, 64])
def test_scales_that_the_first_look_leaves_open(oracle, wgroup):
    """Enough segments that some (one in a hundred or fewer) have two ratios whose errors are too near for the fp32 sums, and rows
    that those sums do not cover: sums of zero, denormal ones, infinite ones, infinities, NaNs, scales out of range; the last
    wavefront is not full. Every byte as from the reference's sums in its order."""
    N, K = 5202, 1024
    w = tensor(N, K, 11 + wgroup)
    rng = np.random.default_rng(wgroup)
    for r, scale in enumerate([1e-38, 1e-30, 1e-20, 1e18, 1e37]):
        w[10 * r + 1] = (rng.standard_normal(K) * scale).astype(f32)
    w[60], w[61], w[62] = 0.0, 0.0, 0.0
    w[60, ::64] = 0.3                     # one element of every group
    w[61, ::64] = np.float32(1e-44)
    w[62, 5] = -2.0
    w[70, 3], w[71, ::64], w[72, :] = np.inf, np.nan, np.nan
    w[N - 1] = np.where(np.arange(K) % 2 == 0, 0.7, -0.7)
    got = rq.quantize_weights(torch.from_numpy(w).to(DEV), rq.TYPE_W4A4, wgroup=wgroup)
    want = oracle.quantize_rows_w(w, wgroup=wgroup)
    assert blocks_equal(got, want), block_diff(got, want)
