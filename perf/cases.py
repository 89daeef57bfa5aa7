"""The work that users of this library have it do, as cases whose time is measured.

Three kinds of program call it. A server multiplies activations by W4A4 / W4A4H weights: one token per step while it
decodes, a handful of tokens when it verifies a draft, hundreds to thousands when it reads a prompt; as single products
or as the seven products of a transformer layer, with q / k / v and gate / up in fused calls. A converter turns fp32
tensors into blocks of either type. A tool that inspects or re-converts a model takes blocks back to fp32.

Shapes: hidden size 5120, attention width 6144 with 1024-wide keys and values, feed-forward width 17408, and the plain
4096 x 1024 product of the reference's CPU path; activations and weights are distributed as in the benchmark (`bench.py`).
"""
import math

import numpy as np
import torch

import ruquant_amd as rq

DEVICE = "cuda:0"

# name -> (K, N): the products of one transformer layer, in the order in which their outputs feed each other
LAYER = {"q": (5120, 6144), "k": (5120, 1024), "v": (5120, 1024), "o": (6144, 5120), "gate": (5120, 17408),
         "up": (5120, 17408), "down": (17408, 5120)}

# Row lengths of the repository's tests and benchmark (H12, H20 and H68 rotations, and powers of two).
ROW_LENGTHS = (1024, 1536, 3072, 4096, 4352, 5120, 6144, 8192, 10240, 17408)


def _product(name, K, N, M, had=True, wgroup=0, acts="normal", clip=1.0, kept=True):
    return {"name": name, "path": "product", "K": K, "N": N, "M": M, "had": had, "wgroup": wgroup, "acts": acts,
            "clip": clip, "kept": kept}


def listed():
    return [
        # The smallest call there is: one token through a small weight of the type without a rotation.
        _product("w4a4_k4096_n1024_m1", 4096, 1024, 1, had=False),
        # One product of a decode step, attention-sized: one token with outlier channels.
        _product("k5120_n5120_m1", 5120, 5120, 1, acts="outliers", clip=0.9),
        # The same token through the feed-forward projection, whose 45 MB of codes are the whole cost.
        _product("k5120_n17408_m1", 5120, 17408, 1, acts="outliers", clip=0.9),
        # A short draft checked by the down projection: the H68 rotation and a ragged token count.
        _product("k17408_n5120_m3", 17408, 5120, 3, acts="relu2"),
        # A decode step of one layer: seven products, four calls, each fed by the one before.
        {"name": "layer_m1", "path": "layer", "M": 1},
        # A batch of drafts (or sixteen sequences decoded together) through one layer.
        {"name": "layer_m16", "path": "layer", "M": 16},
        # A short prompt, or 64 sequences decoded together.
        _product("k5120_n17408_m64", 5120, 17408, 64, acts="student_t", clip=0.85),
        # A prompt through a tensor with one weight scale per 64 inputs and a row count of no round size.
        _product("k5120_n6000_m200_g64", 5120, 6000, 200, wgroup=64, kept=False),
        # A prompt chunk through the feed-forward projection.
        _product("k5120_n17408_m512", 5120, 17408, 512, acts="student_t", clip=0.85, kept=False),
        # The largest work of a server: a whole layer over a long prompt chunk.
        {"name": "layer_m2048", "path": "layer", "M": 2048},
        # A converter: one fp32 tensor of the attention's size to rotated blocks.
        {"name": "quantize_w4a4h_k5120_n6144", "path": "quantize", "K": 5120, "N": 6144, "had": True, "wgroup": 0},
        # A tool that reads a model back: part of a down projection to fp32, through the inverse rotation.
        {"name": "dequantize_w4a4h_k17408_n1280", "path": "dequantize", "K": 17408, "N": 1280, "had": True, "wgroup": 0},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.12:
        return {"path": "layer", "M": _log_int(rng, 1, 2000)}
    K = rng.choice(ROW_LENGTHS)
    had = rng.random() < 0.8
    wgroup = rng.choice((0, 0, 0, 256, 64))
    if kind < 0.30:
        # conversions: bounded by the listed ones' tensors
        path = "quantize" if kind < 0.21 else "dequantize"
        top = (5120 * 6144 if path == "quantize" else 17408 * 1280) // K
        return {"path": path, "K": K, "N": _log_int(rng, top // 16, top), "had": had, "wgroup": wgroup}
    M = _log_int(rng, 1, 2048)
    return {"path": "product", "K": K, "N": _log_int(rng, 256, 17408), "M": M, "had": had, "wgroup": wgroup,
            "acts": rng.choice(("normal", "outliers", "student_t", "relu2")), "clip": rng.choice((1.0, 0.9, 0.85)),
            "kept": M <= 64 or rng.random() < 0.3}


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _weight_blocks(N, K, g, had, wgroup=0, clip=1.0):
    """[N, K / 256] blocks as a model file holds them: codes uniform in 0 .. 15, row scale |N(0.02, 0.005)|; legacy
    header with the row's code sum, or integer weight multipliers 1 .. 15 per 256 or 64 inputs."""
    nb = K // 256
    qs = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, nb, 32), dtype=torch.int32, device=DEVICE, generator=g)
    d = (0.02 + 0.005 * torch.randn((N, 1), device=DEVICE, generator=g)).abs()
    if wgroup:
        mult = torch.randint(1, 16, (N, nb, 4), dtype=torch.int64, device=DEVICE, generator=g)
        if wgroup == 256:
            head = (1 << 30) | mult[..., 0]
        else:
            head = (3 << 29) | mult[..., 0] | mult[..., 1] << 4 | mult[..., 2] << 8 | mult[..., 3] << 12
    else:
        total = torch.zeros((N,), dtype=torch.int64, device=DEVICE)
        for j in range(8):
            nib = (qs >> (4 * j)) & 15
            total += (nib - 16 * (nib >= 8).to(torch.int32)).sum(dim=(1, 2))
        head = total[:, None].expand(N, nb)
    words = torch.empty((N, nb, 36), dtype=torch.int32, device=DEVICE)
    words[:, :, 0] = d.view(torch.int32)
    words[:, :, 1] = head.to(torch.int32)
    words[:, :, 2] = K
    words[:, :, 3] = int(np.float32(clip).view(np.int32)) if clip != 1.0 else 0
    words[:, :, 4:] = qs
    return words.cpu().numpy().view(rq.BLOCK_DTYPE).reshape(N, nb)


def _weight(N, K, g, had, wgroup=0, clip=1.0):
    type_ = rq.TYPE_W4A4H if had else rq.TYPE_W4A4
    return rq.W4A4Weight(_weight_blocks(N, K, g, had, wgroup, clip), type_, DEVICE, keep_blocks=False)


def _activations(kind, M, K, g):
    x = torch.randn((M, K), device=DEVICE, generator=g)
    if kind == "outliers":      # 0.5 % of the channels scaled x20, the same ones for every token
        channels = torch.randperm(K, device=DEVICE, generator=g)[:max(1, round(K * 0.005))]
        x[:, channels] *= 20.0
    elif kind == "student_t":   # Student-t, nu = 4, unit variance
        chi2 = torch.randn((4, M, K), device=DEVICE, generator=g).square().sum(dim=0)
        x = x / (chi2 / 4.0).sqrt() / math.sqrt(2.0)
    elif kind == "relu2":       # behind a squared ReLU: non-negative with a heavy right tail
        x = x.clamp_min(0.0).square()
    return x


def _fp32_weights(N, K, g):
    """A trained linear layer's look: gaussian rows of different widths and a few large entries."""
    w = 0.02 * torch.randn((N, K), device=DEVICE, generator=g)
    w *= 0.5 + torch.rand((N, 1), device=DEVICE, generator=g)
    large = torch.rand((N, K), device=DEVICE, generator=g) < 1e-4
    return torch.where(large, 8.0 * w, w)


def prepare(case, seed):
    g = _generator(seed)
    path = case["path"]
    if path == "product":
        K, N, M = case["K"], case["N"], case["M"]
        w = _weight(N, K, g, case["had"], case["wgroup"], case["clip"])
        state = {"w": w, "x": _activations(case["acts"], M, K, g), "out": None, "workspace": None}
        if case["kept"]:   # a decode loop keeps its buffers; a prompt's length is new every time and it asks for them
            state["out"] = torch.empty((M, N), dtype=torch.float32, device=DEVICE)
            state["workspace"] = w.workspace(M)
    elif path == "layer":
        M = case["M"]
        w = {name: _weight(N, K, g, True) for name, (K, N) in LAYER.items()}
        sizes = [rq.fused_workspace_bytes([w["q"], w["k"], w["v"]], M),
                 rq.fused_workspace_bytes([w["gate"], w["up"]], M),
                 rq.fused_workspace_bytes([w["o"]], M), rq.fused_workspace_bytes([w["down"]], M)]
        state = {"w": w, "x": _activations("normal", M, LAYER["q"][0], g),
                 "out": {name: torch.empty((M, N), dtype=torch.float32, device=DEVICE) for name, (K, N) in LAYER.items()},
                 "workspace": torch.empty(max(sizes), dtype=torch.uint8, device=DEVICE)}
    elif path == "quantize":
        state = {"x": _fp32_weights(case["N"], case["K"], g)}
    else:
        state = {"blocks": _weight_blocks(case["N"], case["K"], g, case["had"], case["wgroup"])}
    state["case"] = case
    return state


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "product":
        return rq.mul_mat(state["w"], state["x"], out=state["out"], workspace=state["workspace"])
    if path == "layer":
        w, o, ws = state["w"], state["out"], state["workspace"]
        rq.mul_mat_fused([w["q"], w["k"], w["v"]], state["x"], outs=[o["q"], o["k"], o["v"]], workspace=ws)
        rq.mul_mat(w["o"], o["q"], out=o["o"], workspace=ws)
        rq.mul_mat_fused([w["gate"], w["up"]], o["o"], outs=[o["gate"], o["up"]], workspace=ws)
        rq.mul_mat(w["down"], o["up"], out=o["down"], workspace=ws)
        return o
    type_ = rq.TYPE_W4A4H if case["had"] else rq.TYPE_W4A4
    if path == "quantize":
        blocks = rq.quantize_weights(state["x"], type_, wgroup=case["wgroup"])
        return blocks.view(np.int32)
    return rq.dequantize(state["blocks"], type_, device=DEVICE)


def _rotation_flops(K):
    p, m = rq.hadamard_factor(K)
    return K * (p + int(math.log2(m)))


def _product_work(K, N, M, had, wgroup, shared_input=False):
    code = N * K // 2 + 4 * N + (N * K // wgroup if wgroup else 0)
    return {"bytes": code + 4 * M * N + (0 if shared_input else 4 * M * K),
            "flops": 2 * M * N * K + (M * _rotation_flops(K) if had and not shared_input else 0)}


def work(case):
    path = case["path"]
    if path == "product":
        return _product_work(case["K"], case["N"], case["M"], case["had"], case["wgroup"])
    if path == "layer":
        # k and v take q's input, up takes gate's: read and rotated once
        parts = [_product_work(K, N, case["M"], True, 0, name in ("k", "v", "up")) for name, (K, N) in LAYER.items()]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    K, N = case["K"], case["N"]
    bytes_ = N * K * 4 + N * (K // 256) * 144
    rotation = N * _rotation_flops(K) if case["had"] else 0
    # a weight is tried at 13 clip ratios: divide, round, clamp, multiply, subtract, square, add
    return {"bytes": bytes_, "flops": rotation + (13 * 8 * N * K if path == "quantize" else N * K)}


def tolerance(case):
    # every path is defined operation by operation and gives the reference's bits
    return "exact"
