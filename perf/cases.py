"""What this package is used for, as a dozen measurable cases and a generator of more of the same ranges.

Four kinds of work, each through the entry points a user's program calls:

    op     vig_amd.batch_bid_fused_chunk_gla, the bidirectional GLA op on [B, H, L, D] tensors; with grad the gradients of
           q, k, v and both directions' gates too (torch.autograd)
    gate   vig_amd.gla_bidir_locality_gate, the op followed by the 3x3 sigmoid locality gate on the (h, w) token grid
    model  the eval forward of a ViG-T / -S / -B on a batch of images (vig_amd.layers)
    train  one training pass of such a model: forward, cross-entropy, backward, in fp32 (the models' own configurations
           train without AMP) or under bf16 autocast

Head shapes are those of the models (Dk 32, Dv 64: a ViG layer; Dk 64, Dv 64: the op's own benchmark), lengths run from a
small image's grid to a 1024 x 1024 image's 4096 tokens and need not be multiples of anything.
"""
import math

import torch
import torch.nn.functional as F

import vig_amd
from vig_amd import layers

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
WIDTH = {"t": 192, "s": 384, "b": 768}  # embedding width of a model; 64 channels of it per head
BUILD = {"t": layers.vig_tiny, "s": layers.vig_small, "b": layers.vig_base}
DEPTH = 12
CLASSES = 1000

# the most a case may hold, as the listed cases do: (batch, head, token) positions of an op call in bf16 inference, and
# the size of a model forward and of a training pass under bf16 autocast (_model_size; fp32 takes up to five times as long)
MOST_POSITIONS = 128 * 6 * 196
MOST_MODEL = 256 * 196 * 384
MOST_TRAIN = 128 * 196 * 384


def _op(name, B, H, L, Dk, dtype="bf16", grad=False):
    return {"name": name, "kind": "op", "B": B, "H": H, "L": L, "Dk": Dk, "dtype": dtype, "grad": grad}


def listed():
    return [
        # one ViG-T layer on one image: the smallest call, latency and host time only
        _op("op_one_image", 1, 3, 196, 32),
        # the op at the ViG-S benchmark shape
        _op("op_vig_s", 128, 6, 196, 64),
        # the 4096 tokens of a 1024 x 1024 image, few sequences
        _op("op_4096_tokens", 8, 3, 4096, 64),
        # fp32 tensors, 14 x 14 patches and a class token (an odd length)
        _op("op_fp32", 32, 6, 197, 64, dtype="fp32"),
        # training the op at the ViG-S benchmark shape
        _op("op_grad_vig_s", 128, 6, 196, 64, grad=True),
        # training on larger images (48 x 48 patches and one token more): states link the segments both ways
        _op("op_grad_2305_tokens", 4, 6, 2305, 32, grad=True),
        # a layer of a model that trains without AMP
        _op("op_grad_fp32", 64, 6, 196, 32, dtype="fp32", grad=True),
        # the op with the locality gate at the ViG-B shape
        {"name": "gate_vig_b", "kind": "gate", "B": 64, "H": 12, "h": 14, "w": 14, "Dk": 64},
        # classifying one image as it arrives
        {"name": "model_t_one_image", "kind": "model", "model": "t", "B": 1, "side": 224},
        # classifying a data set: the throughput batch
        {"name": "model_s_batch_256", "kind": "model", "model": "s", "B": 256, "side": 224},
        # dense 1024 x 1024 input, where linear attention is for
        {"name": "model_t_1024px", "kind": "model", "model": "t", "B": 8, "side": 1024},
        # a training pass under mixed precision
        {"name": "train_s_batch_128", "kind": "train", "model": "s", "B": 128, "side": 224, "amp": True},
    ]


def _model_size(model, side):
    """Activation values of one image's tokens, the wider model's larger products counted in."""
    return (side // 16) ** 2 * WIDTH[model] * max(1, WIDTH[model] // 384)


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["op", "op", "op", "op", "gate", "model", "model", "train"])
    if kind == "op":
        grad, dtype = rng.random() < 0.5, rng.choice(["bf16", "bf16", "fp32"])
        H, L = rng.choice([3, 6, 12]), _log_int(rng, 49, 4097)
        most = max(1, MOST_POSITIONS // (4 if dtype == "fp32" else 1) // (H * L))
        return {"kind": "op", "B": _log_int(rng, 1, most), "H": H, "L": L, "Dk": rng.choice([32, 64]), "dtype": dtype, "grad": grad}
    if kind == "gate":
        H, h, w = rng.choice([3, 6, 12]), rng.randint(7, 32), rng.randint(7, 32)
        return {"kind": "gate", "B": _log_int(rng, 1, max(1, MOST_POSITIONS // (H * h * w))), "H": H, "h": h, "w": w, "Dk": rng.choice([32, 64])}
    model = rng.choice(["t", "s", "b"])
    side = 16 * _log_int(rng, 8, 64 if kind == "model" else 24)
    if kind == "model":
        return {"kind": "model", "model": model, "B": _log_int(rng, 1, max(1, MOST_MODEL // _model_size(model, side))), "side": side}
    amp = rng.random() < 0.5
    most = MOST_TRAIN // (_model_size(model, side) * (1 if amp else 5))
    return {"kind": "train", "model": model, "B": _log_int(rng, 4, max(4, most)), "side": side, "amp": amp}


def _op_inputs(case, L, dtype, gen):
    """q, k, v ~ N(0, 1), keys scaled by Dk^-0.5, each direction's log-gates logsigmoid(N(0, 1)) / 16: what a block of the
    models feeds the op."""
    B, H, Dk = case["B"], case["H"], case["Dk"]
    r = lambda *s: torch.randn(*s, device=DEV, generator=gen)  # noqa: E731
    q, k, v = r(B, H, L, Dk), r(B, H, L, Dk) * Dk ** -0.5, r(B, H, L, 64)
    g = F.logsigmoid(r(2 * B, H, L, Dk)) / 16
    return [t.to(dtype) for t in (q, k, v, g)]


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    if kind == "op":
        dtype = DTYPES[case["dtype"]]
        x = _op_inputs(case, case["L"], dtype, gen)
        state = {"kind": "op", "x": x}
        if case["grad"]:
            for t in x:
                t.requires_grad_()
            state["d_o"] = torch.randn(x[2].shape, device=DEV, generator=gen).to(dtype)
        return state
    if kind == "gate":
        q, k, v, g = _op_inputs(case, case["h"] * case["w"], torch.bfloat16, gen)
        weight = torch.randn(case["H"] * 64, 1, 3, 3, device=DEV, generator=gen) / 3
        return {"kind": "gate", "x": (q, k, v, g[:case["B"]], g[case["B"]:], weight), "hw": (case["h"], case["w"])}
    torch.manual_seed(seed)
    with torch.device(DEV):
        kw = {"drop_path_rate": 0.0} if kind == "train" else {}  # (a pass that can be repeated)
        net = BUILD[case["model"]](img_size=case["side"], num_classes=CLASSES, **kw)
    images = torch.randn(case["B"], 3, case["side"], case["side"], device=DEV, generator=gen)
    if kind == "model":
        return {"kind": "model", "net": net.eval().to(torch.bfloat16), "images": images.to(torch.bfloat16)}
    target = torch.randint(0, CLASSES, (case["B"],), device=DEV, generator=gen)
    return {"kind": "train", "net": net.train(), "images": images, "target": target, "amp": case["amp"]}


def run(state):
    kind = state["kind"]
    if kind == "op":
        o, _ = vig_amd.batch_bid_fused_chunk_gla(*state["x"])
        return (o.detach(),) + torch.autograd.grad(o, state["x"], state["d_o"]) if "d_o" in state else o
    if kind == "gate":
        return vig_amd.gla_bidir_locality_gate(*state["x"], state["hw"])
    if kind == "model":
        return state["net"](state["images"])
    net = state["net"]
    net.zero_grad(set_to_none=True)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=state["amp"]):
        logits = net(state["images"]).float()
        loss = F.cross_entropy(logits, state["target"])
    loss.backward()
    # the gradients as one vector, the way a data-parallel step reduces them
    return {"loss": loss.detach(), "logits": logits.detach(), "grads": torch.cat([p.grad.reshape(-1) for p in net.parameters()])}


def _model_work(case):
    """(operations of one forward, parameters): the products of the layers, the op and the two stem convolutions."""
    C, n = WIDTH[case["model"]], (case["side"] // 16) ** 2
    I = 256 * math.ceil(C * 8 / 3 / 256)
    weights = 2 * C * C + C * C + 16 * C + 16 * C + C * C + 3 * C * I  # qkv, g, both gate layers, o, the MLP's
    token = 2 * weights + 18 * C + 8 * 32 * 64 * (C // 64)
    stem = (case["side"] // 8) ** 2 * C * 243 + n * C * C * 9
    params = DEPTH * (weights + 14 * C) + C * n + C * 243 // 2 + C * C * 9 // 2 + CLASSES * (C + 1)
    return case["B"] * (DEPTH * n * token + stem + 2 * C * CLASSES), params


def work(case):
    kind = case["kind"]
    if kind in ("op", "gate"):
        e = 4 if case.get("dtype") == "fp32" else 2
        Dk, Dv = case["Dk"], 64
        n = case["B"] * case["H"] * (case["L"] if kind == "op" else case["h"] * case["w"])
        moved, ops = 4 * Dk + 2 * Dv, 8 * Dk * Dv  # q, k, two gates, v, o; the state's update and its read-out, twice
        if case.get("grad"):
            moved += 4 * Dk + 2 * Dv  # dq, dk, two gate gradients, dv, do
            ops += 16 * Dk * Dv  # each product's two gradients
        if kind == "gate":
            ops += 18 * Dv
        return {"bytes": n * moved * e, "flops": n * ops}
    ops, params = _model_work(case)
    if kind == "model":
        return {"bytes": 2 * (case["B"] * (3 * case["side"] ** 2 + CLASSES) + params), "flops": ops}
    return {"bytes": 4 * (case["B"] * (3 * case["side"] ** 2 + CLASSES) + 2 * params), "flops": 3 * ops}


def tolerance(case):
    kind = case["kind"]
    if kind == "op":
        return {"rel": 1e-5} if case["dtype"] == "fp32" else {"rel": 1e-2}
    if kind == "gate":
        return {"rel": 1e-2}
    if kind == "model" or case["amp"]:
        return {"rel": 2e-2}  # twelve layers of bf16 activations
    return {"rel": 1e-4}  # twelve layers of 32-bit sums
