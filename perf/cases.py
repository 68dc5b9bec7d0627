"""What the speed of this framework is measured on: its operators on device "vk", called as a program that serves or
trains a quantised model calls them, from one row (a token) to thousands (a prompt, a batch).

  q8      torch._weight_int8pack_mm: the linear layers of a model with int8 weights
  q4      torch._dyn_quant_matmul_4bit: the same with 4-bit weights in groups of `group` values (0: a scale per row)
  f8      the same with float8 weights and activations: the activations are brought to float8 (a scale per row: the
          producer torch.ops.vk.fp8_quant_rowwise; a scale per tensor: a cast), then torch._scaled_mm
  linear  a 16-bit linear layer in training: the product, and both of its gradients
  affine  a tensor to quint8 and back, and through fake quantisation

q8, q4 and f8 run `products` layers one after the other, [k -> n], [n -> k], [k -> n] ..., each on the output of the
layer before it, as the two projections of a model's feed-forward blocks follow each other; every layer has weights of
its own.  `m` is the number of rows.
"""
import math

import torch

import torch_vulkan_amd.backend  # noqa: F401  (registers device "vk")

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # The smallest call: one float32 row against square 4096 x 4096 int8 weights.  Launches and latency.
        dict(name="q8_row_f32", kind="q8", dtype="f32", m=1, k=4096, n=4096, products=2),
        # One token of one sequence through two blocks' projections of 4096 <-> 14336: the weights are the work.
        dict(name="q8_row", kind="q8", dtype="bf16", m=1, k=4096, n=14336, products=4),
        # 64 sequences decoded together, the same projections.
        dict(name="q8_batch", kind="q8", dtype="bf16", m=64, k=4096, n=14336, products=4),
        # A prompt of a length that is no round number, projections of 5120 <-> 13824.
        dict(name="q8_prompt", kind="q8", dtype="bf16", m=1537, k=5120, n=13824, products=2),
        # 4-bit weights, groups of 32, 4096 <-> 11008: one token, 32 sequences, a prompt.
        dict(name="q4_row", kind="q4", dtype="f32", m=1, k=4096, n=11008, group=32, products=4),
        dict(name="q4_batch", kind="q4", dtype="f32", m=32, k=4096, n=11008, group=32, products=4),
        dict(name="q4_prompt", kind="q4", dtype="f32", m=2048, k=4096, n=11008, group=32, products=2),
        # float8, 16 sequences decoded together, 8192 <-> 28672, scales per row.
        dict(name="f8_batch", kind="f8", dtype="bf16", m=16, k=8192, n=28672, scaling="row", products=2),
        # float8, a large square product with one scale per tensor.
        dict(name="f8_square", kind="f8", dtype="bf16", m=8192, k=8192, n=8192, scaling="tensor", products=1),
        # float8, a prompt through the widest projection, scales per row: the largest case.
        dict(name="f8_prompt", kind="f8", dtype="bf16", m=4096, k=8192, n=28672, scaling="row", products=1),
        # A training step of one linear layer on 4096 tokens: y = x w', dx = dy w, dw = dy' x.
        dict(name="linear_train", kind="linear", dtype="bf16", m=4096, k=4096, n=14336),
        # An 11008 x 4096 float32 weight through the quantised-tensor operators and fake quantisation.
        dict(name="affine", kind="affine", m=11008, k=4096),
    ]


# the most multiply-adds a drawn case of a kind takes: those of the kind's largest listed case
MOST = {"q8": 1537 * 5120 * 13824 * 2, "q4": 2048 * 4096 * 11008 * 2, "f8": 4096 * 8192 * 28672, "linear": 4096 * 4096 * 14336}


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _wide(rng, low, high, step):
    return max(low, min(high, step * round(_spread(rng, low, high) / step)))


def draw(rng):
    kind = rng.choice(("q8", "q8", "q8", "q4", "q4", "q4", "f8", "f8", "f8", "linear", "affine"))
    if kind == "affine":
        return dict(kind=kind, m=_spread(rng, 64, 11008), k=rng.randint(512, 4096))
    # model widths are multiples of 64 (of the group size, for 4-bit weights)
    k, n = _wide(rng, 1024, 16384, 64), _wide(rng, 1024, 28672, 64)
    if kind == "linear":
        case = dict(kind=kind, dtype=rng.choice(("bf16", "bf16", "f16")), m=_spread(rng, 128, 8192), k=k, n=n)
        while case["m"] * k * n > MOST[kind]:
            case["m"] //= 2
        return case
    rows = rng.choice(("one", "few", "many"))
    m = {"one": 1, "few": _spread(rng, 2, 64), "many": _spread(rng, 65, 4096)}[rows]
    products = 2 if rows == "many" else 4
    if rng.random() < 0.25:  # a model's last projection: as many columns as its vocabulary has entries, odd ones too
        n, products = rng.randint(16000, 28672), 1
    case = dict(kind=kind, m=m, k=k, n=n, products=products)
    if kind == "q8":
        case["dtype"] = rng.choice(("bf16", "bf16", "f16", "f32"))
    elif kind == "q4":
        case["group"] = rng.choice((32, 32, 64, 128, 0))
        case["dtype"] = rng.choice(("f32", "bf16")) if case["group"] == 0 else "f32"
        if case["group"] == 128:
            case["k"] = k = 128 * (k // 128)
            if products > 1:
                case["n"] = n = 128 * (n // 128)
    else:
        case["scaling"] = rng.choice(("row", "row", "tensor"))
        case["dtype"] = rng.choice(("bf16", "bf16", "bf16", "f16"))
    while case["m"] * k * n * products > MOST[kind]:
        if products > 1:
            case["products"] = products = 1
        else:
            case["m"] //= 2
    return case


class _Source:
    """Seeded values, made on the GPU's own generator and brought to the device through host memory."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, dtype, sd=1.0):
        return (torch.randn(shape, generator=self.g, device="cuda") * sd).to(dtype).cpu().to("vk")

    def uniform(self, shape, dtype, low, high):
        return (torch.rand(shape, generator=self.g, device="cuda") * (high - low) + low).to(dtype).cpu().to("vk")

    def whole(self, shape, dtype, low, high):
        return torch.randint(low, high, shape, generator=self.g, device="cuda", dtype=dtype).cpu().to("vk")


def prepare(case, seed):
    src, kind = _Source(seed), case["kind"]
    if kind == "affine":
        return dict(kind=kind, x=src.normal((case["m"], case["k"]), torch.float32, 3.0))
    dtype, m, k, n = DTYPES[case["dtype"]], case["m"], case["k"], case["n"]
    if kind == "linear":
        return dict(kind=kind, x=src.normal((m, k), dtype), w=src.normal((n, k), dtype, k ** -0.5), dy=src.normal((m, n), dtype))
    layers = []
    for i in range(case["products"]):
        ins, outs = (k, n) if i % 2 == 0 else (n, k)
        if kind == "q8":  # scales so that a layer keeps its input's magnitude
            unit = 1.0 / (74 * math.sqrt(ins))
            layers.append((src.whole((outs, ins), torch.int8, -128, 128), src.uniform((outs,), dtype, 0.5 * unit, 1.5 * unit)))
        elif kind == "q4":
            group = case["group"] or ins
            unit = 1.0 / (4.6 * math.sqrt(ins))
            nibbles, bias = src.whole((outs, ins // 2), torch.uint8, 0, 256), src.normal((outs,), torch.float32, 0.1)
            scales = src.uniform((outs, ins // group), torch.float32, 0.5 * unit, 1.5 * unit)
            layers.append((torch._dyn_quant_pack_4bit_weight(nibbles, scales, bias, group, ins, outs), group, ins, outs))
        elif case["scaling"] == "row":
            w, scale = torch.ops.vk.fp8_quant_rowwise(src.normal((outs, ins), torch.bfloat16, ins ** -0.5), torch.float8_e4m3fn)
            layers.append((w.t(), scale.t()))
        else:
            layers.append((src.normal((outs, ins), torch.float8_e4m3fn).t(), torch.tensor(ins ** -0.5).to("vk")))
    return dict(kind=kind, x=src.normal((m, k), dtype), layers=layers, dtype=dtype, scaling=case.get("scaling"), one=torch.tensor(1.0).to("vk"))


def run(state):
    kind, x = state["kind"], state["x"]
    if kind == "affine":
        q = torch.quantize_per_tensor(x, 0.1, 117, torch.quint8)
        return [q.int_repr(), q.dequantize(), torch.fake_quantize_per_tensor_affine(x, 0.08, 3, -128, 127)]
    if kind == "linear":
        w, dy = state["w"], state["dy"]
        return [torch.mm(x, w.t()), torch.mm(dy, w), torch.mm(dy.t(), x)]
    outputs = []
    for layer in state["layers"]:
        if kind == "q8":
            weight, scales = layer
            x = torch._weight_int8pack_mm(x, weight, scales)
        elif kind == "q4":
            packed, group, ins, outs = layer
            x = torch._dyn_quant_matmul_4bit(x, packed, group, ins, outs)
        elif state["scaling"] == "row":
            weight, scale = layer
            q, row_scales = torch.ops.vk.fp8_quant_rowwise(x, torch.float8_e4m3fn)
            x = torch._scaled_mm(q, weight, row_scales, scale, out_dtype=state["dtype"])
        else:
            weight, scale = layer
            x = torch._scaled_mm(x.to(torch.float8_e4m3fn), weight, state["one"], scale, out_dtype=state["dtype"])
        outputs.append(x)
    return outputs


def work(case):
    kind, m, k = case["kind"], case["m"], case["k"]
    if kind == "affine":  # float32 in, the bytes, and two float32 tensors out
        return {"bytes": m * k * (4 + 1 + 4 + 4), "flops": 0}
    n, item = case["n"], {"f32": 4, "f16": 2, "bf16": 2}[case["dtype"]]
    if kind == "linear":  # x, w, dy in; y, dx, dw out
        return {"bytes": 2 * item * (m * k + n * k + m * n), "flops": 3 * 2 * m * n * k}
    per_layer = 0
    for ins, outs in ((k, n), (n, k))[: min(2, case["products"])]:
        weights = ins * outs
        if kind == "q8":
            weights += item * outs
        elif kind == "q4":
            weights = weights // 2 + 4 * outs * (ins // (case["group"] or ins) + 1)
        elif case["scaling"] == "row":
            weights += 4 * outs
        per_layer += weights + item * m * (ins + outs)
    return {"bytes": per_layer * case["products"] / min(2, case["products"]), "flops": 2 * m * n * k * case["products"]}


def tolerance(case):
    """About four times what was seen against the same chain of layers in 64 bits.  One rounding to bfloat16 (float16)
    is 1.7e-3 (2.1e-4) off as a 2-norm and half an ulp at most, 3.9e-3 (4.9e-4); the roundings of layers in a row add up
    like random ones (2.3e-3 after two, 3.4e-3 after four; largest 1.2e-2, 1.6e-2)."""
    kind, products = case["kind"], case.get("products", 1)
    if kind in ("q4", "affine"):  # integer sums and float32 operations in a fixed order
        return "exact"
    if case["dtype"] == "f32":  # sums of up to 28672 float32 products: up to 5.7e-7 after two layers, largest 4.9e-6
        return {"rel": 3e-6, "max": 3e-5}
    ulp = 1.0 if case["dtype"] == "bf16" else 0.125
    if kind == "f8":
        # an activation next to a rounding boundary of float8 falls to the other side, 2^-3 of it at most, when the layer
        # before it is rounded otherwise: 9.2e-3 after four layers, largest 0.12
        return {"rel": 7e-3 * ulp, "max": 0.25} if products == 1 else {"rel": 0.03, "max": 0.5}
    return {"rel": 7e-3 * ulp * math.sqrt(products), "max": 0.016 * ulp * products}
