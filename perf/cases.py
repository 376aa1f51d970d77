"""The calls whose speed is measured: what programs on this backend spend their time in, from the smallest dispatch to
the largest, through the package's public entry points.

A case names a program (one op, or a whole network as one program) and its sizes.  As in a serving process the program is
serialised and loaded once and kept; what changes from call to call are its inputs, so those come from the seed.  One pass
is one dispatch: device buffers are enqueued and not waited for, host buffers are dispatched blocking."""
import json
import math

import numpy as np
import torch

from torq_compiler_amd import Device, Executable, Program, workloads

WEIGHT_SEED = 1400  # the weights of a program are the same in every process


def listed():
    return [
        # the smallest call: one row through a square int8 layer (a single detection head, the last layer of a classifier)
        dict(name="linear_i8_1x2048x2048", kind="linear_i8", M=1, K=2048, N=2048),
        # a batch of tokens or regions through a wide int8 layer
        dict(name="linear_i8_512x4096x4096", kind="linear_i8", M=512, K=4096, N=4096),
        # the benchmark's headline product
        dict(name="linear_i8_4096x4096x4096", kind="linear_i8", M=4096, K=4096, N=4096),
        # one image of a single-camera pipeline: the 3x3 convolution of the first benchmark configuration
        dict(name="conv_i8_112x112x32_b1", kind="conv_i8", batch=1, size=112, C=32, O=64, window=3, stride=1),
        # a 3x3 convolution of a batch, channels that fill no power of two
        dict(name="conv_i8_56x56x96_b32", kind="conv_i8", batch=32, size=56, C=96, O=96, window=3, stride=1),
        # an image network: one image at a time for latency, ...
        dict(name="mobilenet_v2_b1", kind="image_net", batch=1, resolution=224, width=1.0, host=False),
        # ... a batch that arrives in host memory and whose classes go back there, ...
        dict(name="mobilenet_v2_b32_host", kind="image_net", batch=32, resolution=224, width=1.0, host=True),
        # ... and a large batch for throughput
        dict(name="mobilenet_v2_b256", kind="image_net", batch=256, resolution=224, width=1.0, host=False),
        # a decoder's step: one conversation, and a full batch of them
        dict(name="decoder_step_b1", kind="decoder_step", batch=1, layers=26, hidden=1152, heads=4, head_dim=256, ffn=6912, vocab=262144,
             cache_len=1024),
        dict(name="decoder_step_b32", kind="decoder_step", batch=32, layers=26, hidden=1152, heads=4, head_dim=256, ffn=6912, vocab=262144,
             cache_len=1024),
        # the same decoder reading a prompt: its feed-forward layer over 2048 tokens
        dict(name="linear_bf16_2048x1152x6912", kind="linear_bf16", M=2048, K=1152, N=6912, block=0),
        # a product of two activations with a 16-bit result (attention scores of an int8 network)
        dict(name="matmul_i8_4x1024x128x1024", kind="matmul_i8", B=4, M=1024, K=128, N=1024, out="int16"),
    ]


def _log(rng, low, high, step=1):
    """A whole number from low to high, even over its logarithm, in multiples of `step`."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear_i8", "conv_i8", "image_net", "decoder_step", "linear_bf16", "matmul_i8"])
    while True:
        if kind == "linear_i8":
            ragged = rng.random() < 0.3
            c = dict(M=_log(rng, 1, 4096), K=_log(rng, 64, 8192, 1 if ragged else 16), N=_log(rng, 16, 8192, 1 if ragged else 16))
            fits = c["M"] * c["K"] * c["N"] <= 4096 ** 3
        elif kind == "conv_i8":
            ragged = rng.random() < 0.3
            c = dict(batch=_log(rng, 1, 32), size=_log(rng, 7, 160), C=_log(rng, 3, 512) if ragged else _log(rng, 16, 512, 16),
                     O=_log(rng, 8, 512, 1 if ragged else 8), window=rng.choice([1, 3, 3, 5]), stride=rng.choice([1, 1, 2]))
            fits = work(dict(c, kind=kind))["flops"] <= 4e10
        elif kind == "image_net":
            c = dict(batch=_log(rng, 1, 256), resolution=rng.randrange(96, 225), width=rng.choice([0.5, 0.75, 1.0]), host=rng.random() < 0.3)
            fits = True
        elif kind == "decoder_step":
            c = dict(batch=_log(rng, 1, 32), layers=rng.randrange(1, 7), hidden=_log(rng, 256, 2048, 128), heads=rng.choice([2, 4, 8]),
                     head_dim=rng.choice([64, 128, 256]), ffn=_log(rng, 512, 8192, 128), vocab=_log(rng, 4096, 65536, 16),
                     cache_len=_log(rng, 128, 2048, 8))
            fits = True
        elif kind == "linear_bf16":
            block = rng.choice([0, 0, 32, 128])
            c = dict(M=_log(rng, 1, 4096), K=_log(rng, 128, 8192, block or 8), N=_log(rng, 64, 8192, rng.choice([1, 16])), block=block)
            fits = c["M"] * c["K"] * c["N"] <= 2048 * 1152 * 6912
        else:
            c = dict(B=_log(rng, 1, 16), M=_log(rng, 1, 2048), K=_log(rng, 16, 1024, rng.choice([1, 16])), N=_log(rng, 16, 2048, rng.choice([1, 16])),
                     out=rng.choice(["int8", "int16", "int32"]))
            fits = c["B"] * c["M"] * c["K"] * c["N"] <= 1 << 33
        if fits:
            return dict(c, kind=kind)


# ---- the programs ---------------------------------------------------------------------------------------------------

class _Loaded:
    """A program on the GPU: its executable, and the (shape, element type) of its inputs and outputs in binding order."""

    def __init__(self, program, inputs, outputs):
        self.executable = Executable(_device(), program.serialize())
        self.inputs = inputs
        self.outputs = outputs


_loaded = {}
_the_device = []


def _device():
    if not _the_device:
        _the_device.append(Device(0))
    return _the_device[0]


def _load(case):
    key = json.dumps({k: v for k, v in case.items() if k not in ("name", "host")}, sort_keys=True)
    if key not in _loaded:
        kind = case["kind"]
        if kind == "decoder_step":
            _loaded[key] = _decoder_step(case)
        else:
            if kind == "linear_i8":
                w = workloads.fully_connected_workload(case["M"], case["K"], case["N"], realistic=True, seed=WEIGHT_SEED)
            elif kind == "conv_i8":
                w = workloads.conv2d_workload(N=case["batch"], H=case["size"], W=case["size"], C=case["C"], O=case["O"], KH=case["window"],
                                              KW=case["window"], stride=(case["stride"],) * 2, pad=(case["window"] // 2,) * 4, realistic=True,
                                              seed=WEIGHT_SEED)
            elif kind == "image_net":
                w = workloads.mobilenet_v2_workload(batch=case["batch"], resolution=case["resolution"], width=case["width"], seed=WEIGHT_SEED)
            elif kind == "linear_bf16" and case["block"]:
                w = workloads.expand_weights_workload(case["M"], case["K"], case["N"], block=case["block"], seed=WEIGHT_SEED)
            elif kind == "linear_bf16":
                w = workloads.fully_connected_bf16_workload(case["M"], case["K"], case["N"], seed=WEIGHT_SEED)
            elif case["out"] == "int8":
                # requantised to spread over the int8 range: a sum of K products of two uniform int8 values
                w = workloads.matmul_workload(case["B"], case["M"], case["K"], case["N"], out_dtype=np.int8, shift=32, seed=WEIGHT_SEED,
                                              scale=int(40.0 / (5460.0 * math.sqrt(case["K"])) * 2 ** 32))
            else:
                w = workloads.matmul_workload(case["B"], case["M"], case["K"], case["N"], out_dtype=np.dtype(case["out"]).type, seed=WEIGHT_SEED)
            bf16 = kind == "linear_bf16"
            _loaded[key] = _Loaded(w.program, [(a.shape, torch.bfloat16 if bf16 else torch.int8) for a in w.inputs],
                                   [(s, torch.bfloat16 if bf16 else getattr(torch, np.dtype(d).name)) for s, d in w.outputs])
    return _loaded[key]


def _decoder_step(c):
    """One token for each of `batch` sequences through `layers` layers with block-quantized int8 weights and one key / value
    head, and the vocabulary projection: the ops of a decoder that are this backend's (what lies between them, such as the
    softmax, is not, so scores feed the context product directly and the gate is an add).  Bindings: the embedded tokens,
    key caches [position, dim], value caches [dim, position], logits, new keys, new values."""
    B, L, D, T, hidden, qdim = c["batch"], c["layers"], c["head_dim"], c["cache_len"], c["hidden"], c["heads"] * c["head_dim"]
    gen = torch.Generator(device="cuda").manual_seed(WEIGHT_SEED)
    none = dict(output_zp=0, output_min=workloads.NO_CLAMP[0], output_max=workloads.NO_CLAMP[1])
    zero = np.zeros(1, dtype=np.float32)
    whole, half = (workloads.to_bf16(np.array([v, v], dtype=np.float32)) for v in (1.0, 0.70703125))  # residual sums, the gate
    u16 = np.uint16
    branch = 1.0 / math.sqrt(2 * L)  # what a layer adds to the residual stream, as decoders are initialised
    p = Program()
    p.set_name("decoder_step")
    x = p.binding(0, (B, hidden), u16)
    keys, values = p.binding(1, (L * B, T, D), u16), p.binding(2, (L * B, D, T), u16)
    logits = p.binding(3, (B, c["vocab"]), u16)
    new_keys, new_values = p.binding(4, (L, B, D), u16), p.binding(5, (L, B, D), u16)

    def linear(src, K, N, gain=1.0, init=None):
        w = torch.randint(-128, 128, (K, N), dtype=torch.int8, device="cuda", generator=gen).cpu().numpy()
        scale = (torch.rand(K // 128, N, device="cuda", generator=gen) * 0.5 + 0.75) * (gain / (73.9 * math.sqrt(K)))
        scale = scale.to(torch.bfloat16).view(torch.int16).cpu().numpy().view(u16)
        w16 = p.expand_weights(w, scale, np.zeros((K // 128, N), dtype=np.float32), block_size=128, output_min=none["output_min"],
                               output_max=none["output_max"])
        return p.matmul(src, w16, zero, init=p.tensor((B, N), u16) if init is None else init, shift=0, **none)

    for i in range(L):
        q = linear(x, hidden, qdim, gain=1.0 / 512)
        linear(x, hidden, D, init=p.view(new_keys, (B, D), i * B * D))
        linear(x, hidden, D, init=p.view(new_values, (B, D), i * B * D))
        k = p.transpose(p.view(keys, (B, T, D), i * B * T * D), (0, 2, 1))
        v = p.transpose(p.view(values, (B, D, T), i * B * D * T), (0, 2, 1))
        scores = p.matmul(p.view(q, (B, c["heads"], D)), k, zero, shift=0, **none)
        context = p.matmul(scores, v, zero, shift=0, **none)
        h = p.add(x, linear(p.view(context, (B, qdim)), qdim, hidden, gain=branch), whole, zero, shift_factor=0, **none)
        a = p.add(linear(h, hidden, c["ffn"]), linear(h, hidden, c["ffn"]), half, zero, shift_factor=0, **none)
        x = p.add(h, linear(a, c["ffn"], hidden, gain=branch), whole, zero, shift_factor=0, **none)
    linear(x, hidden, c["vocab"], init=logits)
    bf = torch.bfloat16
    return _Loaded(p, [((B, hidden), bf), ((L * B, T, D), bf), ((L * B, D, T), bf)], [((B, c["vocab"]), bf), ((L, B, D), bf), ((L, B, D), bf)])


# ---- a pass ---------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    loaded = _load(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    inputs = []
    for shape, dtype in loaded.inputs:
        if dtype == torch.bfloat16:
            inputs.append(torch.randn(shape, dtype=torch.float32, device="cuda", generator=gen).to(dtype))
        else:
            inputs.append(torch.randint(-128, 128, shape, dtype=dtype, device="cuda", generator=gen))
    if case.get("host"):
        inputs = [t.cpu().numpy() for t in inputs]
        outputs = [np.empty(shape, dtype=str(dtype).replace("torch.", "")) for shape, dtype in loaded.outputs]
        return dict(executable=loaded.executable, arrays=inputs + outputs, outputs=outputs)
    outputs = [torch.empty(shape, dtype=dtype, device="cuda") for shape, dtype in loaded.outputs]
    buffers = inputs + outputs
    return dict(executable=loaded.executable, buffers=buffers, pointers=[t.data_ptr() for t in buffers],
                lengths=[t.numel() * t.element_size() for t in buffers], outputs=outputs)


def run(state):
    if "arrays" in state:
        state["executable"].run_host(state["arrays"])
    else:
        state["executable"].enqueue_device(state["pointers"], state["lengths"])
    return state["outputs"]


def _out_size(size, stride):
    return -(-size // stride)


def work(case):
    kind = case["kind"]
    if kind == "linear_i8":
        M, K, N = case["M"], case["K"], case["N"]
        return dict(bytes=M * K + N * K + 8 * N + M * N, flops=2 * M * K * N)
    if kind == "conv_i8":
        k, out = case["window"], ((case["size"] + 2 * (case["window"] // 2) - case["window"]) // case["stride"] + 1) ** 2 * case["batch"]
        taps = k * k * case["C"]
        return dict(bytes=case["batch"] * case["size"] ** 2 * case["C"] + taps * case["O"] + 8 * case["O"] + out * case["O"], flops=2 * out * taps * case["O"])
    if kind == "linear_bf16":
        M, K, N = case["M"], case["K"], case["N"]
        weights = N * K + 2 * N * K // case["block"] if case["block"] else 2 * N * K
        return dict(bytes=2 * M * K + weights + 4 * N + 2 * M * N, flops=2 * M * K * N)
    if kind == "matmul_i8":
        B, M, K, N = case["B"], case["M"], case["K"], case["N"]
        return dict(bytes=B * (M * K + K * N + M * N * np.dtype(case["out"]).itemsize), flops=2 * B * M * K * N)
    if kind == "decoder_step":
        B, L, D, T, hidden, ffn = case["batch"], case["layers"], case["head_dim"], case["cache_len"], case["hidden"], case["ffn"]
        q = case["heads"] * D
        weights = L * hidden * (q + 2 * D + q + 3 * ffn) + hidden * case["vocab"]
        return dict(bytes=weights + weights // 64 + 4 * L * B * T * D + 2 * B * hidden + 2 * B * case["vocab"] + 4 * L * B * D,
                    flops=2 * B * weights + 4 * L * B * q * T)
    # image_net: the image, the weights and the classes; every layer's products
    size, ch = _out_size(case["resolution"], 2), lambda v: max(8, int(v * case["width"] + 4) // 8 * 8)
    macs, weights, cin = size * size * ch(32) * 27, ch(32) * 27, ch(32)
    for expand, c, n, s in workloads.MBV2_BLOCKS:
        for i in range(n):
            wide, before, size = cin * expand, size, _out_size(size, s if i == 0 else 1)
            macs += (before ** 2 * cin * wide if expand > 1 else 0) + size ** 2 * wide * (9 + ch(c))
            weights += (cin * wide if expand > 1 else 0) + wide * (9 + ch(c))
            cin = ch(c)
    macs += size ** 2 * cin * 1280 + 1280 * 1000
    weights += cin * 1280 + 1280 * 1000
    return dict(bytes=case["batch"] * (3 * case["resolution"] ** 2 + 1000) + weights, flops=2 * case["batch"] * macs)


def tolerance(case):
    if case["kind"] == "linear_bf16":
        return {"rel": 2e-3, "max": 1.6e-2}  # fp32 sums in another order: a result on a rounding boundary moves by one bf16 step
    if case["kind"] == "decoder_step":
        # such steps carried through the layers that follow: two orders of summation are 0.013 apart after 26 layers
        return {"rel": 4e-3 * math.sqrt(case["layers"]), "max": 4e-2 * math.sqrt(case["layers"])}
    return "exact"
