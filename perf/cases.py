"""Performance cases of the simulator's public entry points.

Each case is one call that a user's program makes: a functional product, a converted layer,
a training step of a hardware-aware layer, or a recurrent sequence.  ``listed`` names the
cases that are always measured and ``draw`` gives more of the same ranges; ``prepare`` makes
what the program holds before the call, ``run`` makes the call, and ``exact`` evaluates the
same model with plain torch in 64 bits.

A case's ``arrays`` names the array geometry and slicing, ``noise`` the device effects.
"""

import hashlib
import math

import torch
from torch import nn
from torch.nn import functional as F

import memfast_amd as memfast

DEVICE = torch.device("cuda", 0)
SEED = 135                     # Config.seed, the base of every matrix's sampling seed
HIGH, LOW = 1e-5, 1e-7         # Config's conductances
_BITS2 = (1, 1, 2, 2, 2)       # INT8 in one sign bit, one bit and three 2-bit slices

# Array geometry, slicing and quantization groups.
ARRAYS = {
    # Config(): 64x64 arrays read whole, one bit per cell and pulse, one scale per row/column.
    "default": dict(),
    # The LeNet-5 checkpoint's configuration: INT4 weights on the default arrays.
    "int4": dict(weight_bits=4),
    # Larger arrays read whole (rows_per_read unset), one bit per cell.
    "whole": dict(array_size=(128, 128), adc_bits=8),
    # 128x128 arrays read 32 rows at a time, 2-bit cells, a scale per read.
    "sliced": dict(input_slice=_BITS2, weight_slice=_BITS2, array_size=(128, 128),
                   rows_per_read=32, weight_quant_gran=(32, 1), input_quant_gran=(1, 32),
                   adc_bits=(6, 7, 7, 8, 8)),
    # The same arrays with a scale per row and output channel (README and GRU workloads).
    "rowwise": dict(input_slice=_BITS2, weight_slice=_BITS2, array_size=(128, 128),
                    rows_per_read=32, adc_bits=7),
    # 256x256 arrays read 64 rows at a time, per-channel weight scales (vision models).
    "vision": dict(input_slice=_BITS2, weight_slice=_BITS2, array_size=(256, 256),
                   rows_per_read=64, weight_quant_gran=(None, 1), adc_bits=8),
    # BFP16 activations in nine slices on INT4 weights in three (LLM linears).
    "llm": dict(activation_bits=16, weight_bits=4, input_slice=(1, 1, 2, 2, 2, 2, 2, 2, 2),
                weight_slice=(1, 1, 2), bw_e=8, adc_bits=(6, 6, 7)),
}

# Device effects.
NOISE = {
    "ideal": dict(write_variation=0.0),
    "write": dict(write_variation=0.02),
    "faults": dict(write_variation=0.02, stuck_at_low=0.0005, stuck_at_high=0.0005),
    "read": dict(write_variation=0.02, read_variation=0.01, adc_nonlinearity=0.1),
    "retention": dict(write_variation=0.02, read_variation=0.01, drift_coefficient=0.05,
                      drift_time=100.0),
    "slice_pair": dict(write_variation=0.02, read_variation=0.01, read_mode="slice_pair"),
    "output": dict(write_variation=0.02, read_variation=0.01, read_mode="output"),
    "voltage": dict(write_variation=0.02, voltage_variation=0.01),
}

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def _case(op, arrays, noise, dtype="float32", **sizes):
    return dict(op=op, arrays=arrays, noise=noise, dtype=dtype, **sizes)


def listed():
    return [
        # The README's first product: the smallest call, all latency.
        dict(_case("mm", "sliced", "write", n=4, k=128, o=32), name="readme_mm"),
        # An ordinary product with a default Simulator; no size is a multiple of an array.
        dict(_case("mm", "default", "write", n=1000, k=1500, o=700), name="default_mm"),
        # A converted bfloat16 Linear under the default configuration, a full training batch
        # of tokens.
        dict(_case("linear", "default", "write", "bfloat16", n=2048, k=2048, o=2048),
             name="default_linear"),
        # Ideal devices (a design's digital baseline) on the default arrays, ragged.
        dict(_case("mm", "default", "ideal", n=777, k=1500, o=1111), name="ideal_mm"),
        # The large ideal product of the benchmark.
        dict(_case("mm", "sliced", "ideal", n=4096, k=4096, o=4096), name="ideal_mm_4096"),
        # The benchmark's noisy product: write and read noise, S-curve converters.
        dict(_case("mm", "sliced", "read", n=4096, k=4096, o=4096), name="noisy_mm_4096"),
        # A ResNet-18 stage-1 convolution at batch 64, with calibrated activations.
        dict(_case("conv", "vision", "faults", batch=64, cin=64, cout=64, size=56, kernel=3,
                   stride=1), name="resnet_conv"),
        # Hardware-aware training of a small classifier layer and of an early convolution:
        # reprogram, forward and backward.
        dict(_case("train_linear", "default", "write", n=128, k=784, o=512),
             name="train_linear"),
        dict(_case("train_conv", "int4", "write", batch=32, cin=32, cout=64, size=16, kernel=3,
                   stride=1), name="train_conv"),
        # The speech GRU: 200 steps that depend on each other.
        dict(_case("gru", "rowwise", "write", batch=32, steps=200, k=40, o=512),
             name="gru_sequence"),
        # An LLM's query projection over a 2048-token prompt, then decoding four sequences
        # through its up projection.
        dict(_case("linear", "llm", "retention", n=2048, k=4096, o=4096), name="llm_prefill"),
        dict(_case("linear", "llm", "retention", n=4, k=4096, o=11008), name="llm_decode"),
    ]


# Slice-MACs of the largest listed case (noisy_mm_4096): no drawn case takes more.
_MOST = 4096**3 * 25
# What a slice-MAC costs beside write noise's: a random draw per conversion, real operands.
_FACTOR = {"output": 16, "slice_pair": 2, "voltage": 2}


def _log(rng, low, high):
    """An integer, spread over the logarithm of [low, high]; one in three a multiple of 64."""
    value = round(math.exp(rng.uniform(math.log(low), math.log(high))))
    return max(64, value // 64 * 64) if value > 96 and rng.random() < 1 / 3 else value


def draw(rng):
    """A case of the listed ones' ranges."""
    while True:
        op = rng.choice(("mm", "mm", "mm", "linear", "linear", "linear", "conv", "conv",
                         "train_linear", "train_conv", "gru"))
        noise = rng.choice(("ideal", "write", "write", "faults", "read", "retention",
                            "slice_pair", "output", "voltage"))
        if op in ("mm", "linear"):
            arrays = rng.choice(("default", "int4", "whole", "sliced", "rowwise", "vision", "llm"))
            case = _case(op, arrays, noise, rng.choice(("float32", "float32", "bfloat16")),
                         n=_log(rng, 1, 4096), k=_log(rng, 64, 11008), o=_log(rng, 32, 11008))
        elif op == "train_linear":
            case = _case(op, rng.choice(("default", "int4", "rowwise")),
                         rng.choice(("ideal", "write", "faults")), n=_log(rng, 8, 1024),
                         k=_log(rng, 64, 4096), o=_log(rng, 10, 4096))
        elif op in ("conv", "train_conv"):
            training = op == "train_conv"
            case = _case(op, rng.choice(("default", "int4", "vision")),
                         rng.choice(("ideal", "write", "faults")),
                         batch=_log(rng, 1, 32 if training else 64),
                         cin=rng.choice((1, 3, 16, 32, 64, 128, 256)),
                         cout=rng.choice((6, 16, 64, 128, 256)), size=rng.randint(7, 56),
                         kernel=rng.choice((1, 3, 5)), stride=rng.choice((1, 1, 2)))
        else:
            case = _case(op, rng.choice(("default", "rowwise")), rng.choice(("ideal", "write")),
                         batch=_log(rng, 1, 64), steps=_log(rng, 8, 200), k=_log(rng, 16, 256),
                         o=_log(rng, 32, 768))
        n, k, _ = _extent(case)
        weighted = _slice_macs(case) * _FACTOR.get(case["noise"], 1)
        # The general read of wide codes with output-mode noise is a reference path.
        if case["arrays"] == "llm" and case["noise"] == "output":
            continue
        if weighted <= _MOST and n * k <= 1 << 28:
            return case


# ---------------------------------------------------------------------------
# Geometry of a case
# ---------------------------------------------------------------------------
def _config(case):
    return memfast.Config(seed=SEED, **ARRAYS[case["arrays"]],
                          nonidealities=memfast.Nonidealities(**NOISE[case["noise"]]))


def _spatial(case):
    """Output height (and width) of a square convolution padded to keep its size."""
    return (case["size"] + 2 * (case["kernel"] // 2) - case["kernel"]) // case["stride"] + 1


def _extent(case):
    """(rows, reduction, columns) of the case's product (a GRU's hidden projections)."""
    if case["op"] in ("conv", "train_conv"):
        return (case["batch"] * _spatial(case)**2, case["cin"] * case["kernel"]**2, case["cout"])
    if case["op"] == "gru":
        return case["batch"] * case["steps"], case["o"], 3 * case["o"]
    return case["n"], case["k"], case["o"]


def _layout(widths, bits):
    """(shift, mask, factor) of each slice, least significant first, of a signed code."""
    widths = (1,) * bits if widths is None else widths
    entries, shift = [], 0
    for position, width in enumerate(reversed(widths)):
        factor = -(1 << shift) if position == len(widths) - 1 else 1 << shift
        entries.append((shift, (1 << width) - 1, factor))
        shift += width
    return entries


def _slices(case):
    arrays = ARRAYS[case["arrays"]]
    return (_layout(arrays.get("input_slice"), arrays.get("activation_bits", 8)),
            _layout(arrays.get("weight_slice"), arrays.get("weight_bits", 8)))


def _slice_macs(case):
    """Multiply-adds of the case's reads: with ideal devices an array's counts are those of
    one integer product, with noise every pair of slices is a product of its own."""
    n, k, o = _extent(case)
    inputs, weights = _slices(case)
    pairs = 1 if case["noise"] == "ideal" else len(inputs) * len(weights)
    macs = n * k * o * pairs
    if case["op"] == "gru":
        macs += n * case["k"] * o * pairs
    return macs


def work(case):
    n, k, o = _extent(case)
    size = 2 if case["dtype"] != "float32" else 4
    flops = 2 * _slice_macs(case)
    weights = k * o
    if case["op"] == "gru":
        weights += case["k"] * o
        moved = size * (n * case["k"] + n * case["o"]) + weights
    elif case["op"] in ("conv", "train_conv"):
        moved = size * (case["batch"] * case["cin"] * case["size"]**2 + n * o)
    else:
        moved = size * (n * k + n * o)
    if case["op"].startswith("train"):
        # Master weights in, their gradient out; the incoming and the input's gradient.
        moved = 2 * moved + 2 * size * weights
        flops += 4 * n * k * o
    elif case["op"] == "mm":
        moved += size * weights            # the operand itself, programmed by the call
    elif case["op"] != "gru":
        moved += weights                   # programmed codes (a byte holds up to 8 bits)
    return {"bytes": moved, "flops": flops}


# ---------------------------------------------------------------------------
# What a program holds, and its call
# ---------------------------------------------------------------------------
class _Inputs:
    """Tensors drawn from one seed, in a fixed order."""

    def __init__(self, case, seed):
        self.case = case
        self.generator = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, device=DEVICE, generator=self.generator)

    def uniform(self, bound, *shape):
        return (torch.rand(*shape, device=DEVICE, generator=self.generator) * 2 - 1) * bound

    def activations(self):
        case = self.case
        if case["op"] in ("conv", "train_conv"):
            # Rectified features, as they reach all but a network's first convolution.
            x = self.normal(case["batch"], case["cin"], case["size"], case["size"]).relu()
        elif case["op"] == "gru":
            x = self.normal(case["steps"], case["batch"], case["k"])
        else:
            x = self.normal(case["n"], case["k"])
            if case["arrays"] == "llm":
                # 1% outlier channels of an LLM's hidden states.
                channels = torch.randperm(case["k"], device=DEVICE, generator=self.generator)
                x[:, channels[:max(1, case["k"] // 100)]] *= 20
        return x.to(DTYPES[case["dtype"]])

    def weights(self):
        """(weight, bias) of the case's layer in PyTorch layout, or the product's right
        operand [K, O] and None."""
        case = self.case
        _, k, o = _extent(case)
        dtype = DTYPES[case["dtype"]]
        if case["op"] == "mm":
            return self.normal(k, o).to(dtype), None
        if case["op"] in ("conv", "train_conv"):
            bound = math.sqrt(2 / k)
            weight = self.normal(o, case["cin"], case["kernel"], case["kernel"]) * bound
        elif case["arrays"] == "llm":
            return (self.normal(o, k) * 0.02).to(dtype), None
        else:
            weight = self.uniform(1 / math.sqrt(k), o, k)
        return weight.to(dtype), self.uniform(1 / math.sqrt(k), o).to(dtype)

    def output_gradient(self):
        case = self.case
        if case["op"] == "train_linear":
            return self.normal(case["n"], case["o"])
        side = _spatial(case)
        return self.normal(case["batch"], case["cout"], side, side)


def _filled(module, weight, bias):
    with torch.no_grad():
        module.weight.copy_(weight)
        if bias is not None:
            module.bias.copy_(bias)
    return module


def _source(case, weight, bias):
    dtype = DTYPES[case["dtype"]]
    if case["op"] in ("conv", "train_conv"):
        layer = nn.Conv2d(case["cin"], case["cout"], case["kernel"], case["stride"],
                          case["kernel"] // 2, bias=bias is not None, device=DEVICE, dtype=dtype)
    else:
        layer = nn.Linear(case["k"], case["o"], bias=bias is not None, device=DEVICE, dtype=dtype)
    return _filled(layer, weight, bias)


def _gru_source(case, inputs):
    gru = nn.GRU(case["k"], case["o"], 1, device=DEVICE)
    bound = 1 / math.sqrt(case["o"])
    with torch.no_grad():
        for parameter in gru.parameters():
            parameter.copy_(inputs.uniform(bound, *parameter.shape))
    return gru


def _input_scale(x):
    """A calibrated fixed activation scale: the largest magnitude over the upper code."""
    return float(x.abs().max()) / 127


def prepare(case, seed):
    inputs = _Inputs(case, seed)
    simulator = memfast.Simulator(_config(case), device=DEVICE)
    op = case["op"]
    x = inputs.activations()
    state = dict(op=op, x=x, simulator=simulator)
    if op == "mm":
        state["rhs"], _ = inputs.weights()
    elif op == "gru":
        state["layer"] = memfast.convert_model(_gru_source(case, inputs), simulator)
    else:
        weight, bias = inputs.weights()
        layer = memfast.convert_model(_source(case, weight, bias), simulator,
                                      training=op.startswith("train"))
        if op == "conv":
            for matrix in layer.matrices:
                matrix.set_input_scale(_input_scale(x))
        if op.startswith("train"):
            state["x"] = x.requires_grad_()
            state["grad"] = inputs.output_gradient()
        state["layer"] = layer
    return state


def run(state):
    op, x = state["op"], state["x"]
    if op == "mm":
        return state["simulator"].mm(x, state["rhs"])
    layer = state["layer"]
    if op == "gru":
        outputs, last = layer(x)
        return dict(outputs=outputs, last=last)
    if not op.startswith("train"):
        return layer(x)
    out = layer(x)
    wanted = (x, layer.weight, layer.bias)
    dx, dw, db = torch.autograd.grad(out, wanted, state["grad"])
    return dict(out=out.detach(), dx=dx, dw=dw, db=db)


# ---------------------------------------------------------------------------
# Tolerances: four times what the present kernels differ from ``exact`` by
# ---------------------------------------------------------------------------
def tolerance(case):
    if case["arrays"] == "llm" and case["noise"] != "ideal":
        # As below, where a count of the leading slices is as large as an output: the outlier
        # channels set the scale, and most activations fill the low slices alone.
        return {"rel": 1e-2, "max": 9.9e-1}
    if case["dtype"] == "bfloat16":
        # One rounding to bfloat16 of the output.
        return {"rel": 8e-3, "max": 5e-1 if case["noise"] != "ideal" else 3e-2}
    if case["op"] == "gru":
        # A changed code of one step enters every later one.
        return {"rel": 2e-3, "max": 5e-2}
    if case["noise"] == "ideal":
        # Integer counts: only the order of FP32 sums over the reads.
        return {"rel": 2e-6, "max": 2e-5}
    # Converters round currents; one that lies within its FP32 error of a half count may go
    # either way, which moves its output by one count of its pair of slices.
    return {"rel": 2e-3, "max": 5e-1}


# ---------------------------------------------------------------------------
# The model in 64 bits
# ---------------------------------------------------------------------------
def _mix(x):
    x = ((x ^ (x >> 16)) * 0x7FEB352D) & 0xFFFFFFFF
    x = ((x ^ (x >> 15)) * 0x846CA68B) & 0xFFFFFFFF
    return x ^ (x >> 16)


def _uniform(address, seed, stream):
    """24-bit uniform of (address, seed, stream), rounded to FP32 as the generator defines."""
    key = _mix((seed ^ (stream * 0x9E3779B9)) & 0xFFFFFFFF)
    high = address >> 32
    folded = _mix(high ^ _mix(seed >> 32))
    folded = folded ^ torch.where(high != 0, _mix(high ^ key), torch.zeros_like(high))
    hashed = _mix((address & 0xFFFFFFFF) ^ folded ^ key)
    return (((hashed >> 8).float() + 0.5) / 16777216).double()


def _normal(address, seed, stream):
    radius = torch.sqrt(-2 * torch.log(_uniform(address, seed, stream)))
    return radius * torch.cos(2 * math.pi * _uniform(address, seed, stream + 1))


def _matrix_seed(name):
    return SEED ^ int.from_bytes(hashlib.sha256(name.encode()).digest()[:4], "little")


def _event_seed(seed, event):
    return (seed ^ _mix(event & 0xFFFFFFFF)) | (_mix(event >> 32) << 32)


class _Model:
    """Quantization, currents, converters and restore of one configuration.  Codes and
    scales follow the precision their quantizer is defined in; the rest is in 64 bits."""

    def __init__(self, case):
        arrays = ARRAYS[case["arrays"]]
        self.a_bits = arrays.get("activation_bits", 8)
        self.w_bits = arrays.get("weight_bits", 8)
        self.bw_e = arrays.get("bw_e")
        self.rows, self.cols = arrays.get("array_size", (64, 64))
        self.step = arrays.get("rows_per_read", self.rows)
        self.inputs, self.weights = _slices(case)
        adc = arrays.get("adc_bits", 6)
        adc = (adc,) * len(self.weights) if isinstance(adc, int) else tuple(reversed(adc))
        self.peaks = [(1 << bits) - 1 for bits in adc]
        self.x_groups = arrays.get("input_quant_gran", (1, None))
        self.w_groups = arrays.get("weight_quant_gran", (None, 1))
        self.noise = NOISE[case["noise"]]

    def quantize(self, value, bits, groups):
        """(codes int64, scale) of ``value`` per rectangular group, both of its shape."""
        dtype = torch.float64 if bits > 8 or self.bw_e is not None else torch.float32
        rows, cols = value.shape
        gr, gc = (min(g, size) if g else size for g, size in zip(groups, value.shape))
        nr, nc = -(-rows // gr), -(-cols // gc)
        blocks = F.pad(value.to(dtype), (0, nc * gc - cols, 0, nr * gr - rows))
        blocks = blocks.reshape(nr, gr, nc, gc)
        # FP32 quotients as FP64 ones rounded once more, which gives the IEEE result.
        blocks = blocks.double()
        peak = blocks.abs().amax((1, 3), keepdim=True)
        upper = (1 << (bits - 1)) - 1
        lower = -upper
        if self.bw_e is None:
            scale = (torch.where(peak > 0, peak, torch.ones_like(peak)) / upper).to(dtype).double()
        else:
            limit = (1 << (self.bw_e - 1)) - 1
            exponent = torch.frexp(peak.clamp_min(torch.finfo(dtype).tiny))[1].double() - 1
            scale = torch.pow(2.0, exponent.clamp(1 - limit, limit) + 2 - bits)
            lower = -upper - 1
        codes = (blocks / scale).to(dtype).round().clamp(lower, upper).long()
        shape = (nr * gr, nc * gc)
        return (codes.reshape(shape)[:rows, :cols],
                scale.expand(blocks.shape).reshape(shape)[:rows, :cols])

    def levels(self, codes, seed, event, c0, c1, p):
        """Conductances [W, kp, c1 - c0] of programmed codes, their cell addresses and the
        read's seed."""
        kp = codes.shape[0]
        row = torch.arange(kp, device=DEVICE)[None, :, None]
        col = torch.arange(c0, c1, device=DEVICE)[None, None, :]
        w = torch.arange(len(self.weights), device=DEVICE)[:, None, None]
        array, tile = row // self.rows, col // self.cols
        cell = (((array * p + tile) * len(self.weights) + w) * self.rows
                + row % self.rows) * self.cols + col % self.cols
        # Nominal levels are the FP32 values that a cell is programmed to.
        table = torch.stack([
            LOW + (HIGH - LOW) * ((codes[:, c0:c1] >> shift) & mask).double() / mask
            for shift, mask, _ in self.weights]).float().double()
        noise = self.noise
        if noise["write_variation"]:
            table = table * torch.exp(noise["write_variation"] * _normal(cell, seed, 10))
        if noise.get("drift_coefficient"):
            table = table * (1 + noise["drift_time"])**-noise["drift_coefficient"]
        low, high = noise.get("stuck_at_low", 0.0), noise.get("stuck_at_high", 0.0)
        if low + high:
            u = _uniform(cell, seed, 30)
            table = torch.where(u < low, LOW, torch.where(u < low + high, HIGH, table))
        read_seed = _event_seed(seed, event)
        if noise.get("read_variation") and noise.get("read_mode", "shared") == "shared":
            table = table * torch.exp(noise["read_variation"] * _normal(cell, read_seed, 20))
        return table, cell, read_seed

    def product(self, qx, sx, qw, sw, name, event=0):
        """Restored outputs [N, O] in FP64 of codes and scales qx, sx [N, K], qw, sw [K, O]."""
        (n, k), o = qx.shape, qw.shape[1]
        m, p = -(-k // self.rows), -(-o // self.cols)
        kp, reads = m * self.rows, m * self.rows // self.step
        starts = (torch.arange(reads, device=DEVICE) * self.step).clamp_max(k - 1)
        xs, ws = sx[:, starts].double().T, sw[starts].double()
        qx = F.pad(qx & ((1 << self.a_bits) - 1), (0, kp - k))
        qw = F.pad(qw & ((1 << self.w_bits) - 1), (0, 0, 0, kp - k))
        noise, seed = self.noise, _matrix_seed(name)
        sigma, mode = noise.get("read_variation", 0.0), noise.get("read_mode", "shared")
        out = torch.empty((n, o), dtype=torch.float64, device=DEVICE)
        width = max(1, min(o, (1 << 26) // (kp * len(self.weights))))
        for c0 in range(0, o, width):
            c1 = min(o, c0 + width)
            table, cell, read_seed = self.levels(qw, seed, event, c0, c1, p)
            height = max(1, (1 << 26) // (reads * (c1 - c0)))
            for n0 in range(0, n, height):
                n1 = min(n, n0 + height)
                out[n0:n1, c0:c1] = self._block(qx, xs, ws, table, cell, read_seed, sigma, mode,
                                                (n0, n1, c0, c1), (m, p, reads))
        return out

    def _block(self, qx, xs, ws, table, cell, read_seed, sigma, mode, block, shape):
        n0, n1, c0, c1 = block
        m, p, reads = shape
        kp = qx.shape[1]
        A, W = len(self.inputs), len(self.weights)
        row = torch.arange(kp, device=DEVICE)[None, :]
        vector = torch.arange(n0, n1, device=DEVICE)[:, None]
        totals = torch.zeros((reads, n1 - n0, c1 - c0), dtype=torch.float64, device=DEVICE)
        for a, (shift, mask, fa) in enumerate(self.inputs):
            digits = ((qx[n0:n1] >> shift) & mask).double()
            if self.noise.get("voltage_variation"):
                address = ((vector * m + row // self.rows) * A + a) * self.rows + row % self.rows
                digits = digits * (1 + self.noise["voltage_variation"]
                                   * _normal(address, read_seed, 40))
            left = digits.reshape(n1 - n0, reads, self.step).transpose(0, 1).contiguous()
            for w, (_, wmask, fw) in enumerate(self.weights):
                g, per_count = table[w], wmask / (HIGH - LOW)
                if sigma and mode == "slice_pair":
                    g = g * torch.exp(sigma * _normal(cell[w] * A + a, read_seed, 20))
                right = g.reshape(reads, self.step, c1 - c0)
                count = left @ ((right - LOW) * per_count)
                if sigma and mode == "output":
                    count += self._output_noise(left, right * per_count, read_seed, sigma, a, w,
                                                block, shape)
                alpha = self.noise.get("adc_nonlinearity", 0.0) / self.peaks[w]
                if alpha:
                    count = count / (1 + (alpha * count).abs())
                totals += count.clamp_(0, self.peaks[w]).round_() * (fa * fw)
        return torch.einsum("gnc,gn,gc->nc", totals, xs[:, n0:n1], ws[:, c0:c1])

    def _output_noise(self, left, right, read_seed, sigma, a, w, block, shape):
        n0, n1, c0, c1 = block
        m, p, reads = shape
        vector = torch.arange(n0, n1, device=DEVICE)[None, :, None]
        read = torch.arange(reads, device=DEVICE)[:, None, None]
        col = torch.arange(c0, c1, device=DEVICE)[None, None, :]
        address = ((((vector * reads + read) * p + col // self.cols) * len(self.inputs) + a)
                   * len(self.weights) + w) * self.cols + col % self.cols
        mean = (left @ right) * math.expm1(0.5 * sigma**2)
        variance = (left.square() @ right.square()) * math.exp(sigma**2) * math.expm1(sigma**2)
        return mean + variance.sqrt() * _normal(address, read_seed, 60)

    def layer(self, x, weight, name, scale=None, event=0):
        """FP64 ``x @ weight.T`` read through the arrays, and both operands' quantized values."""
        qw, sw = self.quantize(weight.T, self.w_bits, self.w_groups)
        if scale is None:
            qx, sx = self.quantize(x, self.a_bits, self.x_groups)
        else:
            sx = torch.full_like(x, scale, dtype=torch.float32)
            qx = (x.double() / sx.double()).float().round().clamp(-127, 127).long()
        out = self.product(qx, sx, qw, sw, name, event)
        return out, qx * sx.double(), qw * sw.double()


def _exact_gru(case, model, x, gru):
    """PyTorch's GRU equations over the two projections' reads; both matrices are read once a
    step, and the state is held in FP32 between steps."""
    steps, batch, _ = x.shape
    names = [f"gru.layer0.direction0.{role}" for role in ("input", "hidden")]
    projected, _, _ = model.layer(x.reshape(steps * batch, -1), gru.weight_ih_l0, names[0])
    projected = (projected + gru.bias_ih_l0.double()).reshape(steps, batch, -1)
    qw, sw = model.quantize(gru.weight_hh_l0.T, model.w_bits, model.w_groups)
    h = torch.zeros((batch, case["o"]), device=DEVICE)
    outputs = []
    for t in range(steps):
        qx, sx = model.quantize(h, model.a_bits, model.x_groups)
        hidden = model.product(qx, sx, qw, sw, names[1], t) + gru.bias_hh_l0.double()
        ir, iz, ic = projected[t].chunk(3, -1)
        hr, hz, hc = hidden.chunk(3, -1)
        update = torch.sigmoid(iz + hz)
        candidate = torch.tanh(ic + torch.sigmoid(ir + hr) * hc)
        state = (1 - update) * candidate + update * h.double()
        outputs.append(state)
        h = state.float()
    return dict(outputs=torch.stack(outputs), last=outputs[-1][None])


@torch.no_grad()
def exact(case, seed):
    inputs, model, op = _Inputs(case, seed), _Model(case), case["op"]
    x = inputs.activations()
    if op == "gru":
        # Sampling the conductances again every step takes long for the larger ones.
        if case["steps"] * case["o"]**2 * len(model.weights) > 1 << 29:
            return None
        return _exact_gru(case, model, x, _gru_source(case, inputs))
    weight, bias = inputs.weights()
    if op == "mm":
        return model.layer(x, weight.T, "matrix.0")[0]
    if op in ("linear", "train_linear"):
        rows, flat = x, weight
    else:
        kernel, pad, stride = case["kernel"], case["kernel"] // 2, case["stride"]
        patches = F.unfold(x, kernel, 1, pad, stride)
        rows, flat = patches.transpose(1, 2).reshape(-1, patches.shape[1]), weight.flatten(1)
    name = "linear" if op in ("linear", "train_linear") else "conv.group0"
    scale = _input_scale(x) if op == "conv" else None
    out, xq, wq = model.layer(rows, flat, name, scale)
    if bias is not None:
        out = out + bias.double()
    side = None if op in ("linear", "train_linear") else _spatial(case)

    def image(value):
        return value.reshape(case["batch"], side * side, -1).transpose(1, 2).reshape(
            case["batch"], -1, side, side)

    if not op.startswith("train"):
        return out if side is None else image(out)
    grad = inputs.output_gradient().double()
    if side is None:
        return dict(out=out, dx=grad @ wq.T, dw=grad.T @ xq, db=grad.sum(0))
    rows_grad = grad.flatten(2).transpose(1, 2).reshape(-1, case["cout"])
    dpatches = (rows_grad @ wq.T).reshape(case["batch"], side * side, -1).transpose(1, 2)
    dx = F.fold(dpatches.contiguous(), (case["size"], case["size"]), kernel, 1, pad, stride)
    return dict(out=image(out), dx=dx, dw=(rows_grad.T @ xq).reshape(weight.shape),
                db=rows_grad.sum(0))
