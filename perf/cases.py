"""Performance cases of the compression-before-swap path.

Each case is one pass of what a training program has the library do with an activation
tensor on its way to the host and back: the fixed-rate ZFP codec and the zero-value
compaction (ZVC) in both directions, and the swap engine that puts the selector and the
pinned copies around them.  Activations are fp32; ZFP runs at 4, 8 and 16 bits per value.

``op`` of a case:
  zfp_compress      field -> stream           (``cuda_compress`` into a kept stream buffer)
  zfp_decompress    stream -> field           (``cuda_decompress`` into a kept tensor)
  zfp_round_trip    both, one after the other
  zvc_round_trip    single-call compaction with a kept workspace, then the expansion
  swap_walk         forward: every tensor of a small stack goes out under the selector;
                    backward: they come back last to first, the next one prefetched
"""
import math

import torch

from cswap_amd import api
from cswap_amd._lib import check, lib
from cswap_amd.swap import AUTO, SwapEngine
from cswap_amd.workloads import field_dims

MB = 1 << 20


def listed():
    return [
        # attention probabilities of a transformer layer, batch 32, sequence 512: the largest tensor that is swapped
        zfp("zfp_compress", "attention_compress", "softmax", 8, 32, 12, 512, 512),
        zfp("zfp_decompress", "attention_decompress", "softmax", 8, 32, 12, 512, 512),
        # hidden states of the same model: the ordinary dense activation
        zfp("zfp_compress", "hidden_compress", "gelu", 8, 1, 32, 512, 768),
        zfp("zfp_decompress", "hidden_decompress", "gelu", 8, 1, 32, 512, 768),
        # its feed-forward activation where 8 bits per value cost too much accuracy
        zfp("zfp_round_trip", "ffn_16bit", "gelu", 16, 1, 32, 512, 3072),
        # one convolution layer's output at 32x32
        zfp("zfp_round_trip", "conv32", "prelu", 8, 64, 64, 32, 32),
        # the last, smallest layers of a convolutional stack: a launch and a lone wavefront's work
        zfp("zfp_round_trip", "conv4_4bit", "leaky", 4, 128, 512, 4, 4),
        # odd feature maps: rows that start on no 16-byte boundary and end inside a block
        zfp("zfp_round_trip", "conv35_odd", "leaky", 8, 64, 192, 35, 35),
        # ReLU outputs, half of them zero: an ordinary layer, a large one, and an odd one that
        # no chunk count divides into whole mask words
        zvc("relu16", 50, 128, 256, 16, 16, True),
        zvc("relu64", 50, 256, 64, 64, 64, True),
        zvc("relu35_odd", 60, 64, 192, 35, 35, False),
        # a stack of ReLU and dense layers through the engine, with the selector choosing
        {"name": "swap_stack", "op": "swap_walk", "d0": 64, "d1": 64, "d2": 32, "levels": 4, "zeros": 55},
    ]


def zfp(op, name, values, rate, d0, d1, d2, d3):
    return {"name": name, "op": op, "values": values, "rate": rate, "d0": d0, "d1": d1, "d2": d2, "d3": d3}


def zvc(name, zeros, d0, d1, d2, d3, fixed_chunks):
    # fixed_chunks: the 16384 chunks of the published format, else as many as the library advises for the size
    return {"name": name, "op": "zvc_round_trip", "zeros": zeros, "d0": d0, "d1": d1, "d2": d2, "d3": d3,
            "fixed_chunks": fixed_chunks}


def draw(rng):
    kind = rng.choice(["zfp", "zfp", "zfp", "zvc", "zvc", "swap"])
    if kind == "swap":
        side = rng.choice([8, 14, 16, 28, 32])
        levels = rng.randint(2, 4)
        channels = rng.choice([32, 48, 64, 96])
        batch = batch_for(log_uniform(rng, 2 * MB, 32 * MB), 4 * channels * side * side)
        return {"op": "swap_walk", "d0": batch, "d1": channels, "d2": side, "levels": levels,
                "zeros": rng.randint(40, 80)}
    if kind == "zvc":
        d2 = d3 = rng.choice([4, 7, 8, 14, 16, 17, 28, 32, 35, 56, 64])
        d1 = rng.choice([32, 48, 64, 96, 128, 192, 256, 320, 512])
        d0 = batch_for(log_uniform(rng, 1 * MB, 256 * MB), 4 * d1 * d2 * d3)
        case = zvc("", rng.randint(30, 90), d0, d1, d2, d3, rng.random() < 0.5)
    else:
        op = rng.choice(["zfp_compress", "zfp_decompress", "zfp_round_trip"])
        rate = rng.choice([4, 8, 8, 8, 16])
        size = log_uniform(rng, 1 * MB, 384 * MB if op != "zfp_round_trip" else 192 * MB)
        form = rng.choice(["conv", "conv", "hidden", "attention"])
        if form == "conv":
            d2 = d3 = rng.choice([4, 7, 8, 14, 16, 17, 28, 32, 35, 56, 64])
            d1 = rng.choice([32, 48, 64, 96, 128, 192, 256, 320, 512])
            values = rng.choice(["prelu", "leaky"])
        elif form == "hidden":
            d1, d2, d3 = 1, rng.choice([49, 128, 196, 197, 256, 384, 512]), rng.choice([192, 256, 384, 768, 1024, 3072])
            values = "gelu"
        else:
            d1, d2 = rng.choice([4, 8, 12, 16]), rng.choice([49, 64, 128, 197, 256, 384, 512])
            d3, values = d2, "softmax"
        d0 = batch_for(size, 4 * d1 * d2 * d3)
        case = zfp(op, "", values, rate, d0, d1, d2, d3)
    del case["name"]
    return case


def batch_for(size, sample_bytes):
    return min(512, max(1, int(size / sample_bytes)))


def log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


# ---------------------------------------------------------------- inputs
def shape_of(case):
    return (case["d0"], case["d1"], case["d2"], case["d3"])


def relu_like(shape, zeros_pct, gen):
    """ReLU(N(mu, 1)) with mu set so that the given share of the values is zero."""
    mu = -math.sqrt(2.0) * float(torch.erfinv(torch.tensor(2.0 * zeros_pct / 100.0 - 1.0, dtype=torch.float64)))
    return torch.randn(shape, generator=gen, device="cuda").add_(mu).clamp_(min=0.0)


def activations(shape, values, gen):
    x = torch.randn(shape, generator=gen, device="cuda")
    if values == "softmax":
        return torch.softmax(x, dim=-1)
    if values == "gelu":
        return torch.nn.functional.gelu(x)
    if values == "prelu":
        return torch.nn.functional.leaky_relu_(x, 0.25)
    scale = torch.rand(shape[1], generator=gen, device="cuda").mul_(3.9).add_(0.1)   # one scale per channel
    return torch.nn.functional.leaky_relu_(x, 0.01).mul_(scale[None, :, None, None])


def stack_shapes(case):
    """Each level of the stack has half the rows and columns and twice the channels of the one before."""
    out = []
    for k in range(case["levels"]):
        side = max(2, case["d2"] >> k)
        out.append((case["d0"], case["d1"] << k, side, side))
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["op"] == "swap_walk":
        xs = [relu_like(s, case["zeros"], gen) if k % 2 == 0 else torch.randn(s, generator=gen, device="cuda")
              for k, s in enumerate(stack_shapes(case))]
        total = sum(4 * x.numel() for x in xs)
        engine = SwapEngine(pinned_bytes=total + 16 * MB, device_bytes=2 * total + 16 * MB)
        return {"op": case["op"], "engine": engine, "xs": xs, "outs": [torch.empty_like(x) for x in xs]}
    if case["op"] == "zvc_round_trip":
        x = relu_like(shape_of(case), case["zeros"], gen)
        n = x.numel()
        process = api.PROCESS if case["fixed_chunks"] else lib().cswap_zvc_pick_process(n)
        _, words, active = api.zvc_geometry(n, process)
        return {"op": case["op"], "x": x, "n": n, "process": process, "active": active,
                "workspace": api.zvc_workspace(process),
                "values": torch.zeros(n, dtype=torch.float32, device="cuda"),   # room for the worst case
                "mask": torch.zeros(words * process, dtype=torch.int32, device="cuda"),
                "begin": torch.zeros(process, dtype=torch.int32, device="cuda"),
                "nnz": torch.zeros(1, dtype=torch.int32, device="cuda"),
                "back": torch.empty_like(x)}
    shape = shape_of(case)
    x = activations(shape, case["values"], gen)
    maxbits = 64 * case["rate"]
    state = {"op": case["op"], "shape": shape, "maxbits": maxbits}
    stream = torch.zeros(api.zfp_stream_capacity(*field_dims(shape), maxbits), dtype=torch.uint8, device="cuda")
    if case["op"] == "zfp_decompress":
        api.cuda_compress(x, maxbits, stream)
        state.update(stream=stream, back=x)      # the decoder fills the tensor that the stream was made from
    else:
        state.update(x=x, stream=stream)
        if case["op"] == "zfp_round_trip":
            state["back"] = torch.empty_like(x)
    return state


# ---------------------------------------------------------------- one pass
def run(state):
    op = state["op"]
    if op == "swap_walk":
        return swap_walk(state["engine"], state["xs"], state["outs"])
    if op == "zvc_round_trip":
        check(lib().cswap_zvc_compress_fused(
            state["x"].data_ptr(), state["n"], state["process"], state["workspace"].data_ptr(),
            state["begin"].data_ptr(), state["nnz"].data_ptr(), state["values"].data_ptr(), state["mask"].data_ptr(),
            torch.cuda.current_stream().cuda_stream), "cswap_zvc_compress_fused")
        api.GPUdecompression(state["values"], state["back"], state["mask"], state["begin"], state["process"])
        # begin has one entry per chunk that holds data; the values array is filled up to nnz
        return [state["nnz"], state["begin"][:state["active"]], state["mask"], state["values"], state["back"]]
    out = []
    if op != "zfp_decompress":
        out.append(api.cuda_compress(state["x"], state["maxbits"], state["stream"]))
    if op != "zfp_compress":
        out.append(api.cuda_decompress(state["stream"], state["shape"], state["maxbits"], state["back"]))
    return out


def swap_walk(engine, xs, outs):
    tickets = [engine.pre(x, AUTO) for x in xs]
    for k in reversed(range(len(xs))):
        if k:
            engine.prefetch(tickets[k - 1])
        engine.swap_in(tickets[k], outs[k])
        engine.release(tickets[k])
    return outs


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Bytes in device memory: every input read once, every output written once.  No matrix work."""
    if case["op"] == "swap_walk":
        return {"bytes": 8 * sum(math.prod(s) for s in stack_shapes(case)), "flops": 0}
    shape = shape_of(case)
    n = math.prod(shape)
    if case["op"] == "zvc_round_trip":
        packed = 4.0 * n * (1.0 - case["zeros"] / 100.0) + n / 8.0     # non-zeros and the bit mask
        return {"bytes": 2 * (4 * n + packed), "flops": 0}
    nx, ny, nz = field_dims(shape)
    stream = -(-nx // 4) * -(-ny // 4) * -(-nz // 4) * 8 * case["rate"]
    return {"bytes": (4 * n + stream) * (2 if case["op"] == "zfp_round_trip" else 1), "flops": 0}


def tolerance(case):
    """Streams, masks and offsets are bytes of a fixed format; a decoded value is one integer times a power of
    two, and the compaction moves values unchanged: every correct implementation gives the same bits."""
    return "exact"
