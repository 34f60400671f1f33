"""The work that users of this package have it do, for timing and for comparing results.

Five kinds of case, each through the public entry points:

* ``gemm``    -- ``quadmul.gemm``: packed int4 x packed int4 -> int32, the drop-in entry point.
* ``linear``  -- ``quadmul_amd.linear.W4A4Linear``: quantise + pack the activations, the GEMM with the scaled 16-bit
  float output, the bias.
* ``mlp``     -- two such layers around a gated activation, captured into a HIP graph and replayed: the
  feed-forward half of a decode step as a serving loop runs it.
* ``quantize`` -- ``quadmul_amd.quantize_pack``: per-row quantisation + packing of float activations or weights.
* ``pack``    -- ``quadmul_amd.pack_int4`` and ``unpack_int4`` on the GPU: int4 values to bytes and back.

Sizes are those of the repository's benchmark and tests: the square and ragged workloads, the
(N, K) pairs of its per-shape table, decode batches of 1 to 64 rows, prefills of 512 to 2048.
"""
import math

import torch

import quadmul
import quadmul_amd
from quadmul_amd.linear import W4A4Linear

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}

# (N, K) of the weight matrices in the repository's shape table and benchmark
WEIGHTS = ((4096, 4096), (11008, 4096), (4096, 11008), (12288, 4096), (8192, 8192), (10240, 8192), (28672, 4096), (6144, 4096),
           (4096, 14336), (8192, 28672))


def listed():
    return [
        # one token through three projections (query, key, value): the smallest calls there are, 8 MiB of weights each
        {"name": "gemm_decode_1_qkv", "kind": "gemm", "m": 1, "n": 4096, "k": 4096, "calls": 3},
        # a batch of sixteen sequences against the longest K of the table: weights from HBM
        {"name": "gemm_decode_16_long_k", "kind": "gemm", "m": 16, "n": 8192, "k": 28672, "calls": 1},
        # an odd number of rows, between the decode and the prefill kernels
        {"name": "gemm_batch_37", "kind": "gemm", "m": 37, "n": 11008, "k": 4096, "calls": 1},
        # a short prefill, a few hundred rows
        {"name": "gemm_prefill_512", "kind": "gemm", "m": 512, "n": 8192, "k": 8192, "calls": 1},
        # the ordinary large product
        {"name": "gemm_square_4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "calls": 1},
        # the largest
        {"name": "gemm_square_8192", "kind": "gemm", "m": 8192, "n": 8192, "k": 8192, "calls": 1},
        # nothing is a multiple of anything: odd M and N, a K that is no multiple of 32
        {"name": "gemm_odd", "kind": "gemm", "m": 1531, "n": 3307, "k": 4100, "calls": 1},
        # one token through one layer, called eagerly: latency and launches count
        {"name": "linear_decode_1", "kind": "linear", "m": 1, "n": 4096, "k": 4096, "dtype": "float16", "bias": False},
        # a prefill of 2048 tokens through the wide projection of an MLP
        {"name": "linear_prefill_2048", "kind": "linear", "m": 2048, "n": 11008, "k": 4096, "dtype": "bfloat16", "bias": True},
        # eight sequences through a feed-forward block, one graph replay
        {"name": "mlp_decode_8_graph", "kind": "mlp", "m": 8, "n": 11008, "k": 4096, "dtype": "float16"},
        # the activations of a prefill, quantised by themselves
        {"name": "quantize_2048", "kind": "quantize", "m": 2048, "k": 8192, "dtype": "bfloat16"},
        # a weight matrix of int4 values packed, and unpacked again to look at it
        {"name": "pack_unpack_8192", "kind": "pack", "m": 8192, "k": 8192},
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("gemm", "linear", "mlp", "quantize", "pack"), weights=(5, 3, 1, 1.5, 1.5))[0]
    dtype = rng.choice(("float16", "bfloat16"))
    if kind in ("gemm", "linear"):
        style = rng.random()
        if style < 0.5:        # a weight of the table, any number of rows
            n, k = rng.choice(WEIGHTS)
        elif style < 0.8:      # any multiples of 32
            n, k = 32 * _log_between(rng, 16, 384), 32 * _log_between(rng, 8, 384)
        else:                  # any N, any even K
            n, k = _log_between(rng, 300, 9000), 2 * _log_between(rng, 150, 4500)
        most = min(8192, int(0.9 * 8192 ** 3 / (n * k)))  # no more work than the largest listed
        m = _log_between(rng, 1, most)
        if kind == "gemm":
            small = n * k < 24e6 and m * n * k < 1e9  # several small calls make one pass
            return {"kind": kind, "m": m, "n": n, "k": k, "calls": 3 if small else 1}
        return {"kind": kind, "m": m, "n": n, "k": k, "dtype": dtype, "bias": rng.random() < 0.5}
    if kind == "mlp":
        n, k = rng.choice(((11008, 4096), (14336, 4096), (28672, 8192)))
        return {"kind": kind, "m": rng.randint(1, 64), "n": n, "k": k, "dtype": "float16"}
    if kind == "quantize":
        return {"kind": kind, "m": _log_between(rng, 1, 8192), "k": 2 * _log_between(rng, 512, 7168), "dtype": rng.choice(("float16", "bfloat16", "float32"))}
    return {"kind": kind, "m": _log_between(rng, 64, 16384), "k": 2 * _log_between(rng, 512, 7168)}


def _packed(gen, rows, k):
    """Uniform int4 values, two to a byte: the repository's own test data."""
    return torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device="cuda", generator=gen).view(torch.int8)


def _activations(gen, rows, k, dtype):
    """Normal values with a few large channels, as the hidden states of a transformer have."""
    x = torch.randn(rows, k, device="cuda", generator=gen)
    loud = torch.randint(0, k, (max(1, k // 512),), device="cuda", generator=gen)
    x[:, loud] *= 6.0
    return x.to(dtype)


def _layer(gen, n, k, dtype, bias):
    weight = torch.randn(n, k, device="cuda", generator=gen) * (1.0 / math.sqrt(k))
    b = torch.randn(n, device="cuda", generator=gen) * 0.1 if bias else None
    return W4A4Linear.from_float(weight.to(dtype), b, out_dtype=dtype)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, m, k = case["kind"], case["m"], case["k"]
    if kind == "gemm":
        n = case["n"]
        weights = [(_packed(gen, n, k), torch.empty(m, n, dtype=torch.int32, device="cuda")) for _ in range(case["calls"])]
        return {"kind": kind, "a": _packed(gen, m, k), "weights": weights, "m": m, "n": n, "k": k}
    if kind == "pack":
        return {"kind": kind, "values": torch.randint(-8, 8, (m, k), dtype=torch.int8, device="cuda", generator=gen)}
    dtype = DTYPES[case["dtype"]]
    x = _activations(gen, m, k, dtype)
    if kind == "quantize":
        return {"kind": kind, "x": x}
    if kind == "linear":
        return {"kind": kind, "x": x, "layer": _layer(gen, case["n"], k, dtype, case["bias"])}

    # the feed-forward block: gate and up projections in one matrix, silu(gate) * up, down projection
    wide, down = _layer(gen, 2 * case["n"], k, dtype, False), _layer(gen, k, case["n"], dtype, False)

    def block(h):
        gate, up = wide(h).chunk(2, dim=-1)
        return down(torch.nn.functional.silu(gate) * up)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        block(x)  # the first call of every kernel, outside the capture
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = block(x)
    return {"kind": kind, "x": x, "y": y, "graph": graph, "wide": wide, "down": down}


def run(state):
    kind = state["kind"]
    if kind == "gemm":
        for b, c in state["weights"]:
            quadmul.gemm(state["a"], b, c, state["m"], state["n"], state["k"])
        return [c for _, c in state["weights"]]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "mlp":
        state["graph"].replay()
        return state["y"]
    if kind == "quantize":
        return quadmul_amd.quantize_pack(state["x"])
    packed = quadmul_amd.pack_int4(state["values"])
    return packed, quadmul_amd.unpack_int4(packed)


def _nibbles(packed):
    """Bytes of int4 pairs -> their values in float64, even k from the low nibble."""
    u = packed.view(torch.uint8).to(torch.int16)
    both = torch.stack((u & 15, u >> 4), dim=-1).reshape(u.shape[0], -1)
    return torch.where(both > 7, both - 16, both).double()


def _bytes(values):
    v = values.to(torch.int16) & 15
    return (v[:, 0::2] | (v[:, 1::2] << 4)).to(torch.uint8).view(torch.int8)


def _rows_to_int4(x):
    """The rule of the quantisation: amax / 7 per row, the multiplication with its inverse in 32 bits where x has no more
    (so the integers are the rule's own, ties too), round to even.  Integers and scales in float64."""
    wide = x if x.dtype == torch.float64 else x.float()
    amax = wide.abs().amax(dim=1, keepdim=True)
    inv = torch.where(amax > 0, 7.0 / amax, torch.zeros_like(amax))
    return torch.round(wide * inv).clamp(-7, 7).double(), amax.double() / 7.0


def _linear64(x, weight, bias=None):
    (xq, xs), (wq, ws) = _rows_to_int4(x), _rows_to_int4(weight)
    y = (xq @ wq.T) * xs * ws.T
    return y if bias is None else y + bias.double()


def exact(case, seed):
    """What ``run`` returns, in 64 bits from the same inputs, with plain torch."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, m, k = case["kind"], case["m"], case["k"]
    if kind == "gemm":
        weights = [_packed(gen, case["n"], k) for _ in range(case["calls"])]
        a = _nibbles(_packed(gen, m, k))
        return [a @ _nibbles(b).T for b in weights]  # below 2^53: the integers themselves
    if kind == "pack":
        values = torch.randint(-8, 8, (m, k), dtype=torch.int8, device="cuda", generator=gen)
        return _bytes(values), values
    dtype = DTYPES[case["dtype"]]
    x = _activations(gen, m, k, dtype)
    if kind == "quantize":
        q, scales = _rows_to_int4(x)
        return _bytes(q), scales[:, 0]

    def drawn(n, k, bias):  # as _layer draws them
        weight = torch.randn(n, k, device="cuda", generator=gen) * (1.0 / math.sqrt(k))
        b = torch.randn(n, device="cuda", generator=gen) * 0.1 if bias else None
        return weight.to(dtype), b if b is None else b.to(dtype)

    if kind == "linear":
        return _linear64(x, *drawn(case["n"], k, case["bias"]))
    wide, down = drawn(2 * case["n"], k, False)[0], drawn(k, case["n"], False)[0]
    gate, up = _linear64(x, wide).chunk(2, dim=-1)
    return _linear64(torch.nn.functional.silu(gate) * up, down)


def work(case):
    kind, m, k = case["kind"], case["m"], case["k"]
    if kind == "gemm":
        n, calls = case["n"], case["calls"]
        return {"bytes": m * k / 2 + calls * (n * k / 2 + 4 * m * n), "flops": calls * 2 * m * n * k}
    if kind == "pack":
        return {"bytes": 3 * m * k, "flops": 0}  # values in; bytes out and in; values out (the bytes are in reach of the caches)
    esz = 4 if case["dtype"] == "float32" else 2
    if kind == "quantize":
        return {"bytes": m * k * (esz + 0.5) + 4 * m, "flops": 3 * m * k}
    n = case["n"]
    if kind == "linear":
        return {"bytes": m * k * esz + n * k / 2 + 4 * n + (esz * n if case["bias"] else 0) + m * n * esz, "flops": 2 * m * n * k}
    return {"bytes": 2 * m * k * esz + 3 * n * k / 2 + 4 * (2 * n + k), "flops": 6 * m * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gemm", "pack"):
        return "exact"
    if kind == "quantize":
        # against the same quantisation in 64 bits: scales 5e-8, and 4e-5 of the bytes on the other side of a tie
        return {"rel": 1e-6, "max": 1e-5, "differ": 2e-4}
    if kind == "linear":
        # the roundings to the 16-bit output, against the same integers scaled in 64 bits: 3e-4 / 2.4e-3, largest 1e-3 / 8e-3
        return {"rel": 1.2e-3, "max": 4e-3} if case["dtype"] == "float16" else {"rel": 1e-2, "max": 3.2e-2}
    # two layers: a rounding of the hidden state moves values of the second quantisation to the other side of a tie
    # (2e-2, largest 0.13, against the whole block in 64 bits)
    return {"rel": 0.03, "max": 0.5}
