"""What a program does with this library, as cases that can be timed and compared.

Kinds (`case["kind"]`), all through the public functions of `qgemm_amd`:

  linear   a quantised linear layer as a server or a training forward pass runs it: the activations arrive in bf16, are
           quantised by `quantize`, and meet weights that were quantised when the model was loaded.  Block scales
           (1 x 128 for activations, 128 x 128 for weights; fp8 or int8) or one scale per matrix (fp8 or int8)
  walk     a decoder's step over its layers: the same with every layer's own weights, captured once as a graph and
           replayed, as servers do; the weights of all layers together do not fit the caches
  product  one product of operands that are quantised already, one scale per matrix (fp8 -> bf16, int8 -> fp32 / int32)
  mm       the block-scaled product on column-major operands (`fp8_mm`)
  plain    the 16-bit product on B stored N x K or K x N
  train    forward and backward of a bf16 linear layer: y = x W^T, dx = dy W, dW = dy^T x in fp32
  encode   quantisation by itself: weights on their way into the library, or activations of a large batch

Sizes are those of the benchmark and the tests, and what lies between and beside them: `draw` takes row counts from one
token to a large prefill, and widths that are multiples of 128 half of the time, otherwise of 8 or of nothing."""
import math

import torch

import qgemm_amd as Q

FP8, I8 = torch.float8_e4m3fn, torch.int8
BLOCK, MATRIX = "block", "matrix"


def listed():
    return [
        # one token of one request through one layer: latency, launches and host work are all there is
        dict(name="one_token_fp8_block", kind="linear", type="fp8", scales=BLOCK, M=1, N=2048, K=1024),
        # sixteen requests, one token each, through 24 layers' weights (352 MB: out of memory every step)
        dict(name="decode_walk_fp8_block", kind="walk", type="fp8", scales=BLOCK, M=16, N=7168, K=2048, layers=24),
        # a small launch-bound 16-bit product
        dict(name="plain_fp16_1024", kind="plain", type="fp16", layout="nk", M=1024, N=1024, K=1024),
        # a mixed batch of prompts: row count and widths as they come, the last K block partial
        dict(name="batch_fp8_block", kind="linear", type="fp8", scales=BLOCK, M=500, N=4608, K=7200),
        # a long prompt through a wide layer, block scales
        dict(name="prefill_fp8_block", kind="linear", type="fp8", scales=BLOCK, M=6144, N=4608, K=7168),
        # the largest product, operands quantised beforehand
        dict(name="product_fp8_8192", kind="product", type="fp8", out="bf16", M=8192, N=8192, K=8192),
        dict(name="product_int8_4096", kind="product", type="int8", out="f32", M=4096, N=4096, K=4096),
        # int8 with one scale per matrix on sizes that are multiples of nothing large
        dict(name="linear_int8_ragged", kind="linear", type="int8", scales=MATRIX, M=1531, N=4100, K=3004),
        # column-major operands, mid-size, rows not a multiple of the tiles
        dict(name="fp8_mm_column_major", kind="mm", M=2080, N=4096, K=4096),
        # a training step's linear layer, whole sizes and ragged ones (the token count is a contraction length in dW)
        dict(name="train_bf16", kind="train", M=4096, N=4096, K=2048),
        dict(name="train_bf16_ragged", kind="train", M=1999, N=3001, K=1000),
        # weights on their way into the library
        dict(name="encode_weights", kind="encode", type="fp8", source="f32", mode="128x128", rows=7168, cols=6144),
    ]


# ---------------------------------------------------------------------------------------------------------------------
# more cases of the same ranges
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, odd=True):
    """A layer's width: a multiple of 128 half of the time, else of 16, 8 or, where `odd`, of nothing."""
    unit = rng.choice([128, 128, 128, 128, 16, 8, 1, 1] if odd else [128, 128, 32])
    return max(unit, _log_int(rng, lo, hi) // unit * unit)


def _at_most(case, flops):
    """The case with its rows cut until its product costs no more than `flops`."""
    unit = 32 if case["kind"] == "mm" else 1
    while 2.0 * case["M"] * case["N"] * case["K"] > flops and case["M"] > unit:
        case["M"] = max(unit, case["M"] // 2 // unit * unit)
    return case


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "walk", "product", "mm", "plain", "train", "encode"])
    if kind == "linear":
        return _at_most(dict(kind=kind, type=rng.choice(["fp8", "fp8", "int8"]), scales=rng.choice([BLOCK, BLOCK, MATRIX]),
                             M=_log_int(rng, 1, 8192), N=_width(rng, 512, 14336), K=_width(rng, 512, 8192)), 4.1e11)
    if kind == "walk":
        return dict(kind=kind, type=rng.choice(["fp8", "int8"]), scales=BLOCK, M=_log_int(rng, 1, 128),
                    N=_width(rng, 1024, 8192, odd=False), K=_width(rng, 1024, 4096, odd=False), layers=rng.choice([12, 16, 20]))
    if kind == "product":
        t = rng.choice(["fp8", "int8"])
        return dict(kind=kind, type=t, out=rng.choice(["bf16", "f32", "i32"]) if t == "int8" else "bf16",
                    M=_log_int(rng, 16, 8192), N=_width(rng, 1024, 8192), K=_width(rng, 512, 8192))
    if kind == "mm":        # the entry takes multiples of 32
        return _at_most(dict(kind=kind, M=max(32, _log_int(rng, 32, 8192) // 32 * 32), N=_width(rng, 512, 8192, odd=False),
                             K=_width(rng, 512, 8192, odd=False)), 4.1e11)
    if kind == "plain":
        return _at_most(dict(kind=kind, type=rng.choice(["fp16", "bf16"]), layout=rng.choice(["nk", "kn"]), M=_log_int(rng, 16, 4096),
                             N=_width(rng, 512, 8192), K=_width(rng, 512, 8192)), 1.4e11)
    if kind == "train":
        return _at_most(dict(kind=kind, M=_log_int(rng, 256, 4096), N=_width(rng, 512, 4096), K=_width(rng, 512, 4096)), 6.8e10)
    return dict(kind="encode", type=rng.choice(["fp8", "fp8", "int8"]), source=rng.choice(["f32", "bf16", "bf16", "fp16"]),
                mode=rng.choice(["1x128", "128x128", "matrix"]), rows=_log_int(rng, 16, 6144), cols=_width(rng, 512, 7168))


# ---------------------------------------------------------------------------------------------------------------------
_TYPES = {"fp8": FP8, "int8": I8, "fp16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "i32": torch.int32}
_MODES = {"1x128": Q.QUANT_BLOCK_1x128, "128x128": Q.QUANT_BLOCK_128x128, "matrix": Q.QUANT_PER_MATRIX}


def _activations(g, rows, cols):
    """Normally distributed, with channels of different size, as layers see them."""
    x = torch.randn(rows, cols, generator=g, device="cuda")
    return x.mul_(torch.exp(0.5 * torch.randn(cols, generator=g, device="cuda")))


def _weights(g, n, k):
    return torch.randn(n, k, generator=g, device="cuda").mul_(k ** -0.5)


def _column_major(t):
    """The same matrix, its columns contiguous."""
    return t.view(torch.uint8).t().contiguous().t().view(t.dtype) if t.element_size() == 1 else t.t().contiguous().t()


def _linear_state(case, g):
    block = case["scales"] == BLOCK
    w, ws = Q.quantize(_weights(g, case["N"], case["K"]), _TYPES[case["type"]], Q.QUANT_BLOCK_128x128 if block else Q.QUANT_PER_MATRIX)
    return dict(x=_activations(g, case["M"], case["K"]).bfloat16(), w=w, ws=ws, type=_TYPES[case["type"]],
                quant=Q.QUANT_BLOCK_1x128 if block else Q.QUANT_PER_MATRIX, scale=Q.SCALE_BLOCK128 if block else Q.SCALE_PER_MATRIX,
                y=torch.empty(case["M"], case["N"], dtype=torch.bfloat16, device="cuda"), sizes=(case["M"], case["N"], case["K"]))


def _linear(s):
    q, qs = Q.quantize(s["x"], s["type"], s["quant"])
    return Q.scaled_gemm(q, s["w"], qs, s["ws"], s["y"], *s["sizes"], s["scale"])


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind, empty = case["kind"], lambda *shape, dtype=torch.bfloat16: torch.empty(*shape, dtype=dtype, device="cuda")
    if kind == "linear":
        return dict(kind=kind, **_linear_state(case, g))
    if kind == "walk":
        layers = [_linear_state(case, g) for _ in range(case["layers"])]
        for s in layers:            # (once outside the capture: it may not allocate the library's workspace)
            _linear(s)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for s in layers:
                _linear(s)
        return dict(kind=kind, layers=layers, graph=graph)
    if kind == "encode":
        x = _activations(g, case["rows"], case["cols"]).to(_TYPES[case["source"]])
        return dict(kind=kind, x=x, type=_TYPES[case["type"]], mode=_MODES[case["mode"]])
    M, N, K = case["M"], case["N"], case["K"]
    if kind == "product":
        a, sa = Q.quantize(_activations(g, M, K), _TYPES[case["type"]])
        b, sb = Q.quantize(_weights(g, N, K), _TYPES[case["type"]])
        return dict(kind=kind, a=a, b=b, sa=sa, sb=sb, c=empty(M, N, dtype=_TYPES[case["out"]]), sizes=(M, N, K))
    if kind == "mm":
        a, sa = Q.quantize(_activations(g, M, K), FP8, Q.QUANT_BLOCK_1x128)
        b, sb = Q.quantize(_weights(g, N, K), FP8, Q.QUANT_BLOCK_128x128)
        return dict(kind=kind, operands=[_column_major(t) for t in (a, b, sa, sb)], c=empty(M, N))
    dtype = _TYPES[case.get("type", "bf16")]
    x, w = _activations(g, M, K).to(dtype), _weights(g, N, K).to(dtype)
    if kind == "plain":
        return dict(kind=kind, a=x, b=w if case["layout"] == "nk" else w.t().contiguous(), layout=case["layout"], c=empty(M, N, dtype=dtype))
    dy = torch.randn(M, N, generator=g, device="cuda").mul_(N ** -0.5).to(dtype)
    return dict(kind=kind, x=x, w=w, dy=dy, y=empty(M, N), dx=empty(M, K), dyt=empty(N, M), dw=empty(N, K, dtype=torch.float32))


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return _linear(state)
    if kind == "walk":
        state["graph"].replay()
        return [s["y"] for s in state["layers"]]
    if kind == "product":
        return Q.scaled_gemm(state["a"], state["b"], state["sa"], state["sb"], state["c"], *state["sizes"], Q.SCALE_PER_MATRIX)
    if kind == "mm":
        return Q.fp8_mm(*state["operands"], state["c"])
    if kind == "plain":
        return Q.gemm(state["a"], state["b"], state["c"], state["layout"])
    if kind == "encode":
        return Q.quantize(state["x"], state["type"], state["mode"])
    Q.gemm(state["x"], state["w"], state["y"], "nk")
    Q.gemm(state["dy"], state["w"], state["dx"], "kn")
    Q.matrix_transpose(state["dy"], state["dyt"])
    Q.gemm(state["dyt"], state["x"], state["dw"], "kn")
    return state["y"], state["dx"], state["dw"]


def work(case):
    """Every input read once, every output written once; what passes between two calls is not counted."""
    kind = case["kind"]
    up = lambda v: -(-v // 128)  # noqa: E731
    if kind == "encode":
        rows, cols = case["rows"], case["cols"]
        scales = {"1x128": rows * up(cols), "128x128": up(rows) * up(cols), "matrix": 1}[case["mode"]]
        return {"bytes": rows * cols * (_TYPES[case["source"]].itemsize + 1) + 4 * scales, "flops": 0}
    M, N, K = case["M"], case["N"], case["K"]
    flops = 2.0 * M * N * K
    if kind in ("linear", "walk"):
        n = case.get("layers", 1)
        scales = 4 * up(N) * up(K) if case["scales"] == BLOCK else 4
        return {"bytes": n * (2 * M * K + N * K + scales + 2 * M * N), "flops": n * flops}
    if kind == "product":
        return {"bytes": M * K + N * K + 8 + M * N * _TYPES[case["out"]].itemsize, "flops": flops}
    if kind == "mm":
        return {"bytes": M * K + N * K + 4 * (M + up(N)) * up(K) + 2 * M * N, "flops": flops}
    if kind == "plain":
        return {"bytes": 2 * (M * K + N * K + M * N), "flops": flops}
    return {"bytes": 2 * (2 * M * K + N * K + 2 * M * N) + 4 * N * K, "flops": 3 * flops}


def tolerance(case):
    """Compared with the same products summed in 64 bits and then rounded once, bf16 and fp16 results differed by 2e-5 to
    5e-5 (2-norm: a last bit here and there), int8 ones by less, fp8 ones by 2.7e-4 (the matrix cores add the 128
    products of a step with fewer bits), int8 sums scaled to fp32 by 4e-8 (the two scales multiplied in another order)."""
    kind = case["kind"]
    if kind == "encode":
        return "exact"                                  # one rounding of one quotient: the bytes are defined
    if kind == "product" and case["out"] == "i32":
        return "exact"
    if kind == "product" and case["type"] == "int8" and case["out"] == "f32":
        return {"rel": 2e-7}
    return {"rel": 1.2e-3 if kind == "mm" or case.get("type") == "fp8" else 3e-4}
