"""What the performance of this package is measured on: the calls a program that uses it makes.

A case names a use (`use`), the sizes and the weight format:

  linear    one `CobaltLinear` call, `y = x W^T (+ bias)`: decode (few rows of x) and prefill (many)
  qkv       the same on a row-fused q | k | v matrix (three column-scale vectors)
  layer     the seven matrices of a decoder layer as its four dependent decode launches
            (`ops.gemv_batch` on q,k,v / o / gate,up / down), called one after the other
  graph     the same for several layers, captured in a HIP graph and replayed, as a decode loop does
  mlp       the gated MLP as `fuse_model` installs it: `forward_act` on the fused gate/up matrix,
            then the down projection
  dequant   the dense weights of a packed matrix
  pack      RAW arrays (mask, codes, scale, zero point, column scale) into a packed module

Sizes are those of the benchmark's Mistral-7B and Gemma-3-27B shaped layers and of its
single-matrix configurations; weights and activations are synthetic.
"""
import math

import torch

from cobalt_amd import format as F
from cobalt_amd import ops
from cobalt_amd.linear import CobaltLinear

DEV = "cuda"
FORMATS = {  # name: (layout, bits, group, keep)
    "sparse4": (F.SPARSE4, 4, 128, None),
    "sparse4x": (F.SPARSE4X, 4, 128, None),
    "dense4": (F.DENSE4, 4, 128, None),
    "dense8": (F.DENSE8, 8, 128, None),
    "blk4": (F.BLK1632_4, 4, 128, 16),
    "blk6": (F.BLK1632_6, 6, 128, 16),
    "dense2g64": (F.DENSEB, 2, 64, None),
    "dense3g128": (F.DENSEB, 3, 128, None),
}
FORMATS.update({f"b{b}k{k}g{g}": (F.BLKC, b, g, k) for b in (2, 3, 4) for k in (10, 16, 23) for g in (64, 128)
                if (b, k, g) != (4, 16, 128)})
GROUPED = [f for f in FORMATS if not f.startswith("sparse")]        # rows of one length: can be fused and batched


def listed():
    return [
        # the smallest projection of a decoder layer, one token: the cost of a call itself
        dict(name="k_proj_m1", use="linear", K=1024, N=4096, M=1, fmt="blk4", dtype="f16", bias=False, tiled=True),
        # one token through a Mistral-7B shaped layer, 3-bit codes at 69 % sparsity, launched from Python
        dict(name="layer_mistral_b3_m1", use="layer", hidden=4096, q=4096, kv=1024, ffn=14336, layers=1, M=1,
             fmt="b3k10g128", dtype="f16"),
        # one token through two Gemma-3-27B shaped layers replayed from a graph: the headline of the benchmark
        dict(name="graph_gemma_m1", use="graph", hidden=5376, q=4096, kv=2048, ffn=21504, layers=2, M=1,
             fmt="blk4", dtype="bf16"),
        # eight sequences decoded together
        dict(name="layer_gemma_m8", use="layer", hidden=5376, q=4096, kv=2048, ffn=21504, layers=1, M=8,
             fmt="blk4", dtype="bf16"),
        # the output projection of a large vocabulary
        dict(name="lm_head_m1", use="linear", K=262144, N=5376, M=1, fmt="dense4", dtype="bf16", bias=False, tiled=True),
        # a matrix of the reference packer's default layout (survivor streams)
        dict(name="sparse4_gate_m1", use="linear", K=21504, N=5376, M=1, fmt="sparse4", dtype="bf16", bias=False,
             tiled=True),
        # a large decode batch or a short prompt through a gated MLP
        dict(name="mlp_mistral_m48", use="mlp", hidden=4096, ffn=14336, M=48, act="silu", fmt="blk4", dtype="f16"),
        # a prompt of odd length on fused q | k | v, 2-bit codes in groups of 64
        dict(name="qkv_mistral_m333", use="qkv", hidden=4096, q=4096, kv=1024, M=333, fmt="b2k16g64", dtype="f16"),
        # a long prompt through the Gemma-3-27B shaped MLP: the prefill headline
        dict(name="mlp_gemma_m2048", use="mlp", hidden=5376, ffn=21504, M=2048, act="gelu_tanh", fmt="blk4",
             dtype="bf16"),
        # a prompt on a matrix kept at eight bits
        dict(name="down_dense8_m512", use="linear", K=4096, N=14336, M=512, fmt="dense8", dtype="f16", bias=True,
             tiled=True),
        # the dense weights back, as a dense twin of the model needs them
        dict(name="dequant_gate", use="dequant", K=14336, N=4096, fmt="blk4", dtype="f16", tiled=True),
        # installing a compressed artifact: RAW arrays to the device image
        dict(name="pack_gate", use="pack", K=14336, N=4096, fmt="blk4", dtype="f16", tiled=True),
    ]


# ------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, lo=1024, hi=28672):
    return max(lo, _log(rng, lo, hi) // 128 * 128)


def _rows(rng, lo=512, hi=65536):
    k = _log(rng, lo, hi)
    return k if rng.random() < 0.4 else max(16, k // 16 * 16)       # odd heights and padded tails among them


def _fmt(rng, names):
    return "blk4" if rng.random() < 0.35 else rng.choice(sorted(names))


def draw(rng):
    use = rng.choice(["linear", "linear", "linear", "linear", "qkv", "layer", "graph", "mlp", "mlp", "dequant", "pack"])
    dtype = rng.choice(["f16", "bf16"])
    if use in ("linear", "qkv", "mlp"):
        M = _log(rng, 1, 8) if rng.random() < 0.45 else _log(rng, 9, 4096)
    if use == "linear":
        fmt = _fmt(rng, FORMATS)
        cap = 1.5e11 if fmt == "dense8" else 7.0e11                 # flops of a drawn pass, below the largest listed
        while True:
            K, N = _rows(rng), _cols(rng)
            if K * N <= 2.4e8 and 2 * M * K * N <= cap:
                break
        return dict(use=use, K=K, N=N, M=M, fmt=fmt, dtype=dtype, bias=rng.random() < 0.3, tiled=rng.random() < 0.85)
    if use in ("dequant", "pack"):
        fmt = _fmt(rng, FORMATS if use == "dequant" else GROUPED)
        while True:
            K, N = _rows(rng), _cols(rng)
            if K * N <= 1.2e8:
                break
        return dict(use=use, K=K, N=N, fmt=fmt, dtype=dtype, tiled=rng.random() < 0.85)
    hidden = _cols(rng, 1024, 6144)
    ffn = max(hidden, int(hidden * rng.uniform(2.5, 4.0)) // 128 * 128)
    q, kv = _cols(rng, hidden // 2, hidden), 128 * rng.choice([2, 4, 8, 12, 16])
    fmt = _fmt(rng, GROUPED)
    if use == "qkv":
        return dict(use=use, hidden=hidden, q=q, kv=kv, M=M, fmt=fmt, dtype=dtype)
    if use == "mlp":
        cap = 1.5e11 if fmt == "dense8" else 7.0e11
        M = max(1, min(M, int(cap / (6.0 * hidden * ffn))))
        return dict(use=use, hidden=hidden, ffn=ffn, M=M, act=rng.choice(["silu", "gelu_tanh"]), fmt=fmt, dtype=dtype)
    return dict(use=use, hidden=hidden, q=q, kv=kv, ffn=ffn, layers=rng.choice([1, 2, 3]) if use == "graph" else 1,
                M=_log(rng, 1, 8), fmt=fmt, dtype=dtype)


# ------------------------------------------------------------------ inputs
def _dt(case):
    return torch.float16 if case["dtype"] == "f16" else torch.bfloat16


def _packed(K, N, fmt, seed):
    layout, bits, group, keep = FORMATS[fmt]
    return F.synth_packed(K, N, layout, bits, group, keep, seed=seed, device=DEV)


def _module(pm, tiled, bias=None):
    lin = CobaltLinear(pm, bias)
    return lin.to_device_order() if tiled else lin


def _x(M, N, dtype, seed):
    """Activations behind a norm: a spread of column magnitudes and a few outlier columns."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    col = torch.exp(0.4 * torch.randn(N, generator=g, device=DEV))
    col[torch.randint(0, N, (max(1, N // 1024),), generator=g, device=DEV)] *= 12.0
    return (torch.randn(M, N, generator=g, device=DEV) * col).to(dtype)


def _layer_shapes(case):
    h, q, kv, f = case["hidden"], case["q"], case["kv"], case["ffn"]
    return [[(q, h), (kv, h), (kv, h)], [(h, q)], [(f, h), (f, h)], [(h, f)]]


def _step(layers):
    out = []
    for phases in layers:
        for pms, x in phases:
            out += ops.gemv_batch(pms, [x] * len(pms))
    return out


def prepare(case, seed):
    use, dt, s = case["use"], _dt(case), 1000 * seed
    st = {"use": use}
    if use == "linear":
        bias = None
        if case["bias"]:
            g = torch.Generator(device=DEV).manual_seed(s + 2)
            bias = torch.randn(case["K"], generator=g, device=DEV).to(dt)
        st["lin"] = _module(_packed(case["K"], case["N"], case["fmt"], s), case["tiled"], bias)
        st["x"] = _x(case["M"], case["N"], dt, s + 1)
    elif use == "qkv":
        h = case["hidden"]
        parts = [_packed(k, h, case["fmt"], s + i) for i, k in enumerate((case["q"], case["kv"], case["kv"]))]
        st["lin"] = _module(F.fuse_rows(parts), True)
        st["x"] = _x(case["M"], h, dt, s + 9)
    elif use == "mlp":
        h, f = case["hidden"], case["ffn"]
        parts = [_packed(f, h, case["fmt"], s + i) for i in range(2)]
        st["gate_up"] = _module(F.fuse_rows(parts, interleave=True), True)
        st["down"] = _module(_packed(h, f, case["fmt"], s + 2), True)
        st["x"], st["act"] = _x(case["M"], h, dt, s + 9), case["act"]
    elif use in ("layer", "graph"):
        layers = []
        for l in range(case["layers"]):
            phases = []
            for i, phase in enumerate(_layer_shapes(case)):
                pms = [_packed(k, n, case["fmt"], s + 50 * l + 5 * i + j).to_tiled() for j, (k, n) in enumerate(phase)]
                phases.append((pms, _x(case["M"], phase[0][1], dt, s + 50 * l + 5 * i + 4)))
            layers.append(phases)
        st["layers"] = layers
        if use == "graph":
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _step(layers)                                       # first launches set kernel attributes: not capturable
            torch.cuda.current_stream().wait_stream(side)
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"]):
                st["out"] = _step(layers)
    elif use == "dequant":
        st["lin"], st["dtype"] = _module(_packed(case["K"], case["N"], case["fmt"], s), case["tiled"]), dt
    else:
        K, N = case["K"], case["N"]
        layout, bits, group, keep = FORMATS[case["fmt"]]
        g = torch.Generator(device=DEV).manual_seed(s)
        kept = torch.ones(K, N, dtype=torch.bool, device=DEV)
        if keep is not None:
            r = torch.rand(K, N // 32, 32, generator=g, device=DEV)
            kept = torch.zeros_like(r, dtype=torch.bool).scatter_(-1, torch.topk(r, keep, dim=-1).indices, True).view(K, N)
        nl = (1 << bits) - 1
        zero = torch.randint(0, nl + 1, (K, N // group), generator=g, device=DEV)
        off = torch.rand(K, N // group, generator=g, device=DEV) < 0.002   # zero points off the code grid: re-derived
        st["raw"] = dict(mask=F.pack_mask(kept), q=torch.randint(0, nl + 1, (K, N), generator=g, device=DEV).to(torch.uint8),
                         scale=(torch.rand(K, N // group, generator=g, device=DEV) * 0.01 + 1e-3).half(),
                         zero=torch.where(off, zero + nl + 1, zero).half(),
                         col_scale=(torch.rand(N, generator=g, device=DEV) * 1.5 + 0.5).half())
        st["kw"] = dict(layout=layout, bits=bits, group=group, keep=keep, tiled=case["tiled"])
    return st


# ------------------------------------------------------------------ one pass
def run(state):
    use = state["use"]
    if use in ("linear", "qkv"):
        return state["lin"](state["x"])
    if use == "mlp":
        h = state["gate_up"].forward_act(state["x"], state["act"])
        return [h, state["down"](h)]
    if use == "layer":
        return _step(state["layers"])
    if use == "graph":
        state["graph"].replay()
        return state["out"]
    if use == "dequant":
        return state["lin"].dequantize(state["dtype"])
    return CobaltLinear.from_raw(**state["raw"], **state["kw"]).blob


# ------------------------------------------------------------------ what a pass cannot do without
def _weight_bytes(K, N, fmt):
    layout, bits, group, keep = FORMATS[fmt]
    if layout in (F.SPARSE4, F.SPARSE4X):
        return K * N / 8 + K * N / 4 + 3 * K * (N // group) + 4 * K
    return K * F.row_stride(layout, N, bits, group, keep) + 3 * K * (N // group)


def _product(K, N, M, fmt):
    return _weight_bytes(K, N, fmt) + 2 * N + 2 * M * N + 2 * M * K, 2.0 * M * K * N


def work(case):
    use, fmt = case["use"], case["fmt"]
    if use in ("dequant", "pack"):
        K, N = case["K"], case["N"]
        if use == "dequant":
            return {"bytes": _weight_bytes(K, N, fmt) + 2 * N + 2 * K * N, "flops": 0}
        group = FORMATS[fmt][2]
        return {"bytes": K * N + K * N / 8 + 4 * K * (N // group) + 4 * N + _weight_bytes(K, N, fmt), "flops": 0}
    M = case["M"]
    if use == "linear":
        parts = [(case["K"], case["N"])]
    elif use == "qkv":
        parts = [(case["q"], case["hidden"]), (case["kv"], case["hidden"]), (case["kv"], case["hidden"])]
    elif use == "mlp":
        parts = [(case["ffn"], case["hidden"])] * 2 + [(case["hidden"], case["ffn"])]
    else:
        parts = [p for phase in _layer_shapes(case) for p in phase] * case["layers"]
    each = [_product(k, n, M, fmt) for k, n in parts]
    return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}


def tolerance(case):
    """Bytes of a packed image and dequantised weights are defined to the bit.  Products are
    accumulated in float32 from operands of at least 11 bits and rounded once to the activation
    type: two correct results differ by the operand rounding (3e-4) and by one step of that type."""
    if case["use"] in ("dequant", "pack"):
        return "exact"
    return {"rel": 2e-3, "max": 3e-2} if case["dtype"] == "f16" else {"rel": 6e-3, "max": 6e-2}
