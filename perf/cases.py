"""Timed cases of the pruned-weight MatMul/Gemm path.

Each case is one pass that a program built on this package makes, through
its public entry points: a session run, a pruned linear layer (float32 or
int8 CSR, 2:4 int8 or bf16), the dense product of a weight above the density
gate, a transformer feed-forward block, or the pruning of a weight at load
time.  The shapes are those of the MLP 784-512-10, BERT-base and Llama-2-7B
layers that the benchmark and the tests use, and ragged sizes between them.
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

from pyflamert_amd import _lib, pfm, rocm, session

# ---- cases -----------------------------------------------------------------


def listed():
    return [
        # The smallest call: one request of a small pruned classifier through
        # InferenceSession, host tensors in and out; launches and copies count.
        {"name": "mlp_session_b32", "kind": "mlp", "batch": 32, "hidden": 512, "sparsity": 0.9, "mode": "strict"},
        # The headline product: a 90 % pruned square weight times 256 columns,
        # bit-exact mode.
        {"name": "csr_f32_4096_n256", "kind": "csr", "M": 4096, "K": 4096, "N": 256, "density": 0.1, "rows": "uniform",
         "values": "f32", "mode": "strict", "form": "spmm"},
        # A ragged weight and batch in fast mode: no extent is a multiple of a
        # tile, the activation is a linear layer's (tokens x features).
        {"name": "csr_f32_ragged_fast", "kind": "csr", "M": 3001, "K": 5003, "N": 99, "density": 0.1,
         "rows": "uniform", "values": "f32", "mode": "fast", "form": "gemm"},
        # Decoding one token: the gate projection of a Llama-2-7B-shaped layer,
        # 70 % pruned with skewed rows, int8 weight-only.
        {"name": "csr_i8_decode_b1", "kind": "csr", "M": 11008, "K": 4096, "N": 1, "density": 0.3, "rows": "skewed",
         "values": "i8", "mode": "fast", "form": "spmm"},
        # Decoding a batch of eight sequences: the down projection.
        {"name": "csr_i8_decode_b8", "kind": "csr", "M": 4096, "K": 11008, "N": 8, "density": 0.3, "rows": "skewed",
         "values": "i8", "mode": "fast", "form": "spmm"},
        # The prompt of the same model: an attention projection of the same
        # kind of weight over 200 tokens.
        {"name": "csr_i8_prefill_t200", "kind": "csr", "M": 4096, "K": 4096, "N": 200, "density": 0.3,
         "rows": "skewed", "values": "i8", "mode": "fast", "form": "gemm"},
        # A BERT-base encoder's feed-forward block, 80 % pruned, 8 x 128
        # tokens, bit-exact products: Gemm + Gelu, Gemm, residual, LayerNorm.
        {"name": "bert_ffn_t1024", "kind": "ffn", "T": 1024, "H": 768, "F": 3072, "density": 0.2, "mode": "strict"},
        # 2:4 int8 with requantised output: a Llama-2-7B gate projection over
        # 512 columns (the statically quantized graph).
        {"name": "sp24_i8_requant_n512", "kind": "sp24_i8", "M": 11008, "K": 4096, "N": 512},
        # 2:4 int8 decode: what a Linear(x) node of a dynamically quantized
        # session runs for a batch of eight: quantize the activation, multiply.
        {"name": "sp24_dynamic_decode_b8", "kind": "sp24_dynamic", "M": 4096, "K": 11008, "T": 8},
        # 2:4 bf16 prefill over an odd number of columns.
        {"name": "sp24_bf16_n500", "kind": "sp24_bf16", "M": 4096, "K": 4096, "N": 500},
        # A weight above the density gate: the dense bit-exact product with
        # bias and Relu.
        {"name": "dense_f32_t512", "kind": "dense", "T": 512, "K": 768, "N": 3072},
        # Load time: prune a dense weight to 90 %, build its CSR and run the
        # first product on it.
        {"name": "prune_and_first_4096", "kind": "prune", "M": 4096, "K": 4096, "N": 64, "sparsity": 0.9,
         "mode": "strict"},
    ]


def draw(rng):
    """One more case of the listed kinds, sizes over their whole ranges."""
    top = {}  # the largest listed work of each kind
    for c in listed():
        w = work(c)
        t = top.setdefault(c["kind"], [0.0, 0.0])
        t[0], t[1] = max(t[0], w["bytes"]), max(t[1], w["flops"])
    kind = rng.choice(["mlp", "csr", "csr", "csr", "csr", "ffn", "sp24_i8", "sp24_dynamic", "sp24_bf16", "dense",
                       "prune"])

    def size(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        if rng.random() < 0.5:  # half of the extents as models have them, half ragged
            n = max(lo, n // 64 * 64) if n >= 64 else n
        return min(max(n, lo), hi)

    while True:
        mode = rng.choice(["strict", "fast"])
        if kind == "mlp":
            c = {"batch": size(1, 64), "hidden": size(64, 512), "sparsity": rng.choice([0.8, 0.9, 0.95])}
        elif kind == "csr":
            c = {"M": size(512, 11008), "K": size(512, 11008), "N": size(1, 512),
                 "density": rng.choice([0.05, 0.1, 0.2, 0.3]), "rows": rng.choice(["uniform", "skewed"]),
                 "values": rng.choice(["f32", "i8"]), "form": rng.choice(["spmm", "gemm"])}
        elif kind == "ffn":
            c = {"T": size(16, 1024), "H": rng.choice([384, 512, 768]), "density": rng.choice([0.1, 0.2])}
            c["F"] = 4 * c["H"]
        elif kind in ("sp24_i8", "sp24_bf16"):
            c = {"M": size(512, 11008), "K": 4 * size(128, 2752), "N": size(1, 512)}
        elif kind == "sp24_dynamic":
            c = {"M": size(512, 11008), "K": 4 * size(128, 2752), "T": size(1, 64)}
        elif kind == "dense":
            c = {"T": size(1, 1024), "K": size(256, 3072), "N": size(256, 3072)}
        else:
            c = {"M": size(512, 8192), "K": size(512, 8192), "N": size(1, 256), "sparsity": rng.choice([0.7, 0.8, 0.9])}
        c["kind"] = kind
        if kind in ("mlp", "csr", "ffn", "prune"):
            c["mode"] = mode
        w = work(c)
        if w["bytes"] <= 1.05 * top[kind][0] and w["flops"] <= 1.05 * top[kind][1]:
            return c


def work(case):
    k = case["kind"]
    if k == "mlp":
        b, h, d = case["batch"], case["hidden"], 1.0 - case["sparsity"]
        nnz = d * (784 * h + 10 * h)
        return {"bytes": 6 * nnz + 4 * (784 * b + 10 * b + h + 10), "flops": 2 * nnz * b}
    if k == "csr":
        M, K, N = case["M"], case["K"], case["N"]
        nnz = case["density"] * M * K
        per = 6 if case["values"] == "f32" else 3
        side = 4 * M if case["values"] == "f32" else 8 * M
        return {"bytes": per * nnz + side + 4 * K * N + 4 * M * N, "flops": 2 * nnz * N}
    if k == "ffn":
        T, H, F = case["T"], case["H"], case["F"]
        nnz = 2 * case["density"] * H * F
        return {"bytes": 6 * nnz + 8 * T * H + 4 * (F + 3 * H), "flops": 2 * nnz * T}
    if k == "sp24_i8":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 0.625 * M * K + K * N + M * N + 4 * M, "flops": M * K * N}
    if k == "sp24_dynamic":
        M, K, T = case["M"], case["K"], case["T"]
        return {"bytes": 0.625 * M * K + 5 * K * T + 4 * M * T + 4 * M, "flops": M * K * T}
    if k == "sp24_bf16":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 1.125 * M * K + 2 * K * N + 4 * M * N, "flops": M * K * N}
    if k == "dense":
        T, K, N = case["T"], case["K"], case["N"]
        return {"bytes": 4 * (T * K + K * N + T * N + N), "flops": 2 * T * K * N}
    M, K, N = case["M"], case["K"], case["N"]
    nnz = (1.0 - case["sparsity"]) * M * K
    return {"bytes": 8 * M * K + 6 * nnz + 4 * N * (M + K), "flops": 2 * nnz * N}


def tolerance(case):
    k = case["kind"]
    # Strict products, int8 accumulators and quantized values are bit-exact by
    # contract; so are masks.  The session's Softmax goes through expf and the
    # block's Gelu through tanhf (a few ulp each); fast mode reassociates
    # float32 sums of up to some thousand terms, and the bf16 product
    # accumulates in float32 in an order of its own.
    if k == "csr" and case["mode"] == "strict" or k in ("sp24_i8", "sp24_dynamic", "dense"):
        return "exact"
    # (against 64 bits fast products are off by 1e-7 to 7e-7, the
    # block's outputs by 3e-7, the bf16 product by 2.4e-7.)
    if k == "prune" and case["mode"] == "strict":
        return "exact"
    return {"rel": 3e-6 if k in ("csr", "prune") else 1e-6 if k == "mlp" else 2e-6}


# ---- inputs (on the GPU, from the seed alone) --------------------------------


@functools.lru_cache(maxsize=None)
def _context():
    """The program's context, on the stream torch works on."""
    ctx = rocm.Context(0)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    return ctx


def _generator(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _pruned(g, M, K, density, rows):
    """(row, column, value) of a pruned weight: each entry kept with the row's
    probability (skewed: lognormal over the rows), values N(0, 0.02)."""
    if rows == "uniform":
        p = torch.full((M, 1), density, device="cuda")
    else:
        w = torch.exp(0.5 * _normal(g, (M, 1)))
        p = (w / w.mean() * density).clamp(max=1.0)
    keep = torch.rand((M, K), generator=g, device="cuda") < p
    r, c = keep.nonzero(as_tuple=True)
    return r, c, _normal(g, (r.numel(),), 0.02)


def _round_half_away(x):
    return torch.sign(x) * torch.floor(torch.abs(x) + 0.5)


def _csr(case, seed):
    """(indptr, column, values, row scales or None, dense float32 or int8 rows)"""
    g = _generator(seed)
    M, K = case["M"], case["K"]
    r, c, v = _pruned(g, M, K, case["density"], case["rows"])
    scale = None
    if case["values"] == "i8":
        top = torch.zeros(M, device="cuda").scatter_reduce_(0, r, v.abs(), "amax")
        scale = torch.where(top > 0, top / 127.0, torch.ones_like(top))
        v = _round_half_away(v / scale[r]).clamp(-127, 127)
        keep = v != 0
        r, c, v = r[keep], c[keep], v[keep]
    count = torch.bincount(r, minlength=M)
    indptr = torch.zeros(M + 1, dtype=torch.int64, device="cuda")
    indptr[1:] = torch.cumsum(count, 0)
    return g, indptr, r, c, v, scale


def _sp24(g, M, K):
    """2:4 weight: N(0, 1), the two largest of every four along K."""
    w = _normal(g, (M, K)).view(M, K // 4, 4)
    keep = torch.zeros_like(w, dtype=torch.bool)
    keep.scatter_(2, w.abs().topk(2, dim=2).indices, True)
    return torch.where(keep, w, torch.zeros_like(w)).view(M, K)


def _sp24_rows(g, M, K):
    """Its per-row symmetric int8 form."""
    w = _sp24(g, M, K)
    top = w.abs().amax(dim=1)
    scale = torch.where(top > 0, top / 127.0, torch.ones_like(top))
    return _round_half_away(w / scale[:, None]).clamp(-128, 127).to(torch.int8), scale


def _mlp(case, seed):
    rng = np.random.default_rng(seed)

    def pruned(o, i):
        w = (rng.standard_normal((o, i)) * 0.05).astype(np.float32)
        w[rng.random((o, i)) < case["sparsity"]] = 0
        return w

    h = case["hidden"]
    w1, w2 = pruned(h, 784), pruned(10, h)
    b1, b2 = ((rng.standard_normal(n) * 0.1).astype(np.float32) for n in (h, 10))
    return w1, b1, w2, b2, rng.random((case["batch"], 784)).astype(np.float32)


def _ffn(case, seed):
    g = _generator(seed)
    T, H, F = case["T"], case["H"], case["F"]

    def pruned(o, i):
        w = _normal(g, (o, i), 0.02)
        return torch.where(torch.rand((o, i), generator=g, device="cuda") < case["density"], w, torch.zeros_like(w))

    return {"w1": pruned(F, H), "w2": pruned(H, F), "b1": _normal(g, (F,), 0.1), "b2": _normal(g, (H,), 0.1),
            "scale": 1.0 + _normal(g, (H,), 0.1), "bias": _normal(g, (H,), 0.1), "x": _normal(g, (T, H))}


def prepare(case, seed):
    k = case["kind"]
    if k == "mlp":
        w1, b1, w2, b2, x = _mlp(case, seed)
        b, h = case["batch"], case["hidden"]
        model = {"name": "mlp", "inputs": [("x", 0, [b, 784])], "outputs": [("y", 0, [b, 10])],
                 "initializers": {"w1": w1, "b1": b1, "w2": w2, "b2": b2},
                 "nodes": [("fc1", "Gemm", ["x", "w1", "b1"], ["h"], {"transB": 1}),
                           ("act", "Relu", ["h"], ["r"], {}),
                           ("fc2", "Gemm", ["r", "w2", "b2"], ["z"], {"transB": 1}),
                           ("prob", "Softmax", ["z"], ["y"], {"axis": 1})]}
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "mlp.pfm")
            pfm.save(model, path)
            return {"run": "mlp", "x": x, "session": session.InferenceSession(
                path, session.SessionOptions(device="rocm", math_mode=case["mode"]))}
    ctx = _context()
    if k == "csr":
        g, indptr, _, c, v, scale = _csr(case, seed)
        M, K, N = case["M"], case["K"], case["N"]
        if scale is None:
            W = ctx.csr_upload(M, K, indptr.cpu().numpy(), c.cpu().numpy(), v.cpu().numpy())
        else:
            W = ctx.csr_upload(M, K, indptr.cpu().numpy(), c.cpu().numpy(), v.to(torch.int8).cpu().numpy(),
                               row_scales=scale.cpu().numpy())
        if case["form"] == "spmm":
            return {"run": "spmm", "W": W, "x": _normal(g, (K, N)), "y": torch.empty((M, N), device="cuda"),
                    "mode": case["mode"]}
        return {"run": "gemm", "W": W, "ctx": ctx, "x": _normal(g, (N, K)), "bias": _normal(g, (M,), 0.1),
                "y": torch.empty((N, M), device="cuda"), "mode": case["mode"]}
    if k == "ffn":
        s = _ffn(case, seed)
        T, H, F = case["T"], case["H"], case["F"]
        s.update(run="ffn", ctx=ctx, mode=case["mode"], w1=ctx.csr_from_dense_dev(s["w1"].data_ptr(), F, H),
                 w2=ctx.csr_from_dense_dev(s["w2"].data_ptr(), H, F), h=torch.empty((T, F), device="cuda"),
                 f=torch.empty((T, H), device="cuda"), r=torch.empty((T, H), device="cuda"),
                 y=torch.empty((T, H), device="cuda"))
        return s
    if k == "prune":
        g = _generator(seed)
        M, K, N = case["M"], case["K"], case["N"]
        return {"run": "prune", "ctx": ctx, "w": _normal(g, (M, K), 0.02), "x": _normal(g, (K, N)),
                "mask": torch.empty((M, K), device="cuda"), "y": torch.empty((M, N), device="cuda"),
                "sparsity": case["sparsity"], "mode": case["mode"]}
    g = _generator(seed)
    if k == "dense":
        T, K, N = case["T"], case["K"], case["N"]
        return {"run": "dense", "ctx": ctx, "x": _normal(g, (T, K)), "w": _normal(g, (K, N), 0.02),
                "bias": _normal(g, (N,), 0.1), "y": torch.empty((T, N), device="cuda")}
    M, K = case["M"], case["K"]
    if k == "sp24_bf16":
        w = _sp24(g, M, K).to(torch.bfloat16)
        x = _normal(g, (K, case["N"])).to(torch.bfloat16)
        return {"run": "bf16", "W": ctx.sp24_pack_dev(w.data_ptr(), M, K, "bf16"), "x": x,
                "y": torch.empty((M, case["N"]), device="cuda")}
    q, scale = _sp24_rows(g, M, K)
    W = ctx.sp24_pack_dev(q.data_ptr(), M, K, "i8", scale.cpu().numpy())
    if k == "sp24_i8":
        x = _round_half_away(_normal(g, (K, case["N"])) / 0.05).clamp(-128, 127).to(torch.int8)
        return {"run": "i8", "W": W, "x": x, "y": torch.empty((M, case["N"]), dtype=torch.int8, device="cuda")}
    T = case["T"]
    return {"run": "dynamic", "W": W, "ctx": ctx, "x": _normal(g, (T, K)),
            "q": torch.empty((T, K), dtype=torch.uint8, device="cuda"),
            "scale": torch.empty(1, device="cuda"), "zero": torch.empty(1, dtype=torch.uint8, device="cuda"),
            "status": torch.empty(1, dtype=torch.int32, device="cuda"), "y": torch.empty((T, M), device="cuda")}


# ---- one pass ------------------------------------------------------------------


def run(s):
    k = s["run"]
    if k == "mlp":
        return s["session"].run(None, {"x": s["x"]})[0]
    y = s["y"]
    if k == "spmm":
        s["W"].spmm_dev(s["x"].data_ptr(), s["x"].shape[1], y.data_ptr(), mode=s["mode"])
        return y
    if k == "gemm":
        T, K = s["x"].shape
        s["ctx"].gemm_csr_dev(s["x"].data_ptr(), T, K, s["W"], y.data_ptr(), C_ptr=s["bias"].data_ptr(),
                              c_size=s["bias"].numel(), mode=s["mode"])
        return y
    if k == "ffn":
        ctx, x = s["ctx"], s["x"]
        T, H = x.shape
        F = s["h"].shape[1]
        ctx.gemm_csr_dev(x.data_ptr(), T, H, s["w1"], s["h"].data_ptr(), C_ptr=s["b1"].data_ptr(), c_size=F,
                         mode=s["mode"], gelu=True)
        ctx.gemm_csr_dev(s["h"].data_ptr(), T, F, s["w2"], s["f"].data_ptr(), C_ptr=s["b2"].data_ptr(), c_size=H,
                         mode=s["mode"])
        ctx.add_dev(s["f"].data_ptr(), (T, H), x.data_ptr(), (T, H), s["r"].data_ptr())
        ctx.layernorm_dev(s["r"].data_ptr(), T, H, s["scale"].data_ptr(), s["bias"].data_ptr(), 1e-12, y.data_ptr())
        return [s["h"], s["f"], y]
    if k == "dense":
        T, K = s["x"].shape
        N = s["w"].shape[1]
        s["ctx"].gemm_dense_dev(s["x"].data_ptr(), T, K, s["w"].data_ptr(), N, y.data_ptr(),
                                C_ptr=s["bias"].data_ptr(), c_size=N, relu=True)
        return y
    if k == "prune":
        ctx = s["ctx"]
        M, K = s["w"].shape
        ctx.magnitude_mask_dev(s["w"].data_ptr(), M * K, s["sparsity"], s["mask"].data_ptr())
        W = ctx.csr_from_dense_dev(s["w"].data_ptr(), M, K, mask_ptr=s["mask"].data_ptr())
        W.spmm_dev(s["x"].data_ptr(), s["x"].shape[1], y.data_ptr(), mode=s["mode"])
        W.free()
        return [s["mask"], y]
    if k == "bf16":
        s["W"].gemm_bf16_dev(s["x"].data_ptr(), s["x"].shape[1], y.data_ptr())
        return y
    if k == "i8":
        s["W"].gemm_i8_dev(s["x"].data_ptr(), s["x"].shape[1], y.data_ptr(), x_scale=0.05, out="i8", out_scale=0.6)
        return y
    ctx, (T, K) = s["ctx"], s["x"].shape
    lib = _lib.load()
    _lib.check(lib.pfr_dynamic_quantize_linear_dev(ctx.handle, s["x"].data_ptr(), T * K, s["q"].data_ptr(),
                                                   s["scale"].data_ptr(), s["zero"].data_ptr(),
                                                   s["status"].data_ptr()))
    _lib.check(lib.pfr_sp24_gemm_qt_dev(ctx.handle, s["W"].handle, s["q"].data_ptr(), _lib.PFR_U8, T, K, 1.0, 0,
                                        s["scale"].data_ptr(), s["zero"].data_ptr(), y.data_ptr(), s["W"].M))
    return [s["q"], s["scale"], s["zero"], y]


# ---- the same in 64 bits ---------------------------------------------------------


def _matmul64(a, b):
    return torch.matmul(a.double().contiguous(), b.double().contiguous())


def exact(case, seed):
    k = case["kind"]
    if k == "mlp":
        w1, b1, w2, b2, x = (a.astype(np.float64) for a in _mlp(case, seed))
        z = np.maximum(x @ w1.T + b1, 0.0) @ w2.T + b2
        e = np.exp(z - z.max(axis=1, keepdims=True))
        return e / e.sum(axis=1, keepdims=True)
    if k == "csr":
        g, _, r, c, v, scale = _csr(case, seed)
        M, K, N = case["M"], case["K"], case["N"]
        if scale is not None:
            v = v * scale[r]  # the float32 weight that the int8 value stands for
        w = torch.zeros((M, K), dtype=torch.float64, device="cuda")
        w[r, c] = v.double()
        if case["form"] == "spmm":
            return _matmul64(w, _normal(g, (K, N)))
        x, bias = _normal(g, (N, K)), _normal(g, (M,), 0.1)
        return _matmul64(x, w.t()) + bias.double()
    if k == "ffn":
        s = {n: a.double() for n, a in _ffn(case, seed).items()}
        h = _matmul64(s["x"], s["w1"].t()) + s["b1"]
        h = 0.5 * h * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (h + 0.044715 * h ** 3)))
        f = _matmul64(h, s["w2"].t()) + s["b2"]
        r = f + s["x"]
        d = r - r.mean(dim=1, keepdim=True)
        y = s["scale"] * d / torch.sqrt((d * d).mean(dim=1, keepdim=True) + 1e-12) + s["bias"]
        return [h, f, y]
    g = _generator(seed)
    if k == "prune":
        M, K, N = case["M"], case["K"], case["N"]
        w, x = _normal(g, (M, K), 0.02), _normal(g, (K, N))
        n, sparsity = M * K, np.float32(case["sparsity"])
        a = w.abs().flatten()
        cut = a.sort().values[min(int(n * float(sparsity)), n - 1)]
        keep = a > cut
        spare = int((~keep).sum()) - int(np.float32(n) * sparsity)  # weights at the cut come back, first ones first
        keep[(a == cut).nonzero().flatten()[:max(spare, 0)]] = True
        return [keep.view(M, K).float(), _matmul64(torch.where(keep.view(M, K), w, torch.zeros_like(w)), x)]
    if k == "dense":
        T, K, N = case["T"], case["K"], case["N"]
        x, w, bias = _normal(g, (T, K)), _normal(g, (K, N), 0.02), _normal(g, (N,), 0.1)
        return (_matmul64(x, w) + bias.double()).clamp(min=0.0)
    M, K = case["M"], case["K"]
    if k == "sp24_bf16":
        w = _sp24(g, M, K).to(torch.bfloat16)
        return _matmul64(w, _normal(g, (K, case["N"])).to(torch.bfloat16))
    q, scale = _sp24_rows(g, M, K)
    if k == "sp24_i8":
        x = _round_half_away(_normal(g, (K, case["N"])) / 0.05).clamp(-128, 127)
        p = _matmul64(q, x) * (scale.double()[:, None] * 0.05) / 0.6
        return _round_half_away(p).clamp(-128, 127).to(torch.int8)
    # the quantized activation is whole numbers, decided by its float32
    # parameters; the product of those numbers is then exact
    x = _normal(g, (case["T"], K))
    lo, hi = x.min().clamp(max=0.0), x.max().clamp(min=0.0)
    step = (hi - lo) / 255.0
    zero = _round_half_away(-lo / step).clamp(0, 255)
    xq = (_round_half_away(x * (1.0 / step)) + zero).clamp(0, 255)
    return [xq.to(torch.uint8), (hi.double() - lo.double()).view(1) / 255.0, zero.to(torch.uint8).view(1),
            _matmul64(xq - zero, q.t()) * (step.double() * scale.double())]
