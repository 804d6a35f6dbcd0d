"""What this backend is timed on: the fused layer kernels, the matrix products,
the attention slots and the whole GPT step, each through the entry point a
training program calls (include/vearo_hip.h, include/vearo_block.h).

A case is a dict: "op" names the path, the other keys are its sizes and
options. Every tensor is f32 (the only type the entry points take); forward
and backward run in one pass, as a training step does. Sizes are those of the
GPT-2-small configuration the benchmark uses ([16, 1024] tokens, width 768,
12 heads, MLP 3072, vocabulary 50257), the smaller models of the tests, and
ragged sizes in between.
"""
import math

import torch

from vearo_amd import _abi as vh

EPS = 1e-5


# ------------------------------------------------------------------- cases --

def listed():
    return [
        # The smallest layer call of the benchmark: 1 MB tensors, bound by launches.
        {"name": "layernorm_2048x128", "op": "layernorm", "rows": 2048, "C": 128},
        # One layernorm of the GPT-2-small step.
        {"name": "layernorm_16384x768", "op": "layernorm", "rows": 16384, "C": 768},
        # The causal attention probabilities of the same step, as the unfused path runs them.
        {"name": "softmax_causal_192x1024", "op": "softmax", "blocks": 192, "T": 1024, "causal": True},
        # The MLP activation with its Linear's bias.
        {"name": "gelu_bias_16384x3072", "op": "gelu_bias", "rows": 16384, "C": 3072},
        # The token embedding under natural-language (Zipf) ids.
        {"name": "embedding_zipf_16384", "op": "embedding", "n": 16384, "V": 50257, "D": 768, "zipf": True},
        # The loss over the whole vocabulary.
        {"name": "cross_entropy_16384x50257", "op": "cross_entropy", "B": 16384, "V": 50257},
        # The MLP's first Linear: the ordinary large product, its two gradients and the bias sum.
        {"name": "linear_16384x768x3072", "op": "linear", "M": 16384, "K": 768, "N": 3072},
        # A Linear on a short ragged batch (one sequence of 1000 tokens).
        {"name": "linear_1000x768x768", "op": "linear", "M": 1000, "K": 768, "N": 768},
        # Attention of the GPT-2-small step, declared causal.
        {"name": "attention_16x12x1024x64", "op": "attention", "B": 16, "H": 12, "S": 1024, "Dk": 64, "mask": False},
        # The BackendOps attention slot with the model's additive -1e9 mask, ragged length.
        {"name": "attention_mask_2x12x333x64", "op": "attention", "B": 2, "H": 12, "S": 333, "Dk": 64, "mask": True},
        # A small model's step, where launches count (the tests' medium model).
        {"name": "gpt_2x128x128", "op": "gpt", "B": 2, "S": 128, "D": 128, "H": 4, "F": 512, "V": 1000},
        # The headline: the GPT-2-small block step, loss and every gradient.
        {"name": "gpt_16x1024x768", "op": "gpt", "B": 16, "S": 1024, "D": 768, "H": 12, "F": 3072, "V": 50257},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["layernorm", "softmax", "gelu_bias", "embedding", "cross_entropy", "linear", "linear",
                     "attention", "gpt"])
    if op in ("layernorm", "gelu_bias"):
        C = _log(rng, 128, 3072)
        if rng.random() < 0.6:
            C = max(4, C // 4 * 4)
        return {"op": op, "rows": _log(rng, 256, 16384), "C": C}
    if op == "softmax":
        T = _log(rng, 64, 1024)
        return {"op": op, "blocks": _log(rng, 2, 192), "T": T, "causal": rng.random() < 0.7}
    if op == "embedding":
        return {"op": op, "n": _log(rng, 256, 16384), "V": _log(rng, 1000, 50257), "D": 4 * _log(rng, 32, 192),
                "zipf": rng.random() < 0.5}
    if op == "cross_entropy":
        return {"op": op, "B": _log(rng, 256, 16384), "V": _log(rng, 1000, 50257)}
    if op == "linear":
        K, N = _log(rng, 128, 3072), _log(rng, 128, 3072)
        if rng.random() < 0.6:
            K, N = K // 16 * 16, N // 16 * 16
        return {"op": op, "M": _log(rng, 256, 16384), "K": K, "N": N}
    if op == "attention":
        return {"op": op, "B": _log(rng, 1, 16), "H": rng.randint(2, 12), "S": _log(rng, 128, 1024),
                "Dk": rng.choice([32, 64, 80]), "mask": rng.random() < 0.5}
    H = rng.choice([4, 8, 12])
    D = H * rng.choice([32, 64])
    return {"op": op, "B": _log(rng, 2, 16), "S": _log(rng, 64, 1024), "D": D, "H": H, "F": 4 * D,
            "V": _log(rng, 1000, 50257)}


# ----------------------------------------------------------------- prepare --

class _Gen:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.empty(shape, device="cuda").normal_(mean, std, generator=self.g)

    def ids(self, n, V, zipf):
        if not zipf:
            return torch.randint(0, V, (n,), device="cuda", generator=self.g).float()
        w = 1.0 / torch.arange(1, V + 1, device="cuda", dtype=torch.float64) ** 1.1
        cum = torch.cumsum(w, 0)
        u = torch.rand(n, device="cuda", dtype=torch.float64, generator=self.g) * cum[-1]
        return torch.searchsorted(cum, u).clamp_(max=V - 1).float()


def _like(*ts):
    return [torch.empty_like(t) for t in ts]


class _Device:
    """A library-owned device buffer as a torch tensor."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _causal_mask(S):
    return torch.triu(torch.full((S, S), -1e9, device="cuda"), 1).reshape(1, 1, S, S)


def _inputs(case, seed):
    """The arrays a pass reads: the same values for run() and exact()."""
    c, g, op = case, _Gen(seed), case["op"]
    if op == "layernorm":
        r, C = c["rows"], c["C"]
        return {"x": g.normal(r, C), "w": g.normal(C, std=0.02, mean=1.0), "b": g.normal(C, std=0.02),
                "dy": g.normal(r, C)}
    if op == "softmax":
        n, T = c["blocks"], c["T"]
        x = g.normal(n, T, T, std=0.125)
        if c["causal"]:
            x.masked_fill_(torch.ones(T, T, dtype=torch.bool, device="cuda").triu_(1), -math.inf)
        return {"x": x, "dy": g.normal(n, T, T)}
    if op == "gelu_bias":
        r, C = c["rows"], c["C"]
        return {"x": g.normal(r, C), "b": g.normal(C, std=0.02), "dy": g.normal(r, C)}
    if op == "embedding":
        return {"ids": g.ids(c["n"], c["V"], c["zipf"]), "w": g.normal(c["V"], c["D"], std=0.02),
                "dy": g.normal(c["n"], c["D"])}
    if op == "cross_entropy":
        return {"x": g.normal(c["B"], c["V"]), "t": g.ids(c["B"], c["V"], False), "go": torch.ones(1, device="cuda")}
    if op == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"x": g.normal(M, K), "w": g.normal(N, K, std=0.02), "b": g.normal(N, std=0.02),
                "dy": g.normal(M, N, std=1e-3)}
    if op == "attention":
        # q, k, v as column blocks of one [B, S, 3, H, Dk] projection, as the model holds them.
        B, H, S, Dk = c["B"], c["H"], c["S"], c["Dk"]
        return {"qkv": g.normal(B, S, 3, H, Dk), "do": g.normal(B, S, H, Dk)}
    from vearo_amd import _block

    cfg = _block.GptConfig(c["B"], c["S"], c["D"], c["H"], c["F"], c["V"], c["S"])
    params = []
    for name, sh in zip(_block.PARAM_NAMES, _block.param_shapes(cfg)):
        params.append(g.normal(*sh, std=0.02, mean=1.0 if name.startswith("ln") and name.endswith("_w") else 0.0))
    n = c["B"] * c["S"]
    return {"cfg": cfg, "params": params, "ids": g.ids(n, c["V"], True), "t": g.ids(n, c["V"], True)}


def _heads(B, S, H, Dk, ld):
    """[B, H, S, Dk] view of [B, S, H, Dk] rows `ld` floats apart."""
    return vh.layout([B, H, S, Dk], [S * ld, Dk, ld, 1])


def _gemm(M, N, K, a, a_s, b, b_s, out, bias=None):
    d = vh.VhGemmDesc()
    d.M, d.N, d.K = M, N, K
    d.a, (d.a_sm, d.a_sk) = a.data_ptr(), a_s
    d.b, (d.b_sk, d.b_sn) = b.data_ptr(), b_s
    d.c, d.c_sm = out.data_ptr(), N
    d.batch[0] = d.batch[1] = 1
    if bias is not None:
        d.e, d.e_sm, d.e_sn = bias.data_ptr(), 0, 1
    d.alpha = 1.0
    return d


def prepare(case, seed):
    vh.init(0)
    c, s, op = case, _inputs(case, seed), case["op"]
    s["case"] = c
    if op == "layernorm":
        s["y"], s["dx"], s["dw"], s["db"] = _like(s["x"], s["x"], s["w"], s["b"])
    elif op == "softmax":
        s["y"], s["dx"] = _like(s["x"], s["x"])
    elif op == "gelu_bias":
        s["y"], s["dx"], s["db"] = _like(s["x"], s["x"], s["b"])
    elif op == "embedding":
        s["y"], s["dw"] = _like(s["dy"], s["w"])
    elif op == "cross_entropy":
        s["loss"], s["dx"] = _like(s["go"], s["x"])
    elif op == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        s["y"], s["dx"], s["dw"], s["db"] = _like(s["dy"], s["x"], s["w"], s["b"])
        s["fwd"] = _gemm(M, N, K, s["x"], (K, 1), s["w"], (1, K), s["y"], s["b"])
        s["bwd_x"] = _gemm(M, K, N, s["dy"], (N, 1), s["w"], (K, 1), s["dx"])
        s["bwd_w"] = _gemm(N, K, M, s["dy"], (1, N), s["x"], (K, 1), s["dw"])
    elif op == "attention":
        B, H, S, Dk = c["B"], c["H"], c["S"], c["Dk"]
        s["lq"], s["lo"] = _heads(B, S, H, Dk, 3 * H * Dk), _heads(B, S, H, Dk, H * Dk)
        s["o"], s["dqkv"] = _like(s["do"], s["qkv"])
        s["mask"] = _causal_mask(S) if c["mask"] else None
        s["lm"] = vh.layout([1, 1, S, S])
    else:
        from vearo_amd import _block

        m = s["model"] = _block.Gpt(s["cfg"])
        shapes = _block.param_shapes(s["cfg"])
        for i, p in enumerate(s.pop("params")):
            torch.as_tensor(_Device(m._ptr(_block.lib.vb_gpt_param, i)[0], shapes[i]), device="cuda").copy_(p)
        m.set_inputs(s.pop("ids").cpu().numpy(), s.pop("t").cpu().numpy())
        # Every gradient but the key bias's, which is zero in exact arithmetic
        # (softmax ignores a shift of a whole row): f32 leaves rounding noise there.
        s["grads"] = {n: torch.as_tensor(_Device(m._ptr(_block.lib.vb_gpt_grad, i)[0], shapes[i]), device="cuda")
                      for i, n in enumerate(_block.PARAM_NAMES) if n != "k_b"}
        s["loss"] = torch.as_tensor(_Device(_block.lib.vb_gpt_loss_ptr(m.h), (1,)), device="cuda")
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- run --

def run(s):
    c, L, ck = s["case"], vh.lib, vh.check
    op = c["op"]
    p = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    if op == "layernorm":
        r, C = c["rows"], c["C"]
        ck(L.vh_layernorm_fwd(p["x"], p["w"], p["b"], p["y"], r, C, EPS, None))
        ck(L.vh_layernorm_bwd(p["x"], p["w"], p["dy"], p["dx"], p["dw"], p["db"], r, C, EPS, None, 0, None))
        return {k: s[k] for k in ("y", "dx", "dw", "db")}
    if op == "softmax":
        rows, T, causal = c["blocks"] * c["T"], c["T"], int(c["causal"])
        ck(L.vh_softmax_fwd(p["x"], p["y"], rows, T, causal, None))
        ck(L.vh_softmax_bwd(p["x"], p["dy"], p["dx"], rows, T, 1, causal, None))
        return {k: s[k] for k in ("y", "dx")}
    if op == "gelu_bias":
        r, C = c["rows"], c["C"]
        ck(L.vh_gelu_bias_fwd(p["x"], p["b"], p["y"], r, C, None))
        ck(L.vh_gelu_bias_bwd(p["x"], p["b"], p["dy"], p["dx"], p["db"], r, C, None, 0, None))
        return {k: s[k] for k in ("y", "dx", "db")}
    if op == "embedding":
        n, V, D = c["n"], c["V"], c["D"]
        ck(L.vh_embedding_fwd(p["ids"], p["w"], p["y"], n, V, D, None))
        ck(L.vh_embedding_bwd(p["ids"], p["dy"], p["dw"], n, V, D, None, 0, None))
        return {k: s[k] for k in ("y", "dw")}
    if op == "cross_entropy":
        B, V = c["B"], c["V"]
        ck(L.vh_cross_entropy_fwd(p["x"], p["t"], p["loss"], B, V, None, 0, None))
        ck(L.vh_cross_entropy_bwd(p["x"], p["t"], p["go"], p["dx"], B, V, None))
        return {k: s[k] for k in ("loss", "dx")}
    if op == "linear":
        for d in (s["fwd"], s["bwd_x"], s["bwd_w"]):
            ck(L.vh_gemm(d, None))
        ck(L.vh_sum_rows(p["dy"], c["M"], c["N"], p["db"], None, 0, None))
        return {k: s[k] for k in ("y", "dx", "dw", "db")}
    if op == "attention":
        step = 4 * c["H"] * c["Dk"]  # bytes from the q block to k's, k's to v's
        q, dq = [p["qkv"] + i * step for i in range(3)], [p["dqkv"] + i * step for i in range(3)]
        lq, lo = s["lq"], s["lo"]
        mask, lm, causal = (p["mask"], s["lm"], 2) if c["mask"] else (None, None, 1)  # 2: VH_ATTN_CAUSAL_AUTO
        ck(L.vh_fused_attention_fwd(q[0], lq, q[1], lq, q[2], lq, mask, lm, causal, p["o"], lo, None, 0, None))
        ck(L.vh_fused_attention_bwd(q[0], lq, q[1], lq, q[2], lq, mask, lm, causal, p["do"], lo, dq[0], lq, dq[1], lq,
                                    dq[2], lq, None, 0, None))
        return {k: s[k] for k in ("o", "dqkv")}
    s["model"].forward_backward(True)
    return {"loss": s["loss"], **s["grads"]}


# ---------------------------------------------------- work, limits, exact --

def work(case):
    c, op = case, case["op"]
    if op == "layernorm":
        n, C = c["rows"] * c["C"], c["C"]
        return {"bytes": 4 * (5 * n + 5 * C), "flops": 0}  # x, w, b -> y; x, w, dy -> dx, dw, db
    if op == "softmax":
        n = c["blocks"] * c["T"] * c["T"]
        live = c["blocks"] * c["T"] * (c["T"] + 1) // 2 if c["causal"] else n
        return {"bytes": 4 * (3 * live + 2 * n), "flops": 0}
    if op == "gelu_bias":
        n, C = c["rows"] * c["C"], c["C"]
        return {"bytes": 4 * (5 * n + 3 * C), "flops": 0}
    if op == "embedding":
        n, V, D = c["n"], c["V"], c["D"]
        hit = V * -math.expm1(n * math.log1p(-1.0 / V))  # distinct rows of uniform ids
        if c["zipf"]:
            w = 1.0 / torch.arange(1, V + 1, dtype=torch.float64) ** 1.1
            hit = float((1 - (1 - w / w.sum()) ** n).sum())
        return {"bytes": 4 * (2 * n + hit * D + 2 * n * D + V * D), "flops": 0}
    if op == "cross_entropy":
        n = c["B"] * c["V"]
        return {"bytes": 4 * (3 * n + 4 * c["B"]), "flops": 0}
    if op == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        # fwd x, w, b -> y; dx: dy, w; dw: dy, x; db: with dy at hand
        return {"bytes": 4 * (3 * M * K + 3 * M * N + 3 * K * N + 2 * N), "flops": 6 * M * K * N}
    if op == "attention":
        B, H, S, Dk = c["B"], c["H"], c["S"], c["Dk"]
        live = S * (S + 1) // 2
        # Two products forward, five backward (the scores again), over the live triangle.
        return {"bytes": 4 * 12 * B * H * S * Dk, "flops": 14 * B * H * live * Dk}
    B, S, D, H, F, V = (c[k] for k in "BSDHFV")
    R, P = B * S, 2 * V * D + S * D + 4 * (D * D + D) + 2 * D * F + F + D + 6 * D
    dense = 2 * R * (4 * D * D + 2 * D * F + V * D)
    attn = 2 * 2 * B * (S * (S + 1) // 2) * D
    return {"bytes": 4 * (2 * P + 2 * R), "flops": 3 * (dense + attn)}


def tolerance(case):
    """f32 throughout: sums of up to ~50000 terms in another order."""
    op = case["op"]
    if op in ("linear", "attention"):
        return {"rel": 4e-6, "max": 2e-4}
    if op == "gpt":
        return {"rel": 2e-5, "max": 2e-3}
    return {"rel": 4e-6, "max": 1e-4}


def _ln(x, w, b):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w, b, EPS)


def _attention(q, k, v):
    """Causal attention over [B, H, S, Dk], one batch entry at a time."""
    S, Dk = q.shape[-2:]
    above = torch.ones(S, S, dtype=torch.bool, device=q.device).triu_(1)
    out = []
    for i in range(q.shape[0]):
        s = (q[i] @ k[i].transpose(1, 2).contiguous()) / math.sqrt(Dk)
        out.append(torch.softmax(s.masked_fill(above, -math.inf), -1) @ v[i])
    return torch.stack(out)


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _grads(out, wrt, upstream):
    return torch.autograd.grad(out, wrt, upstream)


def exact(case, seed):
    c, s, op = case, _inputs(case, seed), case["op"]
    d = {k: v.double() for k, v in s.items() if isinstance(v, torch.Tensor)}
    if op == "layernorm":
        x, w, b = (d[k].requires_grad_() for k in "xwb")
        y = _ln(x, w, b)
        dx, dw, db = _grads(y, (x, w, b), d["dy"])
        return {"y": y, "dx": dx, "dw": dw, "db": db}
    if op == "softmax":
        y = torch.softmax(d["x"], -1)
        dy = d["dy"]
        return {"y": y, "dx": y * (dy - (dy * y).sum(-1, keepdim=True))}
    if op == "gelu_bias":
        x, b = d["x"].requires_grad_(), d["b"].requires_grad_()
        y = _gelu(x + b)
        dx, db = _grads(y, (x, b), d["dy"])
        return {"y": y, "dx": dx, "db": db}
    if op == "embedding":
        i = d["ids"].long()
        return {"y": d["w"][i], "dw": torch.zeros_like(d["w"]).index_add_(0, i, d["dy"])}
    if op == "cross_entropy":
        x, t = d["x"], d["t"].long()
        lse = torch.logsumexp(x, -1, keepdim=True)
        loss = (lse - x.gather(1, t[:, None])).mean().reshape(1)
        dx = x.sub_(lse).exp_()
        dx[torch.arange(len(t), device=t.device), t] -= 1
        return {"loss": loss, "dx": dx.div_(c["B"])}
    if op == "linear":
        x, w, dy = d["x"], d["w"], d["dy"]
        return {"y": x @ w.t() + d["b"], "dx": dy @ w, "dw": dy.t() @ x, "db": dy.sum(0)}
    if op == "attention":
        qkv = d["qkv"].requires_grad_()
        q, k, v = (qkv[:, :, i].transpose(1, 2).contiguous() for i in range(3))
        o = _attention(q, k, v).transpose(1, 2)
        return {"o": o, "dqkv": _grads(o, qkv, d["do"])[0]}
    from vearo_amd._block import PARAM_NAMES

    B, S, D, H = (c[k] for k in "BSDH")
    P = {n: p.double().requires_grad_() for n, p in zip(PARAM_NAMES, s.pop("params"))}
    lin = torch.nn.functional.linear
    h0 = P["wte"][d["ids"].long()].reshape(B, S, D) + P["wpe"][:S]
    a = _ln(h0, P["ln1_w"], P["ln1_b"])
    q, k, v = (lin(a, P[n + "_w"], P[n + "_b"]).reshape(B, S, H, D // H).transpose(1, 2).contiguous() for n in "qkv")
    att = _attention(q, k, v).transpose(1, 2).reshape(B, S, D)
    h1 = h0 + lin(att, P["o_w"], P["o_b"])
    f = _gelu(lin(_ln(h1, P["ln2_w"], P["ln2_b"]), P["fc1_w"], P["fc1_b"]))
    h2 = h1 + lin(f, P["fc2_w"], P["fc2_b"])
    x = lin(_ln(h2, P["lnf_w"], P["lnf_b"]).reshape(B * S, D), P["lm_w"])
    loss = torch.nn.functional.cross_entropy(x, d["t"].long())
    wanted = [n for n in PARAM_NAMES if n != "k_b"]
    grads = torch.autograd.grad(loss, [P[n] for n in wanted])
    return {"loss": loss.detach().reshape(1), **dict(zip(wanted, grads))}
