"""The work a NanoLLM user has this library do, as cases that can be timed and checked.

* ``generate``: a prompt batch is prefilled and continued token by token (``NanoLLM.prefill`` /
  ``decode``), greedily or sampled, down to the tokens and the last step's logits on the host.
* ``prefill``: scoring of prompts -- the logits after each prompt, nothing generated.
* ``window``: the full-window forward (every row's logits), as an evaluation of a text runs it.
* ``dense``: the four projections of a transformer block on rows of activations, with the fused
  epilogues, through the operator API.
* ``mlp_train``, ``attn_train``, ``head_train``: forward and backward of a block's MLP half, of
  its attention layer and of ln_f + tied lm_head + cross entropy + embedding, operator by
  operator as ``Model::Run(input, target)`` issues them.  The AdamW update is not in them: it
  changes the parameters in place, and a case has to give the same answer when it is run again.

Everything is fp32, the library's one data type.  Shapes are c1 .. c5 of ``freeml_amd.synth``
and sizes around them.
"""
import math

import numpy as np
import torch

import freeml_amd as fh
from freeml_amd import synth


def _engine(kind, name, vocab, block, embed, heads, layers, batch, prompt, steps=0, temperature=0.0, top_k=0):
    c = dict(kind=kind, vocab=vocab, block=block, embed=embed, heads=heads, layers=layers, batch=batch,
             prompt=prompt, steps=steps, temperature=temperature, top_k=top_k)
    return dict(c, name=name) if name else c


def _config(name, label, cfg, steps=None):
    s = synth.CONFIGS[cfg]
    h = s["shape"]
    return _engine("generate", name or label, h.vocab, h.block_size, h.n_embed, h.n_head, h.n_layer, s["batch"],
                   s["prompt"], s["n_gen"] - 1 if steps is None else steps)


def listed():
    return [
        # The smallest model: a few tokens of a toy character model, latency only.
        _config(None, "generate_c1_bs1", "c1"),
        # One user typing at a character GPT: the window is filled from a 64-token prompt.
        _config(None, "generate_c2_bs1", "c2"),
        # The same model serving 64 users at once.
        _config(None, "generate_c3_bs64", "c3"),
        # A GPT-2-small-sized model, 8 users, half a context of prompt, the start of the answer.
        _config(None, "generate_c4_bs8", "c4", steps=48),
        # Long context: 4 users with prompts of 3584 tokens.
        _config(None, "generate_c5_bs4", "c5", steps=64),
        # Text generation as it is mostly done: sampled with temperature and top-k, 3 users.
        _engine("generate", "sample_c2_bs3", 65, 256, 384, 6, 6, 3, 37, 100, 0.8, 40),
        # Scoring prompts of an uneven length with a third of the GPT-2-small stack.
        _engine("prefill", "prefill_ragged", 50304, 1024, 768, 12, 4, 5, 777),
        # Evaluation of whole windows of the character GPT.
        _engine("window", "window_c2_bs8", 65, 256, 384, 6, 6, 8, 256),
        # The dense layers of a GPT-2-small block on a ragged number of rows.
        dict(name="dense_768", kind="dense", rows=2500, embed=768),
        # Training of the character GPT, one window: the MLP half of a block.
        dict(name="mlp_train_c2", kind="mlp_train", rows=256, embed=384),
        # Training at GPT-2-small's width and context: the attention layer.
        dict(name="attn_train_c4", kind="attn_train", rows=1024, embed=768, heads=12),
        # Training with the 50304-token vocabulary: ln_f, tied lm_head, cross entropy, embedding.
        dict(name="head_train_c4", kind="head_train", rows=1024, embed=768, vocab=50304),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["generate", "generate", "generate", "prefill", "window", "dense", "mlp_train", "attn_train",
                       "head_train"])
    if kind in ("generate", "prefill", "window"):
        while True:
            head_dim = rng.choice([64, 64, 64, 32, 16])
            embed = rng.choice([64, 128, 192, 256, 320, 384, 512, 640, 768, 1024])
            layers = rng.randint(1, 12)
            vocab = _log_int(rng, 33, 50304)
            block = _log_int(rng, 33, 2048)
            batch = _log_int(rng, 1, 64)
            heads = embed // head_dim
            sampled = kind == "generate" and rng.random() < 0.3
            prompt = block if kind == "window" else rng.randint(1, block)
            steps = rng.randint(0, min(block - prompt, 480 // layers)) if kind == "generate" else 0
            flops = batch * prompt * (24 * layers * embed * embed + 2 * layers * embed * prompt)
            if kind == "window":
                flops += 2 * batch * prompt * vocab * embed
            weights = 4 * (12 * layers * embed * embed + vocab * embed)
            if heads > 16 or batch * block > 16384 or flops > 4e11 or weights > 4e8:
                continue
            if kind == "window" and batch * block * vocab > 16e6:
                continue
            if kind == "generate" and (steps < 1 or weights * steps > 1e10):
                continue
            return _engine(kind, None, vocab, block, embed, heads, layers, batch, prompt, steps,
                           round(rng.uniform(0.5, 1.2), 2) if sampled else 0.0,
                           rng.choice([0, 5, 40]) if sampled else 0)
    embed = 16 * _log_int(rng, 4, 64)
    if kind == "dense":
        return dict(kind=kind, rows=_log_int(rng, 1, 4096), embed=embed)
    if kind == "mlp_train":
        return dict(kind=kind, rows=_log_int(rng, 33, 2048), embed=embed)
    if kind == "attn_train":
        head_dim = rng.choice([64, 64, 32, 16])
        heads = rng.randint(1, min(16, 1024 // head_dim))
        return dict(kind=kind, rows=_log_int(rng, 33, 1024), embed=heads * head_dim, heads=heads)
    return dict(kind=kind, rows=_log_int(rng, 33, 1024), embed=min(embed, 768), vocab=_log_int(rng, 33, 50304))


# ---- inputs ------------------------------------------------------------------------------------

_KINDS = ["generate", "prefill", "window", "dense", "mlp_train", "attn_train", "head_train"]


class _Inputs:
    """Seeded inputs made on the GPU, in one fixed order."""

    def __init__(self, case, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed * 16 + _KINDS.index(case["kind"]))

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(std).add_(mean)

    def ids(self, high, *shape):
        return torch.randint(0, high, shape, generator=self.g, device="cuda")


def _model_inputs(case, seed):
    """Weights of a NanoLLM (std 0.02, tied head) with gains around 1, and the prompts."""
    r = _Inputs(case, seed)
    V, T, C, L = case["vocab"], case["block"], case["embed"], case["layers"]
    w = {"tok": r.normal(V, C, std=0.02), "pos": r.normal(T, C, std=0.02), "lnf": r.normal(C, std=0.1, mean=1.0)}
    w["layers"] = [dict(qkv=r.normal(C, 3 * C, std=0.02), proj=r.normal(C, C, std=0.02),
                        fc=r.normal(C, 4 * C, std=0.02), proj2=r.normal(4 * C, C, std=0.02),
                        ln0=r.normal(C, std=0.1, mean=1.0), ln1=r.normal(C, std=0.1, mean=1.0)) for _ in range(L)]
    return w, r.ids(V, case["batch"], case["prompt"])


def _train_inputs(case, seed):
    """Activations of unit scale, weights of std 0.02, output gradients of a mean loss."""
    r = _Inputs(case, seed)
    M, C = case["rows"], case["embed"]
    if case["kind"] == "dense":
        return dict(x=r.normal(M, C), qkv_w=r.normal(C, 3 * C, std=0.02), y=r.normal(M, C, std=0.3),
                    proj_w=r.normal(C, C, std=0.02), fc_w=r.normal(C, 4 * C, std=0.02),
                    proj2_w=r.normal(4 * C, C, std=0.02), res=r.normal(M, C))
    if case["kind"] == "mlp_train":
        return dict(x=r.normal(M, C), g=r.normal(C, std=0.1, mean=1.0), fc_w=r.normal(C, 4 * C, std=0.02),
                    proj2_w=r.normal(4 * C, C, std=0.02), dy=r.normal(M, C, std=1.0 / M))
    if case["kind"] == "attn_train":
        return dict(x=r.normal(M, C), qkv_w=r.normal(C, 3 * C, std=0.02), proj_w=r.normal(C, C, std=0.02),
                    dy=r.normal(M, C, std=1.0 / M), scale=torch.full((1,), 1.0 / math.sqrt(C // case["heads"]),
                                                                    device="cuda"))
    V = case["vocab"]
    target = r.ids(V, M).float()
    target[M // 2] = -1.0  # a position the loss leaves out
    return dict(x=r.normal(M, C), g=r.normal(C, std=0.1, mean=1.0), tok=r.normal(V, C, std=0.02),
                idx=r.ids(V, M).float(), target=target)


def _buffers(case):
    """Outputs and intermediates of one pass."""
    M, C = case["rows"], case["embed"]

    def e(*shape):
        return torch.empty(*shape, device="cuda")

    if case["kind"] == "dense":
        return dict(qkv=e(M, 3 * C), x1=e(M, C), h=e(M, 4 * C), x2=e(M, C))
    if case["kind"] == "mlp_train":
        return dict(xn=e(M, C), xhat=e(M, C), h=e(M, 4 * C), a=e(M, 4 * C), o=e(M, C), y=e(M, C),
                    dproj2=e(4 * C, C), da=e(M, 4 * C), gd=e(M, 4 * C), dh=e(M, 4 * C), dfc=e(C, 4 * C),
                    dxn=e(M, C), dx=e(M, C), dg=e(C))
    if case["kind"] == "attn_train":
        H = case["heads"]
        hd = C // H
        return dict(qkv=e(M, 3 * C), q=e(M, C), k=e(M, C), v=e(M, C), s=e(H, M, M), att=e(H, M, M),
                    p=[e(M, M) for _ in range(H)], y=e(M, C), out=e(M, C), dproj=e(C, C), dyy=e(M, C),
                    ds=e(H, M, M), dq=e(H, M, hd), dk=e(H, M, hd), dv=e(H, M, hd), dqkv=e(M, 3 * C),
                    dqkv_w=e(C, 3 * C), dx=e(M, C))
    V = case["vocab"]
    return dict(emb=e(M, C), xin=e(M, C), xn=e(M, C), xhat=e(M, C), logits=e(M, V), dlogits=e(M, V), loss=e(1),
                ws=e(M + 1), dxn=e(M, C), dtok=e(V, C), demb=e(V, C), dx=e(M, C), dg=e(C))


def prepare(case, seed):
    fh.init(0)
    if case["kind"] not in ("generate", "prefill", "window"):
        state = dict(case=case, **_train_inputs(case, seed), **_buffers(case))
        torch.cuda.synchronize()  # the library works on a stream of its own
        return state
    w, prompts = _model_inputs(case, seed)

    def host(t):
        return t.cpu().numpy()

    shape = synth.NanoLLMShape(case["vocab"], case["block"], case["embed"], case["heads"], case["layers"])
    tok = host(w["tok"])
    layers = [synth.LayerWeights(host(l["qkv"]), host(l["proj"]), host(l["fc"]), host(l["proj2"]), host(l["ln0"]),
                                 host(l["ln1"])) for l in w["layers"]]
    weights = synth.NanoLLMWeights(shape, tok, host(w["pos"]), layers, host(w["lnf"]), None, tok)
    model = fh.NanoLLM(weights, max_batch=case["batch"])
    if case["temperature"] > 0:
        model.set_sampling(case["temperature"], case["top_k"], seed=7)
    return dict(case=case, model=model, prompts=host(prompts.to(torch.int32)))


# ---- one pass ----------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "window":
        return {"logits": state["model"].forward_window(state["prompts"])}
    if kind == "prefill" or kind == "generate":
        m = state["model"]
        m.prefill(state["prompts"])
        if kind == "generate":
            m.decode(case["steps"])
        return {"tokens": m.tokens(), "logits": m.logits()}
    return _OPS[kind](state, case["rows"], case["embed"])


def _ptrs(s):
    return {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}


def _run_dense(s, M, C):
    p = _ptrs(s)
    fh.gemm_ex(p["x"], C, p["qkv_w"], 3 * C, 0, p["qkv"], 3 * C, M, 3 * C, C)
    fh.gemm_ex(p["y"], C, p["proj_w"], C, 1, p["x1"], C, M, C, C, fh.EPI_RESID, p["res"], C)
    fh.gemm_ex(p["x"], C, p["fc_w"], 4 * C, 0, p["h"], 4 * C, M, 4 * C, C, fh.EPI_GELU)
    fh.gemm_ex(p["h"], 4 * C, p["proj2_w"], C, 0, p["x2"], C, M, C, 4 * C, fh.EPI_RESID, p["res"], C)
    return {k: s[k] for k in ("qkv", "x1", "h", "x2")}


def _run_mlp_train(s, M, C):
    p = _ptrs(s)
    fh.layernorm(p["xn"], p["x"], p["g"], 0, p["xhat"], M, C)
    fh.mul(fh.NONE, p["h"], p["xn"], p["fc_w"], M, 4 * C, C)
    fh.gelu(p["a"], p["h"], M * 4 * C)
    fh.mul(fh.NONE, p["o"], p["a"], p["proj2_w"], M, C, 4 * C)
    fh.add(p["y"], p["x"], p["o"], M * C)
    fh.mul(fh.LEFT, p["dproj2"], p["a"], p["dy"], 4 * C, C, M)
    fh.mul(fh.RIGHT, p["da"], p["dy"], p["proj2_w"], M, 4 * C, C)
    fh.gelu_derivative(p["gd"], p["h"], M * 4 * C)
    fh.per_element_mul(p["dh"], p["da"], p["gd"], M * 4 * C)
    fh.mul(fh.LEFT, p["dfc"], p["xn"], p["dh"], C, 4 * C, M)
    fh.mul(fh.RIGHT, p["dxn"], p["dh"], p["fc_w"], M, C, 4 * C)
    fh.layernorm_backward(p["dx"], p["dxn"], p["x"], p["g"], p["dg"], 0, p["xhat"], 0, M, C)
    fh.add(p["dx"], p["dx"], p["dy"], M * C)
    return {k: s[k] for k in ("y", "dproj2", "dfc", "dg", "dx")}


def _run_attn_train(s, T, C):
    p = _ptrs(s)
    H = s["case"]["heads"]
    hd, tt, th = C // H, T * T, T * (C // H)
    heads = [t.data_ptr() for t in s["p"]]
    fh.mul(fh.NONE, p["qkv"], p["x"], p["qkv_w"], T, 3 * C, C)
    fh.split_qkv(p["q"], p["k"], p["v"], p["qkv"], T, C)
    fh.matmul_strided(fh.RIGHT, p["s"], p["q"], p["k"], T, T, hd, C, 1, C, 1, T, 1, H, hd, hd, tt)
    fh.attention_softmax_heads(heads, 0, p["att"], p["s"], p["scale"], H, T)
    fh.matmul_strided(fh.NONE, p["y"], p["att"], p["v"], T, hd, T, T, 1, C, 1, C, 1, H, tt, hd, hd)
    fh.mul(fh.RIGHT, p["out"], p["y"], p["proj_w"], T, C, C)
    # backward; the all-heads probabilities are read (dV) before dAtt takes their place
    fh.mul(fh.LEFT, p["dproj"], p["dy"], p["y"], C, C, T)
    fh.mul(fh.NONE, p["dyy"], p["dy"], p["proj_w"], T, C, C)
    fh.matmul_strided(fh.LEFT, p["dv"], p["att"], p["dyy"], T, hd, T, T, 1, C, 1, hd, 1, H, tt, hd, th)
    fh.matmul_strided(fh.RIGHT, p["att"], p["dyy"], p["v"], T, T, hd, C, 1, C, 1, T, 1, H, hd, hd, tt)
    fh.attention_softmax_backward_heads(p["ds"], heads, p["att"], p["scale"], H, T)
    fh.matmul_strided(fh.NONE, p["dq"], p["ds"], p["k"], T, hd, T, T, 1, C, 1, hd, 1, H, tt, hd, th)
    fh.matmul_strided(fh.LEFT, p["dk"], p["ds"], p["q"], T, hd, T, T, 1, C, 1, hd, 1, H, tt, hd, th)
    fh.merge_qkv(p["dqkv"], p["dq"], p["dk"], p["dv"], hd, T, H)
    fh.mul(fh.LEFT, p["dqkv_w"], p["x"], p["dqkv"], C, 3 * C, T)
    fh.mul(fh.RIGHT, p["dx"], p["dqkv"], p["qkv_w"], T, C, 3 * C)
    return {k: s[k] for k in ("out", "dproj", "dqkv_w", "dx")}


def _run_head_train(s, M, C):
    p = _ptrs(s)
    V = s["case"]["vocab"]
    fh.gather_rows(p["emb"], p["tok"], p["idx"], C, M, 1, V, 1)
    fh.add(p["xin"], p["x"], p["emb"], M * C)
    fh.layernorm(p["xn"], p["xin"], p["g"], 0, p["xhat"], M, C)
    fh.mul(fh.RIGHT, p["logits"], p["xn"], p["tok"], M, V, C)
    fh.cce_logits(p["dlogits"], p["loss"], p["ws"], p["target"], p["logits"], V, M, 1, 1, 1)
    fh.mul(fh.LEFT, p["dtok"], p["dlogits"], p["xn"], V, C, M)
    fh.mul(fh.NONE, p["dxn"], p["dlogits"], p["tok"], M, C, V)
    fh.layernorm_backward(p["dx"], p["dxn"], p["xin"], p["g"], p["dg"], 0, p["xhat"], 0, M, C)
    fh.fill(p["demb"], 0.0, V * C)
    fh.scatter_add_rows(p["demb"], p["dx"], p["idx"], C, M, 1, V, 1)
    fh.add(p["dtok"], p["dtok"], p["demb"], V * C)
    return {k: s[k] for k in ("logits", "loss", "dtok", "dg", "dx")}


_OPS = {"dense": _run_dense, "mlp_train": _run_mlp_train, "attn_train": _run_attn_train, "head_train": _run_head_train}


# ---- what a pass cannot do without -----------------------------------------------------------------

def work(case):
    """Bytes: inputs once, outputs once; a generated token reads every weight and its sequence's
    cached keys and values again, as it depends on the token before it.  Flops: the products (an
    attention's causal half)."""
    kind = case["kind"]
    if kind in ("generate", "prefill", "window"):
        V, C, L, B, P, n = (case[k] for k in ("vocab", "embed", "layers", "batch", "prompt", "steps"))
        block = 12 * L * C * C
        rows = P if kind == "window" else 1
        flops = B * (2 * P * block + L * 2 * C * P * (P + 1) + rows * 2 * V * C)
        weights = 4 * (block + V * C + 2 * L * C + C)
        nbytes = weights + 4 * B * (P * C * 2 * (L + 1) + rows * V)
        for t in range(P + 1, P + 1 + n):
            flops += B * (2 * block + 4 * L * C * t + 2 * V * C)
            nbytes += weights + 4 * B * (2 * L * C * t + 2 * L * C + 2 * C)
        return {"bytes": nbytes, "flops": flops}
    M, C = case["rows"], case["embed"]
    if kind == "dense":
        return {"bytes": 4 * (12 * C * C + 12 * M * C), "flops": 24 * M * C * C}
    if kind == "mlp_train":
        return {"bytes": 4 * (16 * C * C + 4 * M * C + 2 * C), "flops": 48 * M * C * C}
    if kind == "attn_train":
        return {"bytes": 4 * (8 * C * C + 4 * M * C), "flops": 24 * M * C * C + 12 * C * M * (M + 1) // 2}
    V = case["vocab"]
    return {"bytes": 4 * (2 * V * C + M * V + 2 * M * C + 2 * C + 2 * M), "flops": 6 * M * V * C}


def tolerance(case):
    """About four times the error that fp32 sums show against 64 bits (measured: tokens' logits
    5e-7, long prefills and deep windows 1.6e-6, single layers 3e-7 .. 9e-7, and 4e-6 for the
    input gradient of a 50304-wide lm_head, a sum of that many terms that mostly cancel)."""
    rel = {"generate": 2e-6, "prefill": 8e-6, "window": 8e-6, "dense": 3e-6, "mlp_train": 2e-6, "attn_train": 4e-6,
           "head_train": 1.6e-5}[case["kind"]]
    return {"rel": rel, "max": 100 * rel, "differ": 0.005}


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _ln(x, g):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * g


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


_M64 = (1 << 64) - 1


def _splitmix64(x):
    x = (x + 0x9E3779B97F4A7C15) & _M64
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & _M64
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & _M64
    return x ^ (x >> 31)


def _pick(case, z, pos):
    """Next tokens of logits z (batch x vocab) for position pos: first maximum, or the sampling
    the header of the library states."""
    if case["temperature"] <= 0:
        return z.argmax(-1)
    out = []
    for b, row in enumerate(z.cpu().numpy()):
        p = np.exp((row - row.max()) / np.float64(np.float32(case["temperature"])))
        k = case["top_k"]
        if 0 < k < row.size:
            keep = np.argsort(-row, kind="stable")[:k]
            mask = np.zeros(row.size, bool)
            mask[keep] = True
            p = np.where(mask, p, 0.0)
        u = (_splitmix64(7 ^ _splitmix64((b << 32) | pos)) >> 40) / 16777216.0
        hit = np.nonzero((np.cumsum(p) > u * p.sum()) & (p > 0))[0]
        out.append(int(hit[0]) if hit.size else int(np.nonzero(p)[0][-1]))
    return torch.tensor(out, device=z.device)


def _exact_model(case, seed):
    w, ids = _model_inputs(case, seed)
    w = {k: (v.double() if torch.is_tensor(v) else [{n: t.double() for n, t in l.items()} for l in v])
         for k, v in w.items()}
    C, H, B, P = case["embed"], case["heads"], case["batch"], case["prompt"]
    hd = C // H
    cache = [None] * case["layers"]

    def blocks(x, first):
        rows = x.shape[1]
        mask = None
        if rows > 1:
            mask = torch.full((rows, rows), float("-inf"), device="cuda", dtype=torch.float64).triu(1)
        for i, l in enumerate(w["layers"]):
            q, k, v = (t.reshape(B, rows, H, hd).transpose(1, 2).contiguous()
                       for t in (_ln(x, l["ln0"]) @ l["qkv"]).split(C, -1))
            if first:
                k, v = torch.cat([cache[i][0], k], 2), torch.cat([cache[i][1], v], 2)
            cache[i] = (k, v)
            s = q @ k.transpose(2, 3).contiguous() / math.sqrt(hd)
            if mask is not None:
                s += mask
            y = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(B, rows, C)
            del s
            x = x + y @ l["proj"].t()
            x = x + _gelu(_ln(x, l["ln1"]) @ l["fc"]) @ l["proj2"]
        return x

    def head(x):
        return _ln(x, w["lnf"]) @ w["tok"].t()

    x = blocks(w["tok"][ids] + w["pos"][:P], 0)
    if case["kind"] == "window":
        return {"logits": head(x)}
    z = head(x[:, -1])
    tokens = [_pick(case, z, P)]
    for t in range(P, P + case["steps"]):
        x = blocks((w["tok"][tokens[-1]] + w["pos"][t])[:, None], t)
        z = head(x[:, -1])
        tokens.append(_pick(case, z, t + 1))
    return {"tokens": None, "logits": z}


def _ln_backward(x, g, dy):
    mean = x.mean(-1, keepdim=True)
    inv = 1 / torch.sqrt(((x - mean) ** 2).mean(-1, keepdim=True) + 1e-5)
    xhat = (x - mean) * inv
    dh = dy * g
    dx = inv * (dh - dh.mean(-1, keepdim=True) - xhat * (dh * xhat).mean(-1, keepdim=True))
    return dx, (dy * xhat).sum(0)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("generate", "prefill", "window"):
        return _exact_model(case, seed)
    s = {k: v.double() for k, v in _train_inputs(case, seed).items()}
    x, M, C = s["x"], case["rows"], case["embed"]
    if kind == "dense":
        h = _gelu(x @ s["fc_w"])
        return {"qkv": x @ s["qkv_w"], "x1": s["res"] + s["y"] @ s["proj_w"].t(), "h": h,
                "x2": s["res"] + h @ s["proj2_w"]}
    if kind == "mlp_train":
        xn, dy = _ln(x, s["g"]), s["dy"]
        h = xn @ s["fc_w"]
        a = _gelu(h)
        dh = (dy @ s["proj2_w"].t()) * (0.5 * (1 + torch.erf(h / math.sqrt(2.0)))
                                        + h * torch.exp(-0.5 * h * h) / math.sqrt(2 * math.pi))
        dx, dg = _ln_backward(x, s["g"], dh @ s["fc_w"].t())
        return {"y": x + a @ s["proj2_w"], "dproj2": a.t() @ dy, "dfc": xn.t() @ dh, "dg": dg, "dx": dx + dy}
    if kind == "attn_train":
        H = case["heads"]
        scale = s["scale"]
        q, k, v = (t.reshape(M, H, C // H).transpose(0, 1).contiguous() for t in (x @ s["qkv_w"]).split(C, -1))

        def rows(t):
            return t.transpose(0, 1).reshape(M, C)

        def cols(t):
            return t.transpose(1, 2).contiguous()

        mask = torch.full((M, M), float("-inf"), device="cuda", dtype=torch.float64).triu(1)
        p = torch.softmax(q @ cols(k) * scale + mask, -1)
        y, dy = rows(p @ v), s["dy"]
        dyh = (dy @ s["proj_w"]).reshape(M, H, C // H).transpose(0, 1).contiguous()
        da = dyh @ cols(v)
        ds = p * (da - (da * p).sum(-1, keepdim=True)) * scale
        dqkv = torch.cat([rows(ds @ k), rows(cols(ds) @ q), rows(cols(p) @ dyh)], -1)
        return {"out": y @ s["proj_w"].t(), "dproj": dy.t() @ y, "dqkv_w": x.t() @ dqkv, "dx": dqkv @ s["qkv_w"].t()}
    idx, target = s["idx"].long(), s["target"].long()
    xin = x + s["tok"][idx]
    xn = _ln(xin, s["g"])
    z = xn @ s["tok"].t()
    ok = (target >= 0).double()[:, None]
    onehot = torch.zeros_like(z).scatter_(1, target.clamp(min=0)[:, None], 1.0)
    dz = (onehot - torch.softmax(z, -1)) * ok / ok.sum()
    loss = ((torch.logsumexp(z, -1) - z.gather(1, target.clamp(min=0)[:, None])[:, 0]) * ok[:, 0]).sum() / ok.sum()
    dx, dg = _ln_backward(xin, s["g"], dz @ s["tok"])
    return {"logits": z, "loss": loss.reshape(1), "dtok": (dz.t() @ xn).index_add(0, idx, dx), "dg": dg, "dx": dx}
