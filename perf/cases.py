"""Timing cases of the sparse-autoencoder path: what a program that uses saeflow_amd has it do.

A case is a plain dict: `call` names the entry points that a pass goes through, the rest its
sizes and options. The calls:

  forward    encode_sparse then decode_sparse, as an analysis or steering loop runs a dictionary
             over the tokens it has: interactive single tokens, prompts, full batches.
  features   fused_encode with row counts, dense_to_csr, decode_sparse: a program that works on
             the dense features and on their sparse form.
  encode     ops.encode: dense features alone (for TopK the select and the scatter as well).
  decode     decode_sparse of stored CSR features (an activation cache read back).
  edit       SAE.decode of dense features that the program has changed itself (an ablation), so
             that no row counts are at hand.
  train      forward_train, a reconstruction loss with an L1 penalty, and the gradients of all
             parameters.

The arrays of relu and jumprelu CSR features are as long as the inputs make them, so a pass gives
back their row pointers and, in their place, the reconstruction that every entry of them goes into.

Ranges: 1 to 16384 tokens; d_in 64 to 4096; dictionaries of 1024 to 2^20 features, whole 256-feature
tiles, multiples of 8 and odd ones; fp32, bf16 and fp16; relu, jumprelu and topk.

Weights and tokens follow the recipe of saeflow_amd.workloads: W_enc ~ N(0, 1/d_in), W_dec its
transpose with unit rows, x = b_dec + N(0, 1), so that pre-activations are about N(0, 1); jumprelu
thresholds from log-normal firing frequencies that add up to L0 = 64, relu biases that give the same
mean L0, TopK biases that leave about ten times k positive features a token.
"""

import math
from types import SimpleNamespace

import torch

import saeflow_amd
from saeflow_amd.kernels import dense_to_csr, fused_encode
from saeflow_amd.training import forward_train

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
L0 = 64
LAMBDA = 1e-2        # weight of the L1 penalty of a training step
MOST_FLOPS = 5e12    # of a drawn case: the headline forward
DEVICE = "cuda"


def _case(name, call, activation, dtype, tokens, d_in, d_sae, k=0):
    return {"name": name, "call": call, "activation": activation, "dtype": dtype, "tokens": tokens, "d_in": d_in,
            "d_sae": d_sae, "k": k}


def listed():
    return [
        # one token at a time: interactive inspection, or steering inside a generation loop
        _case("token", "forward", "jumprelu", "bf16", 1, 2304, 16384),
        # one prompt of ordinary length over the headline dictionary
        _case("prompt", "forward", "jumprelu", "bf16", 137, 2304, 65536),
        # the headline batch
        _case("batch", "forward", "jumprelu", "bf16", 16384, 2304, 65536),
        # a few sequences over the largest dictionary (2^20 features)
        _case("wide", "forward", "jumprelu", "bf16", 512, 2304, 1048576),
        # fp32 analysis of a small model's activations: dense features, their CSR, the reconstruction
        _case("small-fp32", "features", "relu", "fp32", 2048, 768, 24576),
        # sizes that fit no tile and no vector: 1000 tokens, an odd dictionary
        _case("odd", "encode", "relu", "bf16", 1000, 1000, 10007),
        # TopK over a wide model and a large dictionary
        _case("topk", "forward", "topk", "fp16", 8192, 4096, 131072, 32),
        # TopK of a small model, dense features wanted
        _case("topk-small", "encode", "topk", "fp32", 300, 768, 12288, 48),
        # stored features read back
        _case("cache-decode", "decode", "jumprelu", "bf16", 4096, 2304, 65536),
        # dense features, edited, decoded
        _case("edit", "edit", "jumprelu", "bf16", 2048, 2304, 16384),
        # one training step of a 16k dictionary
        _case("train", "train", "jumprelu", "bf16", 4096, 2304, 16384),
        # one training step of a small fp32 dictionary
        _case("train-fp32", "train", "relu", "fp32", 777, 768, 8192),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["forward", "forward", "forward", "features", "encode", "decode", "edit", "train"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if call == "train":
        dtype = rng.choice(["bf16", "fp32"])  # fp16 gradients would need a loss scale
    activation = rng.choice(["jumprelu", "jumprelu", "relu", "topk"]) if call in ("forward", "encode", "train") else \
        rng.choice(["jumprelu", "relu"])
    d_in = rng.choice([768, 1024, 2304, 4096, 8 * _log(rng, 8, 512), _log(rng, 64, 4096)])
    d_sae = _log(rng, 1024, 131072 if rng.random() < 0.9 or dtype == "fp32" else 1048576)
    d_sae = {0: d_sae, 1: -(-d_sae // 8) * 8}.get(rng.randrange(4), -(-d_sae // 256) * 256)
    tokens = _log(rng, 1, 16384)
    # fp32 runs at a sixteenth of the 16-bit rate, a training step moves several times the weights,
    # and dense features are bounded to those of the headline batch
    most = MOST_FLOPS * (1 / 16 if dtype == "fp32" else 1) * (1 / 5 if call == "train" else 1)
    tokens = max(1, min(tokens, int(most / (2 * d_in * d_sae)), (1 << 30) // d_sae))
    return {"call": call, "activation": activation, "dtype": dtype, "tokens": tokens, "d_in": d_in, "d_sae": d_sae,
            "k": rng.choice([16, 32, 48, 64]) if activation == "topk" else 0}


# ----------------------------------------------------------------------------- inputs
def _frequencies(d_sae, g):
    """Firing probabilities ~ LogNormal(0, 1.5), scaled to sum to L0, at most one half each."""
    p = torch.exp(1.5 * torch.randn(d_sae, generator=g, device=DEVICE, dtype=torch.float64))
    for _ in range(6):
        p = (p * (L0 / p.sum())).clamp(max=0.5)
    return p


def _sae(case, g):
    """The weights, as the attributes that the entry points read."""
    d_in, d_sae, dtype = case["d_in"], case["d_sae"], DTYPES[case["dtype"]]
    W_enc = torch.randn(d_in, d_sae, generator=g, device=DEVICE) / math.sqrt(d_in)
    b_dec = torch.randn(d_in, generator=g, device=DEVICE) * 0.1
    p = _frequencies(d_sae, g)
    threshold = torch.special.ndtri(1.0 - p).to(dtype) if case["activation"] == "jumprelu" else None
    positive = {"relu": L0, "topk": 10 * case["k"], "jumprelu": d_sae / 2}[case["activation"]]
    b_enc = torch.full((d_sae,), -float(torch.special.ndtri(torch.tensor(1.0 - min(0.5, positive / d_sae)))), device=DEVICE)
    W_dec = W_enc.T / W_enc.norm(dim=0)[:, None]
    return SimpleNamespace(W_enc=W_enc.to(dtype), W_dec=W_dec.contiguous().to(dtype), b_enc=b_enc.to(dtype),
                           b_dec=b_dec.to(dtype), threshold=threshold, activation=case["activation"],
                           k=case["k"] or None), p


def _features(case, p, g):
    """(rows, columns, values) of sparse features with the firing probabilities p, in row order."""
    rows, cols = [], []
    step = max(1, (1 << 28) // case["d_sae"])
    pf = p.float()
    for r in range(0, case["tokens"], step):
        n = min(step, case["tokens"] - r)
        at = (torch.rand(n, case["d_sae"], generator=g, device=DEVICE) < pf).nonzero()
        rows.append(at[:, 0] + r)
        cols.append(at[:, 1])
    rows, cols = torch.cat(rows), torch.cat(cols)
    values = 1.5 + torch.rand(rows.numel(), generator=g, device=DEVICE) * 2
    return rows, cols, values.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    sae, p = _sae(case, g)
    state = {"case": case, "sae": sae}
    dtype, T = DTYPES[case["dtype"]], case["tokens"]
    if case["call"] in ("decode", "edit"):
        rows, cols, values = _features(case, p, g)
        if case["call"] == "decode":
            counts = torch.bincount(rows, minlength=T)
            indptr = torch.zeros(T + 1, dtype=torch.int64, device=DEVICE)
            indptr[1:] = torch.cumsum(counts, 0)
            state["csr"] = (indptr, cols.int(), values)
        else:
            state["f"] = torch.zeros(T, case["d_sae"], dtype=dtype, device=DEVICE)
            state["f"][rows, cols] = values
            module = saeflow_amd.SAE(1, 1, "relu", device=DEVICE, dtype=dtype)
            module.W_dec, module.b_dec = torch.nn.Parameter(sae.W_dec, False), torch.nn.Parameter(sae.b_dec, False)
            state["module"] = module
        return state
    state["x"] = (sae.b_dec.float() + torch.randn(T, case["d_in"], generator=g, device=DEVICE)).to(dtype)
    if case["call"] == "train":
        for name in ("W_enc", "b_enc", "W_dec", "b_dec"):
            getattr(sae, name).requires_grad_(True)
    return state


# ----------------------------------------------------------------------------- one pass
def run(state):
    case, sae = state["case"], state["sae"]
    call = case["call"]
    if call == "forward":
        csr = saeflow_amd.encode_sparse(sae, state["x"])
        x_hat = saeflow_amd.decode_sparse(sae, csr)
        return csr + (x_hat,) if case["activation"] == "topk" else (csr[0], x_hat)
    if call == "features":
        row_nnz = torch.zeros(case["tokens"], dtype=torch.int32, device=state["x"].device)
        f = fused_encode(state["x"], sae.W_enc, sae.b_enc, sae.b_dec, sae.threshold, sae.activation, row_nnz=row_nnz)
        csr = dense_to_csr(f, row_nnz)
        return f, csr[0], saeflow_amd.decode_sparse(sae, csr)
    if call == "encode":
        return saeflow_amd.encode(sae, state["x"])
    if call == "decode":
        return saeflow_amd.decode_sparse(sae, state["csr"])
    if call == "edit":
        return state["module"].decode(state["f"])
    x = state["x"]
    x_hat, (_, _, values) = forward_train(sae, x)
    loss = (x_hat.float() - x.float()).pow(2).sum(-1).mean() + LAMBDA * values.float().abs().sum() / len(x)
    grads = torch.autograd.grad(loss, (sae.W_enc, sae.b_enc, sae.W_dec, sae.b_dec))
    return (x_hat.detach(),) + grads


# ----------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    T, D, N, e = case["tokens"], case["d_in"], case["d_sae"], DTYPES[case["dtype"]].itemsize
    nnz = T * min(case["k"] or L0, N)
    weights, tokens, csr = N * D * e + (2 * N + D) * e, T * D * e, nnz * (4 + e) + (T + 1) * 8
    used = N * (1 - math.exp(-nnz / N)) * D * e  # W_dec rows that some token uses
    encode, gather = 2 * T * D * N, 2 * nnz * D
    return {
        "forward": {"bytes": tokens + weights + csr + used + tokens, "flops": encode + gather},
        "features": {"bytes": tokens + weights + T * N * e + csr + used + tokens, "flops": encode + gather},
        "encode": {"bytes": tokens + weights + T * N * e, "flops": encode},
        "decode": {"bytes": csr + used + tokens, "flops": gather},
        "edit": {"bytes": T * N * e + used + tokens, "flops": gather},
        # weights read and their gradients written; x, x_hat out, its gradient in and out
        "train": {"bytes": 4 * N * D * e + 4 * tokens + 2 * csr, "flops": encode + 4 * gather},
    }[case["call"]]


def tolerance(case):
    """Four times the measured distance from the 64-bit results: that of the storage type's last
    rounding (1.7e-3 in bf16, 2.0e-4 in fp16) or, in fp32, of sums in another order (up to 2.8e-6).
    Gradients pass a second stored tensor (dL/dx_hat): twice that."""
    rel = {"fp32": 1.1e-5, "bf16": 7e-3, "fp16": 8e-4}[case["dtype"]]
    return {"rel": rel * (2 if case["call"] == "train" else 1)}


# ----------------------------------------------------------------------------- 64-bit results
def _chunks(case):
    step = max(1, (1 << 28) // case["d_sae"])
    return [(r, min(r + step, case["tokens"])) for r in range(0, case["tokens"], step)]


def _dense64(case, sae, W, xs):
    """64-bit features of the shifted tokens xs (stored in the weights' type by definition)."""
    f = xs.double() @ W + sae.b_enc.double()
    if case["activation"] == "jumprelu":
        return torch.where(f > sae.threshold.double(), f, 0.0).clamp(min=0.0)
    return f.clamp(min=0.0)


def _kept(case, f):
    """f with all but each row's k largest values zeroed (TopK), and those values in falling order."""
    if case["activation"] != "topk":
        return f, None
    v, i = f.topk(case["k"], dim=-1)
    return torch.zeros_like(f).scatter_(-1, i, v), v


@torch.no_grad()
def exact(case, seed):
    state = prepare(case, seed)
    sae, call, dtype = state["sae"], case["call"], DTYPES[case["dtype"]]
    stored = lambda t: t.to(dtype).double()  # noqa: E731  (a stage's result as the next stage reads it)
    W_dec, b_dec = sae.W_dec.double(), sae.b_dec.double()
    if call == "decode":
        indptr, cols, values = state["csr"]
        out = []
        for lo, hi in _chunks(case):
            a, b = int(indptr[lo]), int(indptr[hi])
            f = torch.zeros(hi - lo, case["d_sae"], dtype=torch.float64, device=DEVICE)
            rows = torch.repeat_interleave(torch.arange(hi - lo, device=DEVICE), indptr[lo + 1:hi + 1] - indptr[lo:hi])
            f[rows, cols[a:b].long()] = values[a:b].double()
            out.append(f @ W_dec + b_dec)
        return torch.cat(out)
    if call == "edit":
        return torch.cat([state["f"][lo:hi].double() @ W_dec + b_dec for lo, hi in _chunks(case)])
    x, W_enc = state["x"], sae.W_enc.double()
    xs = (x.float() - sae.b_dec.float()).to(dtype)
    if call in ("features", "encode"):
        f = torch.cat([_kept(case, _dense64(case, sae, W_enc, xs[lo:hi]))[0] for lo, hi in _chunks(case)])
        if call == "encode":
            return f
        x_hat = torch.cat([stored(f[lo:hi]) @ W_dec + b_dec for lo, hi in _chunks(case)])
        return f, None, x_hat  # (a feature within a rounding of its cut may be counted or not)
    if call == "forward":
        x_hat, tops = [], []
        for lo, hi in _chunks(case):
            f, top = _kept(case, _dense64(case, sae, W_enc, xs[lo:hi]))
            x_hat.append(stored(f) @ W_dec + b_dec)
            tops.append(top)
        # features within a rounding of their cut come and go; TopK's sorted values have one 64-bit result
        x_hat = torch.cat(x_hat)
        return (None, x_hat) if tops[0] is None else (None, None, torch.cat(tops).flatten(), x_hat)
    T = case["tokens"]
    x_hat, d_wenc, d_wdec = [], torch.zeros_like(W_enc), torch.zeros_like(W_dec)
    d_benc, d_bdec = torch.zeros(case["d_sae"], dtype=torch.float64, device=DEVICE), torch.zeros_like(b_dec)
    g_values = stored(torch.tensor(LAMBDA / T, device=DEVICE))
    for lo, hi in _chunks(case):
        f = stored(_kept(case, _dense64(case, sae, W_enc, xs[lo:hi]))[0])
        out = f @ W_dec + b_dec
        x_hat.append(out)
        g = stored((stored(out) - x[lo:hi].double()) * (2.0 / T))
        g_pre = torch.where(f != 0, g @ W_dec.T + g_values, 0.0)
        d_wdec += f.T @ g
        d_wenc += xs[lo:hi].double().T @ g_pre
        d_benc += g_pre.sum(0)
        d_bdec += g.sum(0) - W_enc @ g_pre.sum(0)
    return torch.cat(x_hat), d_wenc, d_benc, d_wdec, d_bdec
