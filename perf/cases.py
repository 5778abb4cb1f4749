"""The measured workloads of the draft-token selection path.

Each case is one call that a speculative-decoding server makes on every draft
block: a single selection step (``lowrank_argmax`` and its e4m3 form), a whole
suffix rollout (``DeLSGraphRunner``, ``MarkovDeLSGraphRunner``,
``DraftCorrectionGraphRunner``), a whole draft block (``DeLSDraftStep``), the
target LM head alone (``lm_head``) and temperature sampling (``sample_rows``).
Shapes are those of the two Qwen3 heads that the benchmark uses (hidden size
2560 with rank 256, 4096 with rank 512; vocabulary 151936) and of the local
head of its draft-block workload (embedding, hidden and correction width 1024,
rank 256, 14 steps); the batch is the number of sequences that one GPU serves
at once.  ``draw`` gives other members of the same families.
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

from __graft_entry__ import load_package

pkg = load_package()

DEV = "cuda:0"
VOCAB = 151936
HEADS = ((2560, 256), (4096, 512))     # (hidden size, rank) of the measured heads
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def listed():
    return [
        # one sequence, one draft position: the smallest call, where latency counts
        dict(name="step_m1", kind="step", M=1, d=2560, r=256, V=VOCAB, base="float32", act="identity", packed=True),
        # the headline step: one block of 16 positions, fp32 base logits
        dict(name="step_m16", kind="step", M=16, d=4096, r=512, V=VOCAB, base="float32", act="identity", packed=True),
        # 40 sequences decoded together, in the runtime's dtype
        dict(name="step_m40", kind="step", M=40, d=4096, r=512, V=VOCAB, base="bfloat16", act="silu", packed=True),
        # a large batch: 32 sequences x 16 positions
        dict(name="step_m512", kind="step", M=512, d=4096, r=512, V=VOCAB, base="bfloat16", act="identity",
             packed=True),
        # e4m3 weights, 8 sequences x 15 positions
        dict(name="step8_m120", kind="step8", M=120, d=4096, r=512, V=VOCAB, base="bfloat16", act="identity"),
        # greedy suffix rollout of a block of 16, batch 8, through the runner's own call
        dict(name="rollout_b8", kind="rollout", B=8, S=14, G=1024, r=256, V=VOCAB),
        # the same for a batch past one MFMA tile of rows
        dict(name="rollout_b24", kind="rollout", B=24, S=14, G=1024, r=256, V=VOCAB),
        # the Markov local head (rank gathered from a table), batch 4
        dict(name="markov_b4", kind="markov", B=4, S=14, r=256, V=VOCAB),
        # the Domino correction of a single sequence
        dict(name="domino_b1", kind="domino", B=1, S=14, P=2, D=4096, G=1024, E=1024, V=VOCAB),
        # a whole draft block of 8 sequences: target LM head, first ids and the rollout
        dict(name="block_b8", kind="block", B=8, k=15, d=4096, G=1024, r=256, V=VOCAB),
        # the target LM head of three sequences' blocks
        dict(name="lm_head_m45", kind="lm_head", M=45, d=4096, V=VOCAB),
        # temperature sampling of 8 blocks' logits
        dict(name="sample_m120", kind="sample", M=120, V=VOCAB, dtype="bfloat16", T=0.7),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "step8", "rollout", "markov", "domino", "block", "lm_head", "sample"))
    # a padded vocabulary (a multiple of 64) mostly, else any size
    V = _log_int(rng, 32000, VOCAB)
    if rng.random() < 0.75:
        V = V // 64 * 64
    if kind in ("step", "step8"):
        d, r = rng.choice(HEADS)
        c = dict(kind=kind, M=_log_int(rng, 1, 512), d=d, r=r, V=V,
                 base=rng.choice(("float32", "bfloat16", "bfloat16", "float16")), act=rng.choice(("identity", "silu")))
        if kind == "step":
            c["packed"] = rng.random() < 0.8
        return c
    if kind == "rollout":
        return dict(kind=kind, B=_log_int(rng, 1, 32), S=rng.randint(4, 15), G=1024, r=rng.choice((256, 256, 512)), V=V)
    if kind == "markov":
        return dict(kind=kind, B=_log_int(rng, 1, 32), S=rng.randint(4, 15), r=rng.choice((128, 256)), V=V)
    if kind == "domino":
        return dict(kind=kind, B=_log_int(rng, 1, 8), S=rng.randint(4, 14), P=rng.randint(1, 3), D=rng.choice((2560, 4096)),
                    G=1024, E=rng.choice((512, 1024)), V=V)
    if kind == "block":
        return dict(kind=kind, B=_log_int(rng, 1, 8), k=rng.choice((8, 15)), d=rng.choice((2560, 4096)), G=1024, r=256, V=V)
    if kind == "lm_head":
        return dict(kind=kind, M=_log_int(rng, 1, 240), d=rng.choice((2560, 4096)), V=V)
    return dict(kind=kind, M=_log_int(rng, 1, 240), V=V, dtype=rng.choice(("float32", "bfloat16", "float16")),
                T=rng.choice((0.6, 0.7, 1.0)))


# ---- inputs (from the seed alone, drawn on the GPU) ---------------------------------


class _Inputs:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        # in pieces of whole rows, so that a large weight needs no large fp32 copy
        out = torch.empty(*shape, dtype=dtype, device=DEV)
        rows = max(1, (1 << 27) // max(1, out[0].numel())) if out.dim() > 1 else out.numel()
        for i in range(0, out.shape[0], rows):
            part = out[i:i + rows]
            part.copy_(torch.randn(part.shape, generator=self.g, device=DEV) * std)
        return out

    def uniform(self, n, hi):
        return torch.rand(n, generator=self.g, device=DEV) * hi

    def ids(self, *shape, high):
        return torch.randint(0, high, shape, generator=self.g, device=DEV)

    def log_prior(self, V, dtype):
        """Log-probabilities of Zipf(1.1) counts, smoothed by one, over permuted ids."""
        k = torch.arange(1, V + 1, dtype=torch.float64, device=DEV)
        counts = torch.round(1e9 * k.pow(-1.1)) + 1.0
        perm = torch.randperm(V, generator=self.g, device=DEV)
        return torch.log(counts / counts.sum())[perm].to(dtype)

    def schedules(self, n):
        """Per-position weights of the correction and of the prior."""
        return self.uniform(n, 0.6), self.uniform(n, 0.6)


def _quantise(W):
    """Per-row absmax e4m3: bytes and fp32 scales."""
    w = W.float()
    scale = w.abs().amax(dim=1) / 448.0
    return (w / scale[:, None]).to(torch.float8_e4m3fn), scale


def _make_step(c, seed):
    x = _Inputs(seed)
    M, d, r, V, dt = c["M"], c["d"], c["r"], c["V"], DTYPES[c["base"]]
    s = dict(h=x.normal(M, d), A=x.normal(r, d, std=0.02), B=x.normal(V, r, std=0.02),
             base=x.normal(M, V, std=3.0, dtype=dt), prior=x.log_prior(V, dt))
    a, b = x.schedules(16)
    rows = torch.arange(M, device=DEV) % 16
    s["alpha"], s["beta"] = a[rows].contiguous(), b[rows].contiguous()
    return s


class _Head(nn.Module):
    """A local head as the DeLS runner reads it: embedding, one GRU layer, rank projection, low-rank LM head."""

    def __init__(self, x, V, G, r):
        super().__init__()
        kw = dict(device=DEV, dtype=torch.bfloat16)
        self.embed_tokens = nn.Embedding(V, G, _weight=x.normal(V, G))
        self.prefix_gru = nn.GRU(G, G, num_layers=1, batch_first=True, bias=False, **kw)
        self.rank_proj = nn.Linear(G, r, bias=False, **kw)
        self.low_rank_lm_head = nn.Linear(r, V, bias=False, **kw)
        self.rank_activation = "silu"
        with torch.no_grad():
            for p in (self.prefix_gru.weight_ih_l0, self.prefix_gru.weight_hh_l0, self.rank_proj.weight,
                      self.low_rank_lm_head.weight):
                p.copy_(x.normal(*p.shape, std=0.02 if p is not self.rank_proj.weight else 0.05))


class _MarkovHead(nn.Module):
    def __init__(self, x, V, r):
        super().__init__()
        self.embedding_weight = nn.Parameter(x.normal(V, r), requires_grad=False)
        self.lm_head_weight = nn.Parameter(x.normal(V, r, std=0.05), requires_grad=False)
        self.vocab_size, self.rank = V, r


class _Draft(nn.Module):
    def __init__(self, x, D, G, E, V):
        super().__init__()
        kw = dict(device=DEV, dtype=torch.bfloat16)
        self.embed_proj = nn.Sequential(nn.Linear(D + G, E, bias=False, **kw), nn.SiLU(),
                                        nn.Linear(E, V, bias=False, **kw))
        self.prefix_gru = nn.GRU(D, G, num_layers=1, batch_first=True, bias=False, **kw)
        with torch.no_grad():
            for p in self.parameters():
                p.copy_(x.normal(*p.shape, std=0.02))


class _Target(nn.Module):
    def __init__(self, x, V, D):
        super().__init__()
        self.model = nn.Module()
        self.model.embed_tokens = nn.Embedding(V, D, _weight=x.normal(V, D))


def _block_hiddens(x, W, B, k, d):
    """Hidden states with a leaning to one token each, from none to clear, as a drafter's have."""
    h = x.normal(B, k, d, dtype=torch.float32)
    w = W[x.ids(B, k, high=W.shape[0])].float()
    lean = x.uniform(B * k, 8.0).view(B, k, 1)
    return (h + lean * w / w.norm(dim=-1, keepdim=True)).to(torch.bfloat16)


def _make(c, seed):
    """The inputs of a case, as plain tensors and modules."""
    kind = c["kind"]
    if kind in ("step", "step8"):
        return _make_step(c, seed)
    x, V = _Inputs(seed), c["V"]
    if kind == "sample":
        return dict(logits=x.normal(c["M"], V, std=3.0, dtype=DTYPES[c["dtype"]]), seed=int(seed) * 2654435761 % 2**63)
    if kind == "lm_head":
        return dict(W=x.normal(V, c["d"], std=0.02), hidden=x.normal(c["M"], c["d"]))
    if kind == "domino":
        B, S, D = c["B"], c["S"], c["D"]
        return dict(draft=_Draft(x, D, c["G"], c["E"], V), target=_Target(x, V, D), prefix=x.ids(B, c["P"], high=V),
                    hiddens=x.normal(B, S, D), base=x.normal(B, S, V, std=3.0))
    B = c["B"]
    S = c["k"] - 1 if kind == "block" else c["S"]
    alpha, beta = x.schedules(S)
    s = dict(alpha=alpha.tolist(), beta=beta.tolist(), prior=x.log_prior(V, torch.bfloat16))
    s["head"] = _MarkovHead(x, V, c["r"]) if kind == "markov" else _Head(x, V, c["G"], c["r"])
    if kind == "block":
        s["W"] = x.normal(V, c["d"], std=0.02)
        s["hiddens"] = _block_hiddens(x, s["W"], B, c["k"], c["d"])
    else:
        s["prefix"] = x.ids(B, 1, high=V)
        s["base"] = x.normal(B, S, V, std=3.0)
    return s


def prepare(case, seed):
    c, s = case, _make(case, seed)
    kind = c["kind"]
    if kind == "step":
        if c["packed"]:
            s["A"], s["B"] = pkg.pack_operand(s["A"]), pkg.pack_operand(s["B"])
        s["act"] = c["act"]
    elif kind == "step8":
        s["A"] = pkg.pack_operand_fp8(*_quantise(s["A"]), "k32")
        s["B"] = pkg.pack_operand_fp8(*_quantise(s["B"]), "k128")
        s["act"] = c["act"]
    elif kind in ("rollout", "markov"):
        cls = pkg.DeLSGraphRunner if kind == "rollout" else pkg.MarkovDeLSGraphRunner
        s["runner"] = cls(local_head=s.pop("head"), batch_size=c["B"], steps=c["S"], vocab_size=c["V"],
                          alpha_values=s["alpha"], beta_values=s["beta"], baseline_logits=s["prior"], device=DEV)
    elif kind == "domino":
        s["runner"] = pkg.DraftCorrectionGraphRunner(
            draft_model=s.pop("draft"), target_model=s.pop("target"), batch_size=c["B"], steps=c["S"],
            hidden_dim=c["D"], gru_hidden_dim=c["G"], vocab_size=c["V"], prefix_token_count=c["P"], device=DEV,
            guidance_alpha=0.8)
    elif kind == "block":
        s["step"] = pkg.DeLSDraftStep(local_head=s.pop("head"), lm_head_weight=s.pop("W"), batch_size=c["B"],
                                      k_draft=c["k"], vocab_size=c["V"], alpha_values=s["alpha"],
                                      beta_values=s["beta"], baseline_logits=s["prior"], device=DEV)
    elif kind == "lm_head":
        s["W"] = pkg.pack_lm_head(s["W"])
    elif kind == "sample":
        s["T"] = c["T"]
    s["kind"] = kind
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        return pkg.lowrank_argmax(s["h"], s["A"], s["B"], s["base"], s["prior"], s["alpha"], s["beta"], act=s["act"])
    if kind == "step8":
        return pkg.lowrank_argmax_fp8(s["h"], s["A"], s["B"], s["base"], s["prior"], s["alpha"], s["beta"],
                                      act=s["act"])
    if kind in ("rollout", "markov"):
        return s["runner"](s["prefix"], s["base"]), s["runner"].static_scores
    if kind == "domino":
        return s["runner"](s["prefix"], s["hiddens"], s["base"]), s["runner"].static_scores
    if kind == "block":
        # the ids, their scores, and the base logits of positions 1 .. k-1 (position 0's are argmaxed, not kept)
        return s["step"](s["hiddens"]), s["step"].static_scores, s["step"].static_base[:, 1:]
    if kind == "lm_head":
        return pkg.lm_head(s["hidden"], s["W"])[0]
    return pkg.sample_rows(s["logits"], s["T"], s["seed"])


def work(case):
    """Every input read once and every output written once; each weight once, though a rollout uses it every step."""
    c, kind, V = case, case["kind"], case["V"]
    if kind in ("step", "step8"):
        M, d, r = c["M"], c["d"], c["r"]
        eb = 4 if c["base"] == "float32" else 2
        wb = r * d + V * r
        wb = 2 * wb if kind == "step" else wb + 4 * (r + V)
        return dict(bytes=wb + M * d * 2 + M * V * eb + V * eb + M * 20, flops=2 * M * r * (d + V))
    if kind == "sample":
        eb = 4 if c["dtype"] == "float32" else 2
        return dict(bytes=c["M"] * V * eb + 12 * c["M"], flops=0)
    if kind == "lm_head":
        M, d = c["M"], c["d"]
        return dict(bytes=2 * (V * d + M * d + M * V), flops=2 * M * V * d)
    B = c["B"]
    if kind == "domino":
        S, P, D, G, E = c["S"], c["P"], c["D"], c["G"], c["E"]
        weights = 3 * G * G + E * (D + G) + V * E
        rows = B * (P + S - 1)
        flops = 2 * B * S * E * (D + G + V) + 2 * rows * 3 * G * G
        return dict(bytes=2 * (weights + rows * 3 * G + B * S * (D + V)) + B * S * 12, flops=flops)
    if kind == "markov":
        S, r = c["S"], c["r"]
        return dict(bytes=2 * (V * r + B * S * r + V + B * S * V) + B * S * 12, flops=2 * B * S * r * V)
    S = c["k"] - 1 if kind == "block" else c["S"]
    G, r = c["G"], c["r"]
    weights = 3 * G * G + r * G + V * r
    nbytes = 2 * (weights + B * S * 3 * G + V + B * S * V) + B * S * 12
    flops = 2 * B * S * (3 * G * G + r * G + r * V)
    if kind == "block":      # the base logits are written for the caller, and need not be read back
        k, d = c["k"], c["d"]
        nbytes += 2 * (V * d + B * k * d) + B * 12
        flops += 2 * B * k * d * V
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind == "lm_head":
        # one bf16 rounding of an fp32 sum: another order of the sum moves a few values by one place
        return {"rel": 1e-3, "max": 0.02}
    if kind == "sample":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}
    if kind == "step8":
        # a bf16 rank value that rounds the other way can move its e4m3 value by one place
        return {"rel": 1e-4, "max": 1e-3, "differ": 0.01}
    if kind == "block":
        # the bf16 base logits
        return {"rel": 1e-3, "max": 0.02, "differ": 0.01}
    if kind in ("rollout", "markov", "domino"):
        # bf16 states: a value that rounds the other way travels through the steps that follow
        return {"rel": 3e-5, "max": 1e-3, "differ": 0.01}
    # a bf16 rank value that rounds the other way moves the scores by a few parts in 1e6
    return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}


# ---- the same results in 64 bits, in plain torch -----------------------------------
# Values that the path holds in bf16 (rank, GRU states, the correction's parts, base
# logits) are rounded to bf16 where it rounds them, from 64-bit sums.


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _act(x, act):
    return x * torch.sigmoid(x) if act == "silu" else x


def _by_vocab(left, W, finish, columns=1 << 14):
    """(max, lowest argmax) of ``finish(left . W^T, columns)`` over the rows of W, in pieces."""
    best = ids = None
    for v in range(0, W.shape[0], columns):
        part = finish(left @ W[v:v + columns].double().t(), slice(v, v + columns))
        val, at = part.max(dim=1)
        at = at + v
        if best is None:
            best, ids = val, at
        else:
            ids = torch.where(val > best, at, ids)
            best = torch.maximum(val, best)
    return best, ids


def _combine(alpha, beta, base, prior):
    """score = dot * alpha + base - beta * prior, for a slice of the vocabulary."""
    return lambda dot, cols: (dot * alpha + base[:, cols].double()) - beta * prior[cols].double()


def _exact_step(c, s):
    h, fp8 = s["h"].double(), c["kind"] == "step8"
    if fp8:
        (qa, sa), (qb, sb) = _quantise(s["A"]), _quantise(s["B"])
        rank = _bf16(_act(_bf16((h @ qa.double().t()) * sa.double()), c["act"]))
        amax = rank.abs().amax(dim=1, keepdim=True).float()
        rank = (rank.float() * (448.0 / amax)).to(torch.float8_e4m3fn).double() * (amax / 448.0).double()
        W = qb.float()
    else:
        rank = _bf16(_act(_bf16(h @ s["A"].double().t()), c["act"]))
        W, sb = s["B"], None
    comb = _combine(s["alpha"].double()[:, None], s["beta"].double()[:, None], s["base"], s["prior"])
    fin = comb if sb is None else (lambda dot, cols: comb(dot * sb[cols].double(), cols))
    best, ids = _by_vocab(rank, W, fin)
    return ids, best


def _gru(gi, h, w_hh, G):
    """One GRU cell on bf16 gate sums; h None is the zero state."""
    gh = _bf16(h @ w_hh.double().t()) if h is not None else torch.zeros_like(gi)
    ir, iz, inn = gi.split(G, dim=1)
    hr, hz, hn = gh.split(G, dim=1)
    r, z = torch.sigmoid(ir + hr), torch.sigmoid(iz + hz)
    n = torch.tanh(inn + r * hn)
    return _bf16((1 - z) * n + (z * h if h is not None else 0.0))


def _gi(embed, w_ih, ids):
    """The bf16 input projection of the ids' embeddings."""
    return _bf16(embed[ids].double() @ w_ih.double().t())


def _exact_rollout(c, s, base, prefix):
    head, B, S = s["head"], c["B"], base.shape[1]
    ids, h, scores = prefix, None, []
    for t in range(S):
        if c["kind"] == "markov":
            rank = head.embedding_weight[ids].double()
            W = head.lm_head_weight
        else:
            gru = head.prefix_gru
            h = _gru(_gi(head.embed_tokens.weight, gru.weight_ih_l0, ids), h, gru.weight_hh_l0, c["G"])
            rank = _bf16(_act(_bf16(h @ head.rank_proj.weight.double().t()), "silu"))
            W = head.low_rank_lm_head.weight
        best, ids = _by_vocab(rank, W, _combine(s["alpha"][t], s["beta"][t], base[:, t], s["prior"]))
        scores.append(best)
    return torch.stack(scores, dim=1)


def _exact_domino(c, s):
    draft, D, G, base = s["draft"], c["D"], c["G"], s["base"]
    w1, w2 = draft.embed_proj[0].weight, draft.embed_proj[2].weight
    gru, embed = draft.prefix_gru, s["target"].model.embed_tokens.weight
    z = _bf16(s["hiddens"].double() @ w1[:, :D].double().t())
    h = None
    for p in range(c["P"]):
        h = _gru(_gi(embed, gru.weight_ih_l0, s["prefix"][:, p]), h, gru.weight_hh_l0, G)
    scores = []
    for t in range(c["S"]):
        mid = _act(z[:, t] + _bf16(h @ w1[:, D:].double().t()), "silu")
        best, ids = _by_vocab(mid, w2, lambda dot, cols: dot * 0.8 + base[:, t, cols].double())
        scores.append(best)
        h = _gru(_gi(embed, gru.weight_ih_l0, ids), h, gru.weight_hh_l0, G)
    return torch.stack(scores, dim=1)


def _philox_bits(M, V, seed):
    """Word v % 4 of Philox4x32-10 at counter (v / 4, m, 0, 0), as int64 [M, V]."""
    mask = 0xFFFFFFFF
    n4 = (V + 3) // 4
    x = [torch.arange(n4, device=DEV)[None, :].expand(M, n4), torch.arange(M, device=DEV)[:, None].expand(M, n4),
         torch.zeros(M, n4, dtype=torch.int64, device=DEV), torch.zeros(M, n4, dtype=torch.int64, device=DEV)]
    k0, k1 = seed & mask, seed >> 32

    def mul(a, k):        # high and low words of a 32 x 32 bit product
        p = a * k
        return (p >> 32) & mask, p & mask

    for _ in range(10):
        h0, l0 = mul(x[0], 0xD2511F53)
        h1, l1 = mul(x[2], 0xCD9E8D57)
        x = [h1 ^ x[1] ^ k0, l1, h0 ^ x[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return torch.stack(x, dim=2).reshape(M, 4 * n4)[:, :V]


def _exact_sample(c, s):
    x = s["logits"]
    y = (x.float() / c["T"]).to(x.dtype).double()
    u = ((_philox_bits(c["M"], c["V"], s["seed"]) >> 9).double() + 0.5) * 2.0 ** -23
    best, ids = (y - torch.log(-torch.log(u))).max(dim=1)
    return ids, best


@torch.no_grad()
def exact(case, seed):
    c, s = case, _make(case, seed)
    kind = c["kind"]
    if kind in ("step", "step8"):
        return _exact_step(c, s)
    if kind == "sample":
        return _exact_sample(c, s)
    if kind == "lm_head":
        return torch.cat([s["hidden"].double() @ s["W"][v:v + 16384].double().t() for v in range(0, c["V"], 16384)],
                         dim=1)
    if kind == "domino":
        return None, _exact_domino(c, s)
    if kind != "block":
        return None, _exact_rollout(c, s, s["base"], s["prefix"][:, 0])
    h = s["hiddens"].double().flatten(0, 1)
    base = torch.cat([h @ s["W"][v:v + 16384].double().t() for v in range(0, c["V"], 16384)], dim=1)
    base = base.view(c["B"], c["k"], c["V"])
    held = base.to(torch.bfloat16)
    first, ids = held[:, 0].double().max(dim=1)
    scores = _exact_rollout(c, s, held[:, 1:], ids)
    return None, torch.cat([first[:, None], scores], dim=1), base[:, 1:]
