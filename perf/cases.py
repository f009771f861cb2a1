"""The work that users have this framework do, as cases to be measured one by one.

A case is a dict of plain values; ``kind`` names the path:

  causal       cuda_causal_rfa on feature maps, forward + backward
  raw          random matrices -> phi(q), phi(k) -> cuda_causal_rfa with a padding mask, forward + backward
  module       a CausalAttention layer, forward + backward with all parameter gradients
  prefill      a CausalAttention layer takes in a prompt and leaves its decoding state
  decode       a CausalAttention layer takes one token per sequence
  cross        an encoder-decoder attention layer (CrossAttentionProjectLayer + CrossAttention), forward + backward
  cross_step   CrossAttention for one target token per sequence against a projected source
  masked       masked_rfa (quadratic form) under a causal mask, forward + backward

Sizes: ``T`` (target) steps, ``S`` source steps, ``B`` sequences, ``H`` heads, ``d`` head width, ``D``
random features per head (phi is 2 * D wide).  All tensors are fp16 (the framework's type), states fp32.
"""
import torch

from rfa_amd import causal_attention as causal
from rfa_amd import cross_attention as cross
from rfa_amd import utils

SCALE = utils.SCALE


def _case(name, kind, T, B, H, d, D, S=0):
    return {"name": name, "kind": kind, "T": T, "S": S, "B": B, "H": H, "d": d, "D": D}


def listed():
    return [
        # the smallest useful call: two short sentences, four heads; launches and host work count
        _case("causal tiny", "causal", 128, 2, 4, 64, 64),
        # language-model training, the attention alone: 8 sequences of 1024 tokens
        _case("causal lm", "causal", 1024, 8, 8, 64, 64),
        # long-context training, the attention alone: wide heads, 16384 tokens
        _case("causal long", "causal", 16384, 2, 16, 128, 128),
        # padded batch of sentences of no round length, from q, k, v to their gradients and sigma's
        _case("raw ragged", "raw", 777, 6, 12, 64, 64),
        # one decoder layer of an ordinary language model in training
        _case("module base", "module", 1024, 8, 8, 64, 64),
        # one layer of a wider model with wide heads in training
        _case("module wide", "module", 512, 16, 8, 128, 128),
        # serving: a batch of 64 prompts of 512 tokens taken in at once
        _case("prefill batch", "prefill", 512, 64, 16, 64, 64),
        # serving: the next token of each of 64 sequences
        _case("decode batch", "decode", 1, 64, 16, 64, 64),
        # interactive use: one prompt decoded with four beams
        _case("decode beam", "decode", 1, 4, 8, 64, 64),
        # translation training: sources up to 512 tokens (padded), targets of 256
        _case("cross train", "cross", 256, 32, 8, 64, 64, S=512),
        # translation decoding: one target token for 32 sentences with five beams each
        _case("cross step", "cross_step", 1, 160, 8, 64, 64),
        # attention with an explicit mask on a batch of sentences
        _case("masked", "masked", 512, 8, 8, 64, 64),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


# kind: how often it is drawn, range of T, of B and the most T * B * H that a drawn case has (that of the listed one of its kind)
_RANGES = {
    "causal": (5, (16, 16384), (1, 32), 2 * 16 * 16384),
    "raw": (2, (16, 2048), (1, 32), 8 * 8 * 1024),
    "module": (3, (16, 2048), (1, 32), 8 * 8 * 1024),
    "prefill": (2, (16, 2048), (1, 64), 64 * 16 * 512),
    "decode": (2, (1, 1), (1, 96), 96 * 16),
    "cross": (2, (16, 512), (1, 48), 32 * 8 * 256),
    "cross_step": (1, (1, 1), (1, 320), 320 * 16),
    "masked": (1, (16, 1024), (1, 16), 8 * 8 * 512),
}


def draw(rng):
    """One more case: any kind, sizes spread over its range, all head widths and feature counts."""
    kinds = sorted(_RANGES)
    kind = rng.choices(kinds, [_RANGES[k][0] for k in kinds])[0]
    _, t_range, b_range, most = _RANGES[kind]
    d, D = rng.choice([(64, 64), (64, 64), (64, 32), (64, 128), (128, 64), (128, 128)])
    H = rng.choice([3, 4, 6, 8, 8, 12, 16]) if d == 64 else rng.choice([2, 4, 6, 8])
    T = _log(rng, *t_range)
    if d == 128 and kind != "causal":
        most //= 2
    # sources up to twice the listed ratio of source to target; they count with the targets
    S = _log(rng, 32, 768) if kind == "cross" else 0
    rows = (T + S) / 3 if S else T
    B = _log(rng, b_range[0], max(b_range[0], min(b_range[1], most / (rows * H))))
    return {"kind": kind, "T": T, "S": S, "B": B, "H": H, "d": d, "D": D}


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _unit(gen, T, B, H, d):
    """Query or key rows of norm 1."""
    x = _randn(gen, T, B, H, d)
    return x / x.norm(dim=-1, keepdim=True)


def _features(x, w):
    """phi(x) in fp32: the feature maps that a causal case starts from."""
    u = torch.einsum("tbhd,hkd->tbhk", x / (x.norm(dim=-1, keepdim=True) + 1e-3), w)
    return SCALE * torch.cat([u.sin(), u.cos()], -1)


def _state(gen, B, H, d, w, steps=256):
    """The fp32 state of B * H heads after ``steps`` keys."""
    k = _features(_unit(gen, steps, B, H, d), w).permute(1, 2, 3, 0).contiguous()
    v = _randn(gen, steps, B, H, d).permute(1, 2, 0, 3).contiguous()
    return torch.matmul(k, v), k.sum(-1)


def _padding(gen, B, length):
    """[B, length] mask of padded keys: lengths spread over the upper half of the range."""
    n = torch.randint((length + 1) // 2, length + 1, (B, 1), generator=gen, device="cuda")
    return torch.arange(length, device="cuda")[None, :] >= n


def _leaf(x):
    return x.half().contiguous().requires_grad_(True)


def _layer(gen, cls, E, H, d, D):
    """A layer in fp16 on the GPU, its weights drawn from ``gen`` at the scale the layer initialises them with."""
    with torch.device("cuda"):
        m = cls(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).to("cuda", torch.float16)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name == "sigma":
                p.copy_(1 + 0.1 * _randn(gen, *p.shape))
            elif p.dim() == 2:
                p.copy_(_randn(gen, *p.shape) / (2 * E) ** 0.5)
            else:
                p.copy_(0.02 * _randn(gen, *p.shape))
    return m


def prepare(case, seed):
    kind, T, S, B, H, d, D = (case[k] for k in ("kind", "T", "S", "B", "H", "d", "D"))
    E = H * d
    gen = torch.Generator("cuda").manual_seed(seed)
    w = _randn(gen, H, D, d)
    st = {"kind": kind, "w": w.half()}
    if kind in ("causal", "masked"):
        w = w.half().float()
        st["in"] = [_leaf(_features(_unit(gen, T, B, H, d), w)), _leaf(_features(_unit(gen, T, B, H, d), w)),
                    _leaf(_randn(gen, T, B, H, d))]
        st["g"] = _randn(gen, T, B, E).half()
        if kind == "masked":
            st["mask"] = torch.full((T, T), float("-inf"), device="cuda").triu(1)
    elif kind == "raw":
        sigma = 1 + 0.1 * _randn(gen, H, 1, d)
        st["in"] = [_leaf(_randn(gen, T, B, H, d)) for _ in range(3)] + [_leaf(sigma)]
        st["g"] = _randn(gen, T, B, E).half()
        st["pad"] = _padding(gen, B, T)
    elif kind == "module":
        st["layer"] = _layer(gen, causal.CausalAttention, E, H, d, D).train()
        st["in"] = [_leaf(_randn(gen, T, B, E))]
        st["g"] = _randn(gen, T, B, E).half()
    elif kind == "prefill":
        st["layer"] = _layer(gen, causal.CausalAttention, E, H, d, D).eval()
        st["x"] = _randn(gen, T, B, E).half()
    elif kind == "decode":
        st["layer"] = _layer(gen, causal.CausalAttention, E, H, d, D).eval()
        st["x"] = _randn(gen, 1, B, E).half()
        st["s"], st["z"] = _state(gen, B, H, d, w)
    elif kind == "cross":
        st["source"] = _layer(gen, cross.CrossAttentionProjectLayer, E, H, d, D).train()
        st["layer"] = _layer(gen, cross.CrossAttention, E, H, d, D).train()
        st["in"] = [_leaf(_randn(gen, S, B, E)), _leaf(_randn(gen, T, B, E))]
        st["g"] = _randn(gen, T, B, E).half()
        st["pad"] = _padding(gen, B, S).transpose(0, 1)[:, :, None, None]
    elif kind == "cross_step":
        st["layer"] = _layer(gen, cross.CrossAttention, E, H, d, D).eval()
        st["x"] = _randn(gen, 1, B, E).half()
        st["state"] = utils.CrossAttentionState(*_state(gen, B, H, d, w), st["w"], 1.0)
    return st


def _backward(out, g, leaves):
    for t in leaves:
        t.grad = None
    out.backward(g)
    return [out.detach()] + [t.grad for t in leaves]


def run(st):
    kind = st["kind"]
    if kind == "causal":
        q, k, v = st["in"]
        return _backward(causal.cuda_causal_rfa(phi_q=q, phi_k=k, v=v), st["g"], st["in"])
    if kind == "raw":
        q, k, v, sigma = st["in"]
        w = utils.build_random_matrices(st["w"], 1.0, sigma, True)
        phi_q = utils.random_project(x=q, random_matrices=w)
        phi_k = utils.random_project(x=k, random_matrices=w)
        out = causal.cuda_causal_rfa(phi_q=phi_q, phi_k=phi_k, v=v, key_padding_mask=st["pad"])
        return _backward(out, st["g"], st["in"])
    if kind == "module":
        layer, (x,) = st["layer"], st["in"]
        return _backward(layer(x, st["w"]), st["g"], [x, *layer.parameters()])
    if kind == "prefill":
        with torch.no_grad():
            state = {}
            out = st["layer"](st["x"], st["w"], saved_state=state)
        return [out, state["prev_s"], state["prev_z"]]
    if kind == "decode":
        with torch.no_grad():
            state = {"prev_s": st["s"], "prev_z": st["z"]}
            out = st["layer"](st["x"], st["w"], saved_state=state)
        return [out, state["prev_s"], state["prev_z"]]
    if kind == "cross":
        source, layer, (enc, query) = st["source"], st["layer"], st["in"]
        state = source(encoder_output=enc, random_matrices=st["w"], mask=st["pad"])
        return _backward(layer(query, state), st["g"], [enc, query, *source.parameters(), *layer.parameters()])
    if kind == "cross_step":
        with torch.no_grad():
            return st["layer"](st["x"], st["state"])
    q, k, v = st["in"]
    return _backward(causal.masked_rfa(phi_q=q, phi_k=k, v=v, attn_mask=st["mask"]), st["g"], st["in"])


def work(case):
    """Inputs once and outputs once; products of the recurrent form (of the lower triangle where masked)."""
    kind, T, S, B, H, d, D = (case[k] for k in ("kind", "T", "S", "B", "H", "d", "D"))
    E, K, N = H * d, 2 * D, B * H
    state = 4 * N * (K * d + K)
    matrices = 2 * H * D * d
    phi, phi_back = 2 * D * d, 4 * D * d                # per row and head
    if kind == "causal":
        return {"bytes": 2 * T * N * (4 * K + 4 * d), "flops": 12.0 * K * d * T * N}
    if kind == "raw":
        return {"bytes": 2 * T * N * 8 * d + matrices + B * T,
                "flops": T * N * (12.0 * K * d + 2 * (phi + phi_back))}
    if kind == "module":
        return {"bytes": 2 * (4 * T * B * E + 8 * E * E) + matrices,
                "flops": T * B * 24.0 * E * E + T * N * (12.0 * K * d + 2 * (phi + phi_back))}
    if kind == "prefill":
        return {"bytes": 2 * (2 * T * B * E + 4 * E * E) + state + matrices,
                "flops": T * B * 8.0 * E * E + T * N * (4.0 * K * d + 2 * phi)}
    if kind == "decode":
        return {"bytes": 2 * (2 * B * E + 4 * E * E) + 2 * state + matrices,
                "flops": B * 8.0 * E * E + N * (4.0 * K * d + 2 * phi)}
    if kind == "cross":
        return {"bytes": 2 * (2 * S * B * E + 4 * T * B * E + 8 * E * E) + matrices + B * S,
                "flops": (S + T) * B * 12.0 * E * E + (S + T) * N * (6.0 * K * d + phi + phi_back)}
    if kind == "cross_step":
        return {"bytes": 2 * (2 * B * E + 2 * E * E) + state + matrices,
                "flops": B * 4.0 * E * E + N * (2.0 * K * d + phi)}
    return {"bytes": 2 * T * N * (4 * K + 4 * d), "flops": N * T * T / 2 * (8.0 * K + 6 * d)}


# Largest relative error of any output against the same path in 64 bits, over the listed cases and drawn ones.
_MEASURED = {"causal": 4.6e-4, "raw": 6.2e-4, "module": 8.3e-4, "prefill": 3.9e-4, "decode": 2.9e-4,
             "cross": 9.7e-4, "cross_step": 2.9e-4, "masked": 5.3e-4}


def tolerance(case):
    kind = case["kind"]
    tol = {"rel": round(4 * _MEASURED[kind], 4)}
    if kind in ("raw", "module"):
        # the gradient jumps where a denominator crosses its clamp at 1: where the feature maps are formed on the
        # way (rounded to fp16), one of the first rows of a sequence may land on the other side of it
        tol["max"] = 0.9
    return tol
