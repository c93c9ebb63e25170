"""Performance cases of the Gated DeltaNet path: what a program that uses this package has it do.

Every case is one call (or one forward and backward) through the public entry points of ``sorernn_amd``:
single-token and multi-token decoding, prefill of a prompt, of a batch and of packed documents, the
training step of the chunked rule, of the layer's prologue and epilogue and of the whole layer, and the
forward of the attention layer's core and of the GDN layer. ``listed()`` gives the fixed cases,
``draw()`` others of the same ranges, ``exact()`` the same results in 64 bits by plain torch.
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

import sorernn_amd as sa
from sorernn_amd.attention import attn_qk_norm_rope, gated_attention
from sorernn_amd.gdn_layer import GatedDeltaNet, GDNLayerConfig

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
EPS = 1e-6
ROPE_THETA = 1e6


def listed():
    return [
        # one user's chat: one token for one sequence, where launches and the host's work count
        {"name": "decode_1", "kind": "decode", "B": 1, "H": 16, "HV": 16, "D": 128, "gate": True, "dtype": "bf16"},
        # a serving batch: one token for each of 64 sequences, 67 MB of fp32 states updated in place
        {"name": "decode_64", "kind": "decode", "B": 64, "H": 16, "HV": 16, "D": 128, "gate": False, "dtype": "bf16"},
        # a few tokens for each of 16 sequences from their stored states (a draft being scored, a short turn)
        {"name": "recurrent_block", "kind": "recurrent", "B": 16, "T": 7, "H": 16, "HV": 16, "D": 128, "l2": True,
         "dtype": "bf16"},
        # the tiny preset in full precision (a reference run, a unit-sized experiment): B=1, T=256, H=4, d=64, fp32
        {"name": "tiny_fp32", "kind": "rule", "B": 1, "T": 256, "docs": 0, "H": 4, "HV": 4, "D": 64, "model": False,
         "h0": False, "final": True, "train": False, "dtype": "fp32"},
        # one user's prompt of 1,000 tokens: the output and the state that decoding continues from
        {"name": "prefill_prompt", "kind": "rule", "B": 1, "T": 1000, "docs": 0, "H": 16, "HV": 16, "D": 128,
         "model": True, "h0": False, "final": True, "train": False, "dtype": "bf16"},
        # the 0.8B-shape prefill of a batch of four, from and to a state: B=4, T=4096, H=16, d=128
        {"name": "prefill_batch", "kind": "rule", "B": 4, "T": 4096, "docs": 0, "H": 16, "HV": 16, "D": 128,
         "model": False, "h0": True, "final": True, "train": False, "dtype": "bf16"},
        # the reference model's call (q/k norm, gate and sigmoid in the kernel) on packed documents of a corpus
        {"name": "prefill_docs", "kind": "rule", "B": 1, "T": 32768, "docs": 53, "H": 16, "HV": 16, "D": 128,
         "model": True, "h0": False, "final": False, "train": False, "dtype": "bf16"},
        # the training step of the rule at the same shape as the batch prefill
        {"name": "train_rule", "kind": "rule", "B": 4, "T": 4096, "docs": 0, "H": 16, "HV": 16, "D": 128,
         "model": True, "h0": False, "final": False, "train": True, "dtype": "bf16"},
        # the training step of what surrounds the rule in the layer, on packed documents: conv + SiLU, the q/k
        # L2 norm and the gated RMSNorm, each with its backward
        {"name": "train_around", "kind": "around", "T": 16384, "docs": 24, "H": 16, "D": 128, "dtype": "bf16"},
        # the attention layer's core between its projections: B=2, T=8192, 16 q and 4 kv heads of 128
        {"name": "attention", "kind": "attention", "B": 2, "T": 8192, "docs": 0, "HQ": 16, "HKV": 4, "D": 128},
        # a training step of the whole GDN layer on 2 x 2048 tokens, hidden 2048
        {"name": "layer_train", "kind": "layer", "B": 2, "T": 2048, "docs": 0, "dm": 2048, "H": 16, "HV": 16,
         "D": 128, "train": True},
        # the forward of the whole GDN layer at the block pair's size: B=2, T=8192, hidden 2048
        {"name": "layer_forward", "kind": "layer", "B": 2, "T": 8192, "docs": 0, "dm": 2048, "H": 16, "HV": 16,
         "D": 128, "train": False},
    ]


# ---------------------------------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------------------------------
def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _heads(rng: random.Random, most: int) -> tuple[int, int]:
    """q/k heads and value heads (a multiple of them): at most `most` value heads."""
    rep = rng.choice([1, 1, 1, 2])
    h = rng.choice([x for x in (1, 2, 4, 8, 10, 16) if x * rep <= most])
    return h, h * rep


def draw(rng: random.Random):
    kind = rng.choice(["decode", "recurrent", "prefill", "prefill", "train", "around", "attention", "layer"])
    d = rng.choice([64, 128, 128])
    if kind == "decode":
        h, hv = _heads(rng, 16)
        return {"kind": "decode", "B": _log_int(rng, 1, 64), "H": h, "HV": hv, "D": d, "gate": rng.random() < 0.5,
                "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if kind == "recurrent":
        h, hv = _heads(rng, 16)
        return {"kind": "recurrent", "B": _log_int(rng, 1, 32), "T": _log_int(rng, 1, 64), "H": h, "HV": hv, "D": d,
                "l2": rng.random() < 0.5, "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    if kind in ("prefill", "train"):
        train = kind == "train"
        h, hv = _heads(rng, 16)
        packed = rng.random() < 0.5
        t = _log_int(rng, 17, 16384 if packed else 8192)
        docs = min(t, _log_int(rng, 1, 40)) if packed else 0
        b = 1 if packed else min(32, _log_int(rng, 1, 16384 // t))
        case = {"kind": "rule", "B": b, "T": t, "docs": docs, "H": h, "HV": hv, "D": d, "model": rng.random() < 0.6,
                "h0": rng.random() < 0.3, "final": rng.random() < 0.5, "train": train, "dtype": "bf16"}
        if not train and not packed and t <= 512 and rng.random() < 0.5:  # full precision is for small runs
            case.update(dtype="fp32", B=min(b, 4))
        return case
    if kind == "around":
        t = _log_int(rng, 50, 16384)
        return {"kind": "around", "T": t, "docs": min(t, _log_int(rng, 1, 40)), "H": rng.choice([1, 4, 10, 16]), "D": d,
                "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    if kind == "attention":
        hkv, rep = rng.choice([(1, 4), (2, 5), (4, 4), (2, 2), (4, 1)])
        packed = rng.random() < 0.4
        t = _log_int(rng, 33, 8192)
        return {"kind": "attention", "B": 1 if packed else rng.choice([1, 2]), "T": t,
                "docs": min(t, _log_int(rng, 1, 24)) if packed else 0, "HQ": hkv * rep, "HKV": hkv, "D": d}
    dm = rng.choice([512, 1280, 2048])
    h = rng.choice([x for x in (4, 8, 10, 16) if x * d <= dm])
    hv = 2 * h if rng.random() < 0.25 and h <= 8 else h
    train = rng.random() < 0.5
    packed = rng.random() < 0.5
    t = _log_int(rng, 33, 2048 if train else 8192)
    return {"kind": "layer", "B": 1 if packed else 2, "T": t, "docs": min(t, _log_int(rng, 1, 16)) if packed else 0,
            "dm": dm, "H": h, "HV": hv, "D": d, "train": train}


# ---------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------
def _lengths(case) -> list[int]:
    """Lengths of a case's packed documents: log-normal as in a text corpus, summing to T exactly."""
    n, total = case["docs"], case["T"]
    rng = random.Random(1000 * n + total)
    raw = [math.exp(rng.gauss(0.0, 0.9)) for _ in range(n)]
    spare = total - n  # every document has at least one token
    lens = [1 + int(spare * r / sum(raw)) for r in raw]
    lens[lens.index(max(lens))] += total - sum(lens)
    return lens


def _bounds(case) -> list[int]:
    if not case.get("docs"):
        return []
    out = [0]
    for n in _lengths(case):
        out.append(out[-1] + n)
    return out


def _cu(case):
    """(cu_seqlens on the GPU, the same on the host), or (None, None)."""
    b = _bounds(case)
    if not b:
        return None, None
    host = torch.tensor(b, dtype=torch.int64)
    return host.to(DEV), host


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device=DEV).to(dtype)


def _rand(gen, *shape):
    return torch.rand(*shape, generator=gen, device=DEV)


def _log_decay(gen, *shape):
    return -F.softplus(_randn(gen, *shape)) * (_rand(gen, *shape) * 3 - 4).exp()


def _gate_params(gen, hv: int):
    """The layer's initialisation: A ~ U(1, 16), dt log-uniform in [1e-3, 1e-1]."""
    a_log = (1 + 15 * _rand(gen, hv)).log()
    dt = (_rand(gen, hv) * (math.log(0.1) - math.log(1e-3)) + math.log(1e-3)).exp()
    return a_log, dt + torch.log(-torch.expm1(-dt))


def _rule_inputs(case, gen):
    b, t, h, hv, d = (case[x] for x in ("B", "T", "H", "HV", "D"))
    dt = DTYPES[case["dtype"]]
    s = {"v": _randn(gen, b, t, hv, d, dtype=dt)}
    if case["model"]:  # as the layer calls the rule: conv + SiLU outputs, raw gate and beta projections
        s["q"], s["k"] = (F.silu(_randn(gen, b, t, h, d)).to(dt) for _ in range(2))
        s["g"], s["beta"] = _randn(gen, b, t, hv, dtype=dt), _randn(gen, b, t, hv, dtype=dt)
        s["A_log"], s["dt_bias"] = _gate_params(gen, hv)
    else:
        s["q"], s["k"] = (F.normalize(_randn(gen, b, t, h, d), dim=-1).to(dt) for _ in range(2))
        s["g"], s["beta"] = _log_decay(gen, b, t, hv), _randn(gen, b, t, hv).sigmoid()
    n = case["docs"] or b
    s["h0"] = 0.02 * _randn(gen, n, hv, d, d) if case["h0"] else None
    if case["train"]:
        s["do"] = _randn(gen, b, t, hv, d, dtype=dt)
        s["dht"] = 0.1 * _randn(gen, n, hv, d, d) if case["final"] else None
    return s


def _around_inputs(case, gen):
    t, h, d = case["T"], case["H"], case["D"]
    c, dt = h * d, DTYPES[case["dtype"]]
    return {
        "x": _randn(gen, 1, t, c, dtype=dt), "w": _rand(gen, c, 4) - 0.5, "dy": _randn(gen, 1, t, c, dtype=dt),
        "qk": F.silu(_randn(gen, 1, t, h, d)).to(dt), "dqk": _randn(gen, 1, t, h, d, dtype=dt),
        "o": _randn(gen, 1, t, h, d, dtype=dt), "gate": _randn(gen, 1, t, h, d, dtype=dt),
        "nw": 1 + 0.1 * _randn(gen, d), "dn": _randn(gen, 1, t, h, d, dtype=dt),
    }


def _attention_inputs(case, gen):
    b, t, hq, hkv, d = (case[x] for x in ("B", "T", "HQ", "HKV", "D"))
    # the fused projection's output, q | gate | k | v side by side
    proj = _randn(gen, b, t, (2 * hq + 2 * hkv) * d, dtype=torch.bfloat16)
    return {"proj": proj, "qw": 1 + 0.1 * _randn(gen, d), "kw": 1 + 0.1 * _randn(gen, d)}


def _split_proj(case, proj):
    nq, nkv = case["HQ"] * case["D"], case["HKV"] * case["D"]
    return proj[..., :nq], proj[..., nq:2 * nq], proj[..., 2 * nq:2 * nq + nkv], proj[..., 2 * nq + nkv:]


def _layer(case, gen):
    cfg = GDNLayerConfig(d_model=case["dm"], gdn_qk_heads=case["H"], gdn_v_heads=case["HV"], gdn_head_dim=case["D"],
                         gdn_kernel_gate=True, gdn_fla_conv=True, fused_norm_gate=True)
    with torch.device(DEV):
        layer = GatedDeltaNet(cfg)
    a_log, dt_bias = _gate_params(gen, case["HV"])
    with torch.no_grad():
        for name, prm in layer.named_parameters():
            if name.endswith("proj.weight"):
                prm.copy_(0.02 * _randn(gen, *prm.shape))
            elif name.startswith("conv"):
                prm.copy_(_rand(gen, *prm.shape) - 0.5)
            elif name == "A_log":
                prm.copy_(a_log)
            elif name == "dt_bias":
                prm.copy_(dt_bias)
            else:
                prm.copy_(1 + 0.1 * _randn(gen, *prm.shape))
    return layer.to(torch.bfloat16)


def _layer_inputs(case, gen):
    layer = _layer(case, gen)
    s = {"layer": layer, "x": _randn(gen, case["B"], case["T"], case["dm"], dtype=torch.bfloat16)}
    if case["train"]:
        s["dy"] = _randn(gen, case["B"], case["T"], case["dm"], dtype=torch.bfloat16)
    return s


def _decode_inputs(case, gen):
    b, h, hv, d = (case[x] for x in ("B", "H", "HV", "D"))
    c, dt = (2 * h + hv) * d, DTYPES[case["dtype"]]
    s = {"x": _randn(gen, b, c, dtype=dt), "conv": _randn(gen, b, c, 4, dtype=dt), "w": _rand(gen, c, 4) - 0.5,
         "state": 0.02 * _randn(gen, b, hv, d, d)}
    if case["gate"]:
        s["g"], s["beta"] = _randn(gen, b, hv, dtype=dt), _randn(gen, b, hv, dtype=dt)
        s["A_log"], s["dt_bias"] = _gate_params(gen, hv)
    else:
        s["g"], s["beta"] = _log_decay(gen, b, hv), _randn(gen, b, hv).sigmoid()
    return s


def _recurrent_inputs(case, gen):
    b, t, h, hv, d = (case[x] for x in ("B", "T", "H", "HV", "D"))
    dt = DTYPES[case["dtype"]]
    mk = (lambda: F.silu(_randn(gen, b, t, h, d)).to(dt)) if case["l2"] else \
        (lambda: F.normalize(_randn(gen, b, t, h, d), dim=-1).to(dt))
    return {"q": mk(), "k": mk(), "v": _randn(gen, b, t, hv, d, dtype=dt), "g": _log_decay(gen, b, t, hv),
            "beta": _randn(gen, b, t, hv).sigmoid(), "state": 0.02 * _randn(gen, b, hv, d, d)}


_INPUTS = {"decode": _decode_inputs, "recurrent": _recurrent_inputs, "rule": _rule_inputs, "around": _around_inputs,
           "attention": _attention_inputs, "layer": _layer_inputs}
_RULE_LEAVES = ("q", "k", "v", "g", "beta", "h0", "A_log", "dt_bias")


def prepare(case, seed):
    s = _INPUTS[case["kind"]](case, _gen(seed))
    s["case"] = case
    if case["kind"] in ("rule", "around", "attention", "layer"):
        s["cu"], s["cu_host"] = _cu(case)
    if case["kind"] == "rule" and case["train"]:
        for name in _RULE_LEAVES:
            if s.get(name) is not None:
                s[name].requires_grad_(True)
    elif case["kind"] == "around":
        for name in ("x", "w", "qk", "o", "gate", "nw"):
            s[name].requires_grad_(True)
    elif case["kind"] == "layer" and case["train"]:
        s["x"].requires_grad_(True)
    return s


# ---------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------
def run(s):
    return _RUN[s["case"]["kind"]](s)


def _run_decode(s):
    case = s["case"]
    gate = dict(use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True, A_log=s["A_log"],
                dt_bias=s["dt_bias"]) if case["gate"] else {}
    o = sa.gated_delta_decode_step(s["x"], s["conv"], s["w"], s["g"], s["beta"], s["state"], case["H"], case["HV"],
                                   case["D"], **gate)
    return [o, s["conv"], s["state"]]


def _run_recurrent(s):
    case = s["case"]
    o, state = sa.fused_recurrent_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"],
                                                   initial_state=s["state"], inplace_final_state=True,
                                                   use_qk_l2norm_in_kernel=case["l2"])
    return [o, state]


def _run_rule(s):
    case = s["case"]
    model = dict(use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True,
                 A_log=s["A_log"], dt_bias=s["dt_bias"]) if case["model"] else {}
    call = lambda: sa.chunk_gated_delta_rule(  # noqa: E731
        s["q"], s["k"], s["v"], s["g"], s["beta"], scale=case["D"] ** -0.5, initial_state=s["h0"],
        output_final_state=case["final"], cu_seqlens=s["cu"], cu_seqlens_cpu=s["cu_host"], **model)
    if not case["train"]:
        with torch.no_grad():
            o, state = call()
        return [o] if state is None else [o, state]
    o, state = call()
    outs, grads = ([o], [s["do"]]) if state is None else ([o, state], [s["do"], s["dht"]])
    leaves = [s[x] for x in _RULE_LEAVES if s.get(x) is not None]
    return [x.detach() for x in outs] + list(torch.autograd.grad(outs, leaves, grads))


def _run_around(s):
    y, _ = sa.causal_conv1d(s["x"], s["w"], activation="silu", cu_seqlens=s["cu"], cu_seqlens_cpu=s["cu_host"])
    n = sa.l2norm(s["qk"])
    z = sa.rms_norm_gated(s["o"], s["gate"], s["nw"], None, eps=EPS)
    grads = torch.autograd.grad([y, n, z], [s[x] for x in ("x", "w", "qk", "o", "gate", "nw")],
                                [s["dy"], s["dqk"], s["dn"]])
    return [y.detach(), n.detach(), z.detach(), *grads]


def _run_attention(s):
    case = s["case"]
    q_in, gate, k_in, v = _split_proj(case, s["proj"])
    with torch.no_grad():
        q, k = attn_qk_norm_rope(q_in, k_in, s["qw"], s["kw"], case["HQ"], case["HKV"], case["D"] // 4, ROPE_THETA, EPS,
                                 s["cu"], s["cu_host"])
        o = gated_attention(q, k, v, gate, s["cu"], s["cu_host"])
    return [q, k, o]


def _run_layer(s):
    layer, x = s["layer"], s["x"]
    if not s["case"]["train"]:
        with torch.no_grad():
            return [layer(x, s["cu"], s["cu_host"])]
    y = layer(x, s["cu"], s["cu_host"])
    return [y.detach(), *torch.autograd.grad(y, [x, *layer.parameters()], s["dy"])]


_RUN = {"decode": _run_decode, "recurrent": _run_recurrent, "rule": _run_rule, "around": _run_around,
        "attention": _run_attention, "layer": _run_layer}


# ---------------------------------------------------------------------------------------------------
# the work of one pass, and the precision that it has
# ---------------------------------------------------------------------------------------------------
def work(case):
    kind, d = case["kind"], case["D"]
    if kind == "decode":
        b, h, hv = case["B"], case["H"], case["HV"]
        c, e = (2 * h + hv) * d, SIZE[case["dtype"]]
        ge = e if case["gate"] else 4
        nbytes = 2 * b * hv * d * d * 4 + b * c * e * (1 + 2 * 4) + c * 16 + b * hv * (d * e + 2 * ge)
        return {"bytes": nbytes, "flops": 6 * b * hv * d * d}
    if kind in ("recurrent", "rule"):
        b, t, h, hv, e = case["B"], case["T"], case["H"], case["HV"], SIZE[case["dtype"]]
        n, tok = case.get("docs") or b, b * t
        ge = e if case.get("model") else 4
        qkv, o, gates = tok * (2 * h + hv) * d * e, tok * hv * d * e, 2 * tok * hv * ge
        states = (2 if kind == "recurrent" else int(case["h0"]) + int(case["final"])) * n * hv * d * d * 4
        # per token and value head: S^T k, S^T q and the rank-1 update
        flops = 6 * tok * hv * d * d
        if case.get("train"):  # the gradients of q, k, v, g, beta and h0 from that of o (and of the final state)
            return {"bytes": 2 * (qkv + o + gates + states), "flops": 3 * flops}
        return {"bytes": qkv + o + gates + states, "flops": flops}
    if kind == "around":
        n = case["T"] * case["H"] * d
        # conv: x, dy -> y, dx; L2 norm: qk, dqk -> n, d(qk); gated norm: o, gate, dn -> z, do, dgate
        return {"bytes": 14 * n * SIZE[case["dtype"]], "flops": 100 * n}
    if kind == "attention":
        b, t, hq, hkv = (case[x] for x in ("B", "T", "HQ", "HKV"))
        lens = _lengths(case) if case["docs"] else [t] * b
        tok = b * t
        # projections in, q and k as they are returned, o
        nbytes = 2 * tok * d * ((2 * hq + 2 * hkv) + (hq + hkv) + hq)
        return {"bytes": nbytes, "flops": 4 * d * hq * sum(n * (n + 1) // 2 for n in lens)}
    b, t, dm, h, hv = (case[x] for x in ("B", "T", "dm", "H", "HV"))
    tok = b * t
    weights = dm * ((2 * h + 2 * hv) * d + 2 * hv) + hv * d * dm
    flops = 2 * tok * weights + 6 * tok * hv * d * d
    nbytes = 2 * (weights + 2 * tok * dm)
    return {"bytes": 2 * nbytes, "flops": 3 * flops} if case["train"] else {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the error of today's outputs against ``exact``: 1.7e-3 is one rounding to bf16, 2.1e-4 one to
    fp16; the chunked rule and its backward have 16-bit matrix operands (2e-3 to 5e-3), a layer several in a row."""
    kind = case["kind"]
    if kind == "decode":  # q, k and v are rounded after the conv, the output once more
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
    if kind == "recurrent":
        return {"rel": {"bf16": 7e-3, "fp16": 1e-3, "fp32": 1e-5}[case["dtype"]]}
    if kind == "rule":
        if case["dtype"] == "fp32":
            return {"rel": 1e-5}
        return {"rel": 2e-2} if case["train"] else {"rel": 1e-2}
    if kind == "around":
        return {"rel": {"bf16": 7e-3, "fp16": 1e-3, "fp32": 1e-5}[case["dtype"]]}
    if kind == "attention":
        return {"rel": 1.2e-2}
    return {"rel": 3e-2 if case["train"] else 2e-2}


# ---------------------------------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------------------------------
def exact(case, seed):
    s = prepare(case, seed)
    s = {k: (x.detach() if torch.is_tensor(x) else x) for k, x in s.items()}
    return _EXACT[case["kind"]](s)


def _mm(a, b):
    return torch.matmul(a, b.contiguous())


def _l2_64(x):
    return x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)


def _segment64(q, k, v, g, beta, scale, state):
    """One sequence, [H, T, d] per head, in chunks of 64 tokens with the triangular system solved exactly."""
    outs = []
    for c0 in range(0, q.shape[1], 64):
        qc, kc, vc, gc, bc = (x[:, c0:c0 + 64] for x in (q, k, v, g, beta))
        n = qc.shape[1]
        cum = gc.cumsum(1)
        low = torch.ones(n, n, dtype=torch.bool, device=q.device).tril()
        decay = (cum[:, :, None] - cum[:, None, :]).masked_fill(~low, -math.inf).exp()
        kt = kc.transpose(1, 2)
        p = (-bc[:, :, None] * decay * _mm(kc, kt)).tril(-1)
        x = bc[:, :, None] * vc - (bc * cum.exp())[:, :, None] * _mm(kc, state)
        m = 1
        while m < n:  # (I - p)^-1 = (I + p)(I + p^2)(I + p^4)...
            x = x + _mm(p, x)
            p = _mm(p, p)
            m *= 2
        outs.append(scale * (cum.exp()[:, :, None] * _mm(qc, state) + _mm(decay * _mm(qc, kt), x)))
        last = cum[:, -1:]
        state = last.exp()[:, :, None] * state + _mm(kt, (last - cum).exp()[:, :, None] * x)
    return torch.cat(outs, 1), state


def _rule64(q, k, v, g, beta, scale, h0, bounds):
    """[B, T, H, d] and [B, T, HV, d] tensors in 64 bits -> o [B, T, HV, d], states [N, HV, d, d]."""
    rep = v.shape[2] // q.shape[2]
    q, k = (x.repeat_interleave(rep, 2) for x in (q, k))
    spans = [(0, a, b) for a, b in zip(bounds[:-1], bounds[1:])] or [(i, 0, q.shape[1]) for i in range(q.shape[0])]
    outs, states = [], []
    for i, (row, a, b) in enumerate(spans):
        qs, ks, vs = (x[row, a:b].transpose(0, 1) for x in (q, k, v))
        gs, bs = (x[row, a:b].transpose(0, 1) for x in (g, beta))
        st = h0[i] if h0 is not None else q.new_zeros(v.shape[2], q.shape[3], v.shape[3])
        o, st = _segment64(qs, ks, vs, gs, bs, scale, st)
        outs.append(o.transpose(0, 1))
        states.append(st)
    o = torch.cat(outs, 0)[None] if bounds else torch.stack(outs, 0)
    return o, torch.stack(states, 0)


def _gates64(g, beta, a_log, dt_bias):
    return -a_log.exp() * F.softplus(g + dt_bias), beta.sigmoid()


def _conv64(x, w, bounds):
    """Causal conv of width 4 + SiLU, [B, T, C], no term from another document."""
    out = x * w[:, 3]
    for j in (1, 2, 3):
        shifted = F.pad(x, (0, 0, j, 0))[:, :x.shape[1]]
        if bounds:
            keep = torch.ones(x.shape[1], dtype=x.dtype, device=x.device)
            for a in bounds[:-1]:
                keep[a:a + j] = 0
            shifted = shifted * keep[:, None]
        out = out + shifted * w[:, 3 - j]
    return F.silu(out)


def _norm64(o, gate, w):
    return o * (o.square().mean(-1, keepdim=True) + EPS).rsqrt() * w * F.silu(gate)


def _exact_decode(s):
    case = s["case"]
    b, h, hv, d = (case[x] for x in ("B", "H", "HV", "D"))
    conv = torch.cat([s["conv"][..., 1:], s["x"].view(b, -1, 1)], -1)
    y = F.silu((conv.double() * s["w"].double()).sum(-1))
    q, k, v = y[:, :h * d].view(b, h, d), y[:, h * d:2 * h * d].view(b, h, d), y[:, 2 * h * d:].view(b, hv, d)
    q, k = (_l2_64(x).repeat_interleave(hv // h, 1) for x in (q, k))
    g, beta = s["g"].double(), s["beta"].double()
    if case["gate"]:
        g, beta = _gates64(g, beta, s["A_log"].double(), s["dt_bias"].double())
    state = s["state"].double() * g.exp()[..., None, None]
    delta = beta[..., None] * (v - (state * k[..., None]).sum(-2))
    state = state + k[..., None] * delta[..., None, :]
    o = d ** -0.5 * (state * q[..., None]).sum(-2)
    return [o[:, None], conv, state]


def _exact_recurrent(s):
    q, k = s["q"].double(), s["k"].double()
    if s["case"]["l2"]:
        q, k = _l2_64(q), _l2_64(k)
    return list(_rule64(q, k, s["v"].double(), s["g"].double(), s["beta"].double(), s["case"]["D"] ** -0.5,
                        s["state"].double(), []))


def _exact_rule(s):
    case = s["case"]
    leaves = {x: s[x].double().requires_grad_(case["train"]) for x in _RULE_LEAVES if s.get(x) is not None}
    q, k, g, beta = (leaves[x] for x in ("q", "k", "g", "beta"))
    if case["model"]:
        q, k = _l2_64(q), _l2_64(k)
        g, beta = _gates64(g, beta, leaves["A_log"], leaves["dt_bias"])
    with torch.set_grad_enabled(case["train"]):
        o, state = _rule64(q, k, leaves["v"], g, beta, case["D"] ** -0.5, leaves.get("h0"), _bounds(case))
        outs = [o, state] if case["final"] else [o]
        if not case["train"]:
            return outs
        cot = [s["do"].double()] + ([s["dht"].double()] if case["final"] else [])
        return [x.detach() for x in outs] + list(torch.autograd.grad(outs, list(leaves.values()), cot))


def _exact_around(s):
    lf = {x: s[x].double().requires_grad_(True) for x in ("x", "w", "qk", "o", "gate", "nw")}
    y = _conv64(lf["x"], lf["w"], _bounds(s["case"]))
    n = _l2_64(lf["qk"])
    z = _norm64(lf["o"], lf["gate"], lf["nw"])
    grads = torch.autograd.grad([y, n, z], list(lf.values()), [s["dy"].double(), s["dqk"].double(), s["dn"].double()])
    return [y.detach(), n.detach(), z.detach(), *grads]


def _exact_attention(s):
    case = s["case"]
    b, t, hq, hkv, d = (case[x] for x in ("B", "T", "HQ", "HKV", "D"))
    rot = d // 4
    q, gate, k, v = (x.double() for x in _split_proj(case, s["proj"]))
    q, k, v, gate = q.view(b, t, hq, d), k.view(b, t, hkv, d), v.view(b, t, hkv, d), gate.view(b, t, hq, d)
    bounds = _bounds(case)
    spans = list(zip(bounds[:-1], bounds[1:])) or [(0, t)]
    pos = torch.cat([torch.arange(n - m, device=DEV) for m, n in spans]).double()
    freq = ROPE_THETA ** (-torch.arange(0, rot, 2, device=DEV).double() / rot)
    ang = pos[:, None] * freq
    cos, sin = (torch.cat([f, f], -1)[None, :, None] for f in (ang.cos(), ang.sin()))

    def turn(x, w):
        x = x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * w.double()
        r = x[..., :rot]
        half = torch.cat([-r[..., rot // 2:], r[..., :rot // 2]], -1)
        return torch.cat([r * cos + half * sin, x[..., rot:]], -1)

    q, k = turn(q, s["qw"]), turn(k, s["kw"])
    o = torch.empty_like(q)
    for row in range(b):
        for m, n in spans:
            ks, vs = (x[row, m:n].transpose(0, 1).repeat_interleave(hq // hkv, 0) for x in (k, v))
            kt = ks.transpose(1, 2).contiguous()
            for a in range(m, n, 1024):
                e = min(a + 1024, n)
                sc = torch.matmul(q[row, a:e].transpose(0, 1), kt[..., :e - m].contiguous()) * d ** -0.5
                late = torch.arange(m, e, device=DEV)[None] > torch.arange(a, e, device=DEV)[:, None]
                pr = sc.masked_fill_(late, -math.inf).softmax(-1)
                o[row, a:e] = torch.matmul(pr, vs[:, :e - m].contiguous()).transpose(0, 1)
    return [q, k, (o * gate.sigmoid()).flatten(2)]


def _exact_layer(s):
    case, layer = s["case"], s["layer"]
    b, t, h, hv, d = (case[x] for x in ("B", "T", "H", "HV", "D"))
    bounds = _bounds(case)
    prm = {n: p.detach().double().requires_grad_(case["train"]) for n, p in layer.named_parameters()}
    x = s["x"].double().requires_grad_(case["train"])
    with torch.set_grad_enabled(case["train"]):
        lin = lambda n, z: z @ prm[n + ".weight"].t()  # noqa: E731
        q = _l2_64(_conv64(lin("q_proj", x), prm["conv_q"], bounds).view(b, t, h, d))
        k = _l2_64(_conv64(lin("k_proj", x), prm["conv_k"], bounds).view(b, t, h, d))
        v = _conv64(lin("v_proj", x), prm["conv_v"], bounds).view(b, t, hv, d)
        g, beta = _gates64(lin("a_proj", x), lin("b_proj", x), prm["A_log"], prm["dt_bias"])
        o, _ = _rule64(q, k, v, g, beta, d ** -0.5, None, bounds)
        y = lin("o_proj", _norm64(o, lin("g_proj", x).view(b, t, hv, d), prm["o_norm.weight"]).flatten(2))
        if not case["train"]:
            return [y]
        return [y.detach(), *torch.autograd.grad(y, [x, *prm.values()], s["dy"].double())]


_EXACT = {"decode": _exact_decode, "recurrent": _exact_recurrent, "rule": _exact_rule, "around": _exact_around,
          "attention": _exact_attention, "layer": _exact_layer}
