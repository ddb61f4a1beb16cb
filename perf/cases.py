"""The work users of this framework have it do, as cases that can be timed and compared.

Each case is one pass through a public entry point on inputs made from a seed:
the routed 4-bit expert layer as a program calls it (decoding, evaluation,
prefill, training), the trainable dense experts, the cache of expert copies and
the 4-bit codec.  Shapes are those of the benchmark (Qwen3-30B-A3B and
Mixtral-8x7B layers), of the OLMoE-1B-7B layer in the tests, and one small
generic layer.

``listed()`` gives the fixed cases, ``draw(rng)`` further ones of the same
ranges, ``prepare`` what a program holds before the call, ``run`` the call,
``work`` what it cannot do without, ``tolerance`` how far another correct
implementation may be, ``exact`` the same outputs from plain torch in 64 bits.
"""
from __future__ import annotations

import math

import torch

from usaf_amd import moe as G
from usaf_amd import olmoe_dml, quantization, qwen3moe_dml
from usaf_amd.expert_cache import ExpertSlotCache
from usaf_amd.moe_loader import SparseGradStore
from usaf_amd.sparse_optim import DeviceLossScale, MomentumSGD, SparseAdam

SHAPES = {  # experts, hidden, intermediate, experts per token
    "qwen3": (128, 2048, 768, 8),
    "mixtral": (8, 4096, 14336, 2),
    "olmoe": (64, 2048, 1024, 8),
    "small": (32, 1024, 512, 4),
}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ACTIVE = 0.005  # share of the weight positions that are trained
PREFIX = "model.layers.0.mlp.experts"


def listed():
    return [
        # one decoded token through a patched Qwen3-MoE block (router and experts): latency and launches
        {"name": "decode_1", "kind": "block", "shape": "qwen3", "T": 1, "dtype": "bf16", "zipf": 0.0},
        # a decode step of a batch of 24 sequences
        {"name": "decode_24", "kind": "block", "shape": "qwen3", "T": 24, "dtype": "bf16", "zipf": 0.0},
        # a small batch on large experts: every expert's weights are read for a few tokens each
        {"name": "decode_mixtral_40", "kind": "experts", "shape": "mixtral", "T": 40, "dtype": "bf16", "zipf": 0.0},
        # scoring one text of odd length in fp16, no gradients
        {"name": "eval_333", "kind": "experts", "shape": "qwen3", "T": 333, "dtype": "fp16", "zipf": 1.1},
        # prefill of a long prompt
        {"name": "prefill_4096", "kind": "experts", "shape": "qwen3", "T": 4096, "dtype": "bf16", "zipf": 0.0},
        # the trainer's microbatch (one sequence of 256 tokens, fp16): forward and backward with
        # trained values over the 4-bit weights and gradients sampled at the active positions
        {"name": "train_256", "kind": "train", "shape": "qwen3", "T": 256, "dtype": "fp16", "zipf": 0.0},
        # a whole training step of the benchmark's layer: block forward and backward, loss scale,
        # finite check, SparseAdam, overlay refresh and the router's optimizer
        {"name": "step_4096", "kind": "step", "shape": "qwen3", "T": 4096, "dtype": "bf16", "zipf": 0.0},
        # backpropagation through a frozen layer of large experts, the benchmark's 8192 tokens
        {"name": "frozen_mixtral_8192", "kind": "frozen", "shape": "mixtral", "T": 8192, "dtype": "bf16", "zipf": 0.0},
        # training dense experts: forward, backward and the experts' full weight gradients
        {"name": "dense_olmoe_512", "kind": "dense", "shape": "olmoe", "T": 512, "dtype": "bf16", "zipf": 0.0},
        # a microbatch on cached fp16 copies of the experts, skewed popularity, two layers in turn
        {"name": "cache_2048", "kind": "cache", "shape": "qwen3", "T": 2048, "dtype": "fp16", "zipf": 1.1, "fits": True},
        # quantizing one expert's weight and reading it back
        {"name": "codec_expert", "kind": "codec", "rows": 768, "cols": 2048, "group": 128, "dtype": "fp16",
         "op": "both"},
        # dequantizing a whole layer's gate and up projections
        {"name": "codec_layer", "kind": "codec", "rows": 128 * 1536, "cols": 2048, "group": 128, "dtype": "bf16",
         "op": "dequantize"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["block", "experts", "experts", "train", "train", "step", "frozen", "dense", "cache", "codec"])
    if kind == "codec":
        cols = _log_int(rng, 64, 4096) if rng.random() < 0.5 else 128 * rng.randint(1, 32)
        rows = _log_int(rng, 16, 200_000_000 // cols)
        return {"kind": kind, "rows": rows, "cols": cols, "group": rng.choice([128, 128, 128, 64, 32]),
                "dtype": rng.choice(["fp16", "bf16"]), "op": rng.choice(["both", "dequantize"])}
    shape = {"train": ["qwen3", "olmoe", "small"], "step": ["qwen3", "olmoe", "small"], "dense": ["olmoe", "small"],
             "cache": ["qwen3", "olmoe"]}.get(kind, ["qwen3", "mixtral", "olmoe", "small"])
    shape = rng.choice(shape)
    lo, hi = {"block": (1, 4096), "experts": (1, 4096), "train": (64, 4096), "step": (64, 4096),
              "frozen": (16, 4096), "dense": (64, 2048), "cache": (64, 4096)}[kind]
    case = {"kind": kind, "shape": shape, "T": _log_int(rng, lo, hi),
            "dtype": "bf16" if kind == "dense" else rng.choice(["bf16", "bf16", "fp16"]),
            "zipf": 0.0 if kind in ("block", "step") else rng.choice([0.0, 0.0, 1.1])}
    if kind == "cache":
        case["fits"] = rng.random() < 0.7
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFF)


def _quantized(gen, numel, group=128, chunk=1 << 26):
    """Codes, scales and zeros of ``numel`` weights ~ N(0, 0.02) in the 4-bit format."""
    groups = -(-numel // group)
    q = torch.empty(groups, group // 2, dtype=torch.int8, device="cuda")
    s = torch.empty(groups, dtype=torch.float16, device="cuda")
    z = torch.empty(groups, dtype=torch.float16, device="cuda")
    for a in range(0, groups, chunk // group):
        b = min(groups, a + chunk // group)
        x = torch.randn(b - a, group, device="cuda", generator=gen).mul_(0.02)
        mn = x.amin(1, keepdim=True)
        step = ((x.amax(1, keepdim=True) - mn) / 15.0).clamp_min_(1e-12)
        codes = x.sub_(mn).div_(step).round_().clamp_(0, 15).to(torch.uint8)
        q[a:b] = (codes[:, 0::2] | (codes[:, 1::2] << 4)).view(torch.int8)
        s[a:b] = step.squeeze(1).half()
        z[a:b] = mn.squeeze(1).half()
    return q, s, z


def _q4(gen, shape):
    q, s, z = _quantized(gen, math.prod(shape))
    return G.Q4Tensor(q, s, z, torch.Size(shape), 128)


def _values(q, s, z, numel):
    """fp16 values of 4-bit groups: fp16(fp16(code * scale) + zero)."""
    raw = q.view(torch.uint8)
    codes = torch.stack([raw & 15, raw >> 4], dim=2).view(raw.shape[0], -1).to(torch.float16)
    return (codes * s.unsqueeze(1) + z.unsqueeze(1)).reshape(-1)[:numel]


def _expert_values(q4, e):
    """Expert e's [rows, cols] slice of a 4-bit tensor, fp16."""
    E, rows, cols = q4.shape
    n = rows * cols // 128
    return _values(q4.q[e * n:(e + 1) * n], q4.s[e * n:(e + 1) * n], q4.z[e * n:(e + 1) * n], rows * cols).view(rows, cols)


def _logits(gen, T, E, zipf):
    """Router logits; zipf > 0: experts drawn with Zipf popularity (Gumbel top-k)."""
    if not zipf:
        return torch.randn(T, E, device="cuda", generator=gen)
    rank = (torch.randperm(E, device="cuda", generator=gen) + 1).float()
    u = torch.rand(T, E, device="cuda", generator=gen).clamp_(1e-12, 1 - 1e-7)
    return -zipf * torch.log(rank) - torch.log(-torch.log(u))


def _routing(gen, T, E, k, zipf, dtype):
    """Routing weights [T, E]: softmax, k largest kept, renormalised."""
    p = torch.softmax(_logits(gen, T, E, zipf), dim=-1)
    val, idx = torch.topk(p, k, dim=-1)
    return torch.zeros_like(p).scatter_(1, idx, val / val.sum(-1, keepdim=True)).to(dtype)


def _positions(gen, numel, chunk=1 << 26):
    """ACTIVE * numel sorted flat positions, uniformly spread."""
    parts = []
    for a in range(0, numel, chunk):
        n = min(chunk, numel - a)
        parts.append((torch.rand(n, device="cuda", generator=gen) < 1.05 * ACTIVE).nonzero().reshape(-1) + a)
    idx = torch.cat(parts)
    return idx[torch.randperm(idx.numel(), device="cuda", generator=gen)[:int(ACTIVE * numel)].sort().values]


class _Router(torch.nn.Module):
    def __init__(self, weight, top_k):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.top_k, self.norm_topk_prob = top_k, True


class _Experts(torch.nn.Module):
    """An expert module as the loader leaves it: 4-bit tensors attached, or dense Parameters."""

    def __init__(self, forward, q4=None, gate_up=None, down=None):
        super().__init__()
        self._forward = forward
        if q4 is not None:
            self._usaf_q4 = q4
        else:
            self.gate_up_proj, self.down_proj = torch.nn.Parameter(gate_up), torch.nn.Parameter(down)

    def forward(self, hidden_states, weights):
        return self._forward(self, hidden_states, weights)


class _Block(torch.nn.Module):
    def __init__(self, gate, experts):
        super().__init__()
        self.gate, self.experts = gate, experts

    def forward(self, hidden_states):
        return qwen3moe_dml.dml_qwen3_moe_block_forward(self, hidden_states)


def _trained(ew, gen, dtype):
    """Active positions, their masters (slices of one buffer), store and overlays of a layer."""
    active, shapes, init = {}, {}, []
    for which, q4 in (("gate_up", ew.gate_up), ("down", ew.down)):
        name = f"{PREFIX}.{which}_proj"
        active[name], shapes[name] = _positions(gen, q4.numel()), tuple(q4.shape)
        init.append(torch.randn(active[name].numel(), device="cuda", generator=gen) * 0.02)
    flat, masters, at = torch.cat(init), {}, 0
    for name, v in zip(active, init):
        masters[name] = torch.nn.Parameter(flat[at:at + v.numel()], requires_grad=False)
        at += v.numel()
    store = SparseGradStore(active, shapes, device="cuda")
    overlays = {n: ew.set_overlay("gate_up" if "gate_up" in n else "down", active[n], masters[n].data, dtype)
                for n in active}
    return active, masters, store, overlays


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    dt = DTYPES[case["dtype"]]
    st = {"case": case}
    if kind == "codec":
        numel = case["rows"] * case["cols"]
        shape = torch.Size([case["rows"], case["cols"]])
        if case["op"] == "both":
            st["w"] = torch.empty(shape, dtype=dt, device="cuda")
            flat = st["w"].view(-1)
            for a in range(0, numel, 1 << 26):
                n = min(1 << 26, numel - a)
                flat[a:a + n] = (torch.randn(n, device="cuda", generator=gen) * 0.02).to(dt)
        else:
            st["q"], st["shape"] = _quantized(gen, numel, case["group"]), shape
        return st
    E, H, I, k = SHAPES[case["shape"]]
    T = case["T"]
    if kind == "dense":
        st["mod"] = _Experts(olmoe_dml.dml_experts_forward,
                             gate_up=(torch.randn(E, 2 * I, H, device="cuda", generator=gen) * 0.02).to(dt),
                             down=(torch.randn(E, H, I, device="cuda", generator=gen) * 0.02).to(dt))
    elif kind == "cache":
        layers = {f"model.layers.{i}.mlp.experts": G.ExpertWeights(_q4(gen, (E, 2 * I, H)), _q4(gen, (E, H, I)))
                  for i in range(2)}
        slot = 2 * 3 * H * I
        st["layers"] = layers
        st["cache"] = ExpertSlotCache(layers, "cuda", max_bytes=(2 * E if case["fits"] else E + E // 2) * slot + slot // 2,
                                      dtype=dt)
    else:
        st["ew"] = ew = G.ExpertWeights(_q4(gen, (E, 2 * I, H)), _q4(gen, (E, H, I)))
    grad = kind in ("train", "step", "frozen", "dense")
    st["x"] = torch.randn(T, H, device="cuda", generator=gen).to(dt).requires_grad_(grad)
    if kind in ("block", "step"):
        router = (torch.randn(E, H, device="cuda", generator=gen) / H ** 0.5).to(dt)
    if kind == "block":
        st["x"] = st["x"].view(1, T, H)
        st["block"] = _Block(_Router(router, k), _Experts(qwen3moe_dml.dml_qwen3_experts_forward,
                                                          q4={"gate_up_proj": ew.gate_up, "down_proj": ew.down}))
    elif kind == "step":
        st["router"] = router.requires_grad_(True)
    elif kind == "cache":
        st["w"] = [_routing(gen, T, E, k, case["zipf"], dt) for _ in range(2)]
    else:
        st["w"] = _routing(gen, T, E, k, case["zipf"], dt).requires_grad_(grad)
    if grad:
        st["dout"] = torch.randn(T, H, device="cuda", generator=gen).to(dt)
    if kind in ("train", "step"):
        st["active"], st["masters"], st["store"], st["overlays"] = _trained(ew, gen, dt)
    if kind == "step":
        st["adam"] = SparseAdam(st["masters"], active_idx=st["active"], lr=2e-4, weight_decay=0.005, compact_params=True)
        st["sgd"] = MomentumSGD([st["router"]], lr=2e-4, momentum=0.9, weight_decay=0.005)
        st["scaler"] = DeviceLossScale(device="cuda")
        st["flags"] = torch.tensor([1, 0], dtype=torch.int32, device="cuda")
        st["dy"], st["cg"] = torch.empty_like(st["dout"]), torch.empty_like(st["store"].flat)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(st):
    return _RUN[st["case"]["kind"]](st)


@torch.no_grad()
def _run_codec(st):
    c = st["case"]
    if c["op"] == "both":
        q, s, z, shape = quantization.quantize_4bit(st["w"], c["group"])
    else:
        (q, s, z), shape = st["q"], st["shape"]
    out = quantization.dequantize_4bit(q, s, z, shape, c["group"], out_dtype=DTYPES[c["dtype"]])
    return {"q": q, "s": s, "z": z, "out": out} if c["op"] == "both" else {"out": out}


@torch.no_grad()
def _run_block(st):
    return {"out": st["block"](st["x"])}


@torch.no_grad()
def _run_experts(st):
    return {"out": G.routed_experts(st["x"], st["w"], st["ew"])}


@torch.no_grad()
def _run_cache(st):
    return {f"out{i}": st["cache"].forward(name, st["x"], w, SHAPES[st["case"]["shape"]][3])
            for i, (name, w) in enumerate(zip(st["layers"], st["w"]))}


def _run_frozen(st):
    st["x"].grad = st["w"].grad = None
    out = G.routed_experts(st["x"], st["w"], st["ew"])
    out.backward(st["dout"])
    return {"out": out.detach(), "dx": st["x"].grad, "dw": st["w"].grad}


def _run_train(st):
    st["x"].grad = st["w"].grad = None
    st["store"].zero_()
    out = G.routed_experts(st["x"], st["w"], st["ew"], capture=(st["store"], PREFIX))
    out.backward(st["dout"])
    return {"out": out.detach(), "dx": st["x"].grad, "dw": st["w"].grad, **_by_role(st["store"].compact)}


def _run_dense(st):
    mod = st["mod"]
    st["x"].grad = st["w"].grad = mod.gate_up_proj.grad = mod.down_proj.grad = None
    out = mod(st["x"], st["w"])
    out.backward(st["dout"])
    return {"out": out.detach(), "dx": st["x"].grad, "dw": st["w"].grad, "d_gate_up": mod.gate_up_proj.grad,
            "d_down": mod.down_proj.grad}


def _run_step(st):
    st["x"].grad = st["router"].grad = None
    store, scaler, flags = st["store"], st["scaler"], st["flags"]
    finite, halt = flags[:1], flags[1:]
    store.zero_()
    out = G.moe_block(st["x"], st["router"], SHAPES[st["case"]["shape"]][3], True, st["ew"], capture=(store, PREFIX),
                      overflow=halt)
    out.backward(scaler.scale_grad(st["dout"], out=st["dy"]))
    scaler.unscale_check(store.flat, st["cg"], finite)
    grads = {n: st["cg"][a:a + c] for n, (a, c) in store.spans.items()}
    router_grad = st["router"].grad
    st["sgd"].step(finite=finite, halt=halt, loss_scale=scaler)
    st["adam"].step(compact_grads=grads, finite=finite, halt=halt)
    for name, ov in st["overlays"].items():
        ov.refresh(st["masters"][name].data)
    scaler.update(finite, halt)
    return {"out": out.detach(), "dx": st["x"].grad, "d_router": router_grad, "router": st["router"].detach(),
            **_by_role(grads), **{"new_" + k: v for k, v in _by_role(st["masters"]).items()}, "flags": flags}


def _by_role(d):
    return {("gate_up" if "gate_up" in n else "down"): v.detach() for n, v in d.items()}


_RUN = {"codec": _run_codec, "block": _run_block, "experts": _run_experts, "cache": _run_cache, "frozen": _run_frozen,
        "train": _run_train, "dense": _run_dense, "step": _run_step}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close another implementation comes
# ---------------------------------------------------------------------------

def work(case):
    if case["kind"] == "codec":
        n = case["rows"] * case["cols"]
        coded = n / 2 + 4 * -(-n // case["group"])
        return {"bytes": 2 * n + coded if case["op"] == "dequantize" else 4 * n + 2 * coded, "flops": 0}
    E, H, I, k = SHAPES[case["shape"]]
    T, kind = case["T"], case["kind"]
    used = E * (1 - (1 - k / E) ** T)  # experts some token selects
    flops = 2 * T * k * 3 * H * I
    weights = used * 3 * H * I * (2 if kind in ("dense", "cache") else 0.53125)
    nbytes = weights + 4 * T * H + 4 * T * E
    if kind in ("block", "step"):
        nbytes += 2 * E * H
        flops += 2 * T * E * H
    if kind == "cache":
        return {"bytes": 2 * nbytes, "flops": 2 * flops}
    if kind in ("frozen", "train", "step", "dense"):
        nbytes += weights + 6 * T * H + 4 * T * E
        flops *= 2
    if kind in ("train", "step"):
        n = ACTIVE * E * 3 * H * I
        nbytes += 12 * n + (28 * n if kind == "step" else 0)
        flops += 2 * T * k * ACTIVE * 3 * H * I
    if kind == "dense":
        nbytes += E * 3 * H * I * 2
        flops += 2 * T * k * 3 * H * I
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "codec":
        return "exact"
    # 16-bit activations between the two projections and at the output
    return {"rel": 2e-3 if case["dtype"] == "fp16" else 1.5e-2}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return None
    st = prepare(case, seed)
    if kind == "codec":
        if case["op"] == "both":
            x = st["w"].reshape(-1).double()
            x = torch.cat([x, x.new_zeros(-x.numel() % case["group"])]).view(-1, case["group"])
            mn = x.amin(1)
            return {"q": None, "s": (x.amax(1) - mn) / 15, "z": mn, "out": None}
        (q, s, z), numel = st["q"], math.prod(st["shape"])
        if numel > 1 << 28:
            return None
        out = torch.empty(numel, dtype=torch.float64, device="cuda")
        g = case["group"]
        for a in range(0, q.shape[0], 1 << 18):
            raw = q[a:a + (1 << 18)].view(torch.uint8)
            codes = torch.stack([raw & 15, raw >> 4], dim=2).view(raw.shape[0], -1).double()
            v = (codes * s[a:a + (1 << 18), None].double() + z[a:a + (1 << 18), None].double()).reshape(-1)
            n = min(v.numel(), numel - a * g)
            out[a * g:a * g + n] = v[:n]
        return {"out": out.view(st["shape"])}
    E, H, I, k = SHAPES[case["shape"]]
    dt = DTYPES[case["dtype"]]
    if kind == "cache":
        return {f"out{i}": _exact_experts(case, st["x"], w, ew)["out"]
                for i, (ew, w) in enumerate(zip(st["layers"].values(), st["w"]))}
    if kind == "block":
        x = st["x"].view(-1, H)
        # the router's output is rounded to the layer's dtype, and the selection is made on that
        logits = (x.double() @ st["block"].gate.weight.double().t()).to(dt)
        p = torch.softmax(logits.double(), dim=-1)
        p = p * (p >= p.topk(k, dim=-1).values[:, -1:])
        out = _exact_experts(case, x, p / p.sum(-1, keepdim=True), st["ew"])["out"]
        return {"out": out.view(st["x"].shape)}
    ew = st["mod"] if kind == "dense" else st["ew"]
    return _exact_experts(case, st["x"].detach(), st["w"].detach(), ew, st.get("dout"), st.get("active"), st.get("masters"))


def _exact_experts(case, x, w, ew, dout=None, active=None, masters=None):
    E, H, I, k = SHAPES[case["shape"]]
    dt = DTYPES[case["dtype"]]
    x, w = x.double(), w.double()
    out = torch.zeros_like(x)
    res = {"out": out}
    if dout is not None:
        dout = dout.double()
        res["dx"], res["dw"] = torch.zeros_like(x), torch.zeros_like(w)
    dense = case["kind"] == "dense"
    if dense:
        res["d_gate_up"] = torch.zeros(E, 2 * I, H, dtype=torch.float64, device="cuda")
        res["d_down"] = torch.zeros(E, H, I, dtype=torch.float64, device="cuda")
    spans = {}
    if active is not None:
        for role, per in (("gate_up", 2 * I * H), ("down", H * I)):
            idx = next(v for n, v in active.items() if role in n)
            edges = torch.searchsorted(idx, torch.arange(E + 1, device="cuda") * per).tolist()
            val = next(v for n, v in masters.items() if role in n).detach().half()
            spans[role] = (idx, val, edges, per)
            res[role] = torch.zeros(idx.numel(), dtype=torch.float64, device="cuda")
    for e in range(E):
        rows = w[:, e].nonzero().reshape(-1)
        if not rows.numel():
            continue
        mats = {}
        for role in ("gate_up", "down"):
            if dense:
                m = getattr(ew, role + "_proj").detach()[e]
            else:
                m = _expert_values(getattr(ew, role), e)
                if role in spans:
                    idx, val, edges, per = spans[role]
                    a, b = edges[e], edges[e + 1]
                    m.view(-1)[idx[a:b] - e * per] = val[a:b]
            mats[role] = m.to(dt).double()
        xe, we = x[rows], w[rows, e:e + 1]
        gate, up = (xe @ mats["gate_up"].t()).split(I, dim=1)
        sig = torch.sigmoid(gate)
        act = gate * sig * up
        y = act @ mats["down"].t()
        out.index_add_(0, rows, y * we)
        if dout is None:
            continue
        de = dout[rows]
        res["dw"][rows, e] = (de * y).sum(1)
        dy = de * we
        dact = dy @ mats["down"]
        dgu = torch.cat([dact * up * (sig * (1 + gate * (1 - sig))), dact * gate * sig], dim=1)
        res["dx"].index_add_(0, rows, dgu @ mats["gate_up"])
        if dense:
            res["d_gate_up"][e], res["d_down"][e] = dgu.t() @ xe, dy.t() @ act
        for role, left, right in (("gate_up", dgu, xe), ("down", dy, act)):
            if role in spans:
                idx, _, edges, per = spans[role]
                a, b = edges[e], edges[e + 1]
                res[role][a:b] = (left.t() @ right).reshape(-1)[idx[a:b] - e * per]
    return res
