"""Workloads of the PSSA inference path, as a program calls it.

Every case goes through the public entry points of `pssa_amd`: whole prompts
and ragged batches of prompts, decode steps, the training forward, and the
single stages a host program dispatches by themselves (retrieval, the dense
scan, the selective scan, a projection).  `listed()` names the cases, `draw()`
gives further ones of the same ranges, `prepare()` makes what a program holds
before the call, `run()` is one call, `work()` what it cannot do without and
`exact()` the same result in 64 bits.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from pssa_amd import HipDevice, ModelWeights, PSSAConfig, PSSALayer, Sequence

# The two models of the benchmark: the 105M-scale one (bf16 weights) and the
# small one the reference runs on its CPU path (fp32).
MODELS = {
    "105m": PSSAConfig(depth=12, d_vocab=16384, d_latent=768, d_state=256, d_mem_key=32, mem_capacity=512),
    "small": PSSAConfig(depth=2, d_vocab=8192, d_latent=128, d_state=64, d_mem_key=128, mem_capacity=512),
}
TAU = 0.1


def listed():
    return [
        # One prompt through the small fp32 model: the smallest whole call.
        {"name": "prefill_small_1x512", "path": "prefill", "model": "small", "dtype": "f32", "lanes": 1, "len": 512},
        # One user's prompt: first token latency of the 105M model.
        {"name": "prefill_105m_1x701", "path": "prefill", "model": "105m", "dtype": "bf16", "lanes": 1, "len": 701},
        # A full batch of prompts: the throughput case.
        {"name": "prefill_105m_32x1024", "path": "prefill", "model": "105m", "dtype": "bf16", "lanes": 32, "len": 1024},
        # Prompts as they arrive in a server: every length its own.
        {"name": "ragged_105m_9", "path": "ragged", "model": "105m", "dtype": "bf16",
         "lens": "817,43,256,611,129,90,377,1000,5"},
        # Batched generation with the plastic write rules, steps replayed as a graph.
        {"name": "decode_105m_256", "path": "decode", "model": "105m", "dtype": "bf16", "lanes": 256, "steps": 16,
         "plastic": True, "temperature": 0.0, "penalty": 1.0},
        # One conversation, sampled with the default penalty: time between tokens.
        {"name": "chat_105m_1", "path": "decode", "model": "105m", "dtype": "bf16", "lanes": 1, "steps": 24,
         "plastic": False, "temperature": 0.8, "penalty": 1.25},
        # Training forward (evaluation loss) of a batch of chunks, some short.
        {"name": "train_105m_16", "path": "train", "model": "105m", "dtype": "bf16",
         "lens": "512,512,480,397,512,301,512,128,512,77,512,256,512,64,512,505"},
        # Exact top-8 read of a whole batch's tokens from one bank of wide keys.
        {"name": "top8_32768x768", "path": "retrieve", "queries": 32768, "count": 512, "d_key": 768, "d_val": 768,
         "top_k": 8},
        # Full soft read, partly filled bank, keys of the model's width.
        {"name": "soft_4001x32", "path": "retrieve", "queries": 4001, "count": 389, "d_key": 32, "d_val": 768,
         "top_k": 0},
        # Dense-transition scan at the benchmark's shape.
        {"name": "dense_64x2048x64", "path": "dense", "batch": 64, "len": 2048, "state": 64},
        # Selective scan of one sequence, host arrays in and out (backend stage).
        {"name": "ssm_509x768x256", "path": "ssm", "len": 509, "d": 768, "s": 256},
        # Projection with a resident weight, host arrays in and out (backend stage).
        {"name": "gemm_1000x1536x768", "path": "gemm", "dtype": "f32", "m": 1000, "n": 1536, "k": 768},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    path = rng.choice(["prefill", "prefill", "ragged", "decode", "decode", "train", "retrieve", "retrieve", "dense",
                       "ssm", "gemm"])
    if path == "prefill":
        small = rng.random() < 0.3
        lanes = _log(rng, 1, 32)
        return {"path": path, "model": "small" if small else "105m", "dtype": "f32" if small else "bf16",
                "lanes": lanes, "len": _log(rng, 8, 1024)}
    if path in ("ragged", "train"):
        n = rng.randint(2, 16)
        return {"path": path, "model": "105m", "dtype": "bf16",
                "lens": ",".join(str(_log(rng, 4, 1024 if path == "ragged" else 512)) for _ in range(n))}
    if path == "decode":
        lanes, sampled = _log(rng, 1, 256), rng.random() < 0.4
        return {"path": path, "model": "105m", "dtype": "bf16", "lanes": lanes, "steps": rng.randint(4, 16),
                "plastic": not sampled, "temperature": 0.8 if sampled else 0.0, "penalty": 1.25 if sampled else 1.0}
    if path == "retrieve":
        top_k = rng.choice([0, 4, 8, 16])
        d_key = rng.choice([32, 64, 100, 128]) if top_k == 0 else rng.choice([64, 128, 260, 384, 768])
        return {"path": path, "queries": _log(rng, 16, 8192 if top_k == 0 else 32768), "count": rng.randint(100, 512),
                "d_key": d_key, "d_val": rng.choice([128, 256, 500, 768]), "top_k": top_k}
    if path == "dense":
        return {"path": path, "batch": _log(rng, 1, 64), "len": _log(rng, 32, 2048), "state": rng.choice([16, 48, 64])}
    if path == "ssm":
        d, s = rng.choice([(128, 64), (256, 16), (768, 256)])
        return {"path": path, "len": _log(rng, 8, 1024), "d": d, "s": s}
    return {"path": "gemm", "dtype": rng.choice(["f32", "bf16"]), "m": _log(rng, 1, 1024),
            "n": rng.choice([32, 128, 500, 768, 1536, 2096]), "k": rng.choice([128, 500, 768, 1536])}


# ---------------------------------------------------------------------------
# What a program holds before the call.


@functools.lru_cache(maxsize=None)
def _device():
    return HipDevice(0)


@functools.lru_cache(maxsize=None)
def _weights(model):
    w = ModelWeights.init(MODELS[model], 0, "baseline")
    w.populate_banks(1)
    return w


def _lens(case):
    return [int(v) for v in case["lens"].split(",")] if "lens" in case else [case["len"]] * case["lanes"]


def _ids(case, seed, lens):
    rng = np.random.default_rng(seed)
    return [rng.integers(0, MODELS[case["model"]].d_vocab, n, dtype=np.uint32) for n in lens]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _ball(gen, n, dim):
    """Rows uniform in direction, norms uniform in [0, 0.9)."""
    v = torch.randn(n, dim, generator=gen, device="cuda", dtype=torch.float32)
    r = torch.rand(n, 1, generator=gen, device="cuda", dtype=torch.float32) * 0.9
    return (v / v.norm(dim=1, keepdim=True) * r).contiguous()


def _bank(case, seed):
    g = _gen(seed)
    keys, values = _ball(g, 512, case["d_key"]), _ball(g, 512, case["d_val"])
    return _ball(g, case["queries"], case["d_key"]), keys, keys.double().square().sum(1).float(), values


def _transitions(case, seed):
    """Orthogonal matrices (two reflections) scaled by U[0.8, 0.99], and drives N(0, 1)."""
    g, (n, L, s) = _gen(seed), (case["batch"], case["len"], case["state"])
    u, v = (torch.nn.functional.normalize(torch.randn(n, L, s, generator=g, device="cuda"), dim=-1) for _ in range(2))
    f = torch.rand(n, L, 1, 1, generator=g, device="cuda") * 0.19 + 0.8
    a = torch.eye(s, device="cuda").expand(n, L, s, s) - 2 * u[..., :, None] * u[..., None, :]
    w = torch.matmul(a, v[..., :, None])
    a = f * (a - 2 * w * v[..., None, :])
    return a.contiguous(), torch.randn(n, L, s, generator=g, device="cuda")


def _scan_inputs(case, seed):
    rng, (L, d, s) = np.random.default_rng(seed), (case["len"], case["d"], case["s"])
    f = np.float32
    delta = np.logaddexp(0.0, rng.normal(0.0, 0.6, (L, d))).astype(f)
    rates = -(1.0 / np.broadcast_to(np.linspace(1.5, 13.0, s), (d, s))).astype(f)
    return {"delta": delta, "b": rng.normal(0, 0.5, (L, s)).astype(f), "x": rng.normal(0, 1, (L, d)).astype(f),
            "rates": rates, "c": rng.normal(0, 0.5, (L, s)).astype(f), "h": rng.normal(0, 0.1, (d, s)).astype(f)}


def _projection(case, seed):
    rng, (m, n, k) = np.random.default_rng(seed), (case["m"], case["n"], case["k"])
    x, w = rng.normal(0, 1, (m, k)).astype(np.float32), rng.normal(0, 0.02, (n, k)).astype(np.float32)
    if case["dtype"] == "bf16":
        w = torch.from_numpy(w).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)
    return x, w


def prepare(case, seed):
    path, dev = case["path"], _device()
    if path in ("prefill", "ragged", "train"):
        lens = _lens(case)
        layer = PSSALayer(dev, _weights(case["model"]), lanes=len(lens), max_tokens=sum(lens),
                          weight_dtype=case["dtype"])
        ids = _ids(case, seed, lens)
        st = {"layer": layer, "ids": np.stack(ids) if path == "prefill" else ids}
        if path == "train":
            st["batch"] = [Sequence(i, q, np.roll(q, -1), True) for i, q in enumerate(ids)]
    elif path == "decode":
        # Every stream stands behind a 48-token prompt.
        ids = np.stack(_ids(case, seed, [49] * case["lanes"]))
        layer = PSSALayer(dev, _weights(case["model"]), lanes=case["lanes"], max_tokens=48 * case["lanes"],
                          weight_dtype=case["dtype"])
        layer.set_repetition_penalty(case["penalty"])
        if case["temperature"] > 0:
            layer.set_sampling(case["temperature"], seed=seed)
        layer.prefill_inference(ids[:, :48], want_logits=False)
        st = {"layer": layer, "first": ids[:, 48].copy()}
    elif path == "retrieve":
        q, keys, norm_sq, values = _bank(case, seed)
        n = case["queries"]
        st = {"dev": dev, "q": q, "keys": keys, "norm_sq": norm_sq, "values": values,
              "val": torch.empty(n, case["d_val"], device="cuda"), "min": torch.empty(n, device="cuda"),
              "idx": torch.empty(n, case["top_k"], dtype=torch.int32, device="cuda") if case["top_k"] else None}
    elif path == "dense":
        a, b = _transitions(case, seed)
        dev.dense_scan_reserve(case["batch"], case["len"], case["state"])
        st = {"dev": dev, "a": a, "b": b, "h": torch.empty_like(b)}
    elif path == "ssm":
        st = {"dev": dev, **_scan_inputs(case, seed)}
    else:
        x, w = _projection(case, seed)
        st = {"dev": dev, "x": x, "w": w}
        # The weight's device copy is keyed by its address: this array's is new.
        dev.invalidate_weights_only([w])
    torch.cuda.synchronize()
    return {"case": dict(case), **st}


def run(state):
    case, path = state["case"], state["case"]["path"]
    if path == "prefill":
        state["layer"].reset_recurrent_state()
        logits = state["layer"].prefill_inference(state["ids"])
        # A small model's conversation is kept by its program; the large one's state stays on the GPU.
        return [logits, state["layer"].get_carry()] if case["model"] == "small" else logits
    if path == "ragged":
        state["layer"].reset_recurrent_state()
        return state["layer"].prefill_ragged(state["ids"])
    if path == "train":
        loss, token_losses = state["layer"].batch_forward(state["batch"], want_token_losses=True)
        return [loss, token_losses]
    if path == "decode":
        ids, logits = state["layer"].decode(case["steps"], first_ids=state["first"], plastic=case["plastic"],
                                            graph=True, want_logits=True)
        return [ids, logits]
    dev = state["dev"]
    if path == "retrieve":
        idx = state["idx"]
        dev.retrieve_resident(state["q"].data_ptr(), case["queries"], state["keys"].data_ptr(),
                              state["norm_sq"].data_ptr(), state["values"].data_ptr(), 512, case["count"],
                              case["d_key"], case["d_val"], TAU, case["top_k"], state["val"].data_ptr(),
                              state["min"].data_ptr(), None if idx is None else idx.data_ptr())
        return [state["val"], state["min"]] + ([] if idx is None else [idx])
    if path == "dense":
        dev.dense_scan_resident(state["a"].data_ptr(), state["b"].data_ptr(), None, case["batch"], case["len"],
                                case["state"], state["h"].data_ptr())
        return state["h"]
    if path == "ssm":
        _, _, _, y, final = dev.ssm_forward(state["delta"], state["b"], state["x"], state["rates"], state["c"],
                                            state["h"], case["len"], case["d"], case["s"], materialize=False)
        return [y, final]
    return dev.try_dispatch_gemm(state["x"], state["w"], case["m"], case["n"], case["k"], w_dtype=case["dtype"],
                                 resident=True)


# ---------------------------------------------------------------------------
# What the path cannot do without.


def _model_work(case, tokens, lanes, passes, heads):
    """`tokens` through the blocks in `passes` passes (each reads the weights
    and advances the carries of `lanes`), and `heads` rows of logits."""
    c, wb = MODELS[case["model"]], 2 if case["dtype"] == "bf16" else 4
    d, s, k, C, r, V = c.d_latent, c.d_state, c.d_mem_key, c.mem_capacity, c.adapter_rank, c.d_vocab
    mac = d * (2 * d + 2 * s + k + r) + d * k + C * k + C * d + d * d + d * r + 4 * d * d
    weights = c.depth * (d * (2 * d + 2 * s + k + r) + k * d + 5 * d * d + C * d + d * r) * wb + V * d * wb
    weights += c.depth * (d * s + C * k) * 4
    flops = c.depth * tokens * (2.0 * mac + 6.0 * d * s) + 2.0 * heads * V * d
    return {"bytes": passes * (weights + 2.0 * lanes * c.depth * d * s * 4) + tokens * d * 4 + heads * V * 4,
            "flops": flops}


def work(case):
    path = case["path"]
    if path in ("prefill", "ragged", "train"):
        lens = _lens(case)
        w = _model_work(case, sum(lens), len(lens), 1, sum(lens) if path == "train" else len(lens))
        if case["model"] == "small":  # the states leave too
            c = MODELS["small"]
            w["bytes"] += 4.0 * len(lens) * c.depth * c.d_latent * c.d_state
        if path == "train":  # one loss per token leaves, the logits stay inside
            w["bytes"] -= 4.0 * sum(lens) * (MODELS[case["model"]].d_vocab - 1)
        return w
    if path == "decode":
        n = case["lanes"] * case["steps"]
        w = _model_work(case, n, case["lanes"], case["steps"], n)
        w["bytes"] -= 4.0 * (n - case["lanes"]) * MODELS[case["model"]].d_vocab  # only the last logits leave
        return w
    if path == "retrieve":
        n, c, dk, dv, k = case["queries"], case["count"], case["d_key"], case["d_val"], case["top_k"]
        return {"bytes": 4.0 * (n * dk + c * (dk + dv + 1) + n * (dv + 1 + k)),
                "flops": 2.0 * n * c * dk + 2.0 * n * (k or c) * dv}
    if path == "dense":
        n = case["batch"] * case["len"]
        return {"bytes": 4.0 * n * (case["state"] ** 2 + 2 * case["state"]), "flops": 2.0 * n * case["state"] ** 2}
    if path == "ssm":
        L, d, s = case["len"], case["d"], case["s"]
        return {"bytes": 4.0 * (3 * L * d + 2 * L * s + 3 * d * s), "flops": 6.0 * L * d * s}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": 4.0 * (m * k + m * n) + (4.0 if case["dtype"] == "f32" else 2.0) * n * k, "flops": 2.0 * m * n * k}


def tolerance(case):
    """About four times the largest error against `exact` over listed and drawn cases; a whole bf16 model is off by
    0.6-1.6% (every operand of twelve layers rounded to eight bits)."""
    path = case["path"]
    if path in ("prefill", "ragged", "decode"):
        return {"rel": 3e-2, "max": 0.6, "differ": 0.0} if case["dtype"] == "bf16" else {"rel": 2e-6, "max": 1.2e-5}
    if path == "train":  # losses near ln(vocab): an error of the logits is small against them
        return {"rel": 8e-5, "max": 2e-3}
    if path == "retrieve":
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.0}
    if path == "dense":
        return {"rel": 1e-6, "max": 2.5e-5}
    if path == "ssm":
        return {"rel": 1e-6, "max": 8e-6}
    return {"rel": 2e-6, "max": 2e-5} if case["dtype"] == "f32" else {"rel": 1e-2, "max": 5e-2}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch.


def _scan64(delta, rates, b, c, x, h):
    """delta, x [n, T, d], b, c [n, T, s], rates [d, s], h [n, d, s] (advanced in place); y [n, T, d]."""
    y = torch.empty_like(delta)
    for t in range(delta.shape[1]):
        dt = delta[:, t, :, None]
        h.mul_((dt * rates).exp_()).add_((delta[:, t] * x[:, t])[..., None] * b[:, t, None, :])
        y[:, t] = torch.matmul(h, c[:, t, :, None])[..., 0]
    return y


def _softmax_read64(q, keys, norm_sq, values, top_k):
    """Poincare distances of q to the bank's keys, softmax weights, values and the least distance."""
    qq = q.square().sum(-1, keepdim=True)
    sq = (qq + keys.square().sum(-1) - 2.0 * q @ keys.T).clamp_min_(0.0)
    if top_k:  # the ranking is defined on the query's 32-bit norm, as the bank's keys have it stored
        qq = qq.float().double()
    dist = 2.0 * torch.asinh((sq / ((1.0 - qq) * (1.0 - norm_sq))).sqrt())
    low = dist.amin(-1, keepdim=True)
    w = torch.exp((low - dist) / TAU)
    if 0 < top_k < dist.shape[-1]:  # ranked by the 32-bit distance, then by the slot
        best = dist.float().sort(dim=-1, stable=True).indices[..., :top_k]
        w = torch.zeros_like(w).scatter(-1, best, w.gather(-1, best))
    return (w / w.sum(-1, keepdim=True)) @ values, low[..., 0]


def _features64(case, seqs):
    """Output rows [n, T, d] of the blocks for the id rows, short ones padded at their ends, the head and the
    blocks' last states."""
    cfg, w, bf16 = MODELS[case["model"]], _weights(case["model"]), case["dtype"] == "bf16"
    T = max(len(q) for q in seqs)
    ids = torch.tensor(np.stack([np.pad(q.astype(np.int64), (0, T - len(q))) for q in seqs]), device="cuda")

    def f64(a):
        return torch.from_numpy(a).to("cuda", torch.float64)

    def mat(a):  # in the model's weight type
        t = torch.from_numpy(a).to("cuda")
        return (t.to(torch.bfloat16) if bf16 else t).double()

    F = torch.nn.functional
    h, carries = f64(w.embed)[ids], []
    for i, b in enumerate(w.blocks):
        x = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-5) * f64(b.norm_gamma) + f64(b.norm_beta)
        delta = F.softplus(x @ mat(b.w_delta).T, threshold=1e9)
        carry = torch.zeros(h.shape[0], cfg.d_latent, cfg.d_state, dtype=torch.float64, device="cuda")
        rates = -F.softplus(f64(b.a_raw), threshold=1e9)
        y = _scan64(delta, rates, x @ mat(b.w_b).T, x @ mat(b.w_c).T, x, carry)
        q = y @ mat(b.w_qh).T + x @ mat(b.w_qx).T
        r = q.norm(dim=-1, keepdim=True)
        q = q * ((r / (1.0 + r)).clamp_max(1.0 - 8.0 * 2.0 ** -23) / r.clamp_min(1e-300))
        n = int(b.mem_count)
        m, _ = _softmax_read64(q, f64(b.mem_keys[:n]), f64(b.mem_norm_sq[:n]), mat(b.mem_values[:n]), 0)
        act = F.silu(x @ mat(b.adapter_down).T) @ mat(b.adapter_up + b.adapter_slow).T
        z = y / math.sqrt(cfg.d_state) + torch.sigmoid(x @ mat(b.w_gate).T) * (m @ mat(b.w_proj).T) + act
        z = z + F.silu(z @ mat(b.mlp_w1).T) @ mat(b.mlp_w2).T
        h = z if i == 0 else h + z / math.sqrt(cfg.depth)
        carries.append(carry.flatten(1).cpu() if case["model"] == "small" else None)
    return h, mat(w.unembed).T / math.sqrt(cfg.d_latent), carries


def exact(case, seed):
    path = case["path"]
    if path in ("prefill", "ragged", "train"):
        seqs = _ids(case, seed, _lens(case))
        h, head, carries = _features64(case, seqs)
        if path != "train":
            logits = (torch.stack([h[i, len(q) - 1] for i, q in enumerate(seqs)]) @ head).cpu().numpy()
            return [logits, torch.stack(carries, 1).numpy()] if case["model"] == "small" else logits
        loss = []
        for i, q in enumerate(seqs):
            target = torch.from_numpy(np.roll(q, -1).astype(np.int64)).cuda()
            loss.append(torch.nn.functional.cross_entropy(h[i, :len(q)] @ head, target, reduction="none"))
        loss = torch.cat(loss).cpu().numpy()
        return [float(loss.mean()), loss]
    if path == "decode":  # every token depends on the choice before it: no value of its own
        return None
    if path == "retrieve":
        q, keys, norm_sq, values = (t.double() for t in _bank(case, seed))
        n = case["count"]
        val, low = _softmax_read64(q, keys[:n], norm_sq[:n], values[:n], case["top_k"])
        return [val, low] + ([None] if case["top_k"] else [])
    if path == "dense":
        a, b = _transitions(case, seed)
        h, out = torch.zeros_like(b[:, 0], dtype=torch.float64), torch.empty_like(b, dtype=torch.float64)
        for t in range(b.shape[1]):
            h = (a[:, t].double() * h[:, None, :]).sum(-1) + b[:, t]
            out[:, t] = h
        return out
    if path == "ssm":
        t = {k: torch.from_numpy(v).to("cuda", torch.float64) for k, v in _scan_inputs(case, seed).items()}
        h = t["h"][None].clone()
        y = _scan64(t["delta"][None], t["rates"], t["b"][None], t["c"][None], t["x"][None], h)
        return [y.reshape(-1).cpu().numpy(), h.reshape(-1).cpu().numpy()]
    x, w = _projection(case, seed)
    w = torch.from_numpy(w) if case["dtype"] == "f32" else torch.from_numpy(w.view(np.int16)).view(torch.bfloat16)
    return (torch.from_numpy(x).to("cuda", torch.float64) @ w.to("cuda", torch.float64).T).reshape(-1).cpu().numpy()
