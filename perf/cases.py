"""What a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values with a "kind":

  router      one token's fused fp16 router: RMSNorm of the residual, logits, top-k, the next layer's
              prediction (every decoded token, every layer)
  router_q8   the same for the checkpoint's 8-bit affine router (bf16)
  glu         one token through the k selected experts of a layer (every decoded token, every
              layer); form "blob" (one blob per expert) or the checkpoint's 9 tensors ("bf16" /
              "fp16" scales and biases)
  codebook    one token through the k selected 2-bit codebook experts of a layer
  prefill     a prompt chunk through one layer: rows sorted by expert, the grouped SwitchGLU, the
              score-weighted combine; forms as glu
  resident    whole decoded tokens through a stack of layers with every expert in HBM
  cached      whole decoded tokens through a stack of layers with 20% of the experts in HBM, the
              misses copied from the pinned host store, next-layer prefetch on

Sizes are those of the repository's workloads: 48 layers of 2048 x 512 (512 experts, top-10), the
checkpoint's 2560 x 640, the codebook model's 3072 x 1536 (240 experts, top-9); prompts up to the
server's 2048-token chunk.  The stacks have fewer layers than the 48 of the workload: a layer costs
the same in each.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

if os.path.join(os.getcwd(), "moe-offload_amd") not in sys.path:
    sys.path.insert(0, os.path.join(os.getcwd(), "moe-offload_amd"))

from moe_offload import _lib, cbformat, cbstack, ops, prefill, q2format, stack, synth  # noqa: E402

GROUP = 64
EPS = 1e-6
MAX_LAYERS = 64          # layer indices of the library; stacks take theirs in turn
PER_STACK = 4


def listed():
    real = {"hidden": 2560, "inter": 640, "n_exp": 512, "k": 10}
    work = {"hidden": 2048, "inter": 512, "n_exp": 512, "k": 10}
    return [
        # the smallest calls: one launch each, on every decoded token's critical path
        {"name": "router_2048", "kind": "router", "hidden": 2048, "n_exp": 512, "k": 10, "m": 12},
        {"name": "router_q8_2560", "kind": "router_q8", "hidden": 2560, "n_exp": 512, "k": 10},
        # decode of one layer's experts, batch 1
        {"name": "glu_blob_2048", "kind": "glu", "form": "blob", **work},
        {"name": "glu_bf16_2560", "kind": "glu", "form": "bf16", **real},
        {"name": "codebook_3072", "kind": "codebook", "hidden": 3072, "inter": 1536, "n_exp": 240, "k": 9},
        # a short prompt through the real model's layer: few rows per expert
        {"name": "prefill_bf16_37", "kind": "prefill", "form": "bf16", "tokens": 37, **real},
        # the ordinary chunk (512 tokens, about 10 rows per expert) in both formats
        {"name": "prefill_blob_512", "kind": "prefill", "form": "blob", "tokens": 512, **work},
        {"name": "prefill_bf16_512", "kind": "prefill", "form": "bf16", "tokens": 512, **real},
        # the server's largest chunk (2048 tokens, about 40 rows per expert)
        {"name": "prefill_bf16_2048", "kind": "prefill", "form": "bf16", "tokens": 2048, **real},
        # odd sizes: a ragged prompt, sizes that are no power of two, few experts with long segments
        {"name": "prefill_fp16_odd", "kind": "prefill", "form": "fp16", "tokens": 777, "hidden": 1152, "inter": 320,
         "n_exp": 100, "k": 6},
        # whole calls: 4 layers; the cached stack decodes 16 tokens, whose experts do not fit its
        # 102 slots a layer, so every token has hits and misses
        {"name": "resident_4x4", "kind": "resident", "layers": 4, "tokens": 4, **work},
        {"name": "cached_4x16", "kind": "cached", "layers": 4, "tokens": 16, **work},
    ]


def _log(rng, lo, hi, step):
    """A multiple of step between lo and hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, step * round(v / step))))


def draw(rng):
    kind = rng.choice(["router", "router_q8", "glu", "glu", "codebook", "prefill", "prefill", "prefill", "resident", "cached"])
    if kind in ("router", "router_q8"):
        n_exp = _log(rng, 33, 1024, 1)
        c = {"kind": kind, "hidden": _log(rng, 512, 4096, 8 if kind == "router" else 64), "n_exp": n_exp,
             "k": rng.randint(1, 16)}
        if kind == "router":
            c["m"] = rng.choice([0, rng.randint(1, 32)])
        return c
    if kind == "codebook":
        return {"kind": kind, "hidden": 256 * rng.randint(2, 16), "inter": 256 * rng.randint(1, 8),
                "n_exp": _log(rng, 16, 240, 1), "k": rng.randint(1, 16)}
    if kind == "glu":
        return {"kind": kind, "form": rng.choice(["blob", "bf16", "fp16"]), "hidden": _log(rng, 512, 4096, 64),
                "inter": _log(rng, 128, 1024, 64), "n_exp": _log(rng, 16, 512, 1), "k": rng.randint(1, 16)}
    if kind == "prefill":
        while True:
            h, i = _log(rng, 256, 2560, 64), _log(rng, 128, 1024, 64)
            if h * i <= 2560 * 640:
                break
        n_exp = _log(rng, 16, 512, 1)
        return {"kind": kind, "form": rng.choice(["blob", "bf16", "fp16"]), "tokens": _log(rng, 2, 2048, 1), "hidden": h,
                "inter": i, "n_exp": n_exp, "k": rng.randint(2, 10)}
    tokens = rng.randint(1, 4) if kind == "resident" else rng.randint(8, 16)
    return {"kind": kind, "layers": rng.randint(2, PER_STACK), "tokens": tokens, "hidden": rng.choice([1024, 2048]),
            "inter": 64 * rng.randint(2, 8), "n_exp": _log(rng, 64, 512, 1), "k": rng.randint(2, 10)}


# ---- inputs -------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _nine(case, g):
    """A layer's 9 pools in role order (gate, up, down: codes, scales, biases), slot = expert."""
    H, I, E = case["hidden"], case["inter"], case["n_exp"]
    dt = torch.bfloat16 if case["form"] == "bf16" else torch.float16
    out = []
    for rows, cols in ((I, H), (I, H), (H, I)):
        w = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, rows, cols // 16), dtype=torch.int32, device="cuda", generator=g)
        s = (torch.randn((E, rows, cols // GROUP), device="cuda", generator=g) * 0.02).to(dt)
        out += [w, s, (-1.5 * s.float()).to(dt)]
    return out


def _u64(values):
    return (ctypes.c_uint64 * 9)(*values)


def _experts(case, g):
    if case["form"] == "blob":
        return {"pool": stack.random_blobs(case["n_exp"], case["hidden"], case["inter"], GROUP, g, torch.device("cuda"))}
    t = _nine(case, g)
    return {"nine": t, "ptrs": _u64([a.data_ptr() for a in t]),
            "slot_bytes": _u64([a[0].numel() * a.element_size() for a in t]), "bf16": int(case["form"] == "bf16")}


def _selection(case, g):
    k, E = min(case["k"], case["n_exp"]), case["n_exp"]
    ids = torch.randperm(E, device="cuda", generator=g)[:k].to(torch.int32)
    s = torch.rand(k, device="cuda", generator=g) + 0.05
    return ids, (s / s.sum()).half()


class _Stack:
    """A decode stack that gives its layers, pools and host store back when it is dropped."""
    taken = 0

    def __init__(self, case, seed):
        base = (_Stack.taken % (MAX_LAYERS // PER_STACK)) * PER_STACK
        _Stack.taken += 1
        resident = case["kind"] == "resident"
        cfg = stack.StackConfig(n_layers=case["layers"], hidden=case["hidden"], n_exp=case["n_exp"], top_k=case["k"],
                                inter=case["inter"], budget_pct=20.0, prefetch=not resident, resident=resident,
                                seed=int(seed), layer_base=base)
        self.st = stack.DecodeStack(cfg, mode="device")
        if not resident:
            self.st.reset_caches()
            self.st.reset_stats()
        self.st.capture_graph()

    def __del__(self):
        if getattr(self, "st", None) is not None:
            self.st.close()


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    s = {"case": case, "seed": int(seed)}
    dev = torch.device("cuda")
    if kind == "router":
        H, E = case["hidden"], case["n_exp"]
        s["w"] = (torch.randn((E, H), device=dev, generator=g) * 0.02).half()
        s["w_next"] = (torch.randn((E, H), device=dev, generator=g) * 0.02).half() if case["m"] else None
        s["norm_w"] = (1.0 + 0.1 * torch.randn(H, device=dev, generator=g)).half()
        s["h"] = torch.randn(H, device=dev, generator=g) * 1.5
        s["x_out"] = torch.empty(H, dtype=torch.float16, device=dev)
        s["k"], s["m"] = min(case["k"], E), min(case["m"], E)
    elif kind == "router_q8":
        H, E = case["hidden"], case["n_exp"]
        s["codes"] = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, H // 4), dtype=torch.int32, device=dev, generator=g)
        s["scales"] = (torch.rand((E, H // GROUP), device=dev, generator=g) * 1e-3).to(torch.bfloat16)
        s["biases"] = (-127.5 * s["scales"].float()).to(torch.bfloat16)
        s["norm_w"] = (1.0 + 0.1 * torch.randn(H, device=dev, generator=g)).to(torch.bfloat16)
        s["h"] = torch.randn(H, device=dev, generator=g) * 1.5
        s["k"] = min(case["k"], E)
        s["ws"] = torch.zeros(int(_lib.lib().moe_router_q8_workspace_bytes(E)), dtype=torch.uint8, device=dev)
        s["xb"] = torch.empty(H, dtype=torch.bfloat16, device=dev)
        s["xh"] = torch.empty(H, dtype=torch.float16, device=dev)
        s["ids"] = torch.empty(s["k"], dtype=torch.int32, device=dev)
        s["scores"] = torch.empty(s["k"], dtype=torch.bfloat16, device=dev)
    elif kind == "glu":
        s.update(_experts(case, g))
        s["ids"], s["scores"] = _selection(case, g)
        s["x"] = torch.randn(case["hidden"], device=dev, generator=g).half()
        s["h_ws"] = torch.empty(s["ids"].numel() * case["inter"], dtype=torch.float16, device=dev)
        s["y"] = torch.empty(case["hidden"], dtype=torch.float32, device=dev)
    elif kind == "codebook":
        s["pool"] = cbstack.gpu_random_blobs(case["n_exp"], case["hidden"], case["inter"], g, dev, 0.01)
        s["grid"] = torch.from_numpy(cbformat.grid()).to(dev)
        s["ids"], s["scores"] = _selection(case, g)
        s["x"] = torch.randn(case["hidden"], device=dev, generator=g).half()
    elif kind == "prefill":
        s.update(_experts(case, g))
        T, k = case["tokens"], min(case["k"], case["n_exp"])
        ids, sc = synth.prefill_routing(T, k, case["n_exp"], seed=int(seed) + 1)
        s["ids_np"] = ids
        s["scores"] = torch.from_numpy(sc).to(dev)
        s["x"] = torch.randn((T, case["hidden"]), device=dev, generator=g).half()
        s["row_token"], s["row_out"], s["seg_start"], s["seg_slot"] = [
            torch.from_numpy(a).to(dev) for a in prefill.resident_plan(ids, k)]
        s["h_ws"] = torch.empty((T * k, case["inter"]), dtype=torch.float16, device=dev)
        s["y"] = torch.empty((T * k, case["hidden"]), dtype=torch.float16, device=dev)
        s["out"] = torch.empty((T, case["hidden"]), dtype=torch.float32, device=dev)
    else:
        s["stack"] = _Stack(case, seed)
        T, H = case["tokens"], case["hidden"]
        s["xs"] = torch.randn((T, H), device=dev, generator=g).half()
        s["out"] = torch.empty((T, H), dtype=torch.float16, device=dev)
        s["logits"] = torch.empty((T, case["n_exp"]), dtype=torch.float32, device=dev)
    return s


# ---- one pass -----------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "router":
        ids, scores, pred = ops.router(s["w"], s["k"], h=s["h"], norm_w=s["norm_w"], eps=EPS, w_next=s["w_next"],
                                       m=s["m"], x_out=s["x_out"])
        return {"ids": ids, "scores": scores, "x": s["x_out"]} | ({} if pred is None else {"pred": pred})
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "router_q8":
        _lib.check(_lib.lib().moe_router_q8_norm(
            s["h"].data_ptr(), s["norm_w"].data_ptr(), EPS, s["xb"].data_ptr(), s["xh"].data_ptr(), s["codes"].data_ptr(),
            s["scales"].data_ptr(), s["biases"].data_ptr(), case["hidden"], case["n_exp"], GROUP, s["k"], 0,
            s["ws"].data_ptr(), s["ids"].data_ptr(), s["scores"].data_ptr(), None, None, stream), "moe_router_q8_norm")
        return {"ids": s["ids"], "scores": s["scores"], "x_bf16": s["xb"], "x_f16": s["xh"]}
    if kind == "glu" and case["form"] == "blob":
        return ops.q2_switch_glu(s["x"], s["pool"], s["ids"], case["hidden"], case["inter"], scores=s["scores"],
                                 residual=s["x"], h_ws=s["h_ws"], out=s["y"])
    if kind == "glu":
        _lib.check(_lib.lib().moe_q2t_switch_glu(
            s["x"].data_ptr(), s["ptrs"], s["slot_bytes"], s["bf16"], case["n_exp"], s["ids"].data_ptr(),
            s["scores"].data_ptr(), s["ids"].numel(), case["hidden"], case["inter"], GROUP, s["x"].data_ptr(),
            s["h_ws"].data_ptr(), s["y"].data_ptr(), 0, stream), "moe_q2t_switch_glu")
        return s["y"]
    if kind == "codebook":
        return ops.cb_moe(s["x"], s["pool"], s["ids"], s["grid"], case["hidden"], case["inter"], scores=s["scores"],
                          residual=s["x"])
    if kind == "prefill":
        if case["form"] == "blob":
            ops.q2_grouped_switch_glu(s["x"], s["row_token"], s["seg_start"], s["pool"], case["hidden"], case["inter"],
                                      row_out=s["row_out"], n_out_rows=s["y"].shape[0], seg_slot=s["seg_slot"],
                                      h_ws=s["h_ws"], out=s["y"])
        else:
            m = s["y"].shape[0]
            _lib.check(_lib.lib().moe_q2t_grouped_switch_glu(
                s["x"].data_ptr(), case["tokens"], s["row_token"].data_ptr(), s["row_out"].data_ptr(), m, m,
                s["seg_start"].data_ptr(), s["seg_slot"].data_ptr(), s["seg_slot"].numel(), s["ptrs"], s["slot_bytes"],
                s["bf16"], case["n_exp"], case["hidden"], case["inter"], GROUP, s["h_ws"].data_ptr(), s["y"].data_ptr(),
                stream), "moe_q2t_grouped_switch_glu")
        return {"rows": s["y"], "out": ops.pair_combine(s["y"], s["scores"], out=s["out"])}
    st = s["stack"].st
    resident = kind == "resident"
    for t in range(case["tokens"]):
        s["out"][t].copy_(st.decode_token(s["xs"][t]))
        if resident:
            s["logits"][t].copy_(st.logits[case["layers"] - 1])
    return {"x": s["out"], "logits": s["logits"]} if resident else {"x": s["out"]}


# ---- what a pass cannot do without ---------------------------------------------------------------

def _expert_bytes(case):
    H, I = case["hidden"], case["inter"]
    return 3 * H * I // 4 + 3 * (H * I // GROUP) * 4


def work(case):
    kind, H = case["kind"], case["hidden"]
    if kind == "router":
        rows = case["n_exp"] * (2 if case["m"] else 1)
        return {"bytes": rows * H * 2 + H * 8, "flops": 2 * rows * H}
    if kind == "router_q8":
        return {"bytes": case["n_exp"] * (H + 4 * (H // GROUP)) + H * 10, "flops": 2 * case["n_exp"] * H}
    I, k, E = case["inter"], min(case["k"], case["n_exp"]), case["n_exp"]
    if kind == "glu":
        return {"bytes": k * _expert_bytes(case) + H * 8, "flops": 6 * k * H * I}
    if kind == "codebook":
        return {"bytes": k * cbformat.expert_bytes(H, I) + H * 8, "flops": 4 * k * H * I}
    if kind == "prefill":
        T = case["tokens"]
        touched = E * (1.0 - (1.0 - k / E) ** T)
        return {"bytes": touched * _expert_bytes(case) + T * H * 2 + T * k * H * 2 + T * H * 4, "flops": 6 * T * k * H * I}
    per = k * _expert_bytes(case) + E * H * 2
    return {"bytes": case["tokens"] * case["layers"] * per, "flops": case["tokens"] * case["layers"] * (6 * k * H * I + 2 * E * H)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("router", "router_q8"):
        return "exact"            # 64-bit sums, each result rounded once to its 16-bit type
    # about four times the distance from exact() that the present kernels show
    if kind == "glu":
        return {"rel": 1.5e-4, "max": 1e-3}    # 32-bit sums; the intermediate rounded to fp16 (3e-5)
    if kind == "codebook":
        return {"rel": 6e-3, "max": 3e-2}      # the intermediate rounded to bf16 (1.6e-3)
    if kind == "prefill":
        return {"rel": 1.6e-3, "max": 1e-2}    # weights, intermediate and rows rounded to fp16 (4e-4)
    # fp16 between the layers (4e-4); where two gates are equal to the last bits, another rounding of
    # the layer before selects the other expert, which moves that token by about 3e-2
    return {"rel": 2e-2, "max": 2e-1}


# ---- the same in 64 bits -------------------------------------------------------------------------

def _q2_rows(w, s, b):
    """int32 codes [rows, K/16], scales and biases [rows, K/64] -> the weights [rows, K] in 64 bits."""
    sh = torch.arange(0, 32, 2, device=w.device, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> sh) & 3).reshape(w.shape[0], -1, GROUP).double()
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(w.shape[0], -1)


def _q2_expert(case, s, e, pool=None):
    """(gate, up, down) of one expert in 64 bits."""
    H, I = case["hidden"], case["inter"]
    if pool is None and "nine" in s:
        t = s["nine"]
        return [_q2_rows(t[3 * p][e], t[3 * p + 1][e], t[3 * p + 2][e]) for p in range(3)]
    blob = (s["pool"] if pool is None else pool)[e]
    o = q2format.blob_offsets(H, I, GROUP)
    out = []
    for name, rows, cols in (("gate", I, H), ("up", I, H), ("down", H, I)):
        w = blob[o[name + "_codes"]:o[name + "_codes"] + rows * cols // 4].view(torch.int32).reshape(rows, cols // 16)
        n = rows * (cols // GROUP)
        sb = blob[o[name + "_sb"]:o[name + "_sb"] + 4 * n].view(torch.float16).reshape(rows, cols // GROUP, 2)
        out.append(_q2_rows(w, sb[..., 0], sb[..., 1]))
    return out


def _swiglu(x, gate, up, down):
    g, u = x @ gate.T, x @ up.T
    return (g / (1.0 + torch.exp(-g)) * u) @ down.T


def _np64(t):
    return t.detach().double().cpu().numpy()


def _bf16(v):
    """64-bit values rounded once, to nearest even, to bf16 (normal range)."""
    b = np.ascontiguousarray(np.asarray(v, np.float64)).view(np.int64)
    r = ((b + (1 << 44) - 1 + ((b >> 45) & 1)) >> 45) << 45
    return r.view(np.float64)


def _f16(v):
    return np.asarray(v, np.float64).astype(np.float16).astype(np.float64)


def _norm(h, norm_w, rnd):
    h = _np64(h)
    return rnd(h / np.sqrt(np.mean(h * h) + np.float64(np.float32(EPS))) * _np64(norm_w))


def _route(logits, k, rnd):
    """The router's rule: ids in ascending order of the rounded gates (equal gates by id), scores."""
    g = np.exp(logits - logits.max())
    g = rnd(g / g.sum())
    ids = np.argsort(g, kind="stable")[-k:]
    total = np.float64(0)
    for j in ids:
        total = rnd(total + g[j])
    return ids, rnd(g[ids] / total)


def _predict(logits, m):
    top = np.argsort(logits + 0.0, kind="stable")[-m:]
    return np.array(sorted(top.tolist(), key=lambda e: (-logits[e], e)))


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "router":
        x = _norm(s["h"], s["norm_w"], _f16)
        ids, sc = _route(_f16(_np64(s["w"]) @ x), s["k"], _f16)
        out = {"ids": ids.astype(np.int32), "scores": sc.astype(np.float16), "x": x.astype(np.float16)}
        if s["w_next"] is not None:
            out["pred"] = _predict(_f16(_np64(s["w_next"]) @ x), s["m"]).astype(np.int32)
        return out
    if kind == "router_q8":
        x = _norm(s["h"], s["norm_w"], _bf16)
        q = s["codes"].cpu().numpy().view(np.uint8).reshape(case["n_exp"], -1, GROUP).astype(np.float64)
        w = q * _np64(s["scales"])[..., None] + _np64(s["biases"])[..., None]
        ids, sc = _route(_bf16(w.reshape(case["n_exp"], -1) @ x), s["k"], _bf16)
        return {"ids": ids.astype(np.int32), "scores": torch.from_numpy(sc).to(torch.bfloat16),
                "x_bf16": torch.from_numpy(x).to(torch.bfloat16), "x_f16": x.astype(np.float16)}
    if kind == "glu":
        x = s["x"].double()
        y = x.clone()
        for e, sc in zip(s["ids"].tolist(), s["scores"].double().tolist()):
            y += sc * _swiglu(x[None], *_q2_expert(case, s, e))[0]
        return y
    if kind == "codebook":
        x, pool = s["x"].double(), s["pool"].cpu().numpy()
        y = x.clone()
        grid = cbformat.grid().astype(np.float64)

        def rows(idx, sign7, sub, d):
            s7 = sign7[..., None] >> np.arange(7) & 1
            sg = np.concatenate([s7, s7.sum(-1, keepdims=True) & 1], -1)
            v = grid[idx] * (1 - 2 * sg)
            scale = np.repeat(d.astype(np.float64), 8, axis=1) * (2 * sub + 1) / 8
            return torch.from_numpy((v.reshape(idx.shape[0], -1, 32) * scale[..., None]).reshape(idx.shape[0], -1)).cuda()

        for e, sc in zip(s["ids"].tolist(), s["scores"].double().tolist()):
            up, down = (rows(*m) for m in cbformat.from_blob(pool[e], case["hidden"], case["inter"]))
            y += sc * (torch.relu(x @ up.T) ** 2 @ down.T)
        return y
    if kind == "prefill":
        x = s["x"].double()
        flat = torch.from_numpy(s["ids_np"].reshape(-1).astype(np.int64)).cuda()
        k = s["ids_np"].shape[1]
        y = torch.zeros(s["y"].shape, dtype=torch.float64, device="cuda")
        for e in np.unique(s["ids_np"]).tolist():
            at = (flat == e).nonzero()[:, 0]
            y[at] = _swiglu(x[at // k], *_q2_expert(case, s, e))
        sc = s["scores"].double()
        return {"rows": y, "out": (y.reshape(sc.shape[0], k, -1) * sc[..., None]).sum(1)}
    # whole tokens, rounded where the stack's own buffers between the layers are 16 bits
    st, L = s["stack"].st, case["layers"]
    xs, lg = [], []
    for t in range(case["tokens"]):
        x = s["xs"][t]
        for l in range(L):
            logits = _f16(_np64(st.router_w[l]) @ _np64(x))
            ids, sc = _route(logits, case["k"], _f16)
            h, xd = x.double(), x.double()[None]
            if kind == "resident" or l == 0:
                pool = st.full_pools[l] if kind == "resident" else st.pool0
            else:
                pool = st.store.tensor(l)
            for e, v in zip(ids.tolist(), sc.tolist()):
                one = {0: pool[e].to("cuda")}
                h = h + v * _swiglu(xd, *_q2_expert(case, {}, 0, pool=one))[0]
            x = torch.from_numpy(_norm(h, st.norm_w[l], _f16)).half().cuda()
        xs.append(x.double())
        lg.append(torch.from_numpy(logits).cuda())
    out = {"x": torch.stack(xs)}
    return out | {"logits": torch.stack(lg)} if kind == "resident" else out
