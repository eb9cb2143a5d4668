"""Performance cases of the MoE expert path, through the package's public calls.

A case is a dict of plain values. `listed()` names the fixed ones, `draw(rng)`
gives more of the same ranges, `prepare` builds what a program holds before the
call, `run` is one pass, `work` the bytes and operations a pass cannot do
without, `tolerance` the error another correct implementation at the same
precision shows, `exact` the outputs in 64 bits from the quantized bytes alone.

Weights are N(0, 0.02) quantized by the package's generator (as in bench.py),
activations N(0, 1), router logits carry a Zipf(1.1) popularity bias.
"""
import math

import numpy as np
import torch

import fomoe_amd as FA

DEV = "cuda"
TYPES = {"q4_k": FA.Q4_K, "q5_k": FA.Q5_K, "q6_k": FA.Q6_K, "q8_0": FA.Q8_0, "mxfp4": FA.MXFP4}
W_STD, ZIPF_S, EPS = 0.02, 1.1, 1e-6
_SHARED_GPU = None


class _Context(FA.Gpu):
    def __del__(self):
        self.close()


def _gpu():
    """The process's context (one per program; a captured stack keeps its own)."""
    global _SHARED_GPU
    if _SHARED_GPU is None:
        _SHARED_GPU = _Context()
    return _SHARED_GPU


# ------------------------------------------------------------------ cases
def listed():
    return [
        # one expert gate projection by itself: the smallest call, launch and latency
        {"name": "matvec_q4k_one", "kind": "matvec", "type": "q4_k", "M": 1024, "K": 4096, "n": 1, "one_x": True},
        # a rotation over 512 expert down projections, the headline benchmark's sweep
        {"name": "matvec_q6k_rotation", "kind": "matvec", "type": "q6_k", "M": 4096, "K": 1024, "n": 512, "one_x": True},
        # a batch of matrices in a shape nothing is tuned for, each with its own x
        {"name": "matvec_q5k_ragged", "kind": "matvec", "type": "q5_k", "M": 1000, "K": 2816, "n": 24, "one_x": False},
        # one decoded token through four MoE layers, one call per layer (top-10 of 512, shared expert)
        {"name": "layer_512", "kind": "layer", "layers": 4, "E": 512, "k": 10, "H": 4096, "F": 1024, "gate": "q4_k",
         "down": "q6_k", "shared": "same", "gate_vec": False},
        # the usual mixed file: Q5_K routed down projections, a Q8_0 shared down projection, gated shared expert
        {"name": "layer_512_mixed", "kind": "layer", "layers": 4, "E": 512, "k": 10, "H": 4096, "F": 1024,
         "gate": "q4_k", "down": "q5_k", "shared": "q8_0_down", "gate_vec": True},
        # a smaller MoE without a shared expert
        {"name": "layer_128", "kind": "layer", "layers": 4, "E": 128, "k": 8, "H": 2048, "F": 768, "gate": "q4_k",
         "down": "q6_k", "shared": "none", "gate_vec": False},
        # one decode step through a resident stack, the captured graph replayed per token
        {"name": "stack_512", "kind": "stack", "layers": 6, "E": 512, "k": 10, "H": 4096, "F": 1024, "gate": "q4_k",
         "down": "q6_k", "shared": "same", "gate_vec": False},
        # a short prompt (or a small decode batch) through one layer
        {"name": "prefill_16", "kind": "prefill", "T": 16, "E": 512, "k": 10, "H": 4096, "F": 1024, "gate": "q4_k",
         "down": "q6_k", "shared": "same", "gate_vec": False, "residual": False},
        # the benchmark's prompt
        {"name": "prefill_512", "kind": "prefill", "T": 512, "E": 512, "k": 10, "H": 4096, "F": 1024, "gate": "q4_k",
         "down": "q6_k", "shared": "same", "gate_vec": False, "residual": False},
        # a long prompt, where the matrix work counts
        {"name": "prefill_4096", "kind": "prefill", "T": 4096, "E": 512, "k": 10, "H": 4096, "F": 1024,
         "gate": "q4_k", "down": "q6_k", "shared": "same", "gate_vec": False, "residual": True},
        # an odd number of tokens through a smaller MoE in other types
        {"name": "prefill_203_q5k", "kind": "prefill", "T": 203, "E": 64, "k": 6, "H": 2048, "F": 1536, "gate": "q5_k",
         "down": "q8_0", "shared": "same", "gate_vec": True, "residual": True},
        # the drop-in call: ten experts' blobs in host memory, copied to the device on every call
        {"name": "expert_ffn_host", "kind": "ffn", "n": 10, "H": 4096, "F": 1024, "gate": "q4_k", "down": "q6_k"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "layer", "layer", "stack", "prefill", "prefill", "prefill", "ffn"])
    if kind == "matvec":
        t = rng.choice(["q4_k", "q5_k", "q6_k", "q8_0", "mxfp4"])
        M, K = _log_int(rng, 64, 4096), 256 * _log_int(rng, 1, 32)
        most = max(1, min(512, 1_700_000_000 // (M * FA.row_bytes(TYPES[t], K))))
        return {"kind": kind, "type": t, "M": M, "K": K, "n": _log_int(rng, 1, most), "one_x": rng.random() < 0.5}
    if kind == "ffn":
        H, F = 256 * rng.randint(4, 16), 256 * rng.randint(1, 4)
        return {"kind": kind, "n": rng.randint(1, 10), "H": H, "F": F, "gate": rng.choice(["q4_k", "q5_k"]),
                "down": rng.choice(["q4_k", "q5_k", "q6_k"])}
    E = _log_int(rng, 16, 512)
    c = {"kind": kind, "E": E, "k": rng.randint(2, 10), "H": rng.choice([1024, 1536, 2048, 3072, 4096, 4096]),
         "F": rng.choice([512, 768, 1024, 1024, 1280, 1536]), "gate": rng.choice(["q4_k", "q4_k", "q4_k", "q5_k", "q6_k"]),
         "down": rng.choice(["q6_k", "q6_k", "q5_k", "q4_k", "q8_0"]), "shared": rng.choice(["same", "same", "none", "q8_0_down"]),
         "gate_vec": rng.random() < 0.5}
    if kind == "prefill":
        c["residual"] = rng.random() < 0.5
        most = 4096 * 10 * 4096 * 1024 // (c["k"] * c["H"] * c["F"])
        c["T"] = _log_int(rng, 2, max(2, min(4096, most)))
    else:
        blob = _blob(c)["stride"] * (E + 1)
        c["layers"] = max(1, min(rng.randint(2, 6), 17_000_000_000 // blob))
    return c


# ------------------------------------------------------------------ layouts
def _blob(c):
    """Types, sizes and offsets of one expert blob gate | up | down, and of the shared one."""
    H, F = c["H"], c["F"]
    g, d = TYPES[c["gate"]], TYPES[c["down"]]
    gs, ds = F * FA.row_bytes(g, H), H * FA.row_bytes(d, F)
    sd = FA.Q8_0 if c.get("shared") == "q8_0_down" else d
    return {"g": g, "d": d, "sd": sd, "gs": gs, "ds": ds, "stride": (2 * gs + ds + 4095) // 4096 * 4096,
            "shared_bytes": 2 * gs + H * FA.row_bytes(sd, F)}


def _has_shared(c):
    return c.get("shared", "none") != "none"


def _zipf(E, seed):
    r = np.random.RandomState(seed % (1 << 31))
    b = np.empty(E, np.float32)
    b[r.permutation(E)] = -ZIPF_S * np.log(np.arange(1, E + 1))
    return b


def _touched(c):
    """Distinct experts the tokens of a prefill reach (mean over a few draws of the same routing statistics)."""
    E, k, T = c["E"], c["k"], c["T"]
    r = np.random.RandomState(7)
    n = []
    for i in range(3):
        z = r.randn(min(T, 2048), E) * (W_STD * math.sqrt(c["H"])) + _zipf(E, i)
        n.append(len(np.unique(np.argpartition(z, E - min(k, E), axis=1)[:, E - min(k, E):])))
    return float(np.mean(n))


def work(c):
    if c["kind"] == "matvec":
        M, K, n = c["M"], c["K"], c["n"]
        return {"bytes": n * (M * FA.row_bytes(TYPES[c["type"]], K) + 4 * M) + 4 * K * (1 if c["one_x"] else n),
                "flops": 2 * n * M * K}
    b, H, F = _blob(c), c["H"], c["F"]
    if c["kind"] == "ffn":
        return {"bytes": c["n"] * (2 * b["gs"] + b["ds"]) + 8 * H, "flops": 6 * c["n"] * H * F}
    E, k = c["E"], min(c["k"], c["E"])
    sh = _has_shared(c)
    expert = 2 * b["gs"] + b["ds"]
    if c["kind"] == "prefill":
        T = c["T"]
        return {"bytes": 4 * E * H + _touched(c) * expert + (b["shared_bytes"] if sh else 0) + T * H * 6,
                "flops": 2 * T * E * H + 6 * T * (k + sh) * H * F}
    one = 4 * E * H + k * expert + (b["shared_bytes"] if sh else 0) + 8 * H
    return {"bytes": c["layers"] * one, "flops": c["layers"] * (2 * E * H + 6 * (k + sh) * H * F)}


def tolerance(c):
    # each about four times the error against `exact` that the path shows over these ranges
    if c["kind"] == "prefill":
        # fp16 down operands (2^-11 relative each): 3.6e-4 with Q4_K gate/up; gate/up of another type multiplies
        # bf16 weights (2^-9): 6.5e-4 beside a residual of the tokens' size, about 1.5e-3 without
        return {"rel": 1.5e-3} if c["gate"] == "q4_k" else {"rel": 6e-3}
    # fp32 sums: a matvec 3.0e-7, an expert FFN 5.5e-7, a layer or a stack 8.4e-7
    return {"rel": {"matvec": 1.2e-6, "ffn": 2.2e-6}.get(c["kind"], 3.5e-6)}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _weights(gpu, t, seed, stream0, step, M, K, n, dst, stride):
    """n matrices [M x K] of type t at dst (device address), stride bytes apart."""
    gpu.synth_quant(t, seed, stream0, step, W_STD, M, K, n, dst, stride)


def _layer(gpu, c, seed, index):
    """One resident MoE layer: its descriptor and the tensors behind it."""
    E, H, F, b = c["E"], c["H"], c["F"], _blob(c)
    experts = torch.zeros(E * b["stride"] + b["shared_bytes"], dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    base, st = experts.data_ptr(), (index + 1) << 24
    for kind, off, t, M, K in ((0, 0, b["g"], F, H), (1, b["gs"], b["g"], F, H), (2, 2 * b["gs"], b["d"], H, F)):
        _weights(gpu, t, seed, st | kind, 16, M, K, E, base + off, b["stride"])
        if _has_shared(c):
            _weights(gpu, b["sd"] if kind == 2 else t, seed, st | (E << 4) | kind, 16, M, K, 1, base + E * b["stride"] + off, 0)
    g = _gen(seed * 64 + index)
    k = {"experts": experts, "router": torch.randn(E, H, generator=g, device=DEV) * W_STD,
         "bias": torch.from_numpy(_zipf(E, seed * 64 + index)).to(DEV),
         "norm": 1 + 0.1 * torch.randn(H, generator=g, device=DEV),
         "vec": torch.randn(H, generator=g, device=DEV) * W_STD}
    d = FA.MoeLayer()
    d.n_embd, d.inter, d.n_experts, d.k = H, F, E, min(c["k"], E)
    d.gate_type = d.up_type = b["g"]
    d.down_type = b["d"]
    d.gate_size = d.up_size = b["gs"]
    d.expert_stride = b["stride"]
    d.router, d.router_bias, d.experts = k["router"].data_ptr(), k["bias"].data_ptr(), base
    d.norm_w, d.eps = k["norm"].data_ptr(), EPS
    if _has_shared(c):
        d.shared = base + E * b["stride"]
        d.shared_inter, d.shared_gate_size, d.shared_up_size = F, b["gs"], b["gs"]
        d.shared_gate_type = d.shared_up_type = b["g"]
        d.shared_down_type = b["sd"]
        d.shared_gate_vec = k["vec"].data_ptr() if c["gate_vec"] else None
    k["desc"] = d
    return k


def _blobs(gpu, c, seed):
    b = _blob(c)
    bytes_ = 2 * b["gs"] + b["ds"]
    dev = torch.zeros(c["n"] * bytes_, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    for kind, off, t, M, K in ((0, 0, b["g"], c["F"], c["H"]), (1, b["gs"], b["g"], c["F"], c["H"]),
                               (2, 2 * b["gs"], b["d"], c["H"], c["F"])):
        _weights(gpu, t, seed, kind, 16, M, K, c["n"], dev.data_ptr() + off, bytes_)
    gpu.sync()
    return dev, bytes_


def prepare(c, seed):
    g = _gen(seed)
    if c["kind"] == "stack":
        gpu = _Context()   # a captured graph belongs to its context
    else:
        gpu = _gpu()
    s = {"case": c, "gpu": gpu}
    if c["kind"] == "matvec":
        t, M, K, n = TYPES[c["type"]], c["M"], c["K"], c["n"]
        stride = M * FA.row_bytes(t, K)
        s["W"] = torch.empty(n * stride, dtype=torch.uint8, device=DEV)
        if t == FA.MXFP4:   # no quantizer for it: random codes, block exponents of weights of this size
            blk = torch.randint(0, 256, (n * stride // 17, 17), dtype=torch.uint8, device=DEV, generator=g)
            blk[:, 0] = torch.randint(118, 123, (blk.shape[0],), dtype=torch.uint8, device=DEV, generator=g)
            s["W"].copy_(blk.reshape(-1))
        s["x"] = torch.randn(1 if c["one_x"] else n, K, generator=g, device=DEV)
        s["y"] = torch.zeros(n, M, device=DEV)
        torch.cuda.synchronize()
        if t != FA.MXFP4:
            _weights(gpu, t, seed, 0, 16, M, K, n, s["W"].data_ptr(), stride)
    elif c["kind"] == "ffn":
        dev, nbytes = _blobs(gpu, c, seed)
        s["host"] = [b.copy() for b in dev.cpu().numpy().reshape(c["n"], nbytes)]
        s["h"] = torch.randn(c["H"], generator=g, device=DEV).cpu().numpy()
        w = torch.rand(c["n"], generator=g, device=DEV).cpu().numpy()
        s["scores"] = (w / w.sum()).astype(np.float32)
    else:
        s["layers"] = [_layer(gpu, c, seed, i) for i in range(c.get("layers", 1))]
        if c["kind"] == "prefill":
            s["x"] = torch.randn(c["T"], c["H"], generator=g, device=DEV).bfloat16()
            s["out"] = torch.zeros(c["T"], c["H"], device=DEV)
        else:
            s["x"] = torch.randn(c["H"], generator=g, device=DEV)
            s["out"] = torch.zeros(len(s["layers"]), c["H"], device=DEV)
    gpu.sync()
    torch.cuda.synchronize()
    return s


def run(s):
    c, gpu = s["case"], s["gpu"]
    if c["kind"] == "matvec":
        M, K = c["M"], c["K"]
        if c["n"] == 1:
            gpu.matvec(TYPES[c["type"]], s["W"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(), M, K)
        else:
            gpu.matvec_batched(TYPES[c["type"]], s["W"].data_ptr(), M * FA.row_bytes(TYPES[c["type"]], K), c["n"],
                               s["x"].data_ptr(), 0 if c["one_x"] else K, s["y"].data_ptr(), M, M, K)
        return s["y"]
    if c["kind"] == "ffn":
        b = _blob(c)
        rc, out = gpu.expert_ffn(s["h"], s["host"], s["scores"], c["H"], c["F"], b["gs"], b["gs"], 2 * b["gs"] + b["ds"],
                                 b["g"], b["g"], b["d"])
        if rc != 0:
            raise RuntimeError("gpu_expert_ffn refused the call")
        return out
    if c["kind"] == "prefill":
        gpu.moe_prefill(s["layers"][0]["desc"], s["x"].data_ptr(), c["T"], s["out"].data_ptr(),
                        FA.MOE_RESIDUAL if c["residual"] else 0)
        return s["out"]
    if c["kind"] == "stack":
        gpu.stack_decode([k["desc"] for k in s["layers"]], s["x"].data_ptr(), 1)
        return s["x"]
    x, H4 = s["x"].data_ptr(), 4 * c["H"]
    for i, k in enumerate(s["layers"]):   # each layer's output is the next one's input
        gpu.moe_layer(k["desc"], x, s["out"].data_ptr() + i * H4, FA.MOE_NORM | FA.MOE_RESIDUAL)
        x = s["out"].data_ptr() + i * H4
    return s["out"]


# ------------------------------------------------------------------ 64-bit outputs
def _half(b):
    """Pairs of bytes [..., 2] as the fp16 numbers they hold, in 64 bits."""
    return b.contiguous().view(torch.float16).squeeze(-1).double()


def _k_scales(b):
    """The eight 6-bit (scale, min) pairs of Q4_K / Q5_K blocks from their 12 scale bytes."""
    b = b.int()
    lo, mid, hi = b[:, 0:4], b[:, 4:8], b[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _dequant(t, raw, M, K):
    """[M x K] in 64 bits from the bytes of a GGUF-format matrix."""
    if t == FA.Q8_0:
        b = raw.reshape(-1, 34)
        return (_half(b[:, :2])[:, None] * b[:, 2:].contiguous().view(torch.int8).double()).reshape(M, K)
    if t == FA.MXFP4:
        b = raw.reshape(-1, 17)
        table = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, 0, -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device=raw.device)
        q = torch.cat([b[:, 1:] & 15, b[:, 1:] >> 4], 1)
        return (torch.pow(2.0, b[:, :1].double() - 127) * table[q.long()]).reshape(M, K)
    if t == FA.Q6_K:
        b = raw.reshape(-1, 210)
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32).int(), b[:, 128:192].reshape(-1, 2, 32).int()
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return (_half(b[:, 208:210])[:, None, None] * sc[:, :, None] * (q.reshape(-1, 16, 16).double() - 32)).reshape(M, K)
    b = raw.reshape(-1, 144 if t == FA.Q4_K else 176)
    sc, mn = _k_scales(b[:, 4:16])
    qs = b[:, -128:].reshape(-1, 4, 32).int()
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if t == FA.Q5_K:
        bits = torch.arange(8, device=raw.device, dtype=torch.int32)[None, :, None]
        q = q + (((b[:, 16:48].int()[:, None, :] >> bits) & 1) << 4)
    d, dm = _half(b[:, :2])[:, None, None], _half(b[:, 2:4])[:, None, None]
    return (d * sc[:, :, None] * q.double() - dm * mn[:, :, None]).reshape(M, K)


def _ffn64(raw, b, g, d, X, H, F):
    """silu(X Wg^T) * (X Wu^T) Wd^T of one blob, X [n x H] in 64 bits."""
    gate = X @ _dequant(g, raw[:b["gs"]], F, H).T
    up = X @ _dequant(g, raw[b["gs"]:2 * b["gs"]], F, H).T
    return (gate * torch.sigmoid(gate) * up) @ _dequant(d, raw[2 * b["gs"]:2 * b["gs"] + H * FA.row_bytes(d, F)], H, F).T


def _moe64(c, k, X):
    """The MoE block of the tokens X [n x H] (64 bits): top-k of the softmax, renormalised, experts, shared expert."""
    b, E, H, F = _blob(c), c["E"], c["H"], c["F"]
    p = torch.softmax(X @ k["router"].double().T + k["bias"].double(), 1)
    w, ids = torch.topk(p, min(c["k"], E), 1)
    w = w / w.sum(1, keepdim=True)
    out = torch.zeros_like(X)
    for e in torch.unique(ids).tolist():
        t, r = torch.nonzero(ids == e, as_tuple=True)
        raw = k["experts"][e * b["stride"]:]
        out.index_add_(0, t, w[t, r][:, None] * _ffn64(raw, b, b["g"], b["d"], X[t], H, F))
    if _has_shared(c):
        sw = torch.sigmoid(X @ k["vec"].double())[:, None] if c["gate_vec"] else 1.0
        out += sw * _ffn64(k["experts"][E * b["stride"]:], b, b["g"], b["sd"], X, H, F)
    return out


def exact(c, seed):
    s = prepare(c, seed)
    if c["kind"] == "matvec":
        t, M, K, n = TYPES[c["type"]], c["M"], c["K"], c["n"]
        W, x = s["W"].reshape(n, -1), s["x"].double()
        return torch.stack([_dequant(t, W[i], M, K) @ x[0 if c["one_x"] else i] for i in range(n)])
    if c["kind"] == "ffn":
        b, h = _blob(c), torch.from_numpy(s["h"]).to(DEV).double()[None]
        out = torch.zeros_like(h)
        for w, blob in zip(s["scores"], s["host"]):
            out += float(w) * _ffn64(torch.from_numpy(blob).to(DEV), b, b["g"], b["d"], h, c["H"], c["F"])
        return out[0].cpu().numpy()
    x = s["x"].double()
    if c["kind"] == "prefill":
        y = _moe64(c, s["layers"][0], x)
        return y + x if c["residual"] else y
    outs, x = [], x[None]
    for k in s["layers"]:
        h = x / torch.sqrt((x * x).mean() + EPS) * k["norm"].double()
        x = x + _moe64(c, k, h)
        outs.append(x[0])
    return outs[-1] if c["kind"] == "stack" else torch.stack(outs)
