"""The work a user of this backend has it do, as measurable cases.

Each case is one call (or one burst of calls) of the package's public entry
points over weights resident in HBM.  Kinds:

* ``burst_qkv``   the contract's burst: q, k and v of one layer over one host
  activation, then their waits (zlm's executor, once per layer and token);
* ``burst_mlp``   the contract's fused MLP (gate_up + down) and its wait;
* ``host_gemv``   the contract's synchronous GEMV (the lm_head: host logits);
* ``host_matmul`` the contract's synchronous matrix product over host rows
  (short prompts and verification batches);
* ``gemv``        one GEMV form on device buffers (plain, norm, normed
  gate_up, gate_up, residual), as the decode step enqueues them;
* ``matmul``      the matrix product on device buffers: 2..32 tokens of a
  verification batch up to the thousands of a prompt;
* ``attention``   the fused decode attention block over an f16 KV cache;
* ``step``        a whole decode step of a Qwen3-shaped model replayed from
  its graph, logits to the host.

Weights are raw GGUF blocks made on the GPU from the seed (scales |N(0,1)| *
0.02 as f16, uniform quants: the distributions of the package's synthetic
weights), activations N(0, 1).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from zlm_amd import decode as zdec
from zlm_amd import device as zd

TYPES = {"q4_0": zd.Q4_0, "q4_1": zd.Q4_1, "q8_0": zd.Q8_0, "q4_k": zd.Q4_K, "q6_k": zd.Q6_K, "f32": zd.F32,
         "f16": zd.F16, "bf16": zd.BF16}
BLOCK = {"q4_0": (32, 18), "q4_1": (32, 20), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210),
         "f32": (1, 4), "f16": (1, 2), "bf16": (1, 2)}
MATMUL_TYPES = ("q4_0", "q8_0", "q4_1", "q4_k")
FORMS = {"plain": zd.FORM_PLAIN, "pair": zd.FORM_PAIR, "norm": zd.FORM_NORM, "normpair": zd.FORM_NORMPAIR,
         "resid": zd.FORM_RESID}
ACTS = {"silu": zd.SILU, "gelu": zd.GELU}
EPS = 1e-6
ROPE_BASE = 1_000_000.0
FP_TOKENS = 2  # matrix products of up to two tokens multiply the activations as they are; past that, as q8 blocks

_dev = None


def _device() -> zd.Device:
    global _dev
    if _dev is None:
        _dev = zd.Device()
        if not _dev.available():
            raise RuntimeError(_dev.last_error())
    return _dev


def listed():
    return [
        # one layer's q, k, v of Qwen3-8B at batch 1, through the contract: the smallest calls of a token
        {"name": "qkv_burst_q4_0", "kind": "burst_qkv", "quant": "q4_0", "k": 4096, "q_rows": 4096, "kv_rows": 1024},
        # one layer's MLP of a 3840-wide model in the usual k-quant mix, through the contract
        {"name": "mlp_burst_q4_k_q6_k", "kind": "burst_mlp", "quant": "q4_k", "down": "q6_k", "k": 3840,
         "ffn": 15360, "act": "gelu"},
        # that model's lm_head, logits to the host
        {"name": "head_host_q6_k", "kind": "host_gemv", "quant": "q6_k", "rows": 262144, "k": 3840},
        # the attention output projection with the residual, 4096-wide model
        {"name": "o_resid_q4_0", "kind": "gemv", "form": "resid", "quant": "q4_0", "rows": 4096, "k": 4096,
         "act": "silu"},
        # the benchmark's Q8_0 FFN projection
        {"name": "gate_q8_0", "kind": "gemv", "form": "plain", "quant": "q8_0", "rows": 12288, "k": 4096,
         "act": "silu"},
        # the decode step's normed gate_up
        {"name": "norm_gate_up_q4_0", "kind": "gemv", "form": "normpair", "quant": "q4_0", "rows": 12288, "k": 4096,
         "act": "silu"},
        # a verification batch of eight tokens through the contract
        {"name": "verify_host_q4_0_m8", "kind": "host_matmul", "quant": "q4_0", "rows": 12288, "k": 4096, "m": 8},
        # the lm_head of a verification batch of five
        {"name": "verify_head_q4_k_m5", "kind": "matmul", "quant": "q4_k", "rows": 262144, "k": 3840, "m": 5},
        # a 512-token prompt through an FFN projection
        {"name": "prefill_q4_0_m512", "kind": "matmul", "quant": "q4_0", "rows": 12288, "k": 4096, "m": 512},
        # a long ragged prompt through a k-quant FFN projection
        {"name": "prefill_q4_k_m1999", "kind": "matmul", "quant": "q4_k", "rows": 15360, "k": 3840, "m": 1999},
        # the decode attention block at 8000 cached positions
        {"name": "attention_8000", "kind": "attention", "n_heads": 32, "n_kv": 8, "max_seq": 32768, "pos": 7999},
        # one token of Qwen3-8B at 2048 cached positions
        {"name": "step_qwen3_8b", "kind": "step", "n_layers": 36, "hidden": 4096, "n_heads": 32, "n_kv": 8,
         "ffn": 12288, "vocab": 151936, "max_seq": 2048, "pos": 2047},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k(rng, quant, lo, hi):
    be = max(32, BLOCK[quant][0])
    return max(be, _log(rng, lo, hi) // be * be)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "burst_qkv", "burst_mlp", "host_gemv", "host_matmul", "matmul",
                       "matmul", "matmul", "matmul", "attention", "step"])
    if kind == "gemv":
        quant = rng.choice(["q4_0", "q8_0", "q4_k", "q6_k", "q4_1", "f16", "bf16"])
        rows, k = _log(rng, 256, 160000), _k(rng, quant, 1024, 16384)
        return {"kind": kind, "form": rng.choice(sorted(FORMS)), "quant": quant,
                "rows": min(rows, int(4e8 / k)), "k": k, "act": rng.choice(sorted(ACTS))}
    if kind == "burst_qkv":
        quant = rng.choice(["q4_0", "q8_0", "q4_k", "q6_k"])
        k = _k(rng, quant, 1024, 8192)
        return {"kind": kind, "quant": quant, "k": k, "q_rows": 128 * rng.randint(8, 64),
                "kv_rows": 128 * rng.randint(1, 16)}
    if kind == "burst_mlp":
        quant, down = rng.choice([("q4_0", "q4_0"), ("q8_0", "q8_0"), ("q4_k", "q6_k"), ("q4_k", "q4_k")])
        return {"kind": kind, "quant": quant, "down": down, "k": _k(rng, down, 1024, 8192),
                "ffn": 256 * _log(rng, 8, 72), "act": rng.choice(sorted(ACTS))}
    if kind == "host_gemv":
        quant = rng.choice(["q4_0", "q8_0", "q4_k", "q6_k", "f16"])
        return {"kind": kind, "quant": quant, "rows": _log(rng, 1024, 160000), "k": _k(rng, quant, 1024, 4096)}
    if kind == "attention":
        max_seq = 2048 * 2 ** rng.randint(0, 4)
        n_kv = rng.choice([2, 4, 8])
        return {"kind": kind, "n_heads": n_kv * rng.choice([1, 2, 4]), "n_kv": n_kv, "max_seq": max_seq,
                "pos": min(_log(rng, 64, max_seq), max_seq) - 1}
    if kind == "step":
        max_seq = rng.choice([512, 2048, 4096])
        n_kv = rng.choice([2, 4, 8])
        return {"kind": kind, "n_layers": rng.randint(1, 8), "hidden": 128 * rng.randint(4, 40),
                "n_heads": n_kv * rng.choice([2, 4]), "n_kv": n_kv, "ffn": 256 * rng.randint(4, 48),
                "vocab": _log(rng, 8000, 152000), "max_seq": max_seq, "pos": rng.randrange(max_seq)}
    quant = rng.choice(MATMUL_TYPES)
    few = kind == "host_matmul" or rng.random() < 0.4
    k = _k(rng, quant, 1024, 16384)
    m = _log(rng, 2, 64) if few else _log(rng, 33, 2048)
    rows = _log(rng, 512, 160000 if few and kind == "matmul" else 20000)
    return {"kind": kind, "quant": quant, "rows": max(64, min(rows, int(6e8 / k), int(1.1e11 / (k * m)))), "k": k, "m": m}


# ---- inputs ---------------------------------------------------------------------


class _Inputs:
    """The seeded stream of a case: the same tensors in the same order for prepare() and exact()."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.gen, device="cuda", dtype=torch.float32)

    def _bytes(self, n, width):
        return torch.randint(0, 256, (n, width), generator=self.gen, device="cuda", dtype=torch.uint8)

    def _f16(self, n, scale):
        return (self.normal(n).abs_() * scale).half().view(torch.uint8).reshape(n, 2)

    def weight(self, quant, rows, k):
        """Raw GGUF blocks (n_blocks x block bytes, uint8, on the GPU) of a rows x k weight."""
        be, _ = BLOCK[quant]
        n = rows * (k // be)
        if quant == "q4_0":
            return torch.cat([self._f16(n, 0.02), self._bytes(n, 16)], 1)
        if quant == "q4_1":
            lo = (self.normal(n).abs_() * -0.1).half().view(torch.uint8).reshape(n, 2)
            return torch.cat([self._f16(n, 0.02), lo, self._bytes(n, 16)], 1)
        if quant == "q8_0":
            q = torch.randint(-127, 128, (n, 32), generator=self.gen, device="cuda", dtype=torch.int8)
            return torch.cat([self._f16(n, 0.01), q.view(torch.uint8)], 1)
        if quant == "q4_k":
            return torch.cat([self._f16(n, 0.02), self._f16(n, 0.02), self._bytes(n, 140)], 1)
        if quant == "q6_k":
            return torch.cat([self._bytes(n, 208), self._f16(n, 0.02)], 1)
        w = self.normal(n) * 0.02
        return (w if quant == "f32" else w.half() if quant == "f16" else w.bfloat16()).view(torch.uint8).reshape(n, -1)


def _host(t):
    return t.reshape(-1).cpu().numpy()


class _State:
    """What a program keeps: its residents and buffers (residents are given back with it)."""

    def __init__(self, case):
        self.case, self.dev, self.residents, self.model, self.graph = case, _device(), [], None, None

    def resident(self, raw):
        r = self.dev.upload_resident(_host(raw))
        if r is None:
            raise RuntimeError(self.dev.last_error())
        self.residents.append(r)
        return r

    def __del__(self):
        if self.graph is not None:
            self.dev.graph_destroy(self.graph)
        if self.model is not None:
            self.model.free()
        for r in self.residents:
            self.dev.free_resident(r)


def _step_config(c):
    return zdec.DecodeConfig(n_layers=c["n_layers"], hidden=c["hidden"], n_heads=c["n_heads"], n_kv_heads=c["n_kv"],
                             head_dim=128, ffn=c["ffn"], vocab=c["vocab"], max_seq=c["max_seq"], eps=EPS,
                             freq_base=ROPE_BASE)


def _step_layer(g, c):
    """One layer's tensors, in the stream's order."""
    kv = 128 * c["n_kv"]
    qr = 128 * c["n_heads"]
    return {"qkv": g.weight("q4_0", qr + 2 * kv, c["hidden"]), "o": g.weight("q4_0", c["hidden"], qr),
            "gate": g.weight("q4_0", c["ffn"], c["hidden"]), "up": g.weight("q4_0", c["ffn"], c["hidden"]),
            "down": g.weight("q4_0", c["hidden"], c["ffn"]),
            "attn_norm": 1 + 0.1 * g.normal(c["hidden"]), "ffn_norm": 1 + 0.1 * g.normal(c["hidden"]),
            "q_norm": 1 + 0.1 * g.normal(128), "k_norm": 1 + 0.1 * g.normal(128),
            "k_cache": g.normal(c["n_kv"], c["max_seq"], 128).half(),
            "v_cache": g.normal(c["n_kv"], c["max_seq"], 128).half()}


def prepare(case, seed):
    c, g, s = case, _Inputs(seed), _State(case)
    kind = c["kind"]
    if kind == "burst_qkv":
        s.q, s.k, s.v = (s.resident(g.weight(c["quant"], r, c["k"])) for r in (c["q_rows"], c["kv_rows"], c["kv_rows"]))
        s.x = _host(g.normal(c["k"]))
        s.out = [np.empty(r, np.float32) for r in (c["q_rows"], c["kv_rows"], c["kv_rows"])]
    elif kind == "burst_mlp":
        s.gate, s.up = (s.resident(g.weight(c["quant"], c["ffn"], c["k"])) for _ in range(2))
        s.down = s.resident(g.weight(c["down"], c["k"], c["ffn"]))
        s.x = _host(g.normal(c["k"]))
        s.out = np.empty(c["k"], np.float32)
    elif kind in ("host_gemv", "host_matmul"):
        m = c.get("m", 1)
        s.w = s.resident(g.weight(c["quant"], c["rows"], c["k"]))
        s.x = _host(g.normal(m, c["k"]))
        s.out = np.empty(m * c["rows"], np.float32)
    elif kind == "gemv":
        s.w = s.resident(g.weight(c["quant"], c["rows"], c["k"]))
        s.x = g.normal(c["k"])
        s.up = s.resident(g.weight(c["quant"], c["rows"], c["k"])) if "pair" in c["form"] else None
        s.norm = 1 + 0.1 * g.normal(c["k"])
        s.res = g.normal(c["rows"])
        s.out = torch.empty(c["rows"], device="cuda")
    elif kind == "matmul":
        s.w = s.resident(g.weight(c["quant"], c["rows"], c["k"]))
        s.x = g.normal(c["m"], c["k"])
        s.out = torch.empty(c["m"], c["rows"], device="cuda")
    elif kind == "attention":
        heads = c["n_heads"] + 2 * c["n_kv"]
        s.qkv = g.normal(heads * 128)
        s.qn, s.kn = 1 + 0.1 * g.normal(128), 1 + 0.1 * g.normal(128)
        s.kc, s.vc = (g.normal(c["n_kv"], c["max_seq"], 128).half() for _ in range(2))
        s.pos = torch.tensor([c["pos"], 0, 0, 0], dtype=torch.int32, device="cuda")
        s.window = 128
        while s.window < c["pos"] + 1:
            s.window *= 2
        s.window = min(s.window, c["max_seq"])
        s.out = torch.empty(c["n_heads"] * 128, device="cuda")
    elif kind == "step":
        layers = [{n: t.cpu().numpy() if t.dtype == torch.float16 else _host(t) for n, t in _step_layer(g, c).items()}
                  for _ in range(c["n_layers"])]
        host = {"layers": layers, "lm_head": _host(g.weight("q8_0", c["vocab"], c["hidden"])),
                "out_norm": _host(1 + 0.1 * g.normal(c["hidden"]))}
        s.x = _host(g.normal(c["hidden"]))
        s.model = zdec.DecodeModel(s.dev, _step_config(c), host)
        window = s.model.window_for(c["pos"])
        s.model.step(s.x, c["pos"], window)  # a step runs eagerly before its capture
        s.graph = s.model.capture(window)
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()  # the backend has a stream of its own
    return s


# ---- one pass -------------------------------------------------------------------


def _ok(dev, flag):
    if not flag:
        raise RuntimeError(dev.last_error())


def run(state):
    s, c, d = state, state.case, state.dev
    kind = c["kind"]
    if kind == "burst_qkv":
        q = zd.quant(TYPES[c["quant"]])
        ops = ((s.q, c["q_rows"]), (s.k, c["kv_rows"]), (s.v, c["kv_rows"]))
        hs = [d.mat_vec_resident_burst_async(r, q, rows, c["k"], s.x, i == 0) for i, (r, rows) in enumerate(ops)]
        for h, (_, rows), out in zip(hs, ops, s.out):
            _ok(d, h is not None and d.wait_resident(h, out, rows))
    elif kind == "burst_mlp":
        h = d.mat_vec_mlp_pair_resident_burst_async(s.gate, s.up, s.down, zd.quant(TYPES[c["quant"]]),
                                                    zd.quant(TYPES[c["down"]]), c["k"], c["k"], c["ffn"], s.x,
                                                    ACTS[c["act"]], 0, True)
        _ok(d, h is not None and d.wait_resident(h, s.out, c["k"]))
    elif kind == "host_gemv":
        _ok(d, d.mat_vec_resident(s.w, zd.quant(TYPES[c["quant"]]), c["rows"], c["k"], s.x, s.out))
    elif kind == "host_matmul":
        _ok(d, d.mat_mul_resident(s.w, zd.quant(TYPES[c["quant"]]), c["rows"], c["k"], c["m"], s.x, s.out))
    elif kind == "gemv":
        q = zd.quant(TYPES[c["quant"]])
        if c["form"] == "plain":
            _ok(d, d.mat_vec_enqueue(s.w, q, c["rows"], c["k"], s.x.data_ptr(), s.out.data_ptr()))
        else:
            _ok(d, d.gemv_op_enqueue(FORMS[c["form"]], q, s.w, c["rows"], c["k"], s.x.data_ptr(), s.out.data_ptr(),
                                     w_up=s.up, norm_w=s.norm.data_ptr(), eps=EPS, act=ACTS[c["act"]],
                                     res=s.res.data_ptr()))
    elif kind == "matmul":
        _ok(d, d.mat_mul_enqueue(s.w, zd.quant(TYPES[c["quant"]]), c["rows"], c["k"], c["m"], s.x.data_ptr(),
                                 s.out.data_ptr()))
    elif kind == "attention":
        _ok(d, d.attention_decode_window_enqueue(
            s.qkv.data_ptr(), s.qn.data_ptr(), s.kn.data_ptr(), c["n_heads"], c["n_kv"], 128, EPS, ROPE_BASE,
            s.pos.data_ptr(), s.kc.data_ptr(), s.vc.data_ptr(), c["max_seq"], s.window, 128 ** -0.5,
            s.out.data_ptr()))
        return {"out": s.out, "k_cache": s.kc, "v_cache": s.vc}
    elif kind == "step":
        s.model.set_input(s.x, c["pos"])
        d.graph_launch(s.graph, 1)
        return s.model.logits_host()
    return s.out


# ---- what a pass cannot do without ------------------------------------------------


def _wbytes(quant, rows, k):
    be, bb = BLOCK[quant]
    return rows * (k // be) * bb


def work(case):
    c = case
    kind = c["kind"]
    if kind == "burst_qkv":
        rows = c["q_rows"] + 2 * c["kv_rows"]
        return {"bytes": _wbytes(c["quant"], rows, c["k"]) + 4 * (c["k"] + rows), "flops": 2 * rows * c["k"]}
    if kind == "burst_mlp":
        return {"bytes": _wbytes(c["quant"], 2 * c["ffn"], c["k"]) + _wbytes(c["down"], c["k"], c["ffn"]) + 8 * c["k"],
                "flops": 6 * c["ffn"] * c["k"]}
    if kind == "gemv":
        n = 2 if "pair" in c["form"] else 1
        vec = c["k"] * (2 if "norm" in c["form"] else 1) + c["rows"] * (2 if c["form"] == "resid" else 1)
        return {"bytes": n * _wbytes(c["quant"], c["rows"], c["k"]) + 4 * vec, "flops": 2 * n * c["rows"] * c["k"]}
    if kind in ("matmul", "host_matmul", "host_gemv"):
        m = c.get("m", 1)
        return {"bytes": _wbytes(c["quant"], c["rows"], c["k"]) + 4 * m * (c["k"] + c["rows"]),
                "flops": 2 * m * c["rows"] * c["k"]}
    if kind == "attention":
        n = c["pos"] + 1
        return {"bytes": 4 * 128 * n * c["n_kv"] + 4 * 128 * (2 * c["n_heads"] + 2 * c["n_kv"]),
                "flops": 4 * 128 * n * c["n_heads"]}
    per = (128 * (c["n_heads"] + 2 * c["n_kv"]) * c["hidden"] + 128 * c["n_heads"] * c["hidden"]
           + 3 * c["ffn"] * c["hidden"])
    kv = 4 * 128 * c["n_kv"] * (c["pos"] + 1)
    return {"bytes": c["n_layers"] * (per // 32 * 18 + kv) + _wbytes("q8_0", c["vocab"], c["hidden"])
            + 4 * (c["hidden"] + c["vocab"]),
            "flops": 2 * (c["n_layers"] * per + c["vocab"] * c["hidden"])}


def tolerance(case):
    """About four times what is seen against the 64-bit result: 2e-7 for the 32-bit sums over exact block dots, 2.5e-6
    where x is staged as int8 planes (2^-20 of a block's largest value) instead of fp32 -- either is a correct form of
    the one-token products --, 5e-5 for the attention (its rotary angles are 32-bit products of the position) and up to
    2e-5 for a whole step."""
    if case["kind"] in ("matmul", "host_matmul"):
        return {"rel": 1e-6 if case["m"] > FP_TOKENS else 1e-5}
    return {"attention": {"rel": 2e-4}, "step": {"rel": 1e-4}}.get(case["kind"], {"rel": 1e-5})


# ---- the same in 64 bits ------------------------------------------------------------


def _h(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(quant, raw):
    """Block values (n_blocks x block elements) in float64 of raw GGUF blocks."""
    n = raw.shape[0]
    if quant in ("q4_0", "q4_1"):
        q = raw[:, -16:]
        nib = torch.cat([q & 15, q >> 4], 1).double()
        return (nib - 8) * _h(raw[:, 0:2]) if quant == "q4_0" else nib * _h(raw[:, 0:2]) + _h(raw[:, 2:4])
    if quant == "q8_0":
        return raw[:, 2:].contiguous().view(torch.int8).double() * _h(raw[:, 0:2])
    if quant == "q4_k":
        d, dmin, p, qs = _h(raw[:, 0:2]), _h(raw[:, 2:4]), raw[:, 4:16], raw[:, 16:]
        sc = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1).double()
        qs = qs.reshape(n, 4, 32)
        nib = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32).double()
        return (nib * (d * sc)[:, :, None] - (dmin * mn)[:, :, None]).reshape(n, 256)
    if quant == "q6_k":
        ql, qh = raw[:, 0:128].reshape(n, 2, 64), raw[:, 128:192].reshape(n, 2, 32)
        sc, d = raw[:, 192:208].contiguous().view(torch.int8).double(), _h(raw[:, 208:210])
        parts = [(ql[:, :, 0:32] & 15) | ((qh & 3) << 4), (ql[:, :, 32:64] & 15) | (((qh >> 2) & 3) << 4),
                 (ql[:, :, 0:32] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 32:64] >> 4) | ((qh >> 6) << 4)]
        q = torch.stack(parts, 2).reshape(n, 16, 16).double() - 32
        return (q * (d * sc)[:, :, None]).reshape(n, 256)
    kind = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[quant]
    return raw.contiguous().view(kind).double()


def _times(quant, raw, rows, k, x):
    """x (m x k, float64) times the weight's transpose: m x rows."""
    per = k // BLOCK[quant][0]
    step = max(1, (1 << 26) // k)
    out = [x @ _dequant(quant, raw[r * per:min(rows, r + step) * per]).reshape(-1, k).T for r in range(0, rows, step)]
    return torch.cat(out, 1)


def _q8(x):
    """The q8 blocks' values of x (m x k, float32): d = amax / 127 and q = round-half-away(x / d), formed in 32 bits."""
    b = x.cpu().numpy().reshape(-1, 32)
    d = np.abs(b).max(1, keepdims=True) / np.float32(127)
    with np.errstate(divide="ignore"):
        inv = np.where(d != 0, np.float32(1) / d, np.float32(0)).astype(np.float32)
    v = (b * inv).astype(np.float64)
    q = np.clip(np.sign(v) * np.floor(np.abs(v) + 0.5), -127, 127)
    return torch.from_numpy((q * d.astype(np.float64)).reshape(x.shape)).cuda()


def _act(name, g, u):
    if name == "silu":
        return g / (1 + torch.exp(-g)) * u
    return 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3))) * u


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(h, pos):
    i = torch.arange(64, dtype=torch.float32)
    inv = torch.tensor(np.power(np.float32(ROPE_BASE), (np.float32(-2) * i.numpy() / np.float32(128))).astype(np.float32))
    a = (torch.tensor(float(pos), dtype=torch.float32) * inv).double().cuda()  # the angle is a 32-bit product
    x0, x1 = h[:, :64], h[:, 64:]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()], 1)


def _attend(qkv, qn, kn, kc, vc, n_heads, n_kv, pos):
    """(heads, k cache, v cache) after the block at `pos`: caches in their own f16."""
    h = qkv.double().reshape(-1, 128)
    q = _rope(_rms(h[:n_heads], qn), pos)
    k = _rope(_rms(h[n_heads:n_heads + n_kv], kn), pos)
    kc, vc = kc.clone(), vc.clone()
    kc[:, pos], vc[:, pos] = k.half(), h[n_heads + n_kv:].half()
    K, V = kc[:, :pos + 1].double(), vc[:, :pos + 1].double()
    s = torch.matmul(q.reshape(n_kv, -1, 128), K.transpose(1, 2).contiguous()) * 128 ** -0.5
    return torch.matmul(torch.softmax(s, -1), V).reshape(-1), kc, vc


def exact(case, seed):
    c, g = case, _Inputs(seed)
    kind = c["kind"]
    if kind == "burst_qkv":
        rows = (c["q_rows"], c["kv_rows"], c["kv_rows"])
        w = [g.weight(c["quant"], r, c["k"]) for r in rows]
        x = g.normal(c["k"]).double()[None]
        return [_times(c["quant"], t, r, c["k"], x)[0] for t, r in zip(w, rows)]
    if kind == "burst_mlp":
        gate, up = (g.weight(c["quant"], c["ffn"], c["k"]) for _ in range(2))
        down = g.weight(c["down"], c["k"], c["ffn"])
        x = g.normal(c["k"]).double()[None]
        mid = _act(c["act"], *(_times(c["quant"], t, c["ffn"], c["k"], x) for t in (gate, up)))
        return _times(c["down"], down, c["k"], c["ffn"], mid)[0]
    if kind in ("host_gemv", "host_matmul", "matmul"):
        m = c.get("m", 1)
        w, x = g.weight(c["quant"], c["rows"], c["k"]), g.normal(m, c["k"])
        y = _times(c["quant"], w, c["rows"], c["k"], x.double() if m <= FP_TOKENS else _q8(x))
        return y if kind == "matmul" else y.reshape(-1)
    if kind == "gemv":
        w, x = g.weight(c["quant"], c["rows"], c["k"]), g.normal(c["k"])
        up = g.weight(c["quant"], c["rows"], c["k"]) if "pair" in c["form"] else None
        norm, res = 1 + 0.1 * g.normal(c["k"]), g.normal(c["rows"])
        x = x.double()[None]
        x = _rms(x, norm) if "norm" in c["form"] else x
        y = _times(c["quant"], w, c["rows"], c["k"], x)
        if up is not None:
            y = _act(c["act"], y, _times(c["quant"], up, c["rows"], c["k"], x))
        return (y + res.double() if c["form"] == "resid" else y)[0]
    if kind == "attention":
        qkv = g.normal((c["n_heads"] + 2 * c["n_kv"]) * 128)
        qn, kn = 1 + 0.1 * g.normal(128), 1 + 0.1 * g.normal(128)
        kc, vc = (g.normal(c["n_kv"], c["max_seq"], 128).half() for _ in range(2))
        out, kc, vc = _attend(qkv, qn, kn, kc, vc, c["n_heads"], c["n_kv"], c["pos"])
        return {"out": out, "k_cache": kc.double(), "v_cache": vc.double()}
    # a whole step: the layers' tensors are made in the stream's order and the input comes last, so they wait on the host
    layers = [{n: t.cpu() for n, t in _step_layer(g, c).items()} for _ in range(c["n_layers"])]
    head, out_norm = g.weight("q8_0", c["vocab"], c["hidden"]), 1 + 0.1 * g.normal(c["hidden"])
    h = g.normal(c["hidden"]).double()[None]
    qr = 128 * c["n_heads"]
    for L in layers:
        L = {n: t.cuda() for n, t in L.items()}
        qkv = _times("q4_0", L["qkv"], qr + 256 * c["n_kv"], c["hidden"], _rms(h, L["attn_norm"]))
        att, _, _ = _attend(qkv, L["q_norm"], L["k_norm"], L["k_cache"], L["v_cache"], c["n_heads"], c["n_kv"], c["pos"])
        h = h + _times("q4_0", L["o"], c["hidden"], qr, att[None])
        n = _rms(h, L["ffn_norm"])
        mid = _act("silu", *(_times("q4_0", L[t], c["ffn"], c["hidden"], n) for t in ("gate", "up")))
        h = h + _times("q4_0", L["down"], c["hidden"], c["ffn"], mid)
    return _times("q8_0", head, c["vocab"], c["hidden"], _rms(h, out_norm))[0]
