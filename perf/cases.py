"""The work whose speed is followed: what a user of the library has it do, through its public
entry points (include/switch_gpu.h, bound by switch-l4t-gpu_amd/sgpu.py).

Kinds of case and the use each stands for:
  sgemm     C = A B in fp32 through sgpu_sgemm_opt: the harness's squares (256 to 4096), its
            ragged 1023x1025x997, and products with odd sides
  gemv      one batch-1 product through sgpu_gemv_h / _hh / _warp_b: a vocabulary head or a
            projection that a host launches by itself
  layer     the four products of one Qwen2.5-0.5B decode layer, one call each: a host that
            keeps the reference's per-layer sequence
  batched   sgpu_gemv_multi: a projection of a prompt's rows (GPT-2 124M's shapes and others)
  prompt    a whole prompt through a decode engine, its last row's logits back
  request   a prompt and greedy tokens through an engine, with the logits that follow them
  chat      an engine whose cache holds a long conversation: the next positions one by one,
            each position's logits back on the host, as a sampling loop calls it

Models are random-init at the repository's own dimensions: Qwen2.5-0.5B (fp16 weights) and
GPT-2 124M (fp32 weights), with norm gains near one as trained models have them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "switch-l4t-gpu_amd"))
import sgpu  # noqa: E402

QWEN = dict(V=151936, C=896, NL=24, NH=14, NKV=2, HD=64, FC=4864, CTX=8192, eps=1e-6, theta=1e6)
GPT2 = dict(V=50257, C=768, NL=12, NH=12, HD=64, FC=3072, CTX=1024, eps=1e-5)
QWEN_LAYER = [("qkv", 896, 1152, True), ("o", 896, 896, False), ("gate_up", 896, 9728, False), ("down", 4864, 896, False)]

# The largest drawn sizes: no drawn case costs more than the largest listed one of its kind.
SGEMM_FLOP = 2 * 4096**3
GEMV_WEIGHTS = 151936 * 896


def listed():
    return [
        # the smallest product of the harness: launch and latency
        {"name": "sgemm_256", "kind": "sgemm", "M": 256, "N": 256, "K": 256},
        # the reference harness's ragged verification shape
        {"name": "sgemm_ragged", "kind": "sgemm", "M": 1023, "N": 1025, "K": 997},
        # an ordinary product with odd sides
        {"name": "sgemm_odd_2k", "kind": "sgemm", "M": 2047, "N": 2049, "K": 2048},
        # the harness's headline product
        {"name": "sgemm_4096", "kind": "sgemm", "M": 4096, "N": 4096, "K": 4096},
        # the vocabulary head of Qwen2.5-0.5B: the largest batch-1 product
        {"name": "gemv_lm_head", "kind": "gemv", "weights": "f16", "x": "f32", "K": 896, "N": 151936, "bias": False},
        # one decode layer's products, called one by one
        {"name": "qwen_layer_gemvs", "kind": "layer"},
        # a short prompt's rows through GPT-2's widest projection
        {"name": "batched_fc_100", "kind": "batched", "K": 768, "N": 3072, "T": 100},
        # an ordinary prompt (a question with some context)
        {"name": "qwen_prompt_500", "kind": "prompt", "model": "qwen", "T": 500},
        # a long prompt (a document)
        {"name": "qwen_prompt_3001", "kind": "prompt", "model": "qwen", "T": 3001},
        # a short question and its answer
        {"name": "qwen_request_32_64", "kind": "request", "model": "qwen", "T": 32, "gen": 64},
        # a text and its continuation on the fp32 model
        {"name": "gpt2_request_300_32", "kind": "request", "model": "gpt2", "T": 300, "gen": 32},
        # the end of a long conversation, sampled on the host
        {"name": "qwen_chat_4000", "kind": "chat", "model": "qwen", "T": 4000, "gen": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sgemm", "sgemm", "gemv", "batched", "prompt", "prompt", "request", "chat"])
    if kind == "sgemm":
        while True:
            M, N, K = (_log(rng, 64, 8192) for _ in range(3))
            if rng.random() < 0.4:                          # whole tiles, as weight matrices have them
                M, N, K = (max(64, 64 * round(v / 64)) for v in (M, N, K))
            if 2 * M * N * K <= SGEMM_FLOP:
                return {"kind": kind, "M": M, "N": N, "K": K}
    if kind == "gemv":
        w, x = rng.choice([("f16", "f32"), ("f16", "f16"), ("f32", "f32")])
        while True:
            K, N = _log(rng, 256, 8192), _log(rng, 256, 160000)
            if rng.random() < 0.8:                          # most weight rows are whole 16-byte segments
                K = 8 * round(K / 8)
            if 2**18 <= N * K <= GEMV_WEIGHTS:
                return {"kind": kind, "weights": w, "x": x, "K": K, "N": N, "bias": rng.random() < 0.5}
    if kind == "batched":
        K, N = rng.choice([(768, 2304), (768, 768), (768, 3072), (3072, 768), (896, 4864), (4096, 4096), (1000, 3001)])
        return {"kind": kind, "K": K, "N": N, "T": _log(rng, 1, 1024)}
    model = "qwen" if kind == "chat" else rng.choice(["qwen", "qwen", "gpt2"])
    if kind == "prompt":
        return {"kind": kind, "model": model, "T": _log(rng, 8, 3000 if model == "qwen" else 1000)}
    if kind == "request":
        return {"kind": kind, "model": model, "T": _log(rng, 1, 900), "gen": _log(rng, 4, 100)}
    return {"kind": kind, "model": model, "T": _log(rng, 64, 8000), "gen": rng.randint(2, 12)}


# ---- inputs ----
def _rng(seed, salt):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + salt)


def _normal(shape, g, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)


def _uniform(shape, g):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32).mul_(2.0).sub_(1.0)


def _sgemm_inputs(case, seed):
    g = _rng(seed, 1)
    return _uniform((case["M"], case["K"]), g), _uniform((case["K"], case["N"]), g)


def _gemv_inputs(case, seed):
    g = _rng(seed, 2)
    W = _normal((case["N"], case["K"]), g, 0.02)
    x = _normal((case["K"],), g)
    b = _normal((case["N"],), g, 0.02) if case["bias"] else None
    return W.half() if case["weights"] == "f16" else W, x.half() if case["x"] == "f16" else x, b


def _layer_inputs(seed):
    g = _rng(seed, 3)
    return [(_normal((N, K), g, 0.02).half(), _normal((K,), g), _normal((N,), g, 0.02) if bias else None)
            for _, K, N, bias in QWEN_LAYER]


def _batched_inputs(case, seed):
    g = _rng(seed, 4)
    return (_normal((case["N"], case["K"]), g, 0.02), _normal((case["T"], case["K"]), g),
            _normal((case["N"],), g, 0.02))


def _qwen_weights(seed):
    """The tensors of the flat weight file in its order: name -> fp16 tensor on the GPU."""
    m, g = QWEN, _rng(seed, 5)
    C, FC, KVD = m["C"], m["FC"], m["NKV"] * m["HD"]
    Q = C + 2 * KVD

    def half(n, std, mean=0.0):
        return _normal(n, g, std, mean).half()

    layers = [dict(ln1=half((C,), 0.1, 1.0), qkv=half((Q, C), 0.04), qkvb=half((Q,), 0.02), o=half((C, C), 0.02),
                   ln2=half((C,), 0.1, 1.0), gateup=half((2 * FC, C), 0.02), down=half((C, FC), 0.02))
              for _ in range(m["NL"])]
    return dict(emb=half((m["V"], C), 0.02), layers=layers, lnf=half((C,), 0.1, 1.0))


def _rope_tables():
    m = QWEN
    h2 = m["HD"] // 2
    ang = np.arange(m["CTX"], dtype=np.float64)[:, None] * m["theta"] ** (-2.0 * np.arange(h2) / m["HD"])
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def _qwen_blob(seed):
    w = _qwen_weights(seed)
    parts = [w["emb"].reshape(-1).view(torch.uint8)]
    parts += [torch.from_numpy(t.reshape(-1)).cuda().view(torch.uint8) for t in _rope_tables()]
    for lw in w["layers"]:
        parts += [lw[k].reshape(-1).view(torch.uint8) for k in ("ln1", "qkv", "qkvb", "o", "ln2", "gateup", "down")]
    parts.append(w["lnf"].view(torch.uint8))
    return torch.cat(parts).cpu().numpy()


def _gpt2_weights(seed):
    m, g = GPT2, _rng(seed, 6)
    C, FC = m["C"], m["FC"]
    layers = [dict(ln1w=_normal((C,), g, 0.1, 1.0), ln1b=_normal((C,), g, 0.02), qkvw=_normal((3 * C, C), g, 0.04),
                   qkvb=_normal((3 * C,), g, 0.02), aow=_normal((C, C), g, 0.02), aob=_normal((C,), g, 0.02),
                   ln2w=_normal((C,), g, 0.1, 1.0), ln2b=_normal((C,), g, 0.02), fcw=_normal((FC, C), g, 0.02),
                   fcb=_normal((FC,), g, 0.02), projw=_normal((C, FC), g, 0.02), projb=_normal((C,), g, 0.02))
              for _ in range(m["NL"])]
    return dict(wte=_normal((m["V"], C), g, 0.02), wpe=_normal((m["CTX"], C), g, 0.01), layers=layers,
                lnfw=_normal((C,), g, 0.1, 1.0), lnfb=_normal((C,), g, 0.02))


def _gpt2_blob(seed):
    w = _gpt2_weights(seed)
    parts = [w["wte"], w["wpe"]] + [t for lw in w["layers"] for t in lw.values()] + [w["lnfw"], w["lnfb"]]
    return torch.cat([t.reshape(-1) for t in parts]).cpu().numpy()


def _ids(case, seed):
    """The prompt, then (for a chat) the tokens of the positions after it."""
    V = (QWEN if case["model"] == "qwen" else GPT2)["V"]
    return np.random.RandomState(seed % (1 << 32)).randint(0, V, case["T"] + case.get("gen", 0)).astype(np.int32)


def _engine(case, seed):
    if case["model"] == "qwen":
        return sgpu.QwenEngine(sgpu.qwen_cfg(**QWEN), _qwen_blob(seed), sgpu.QWEN_PATH_GRAPH)
    return sgpu.Gpt2Engine(sgpu.gpt2_cfg(**GPT2), _gpt2_blob(seed), sgpu.GPT2_PATH_GRAPH)


def prepare(case, seed):
    sgpu.init(0)
    kind = case["kind"]
    state = {"kind": kind, "case": case}
    if kind == "sgemm":
        A, B = _sgemm_inputs(case, seed)
        state.update(A=A, B=B, C=torch.empty((case["M"], case["N"]), device="cuda"))
    elif kind == "gemv":
        W, x, b = _gemv_inputs(case, seed)
        state.update(W=W, x=x, b=b, y=torch.empty((case["N"],), device="cuda"))
    elif kind == "layer":
        state["calls"] = [(W, x, b, torch.empty((W.shape[0],), device="cuda")) for W, x, b in _layer_inputs(seed)]
    elif kind == "batched":
        W, X, b = _batched_inputs(case, seed)
        state.update(W=W, X=X, b=b, Y=torch.empty((case["T"], case["N"]), device="cuda"))
    else:
        ids = _ids(case, seed)
        e = _engine(case, seed)
        state.update(engine=e, ids=ids)
        if kind == "chat":
            e.prefill(ids[:case["T"]])
            state["logits"] = np.empty((case["gen"], e.cfg.V), np.float32)
    return state


def _ptr(t):
    return None if t is None else t.data_ptr()


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "sgemm":
        sgpu.call("sgpu_sgemm_opt", _ptr(state["A"]), _ptr(state["B"]), _ptr(state["C"]), case["M"], case["N"], case["K"],
                  None)
        return state["C"]
    if kind == "gemv":
        name = "sgpu_gemv_warp_b" if case["weights"] == "f32" else "sgpu_gemv_hh" if case["x"] == "f16" else "sgpu_gemv_h"
        sgpu.call(name, _ptr(state["W"]), _ptr(state["x"]), _ptr(state["b"]), _ptr(state["y"]), case["K"], case["N"], None)
        return state["y"]
    if kind == "layer":
        for W, x, b, y in state["calls"]:
            sgpu.call("sgpu_gemv_h", _ptr(W), _ptr(x), _ptr(b), _ptr(y), W.shape[1], W.shape[0], None)
        return [y for _, _, _, y in state["calls"]]
    if kind == "batched":
        sgpu.call("sgpu_gemv_multi", _ptr(state["W"]), _ptr(state["X"]), _ptr(state["b"]), _ptr(state["Y"]), case["K"],
                  case["N"], case["T"], None)
        return state["Y"]
    e, ids, T = state["engine"], state["ids"], case["T"]
    if kind == "prompt":
        return e.prefill(ids)
    if kind == "request":
        tokens = e.generate(ids[:T], case["gen"])
        return {"tokens": tokens, "logits": e.forward(int(tokens[-1]), T + case["gen"])}
    out = state["logits"]                                   # chat
    forward = "sgpu_qwen_forward" if case["model"] == "qwen" else "sgpu_gpt2_forward"
    for i in range(case["gen"]):
        sgpu.call(forward, e.h, int(ids[T + i]), T + i, 1, out[i].ctypes.data)
    return out


# ---- work and tolerance ----
def _model_work(case):
    """(bytes, flops) of the layers' weights, of the head, and the attention's per cached position and row."""
    if case["model"] == "qwen":
        m, b = QWEN, 2
        KVD = m["NKV"] * m["HD"]
        layer = m["C"] * (m["C"] + 2 * KVD) + m["C"] ** 2 + 3 * m["C"] * m["FC"]
    else:
        m, b = GPT2, 4
        KVD = m["C"]
        layer = 4 * m["C"] ** 2 + 2 * m["C"] * m["FC"]
    return m, b, m["NL"] * layer, m["V"] * m["C"], m["NL"] * 2 * KVD * 4, m["NL"] * 4 * m["NH"] * m["HD"]


def work(case):
    kind = case["kind"]
    if kind == "sgemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    if kind == "gemv":
        N, K = case["N"], case["K"]
        w, x = (4 if case[k] == "f32" else 2 for k in ("weights", "x"))
        return {"bytes": w * N * K + x * K + 4 * N * (2 if case["bias"] else 1), "flops": 2 * N * K}
    if kind == "layer":
        return {"bytes": sum(2 * N * K + 4 * K + 4 * N * (2 if b else 1) for _, K, N, b in QWEN_LAYER),
                "flops": sum(2 * N * K for _, K, N, _ in QWEN_LAYER)}
    if kind == "batched":
        N, K, T = case["N"], case["K"], case["T"]
        return {"bytes": 4 * (N * K + T * K + T * N + N), "flops": 2 * N * K * T}
    m, b, layers, head, kv, att = _model_work(case)
    T, gen = case["T"], case.get("gen", 0)
    prompt_b = b * (layers + head) + kv * T + b * m["C"] * T + 4 * m["V"]
    prompt_f = 2 * layers * T + 2 * head + att * T * (T + 1) // 2
    steps = gen if kind != "request" else gen + 1
    step_b = sum(b * (layers + head) + kv * (T + i + 1) for i in range(steps))
    step_f = sum(2 * (layers + head) + att * (T + i + 1) for i in range(steps))
    if kind == "prompt":
        return {"bytes": prompt_b, "flops": prompt_f}
    if kind == "request":
        return {"bytes": prompt_b + step_b, "flops": prompt_f + step_f}
    return {"bytes": step_b + 4 * m["V"] * steps, "flops": step_f}


def tolerance(case):
    # fp32 products and sums everywhere: about four times the largest distance from exact()
    # measured over the listed and drawn cases (sgemm 5.7e-7 at K 4096, more at longer K; gemv
    # 1.5e-7; batched 4.3e-7 at K 4096; engines 1.1e-6)
    return {"rel": {"sgemm": 4e-6, "gemv": 1e-6, "layer": 1e-6, "batched": 2e-6}.get(case["kind"], 5e-6)}


# ---- the same in 64 bits ----
def _h(t):
    """fp16 weights as the engines read them: subnormal codes are zero."""
    d = t.double()
    return torch.where(d.abs() < 2.0**-14, torch.zeros_like(d), d)


def _attend(q, k, v, NH, NKV, HD, first):
    """Rows first.. of q (rows x NH*HD) over the cached rows of k and v, causal."""
    out = torch.empty_like(q)
    n, rows = k.shape[0], q.shape[0]
    mask = torch.arange(n, device=q.device)[None, :] > first + torch.arange(rows, device=q.device)[:, None]
    for h in range(NH):
        g = h // (NH // NKV)
        s = q[:, h * HD:(h + 1) * HD] @ k[:, g * HD:(g + 1) * HD].t().contiguous() / math.sqrt(HD)
        p = torch.softmax(s.masked_fill_(mask, -math.inf), 1)
        out[:, h * HD:(h + 1) * HD] = p @ v[:, g * HD:(g + 1) * HD].contiguous()
    return out


class _Qwen64:
    def __init__(self, seed):
        w = _qwen_weights(seed)
        self.m, self.emb, self.lnf = QWEN, _h(w["emb"]), _h(w["lnf"])
        self.layers = [{k: _h(t) for k, t in lw.items()} for lw in w["layers"]]
        self.cos, self.sin = (torch.from_numpy(t).cuda().double() for t in _rope_tables())
        kvd = QWEN["NKV"] * QWEN["HD"]
        self.cache = [[torch.empty((0, kvd), device="cuda", dtype=torch.float64)] * 2 for _ in self.layers]
        self.eps = float(np.float32(QWEN["eps"]))

    def rms(self, x, w):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + self.eps) * w

    def rope(self, x, pos, heads):
        h2 = self.m["HD"] // 2
        x = x.reshape(x.shape[0], heads, 2, h2)
        c, s = self.cos[pos:pos + x.shape[0], None], self.sin[pos:pos + x.shape[0], None]
        a, b = x[:, :, 0], x[:, :, 1]
        return torch.stack([a * c - b * s, a * s + b * c], 2).reshape(x.shape[0], -1)

    def rows(self, ids, pos):
        m = self.m
        C, kvd = m["C"], m["NKV"] * m["HD"]
        x = self.emb[torch.as_tensor(np.asarray(ids, np.int64), device="cuda")]
        for lw, kv in zip(self.layers, self.cache):
            y = self.rms(x, lw["ln1"]) @ lw["qkv"].t() + lw["qkvb"]
            q, k = self.rope(y[:, :C], pos, m["NH"]), self.rope(y[:, C:C + kvd], pos, m["NKV"])
            kv[0], kv[1] = torch.cat([kv[0], k]), torch.cat([kv[1], y[:, C + kvd:]])
            x = x + _attend(q, kv[0], kv[1], m["NH"], m["NKV"], m["HD"], pos) @ lw["o"].t()
            y = self.rms(x, lw["ln2"]) @ lw["gateup"].t()
            x = x + (torch.nn.functional.silu(y[:, :m["FC"]]) * y[:, m["FC"]:]) @ lw["down"].t()
        return self.rms(x[-1:], self.lnf)[0] @ self.emb.t()


class _Gpt264:
    def __init__(self, seed):
        w = _gpt2_weights(seed)
        self.w = {k: t.double() for k, t in w.items() if k != "layers"}
        self.layers = [{k: t.double() for k, t in lw.items()} for lw in w["layers"]]
        self.cache = [[torch.empty((0, GPT2["C"]), device="cuda", dtype=torch.float64)] * 2 for _ in self.layers]
        self.eps = float(np.float32(GPT2["eps"]))

    def ln(self, x, w, b):
        return torch.nn.functional.layer_norm(x, (x.shape[1],), w, b, self.eps)

    def rows(self, ids, pos):
        m, C = GPT2, GPT2["C"]
        n = len(ids)
        x = self.w["wte"][torch.as_tensor(np.asarray(ids, np.int64), device="cuda")] + self.w["wpe"][pos:pos + n]
        for lw, kv in zip(self.layers, self.cache):
            y = self.ln(x, lw["ln1w"], lw["ln1b"]) @ lw["qkvw"].t() + lw["qkvb"]
            kv[0], kv[1] = torch.cat([kv[0], y[:, C:2 * C]]), torch.cat([kv[1], y[:, 2 * C:]])
            x = x + _attend(y[:, :C], kv[0], kv[1], m["NH"], m["NH"], m["HD"], pos) @ lw["aow"].t() + lw["aob"]
            y = self.ln(x, lw["ln2w"], lw["ln2b"]) @ lw["fcw"].t() + lw["fcb"]
            y = 0.5 * y * (1.0 + torch.tanh(float(np.float32(0.7978845608)) * (y + float(np.float32(0.044715)) * y**3)))
            x = x + y @ lw["projw"].t() + lw["projb"]
        return self.ln(x[-1:], self.w["lnfw"], self.w["lnfb"])[0] @ self.w["wte"].t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sgemm":
        A, B = _sgemm_inputs(case, seed)
        return A.double() @ B.double()
    if kind in ("gemv", "layer"):
        calls = [_gemv_inputs(case, seed)] if kind == "gemv" else _layer_inputs(seed)
        out = []
        for W, x, b in calls:
            y = torch.cat([(_h(w) if w.dtype == torch.float16 else w.double()) @ (_h(x) if x.dtype == torch.float16 else x.double())
                           for w in W.split(16384)])
            out.append(y if b is None else y + b.double())
        return out[0] if kind == "gemv" else out
    if kind == "batched":
        W, X, b = _batched_inputs(case, seed)
        return X.double() @ W.double().t() + b.double()
    ids, T = _ids(case, seed), case["T"]
    model = _Qwen64(seed) if case["model"] == "qwen" else _Gpt264(seed)
    logits = model.rows(ids[:T], 0)
    if kind == "prompt":
        return logits
    if kind == "request":
        for i in range(case["gen"] + 1):                    # each greedy token, the last one's logits
            logits = model.rows([int(logits.argmax())], T + i)
        return {"tokens": None, "logits": logits}
    return torch.stack([model.rows(ids[T + i:T + i + 1], T + i) for i in range(case["gen"])])
