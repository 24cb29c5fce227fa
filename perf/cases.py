"""The work that this package's users have it do, as cases that can be timed: the token loop of a LLaMA-2-7B shaped model
(prompts, single-token passes, both one after the other, in both summation orders), the operator-by-operator path
(Backend::submit), and single quantized MatMuls through the C ABI.  Model shape, weight types and context lengths are those of
the configurations in BASELINE.json, the odd sizes between them those of a conversation that goes on.

A case is a dict of plain values:
  kind      "prompt": one pass over `tokens` tokens on top of `past` cached ones, logits of the last token
            "decode": `steps` greedy single-token passes on the device on top of `past` cached tokens
            "generate": a prompt of `tokens` tokens and `steps` greedy tokens after it, as the command line tool does it
            "submit": one single-token pass operator by operator through Backend::submit on top of `past` cached tokens
            "matmul": one MatMul of a `rows` x `cols` weight matrix by `batch` activation rows through the C ABI
  model     weights: "q4_0" (Q4_0, Q6_K head), "q8_0", "q4_k_m" (Q4_K with Q6_K attn_v, ffn_down and head); matmul: `wtype`
  order     summation order of the model's passes: 1 (the host backend's, the default) or 0 (the backend's own)
"""
import ctypes as C
import math

import numpy as np
import torch

from spy_amd import _lib as H
from spy_amd import backend_driver as B
from spy_amd import model as M

TYPES = {"q4_0": H.Q4_0, "q8_0": H.Q8_0, "q4_k": H.Q4_K, "q6_k": H.Q6_K}
SUBMIT_LAYERS = 4                                                            # layers of the operator path's model (its weights come from host memory)


def listed():
    return [
        # the headline configuration: greedy decoding with 4096 tokens in the cache
        {"name": "decode_q4_0_4096", "kind": "decode", "model": "q4_0", "order": 1, "past": 4096, "steps": 16},
        # the shortest session: 8 prompt tokens, 32 generated ones
        {"name": "generate_q4_0_8_32", "kind": "generate", "model": "q4_0", "order": 1, "tokens": 8, "steps": 32},
        # a document as the prompt: the longest pass
        {"name": "prompt_q4_0_4096", "kind": "prompt", "model": "q4_0", "order": 1, "past": 0, "tokens": 4096},
        # the next turn of a conversation: a short, ragged prompt on a filled cache
        {"name": "prompt_q4_0_77_on_1000", "kind": "prompt", "model": "q4_0", "order": 1, "past": 1000, "tokens": 77},
        # a medium prompt and an answer to it, Q8_0 weights
        {"name": "generate_q8_0_512_24", "kind": "generate", "model": "q8_0", "order": 1, "tokens": 512, "steps": 24},
        # the mixed K-quant model: its prompt ...
        {"name": "prompt_q4_k_m_2048", "kind": "prompt", "model": "q4_k_m", "order": 1, "past": 0, "tokens": 2048},
        # ... and the decoding after it
        {"name": "decode_q4_k_m_2048", "kind": "decode", "model": "q4_k_m", "order": 1, "past": 2048, "steps": 16},
        # the backend's own summation order, chosen for speed
        {"name": "decode_q4_0_4096_own", "kind": "decode", "model": "q4_0", "order": 0, "past": 4096, "steps": 16},
        {"name": "prompt_q4_0_1000_own", "kind": "prompt", "model": "q4_0", "order": 0, "past": 0, "tokens": 1000},
        # a graph that an existing scheduler runs operator by operator
        {"name": "submit_q4_0_512", "kind": "submit", "model": "q4_0", "past": 512},
        # single operators: one activation row (the smallest call) and a batch of them
        {"name": "matmul_q4_0_11008_1", "kind": "matmul", "wtype": "q4_0", "rows": 11008, "cols": 4096, "batch": 1},
        {"name": "matmul_q4_k_11008_128", "kind": "matmul", "wtype": "q4_k", "rows": 11008, "cols": 4096, "batch": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "generate", "submit", "matmul", "matmul"])
    if kind == "matmul":
        wtype = rng.choice(sorted(TYPES))
        rows, cols = 32 * _log(rng, 8192 / 32, 32000 / 32), 256 * _log(rng, 16, 43)      # around the model's weight shapes, tiles with remainders among them
        return {"kind": kind, "wtype": wtype, "rows": rows, "cols": cols, "batch": rng.choice([1, _log(rng, 2, 512)])}
    if kind == "submit":
        return {"kind": kind, "model": "q4_0", "past": _log(rng, 8, 1024)}
    model = rng.choice(["q4_0", "q4_0", "q8_0", "q4_k_m"])
    if kind == "generate":
        return {"kind": kind, "model": model, "order": 1, "tokens": _log(rng, 2, 512), "steps": _log(rng, 8, 32)}
    order = rng.choice([1, 1, 1, 0])
    if kind == "decode":
        return {"kind": kind, "model": model, "order": order, "past": _log(rng, 8, 4096), "steps": _log(rng, 8, 32)}
    tokens = _log(rng, 2, 3000)
    return {"kind": kind, "model": model, "order": order, "past": rng.choice([0, _log(rng, 16, 1200)]), "tokens": tokens}


# ---- weights: bell-shaped quants and scales of the size that N(0, 0.02) weights have, made on the GPU in the native block layouts ----
def _bell(gen, shape, std, mean, lo, hi, dtype=torch.uint8):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float16).mul_(std).add_(mean).round_().clamp_(lo, hi).to(dtype)


def _scale(gen, n, size):
    return (torch.rand((n, 1), generator=gen, device="cuda") * 0.4 + 0.8).mul_(size).half()


def _bytes(x):
    return x.contiguous().view(torch.uint8)


def _blocks(gen, t, n):
    """n weights as the bytes of native blocks of type t"""
    nb = n // H.BLOCK_SIZE[t]
    if t == H.Q4_0:                                          # scale, 16 bytes of nibbles (low: elements 0..15, high: 16..31)
        q = _bell(gen, (nb, 32), 2.6, 8.0, 0, 15)
        parts = [_bytes(_scale(gen, nb, 0.02 / 2.6)), q[:, :16] | (q[:, 16:] << 4)]
    elif t == H.Q8_0:                                        # scale, 32 signed bytes
        parts = [_bytes(_scale(gen, nb, 0.02 / 45)), _bell(gen, (nb, 32), 45.0, 0.0, -127, 127, torch.int8).view(torch.uint8)]
    elif t == H.Q4_K:                                        # d, dmin, eight 6-bit scales and minima in 12 bytes, 128 bytes of nibbles
        d = _scale(gen, nb, 0.02 / 2.6 / 48)
        s = torch.randint(32, 64, (nb, 8), generator=gen, device="cuda", dtype=torch.uint8)     # scale and minimum alike: zero mean
        a, b = s[:, :4], s[:, 4:]
        top = a | ((b >> 4) << 6)
        parts = [_bytes(d), _bytes((d.float() * 7.5).half()), top, top, (b & 15) | ((b & 15) << 4)]
        q = _bell(gen, (nb, 4, 2, 32), 2.6, 7.5, 0, 15)
        parts.append((q[:, :, 0] | (q[:, :, 1] << 4)).reshape(nb, 128))
    else:                                                    # Q6_K: low nibbles, high pairs of bits, 16 signed scales, d
        q = _bell(gen, (nb, 2, 4, 32), 10.0, 32.0, 0, 63)
        lo, hi = q & 15, q >> 4
        ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], dim=2)
        qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
        s = torch.randint(64, 128, (nb, 16), generator=gen, device="cuda").mul_(torch.randint(0, 2, (nb, 16), generator=gen, device="cuda").mul_(2).sub_(1))
        parts = [ql.reshape(nb, 128), qh.reshape(nb, 64), s.to(torch.int8).view(torch.uint8), _bytes(_scale(gen, nb, 0.02 / 10 / 96))]
    return torch.cat(parts, dim=1).reshape(-1)


def _config(model, n_ctx, **kw):
    if model == "q4_0":
        return M.Config.llama2_7b(n_ctx=n_ctx, wtype=H.Q4_0, t_out=H.Q6_K, **kw)
    if model == "q8_0":
        return M.Config.llama2_7b(n_ctx=n_ctx, wtype=H.Q8_0, **kw)
    return M.Config.llama2_7b(n_ctx=n_ctx, wtype=H.Q4_K, t_out=H.Q6_K, tensor_types={"attn_v": H.Q6_K, "ffn_down": H.Q6_K}, **kw)


def _weights(cfg, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    out = {}
    for name, (t, rows, cols) in cfg.tensor_shapes().items():
        if "norm" in name:
            out[name] = torch.randn(cols, generator=gen, device="cuda").mul_(0.1).add_(1.0)
        elif t == H.F32:
            out[name] = torch.randn(rows * cols, generator=gen, device="cuda")
        else:
            out[name] = _blocks(gen, t, rows * cols)
            if name == "token_embd.weight":                  # Q8_0 table, embeddings ~ N(0, 1)
                d = out[name].view(-1, 34)
                d[:, :2] = _bytes((d[:, :2].contiguous().view(torch.float16).float() * 50.0).half())
    return out


class _DeviceArray:
    """An engine's own buffer as the outputs see it; keeps the engine alive."""

    def __init__(self, owner, ptr, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (ptr, False), "version": 2}


class _Model:
    """A model whose weights lie in device memory already, through the C ABI's token loop."""

    def __init__(self, cfg, seed, order):
        H.init(0)
        self.cfg, self.L = cfg, H.load()
        self.dev = _weights(cfg, seed)
        torch.cuda.synchronize()
        self.layers = (H.LlamaLayer * cfg.n_layer)()
        for i in range(cfg.n_layer):
            for field, name in (("attn_norm", "attn_norm"), ("ffn_norm", "ffn_norm"), ("wq", "attn_q"), ("wk", "attn_k"), ("wv", "attn_v"),
                                ("wo", "attn_output"), ("w_gate", "ffn_gate"), ("w_up", "ffn_up"), ("w_down", "ffn_down")):
                setattr(self.layers[i], field, self.dev["blk.%d.%s.weight" % (i, name)].data_ptr())
            for field, name in (("t_wq", "attn_q"), ("t_wk", "attn_k"), ("t_wv", "attn_v"), ("t_wo", "attn_output"), ("t_gate", "ffn_gate"),
                                ("t_up", "ffn_up"), ("t_down", "ffn_down")):
                setattr(self.layers[i], field, cfg.tensor_types.get(name, 0))
        self.desc = H.LlamaDesc(cfg.n_layer, cfg.n_embd, cfg.n_head, cfg.n_ff, cfg.n_vocab, cfg.n_ctx, cfg.eps, cfg.rope_freq_base, cfg.wtype,
                                self.dev["token_embd.weight"].data_ptr(), cfg.t_tok_embd, self.dev["output_norm.weight"].data_ptr(),
                                self.dev["output.weight"].data_ptr(), cfg.t_out, self.layers)
        h = C.c_void_p()
        H.check(self.L.spy_hip_llama_create(C.byref(self.desc), C.byref(h)), "spy_hip_llama_create")
        self.handle = h
        self.order = order

    def set_order(self, order):
        H.check(self.L.spy_hip_llama_set_order(self.handle, order), "spy_hip_llama_set_order")

    def forward_last(self, tokens, past):
        logits = np.empty(self.cfg.n_vocab, dtype=np.float32)
        H.check(self.L.spy_hip_llama_forward_last(self.handle, None, tokens.ctypes.data, len(tokens), past, logits.ctypes.data), "spy_hip_llama_forward_last")
        return logits

    def decode(self, first, past, steps):
        tokens = np.empty(steps, dtype=np.int32)
        H.check(self.L.spy_hip_llama_decode_greedy(self.handle, None, first, past, steps, tokens.ctypes.data, 1), "spy_hip_llama_decode_greedy")
        return tokens

    def buffer(self, name, layer, typestr):
        p, n = C.c_void_p(), C.c_size_t()
        H.check(self.L.spy_hip_llama_buffer(self.handle, name.encode(), layer, C.byref(p), C.byref(n)), "spy_hip_llama_buffer")
        return torch.as_tensor(_DeviceArray(self, p.value, n.value // int(typestr[2:]), typestr), device="cuda")

    def updated(self):
        """what a pass leaves behind: the last layer's caches"""
        last = self.cfg.n_layer - 1
        return {"k_cache": self.buffer("k_cache", last, "<f2"), "v_cache": self.buffer("v_cache", last, "<f2")}

    def __del__(self):
        if getattr(self, "handle", None):
            self.L.spy_hip_llama_destroy(self.handle)
            self.handle = None


def _ctx(n):
    return (n + 63) // 64 * 64


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "matmul":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        H.init(0)
        wt, rows, cols, batch = TYPES[case["wtype"]], case["rows"], case["cols"], case["batch"]
        w = _blocks(gen, wt, rows * cols)
        x = torch.randn((batch, cols), generator=gen, device="cuda")
        out = torch.empty((batch, rows), device="cuda")
        tw, tx, to = H.tensor(w.data_ptr(), wt, [cols, rows]), H.tensor(x.data_ptr(), H.F32, [cols, batch]), H.tensor(out.data_ptr(), H.F32, [rows, batch])
        need = H.load().spy_hip_op_matmul_scratch_size(C.byref(tw), C.byref(tx))
        scratch = torch.empty(max(need, 1), device="cuda", dtype=torch.uint8)
        torch.cuda.synchronize()
        return {"kind": kind, "call": H.load().spy_hip_op_matmul, "args": (None, C.byref(tw), C.byref(tx), C.byref(to), scratch.data_ptr(), need), "out": out,
                "keep": (w, x, scratch, tw, tx, to)}
    if kind == "submit":
        past = case["past"]
        cfg = _config(case["model"], _ctx(past + 8), t_tok_embd=H.Q8_0)
        cfg.n_layer = SUBMIT_LAYERS
        host = {k: v.view(torch.uint8).cpu().numpy() for k, v in _weights(cfg, seed).items()}
        m = B.HostModel(cfg, host)
        tokens = rng.integers(0, cfg.n_vocab, past + 1).astype(np.int32)
        m.forward(tokens[:past], 0)
        return {"kind": kind, "m": m, "token": tokens[past:], "past": past}
    past, tokens, steps = case.get("past", 0), case.get("tokens", 0), case.get("steps", 0)
    m = _Model(_config(case["model"], _ctx(past + tokens + steps + 8)), seed, case["order"])
    ids = rng.integers(0, m.cfg.n_vocab, past + tokens + 1).astype(np.int32)
    if past:                                                 # the conversation so far, in the default order: the same caches for both orders
        m.forward_last(ids[:past], 0)
    m.set_order(case["order"])
    return {"kind": kind, "m": m, "tokens": np.ascontiguousarray(ids[past:past + tokens]), "first": int(ids[-1]), "past": past, "steps": steps}


def run(state):
    kind = state["kind"]
    if kind == "matmul":
        H.check(state["call"](*state["args"]), "spy_hip_op_matmul")
        return state["out"]
    m = state["m"]
    if kind == "submit":
        return m.forward(state["token"], state["past"])
    out = m.updated()
    if kind == "decode":
        out["tokens"] = m.decode(state["first"], state["past"], state["steps"])
        out["logits"] = m.buffer("logits", 0, "<f4")
    else:
        out["logits"] = m.forward_last(state["tokens"], state["past"])
        if kind == "generate":
            first = int(np.argmax(out["logits"]))
            out["tokens"] = m.decode(first, len(state["tokens"]), state["steps"])
    return out


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        wt, rows, cols, batch = TYPES[case["wtype"]], case["rows"], case["cols"], case["batch"]
        return {"bytes": H.row_size(wt, rows * cols) + 4 * batch * (rows + cols), "flops": 2 * rows * cols * batch}
    cfg = _config(case["model"], 64)
    if kind == "submit":
        cfg.n_layer = SUBMIT_LAYERS
    d, F, V, L = cfg.n_embd, cfg.n_ff, cfg.n_vocab, cfg.n_layer
    params, head, kv = L * (4 * d * d + 3 * d * F), V * d, 4 * d * L           # kv: bytes of K and V per cached token

    def step(n_kv):
        return cfg.weight_bytes() + kv * n_kv, 2 * (params + head) + 4 * d * L * n_kv

    def prompt(past, t):
        return cfg.weight_bytes() + kv * (past + t) + 4 * V, 2 * (params * t + head) + 4 * d * L * (t * past + t * (t + 1) // 2)

    parts = []
    if kind in ("prompt", "generate"):
        parts.append(prompt(case.get("past", 0), case["tokens"]))
    if kind in ("decode", "generate"):
        n0 = case.get("past", 0) + case.get("tokens", 0)
        parts += [step(n0 + i + 1) for i in range(case["steps"])]
    if kind == "submit":
        parts.append(step(case["past"] + 1))
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    if case["kind"] == "matmul":
        return {"rel": 1e-5}                                 # fp32 sums of exact block dots
    if case.get("order") == 1:
        return "exact"                                       # the host backend's summation order: the same bits
    # Every MatMul rounds its activations to 8 bits, so a last-bit difference upstream moves some of them by a whole quantization
    # step, layer after layer; the greedy tokens of the own order are those of its own arithmetic.
    return {"rel": 2e-2} if case["kind"] != "decode" else {"rel": 2e-2, "differ": 0.0}
