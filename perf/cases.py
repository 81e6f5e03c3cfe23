"""The work this framework is measured on: models and operators as a program uses them, over the range of their sizes.

A model case is one turn of a conversation: the cache holds `past` positions, `rows` prompt tokens come in, `steps` tokens are decoded
greedily, each read back by the host.  rows = 0 is decoding alone, steps = 0 a prompt alone.  Weights are random at the scale that keeps
a layer's output beside its input, as in a trained model; embedding and output table are one, so the greedy token is the token fed, by a
margin no rounding reaches.  Outputs: the logits, the tokens, and of GGUF models the last layer's cache, which every layer before it has a
part in.  exact() evaluates the same models in 64 bits, without the rounding of activations to 8 bits that belongs to Q4_K products here.
"""
import json
import math
import os
import shutil
import tempfile

import numpy as np
import torch

Q5_0, Q8_0, Q4_K, Q5_K, Q6_K = 6, 8, 12, 13, 14
BLOCK = {Q5_0: (32, 22), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}
TYPES = {"Q5_0": Q5_0, "Q8_0": Q8_0, "Q4_K": Q4_K, "Q5_K": Q5_K, "Q6_K": Q6_K}
MATRICES = ("q", "k", "v", "o", "gate", "up", "down")

# GGUF shapes: the benchmark's families, and a small model of generic sizes
GGUF = {
    "small": dict(vocab=32000, hidden=1024, n_layers=16, n_heads=16, n_kv_heads=4, head_dim=64, inter=2816, rope_base=1e4, eps=1e-5,
                  rope_interleaved=True),
    "qwen3_4b": dict(vocab=151936, hidden=2560, n_layers=36, n_heads=32, n_kv_heads=8, head_dim=128, inter=9728, rope_base=1e6, eps=1e-6),
    "llama3_8b": dict(vocab=128256, hidden=4096, n_layers=32, n_heads=32, n_kv_heads=8, head_dim=128, inter=14336, rope_base=5e5, eps=1e-5,
                      rope_interleaved=True),
    "qwen25_7b": dict(vocab=152064, hidden=3584, n_layers=28, n_heads=28, n_kv_heads=4, head_dim=128, inter=18944, rope_base=1e6, eps=1e-6),
    "gemma3_4b": dict(vocab=262144, hidden=2560, n_layers=34, n_heads=8, n_kv_heads=4, head_dim=256, inter=10240, rope_base=1e6, eps=1e-6,
                      scale_embeddings=True, ffn_gelu=True, swa_window=1024, swa_pattern=6, rope_swa_base=1e4, rope_scale=8.0),
}
QK_NORM = ("qwen3_4b", "gemma3_4b")
# model folders: widths of the benchmark's Tovasun and Nadozen models, with fewer layers and a smaller vocabulary so that a new model is
# quickly written and read
FOLDER = {1024: dict(heads=16, kv_heads=4, dim=64, ff=2816, rank=256, rot=32), 2560: dict(heads=32, kv_heads=8, dim=128, ff=9728, rank=512, rot=64),
          4096: dict(heads=32, kv_heads=8, dim=128, ff=14336, rank=512, rot=64)}
FOLDER_VOCAB = 8192


def _model(name, design, layers, past, rows, steps, width=0):
    return {"name": name, "kind": "model", "design": design, "width": width, "layers": layers, "past": past, "rows": rows, "steps": steps}


def listed():
    return [
        # one product through the type dispatcher, as a program with its own layers calls it: a gate projection of a Q8_0 file
        {"name": "gemv q8_0 9728x2560", "kind": "gemv", "type": "Q8_0", "rows": 9728, "cols": 2560},
        # the shortest call of a chat loop: a sampled token from logits that are there
        {"name": "sample 151936", "kind": "sample", "vocab": 151936, "top_k": 40, "top_p": 0.9, "temperature": 0.8, "penalty": 1.1},
        # a small model answering at the start of a conversation: launches count
        _model("steps small past 77", "small", 16, 77, 0, 8),
        # the ordinary case: a 4B model two pages into a conversation, and far into a long one
        _model("steps qwen3_4b past 2048", "qwen3_4b", 36, 2048, 0, 8),
        _model("steps qwen3_4b past 32411", "qwen3_4b", 24, 32411, 0, 8),
        # prompts: a short question, a page with its instructions, and a document in two chunks on a wider model
        _model("prompt qwen3_4b 19", "qwen3_4b", 36, 0, 19, 0),
        _model("prompt qwen3_4b 509", "qwen3_4b", 36, 0, 509, 0),
        _model("prompt llama3_8b 3001", "llama3_8b", 16, 0, 3001, 0),
        # layers described one by one, bfloat16: decoding and prompts of both designs (recurrent state starts with the prompt)
        _model("steps tovasun past 1500", "tovasun", 4, 1500, 0, 8, 2560),
        _model("prompt tovasun 1030", "tovasun", 4, 0, 1030, 0, 2560),
        _model("turn nadozen 30 + 24", "nadozen", 4, 0, 30, 24, 2560),
        _model("prompt nadozen 2048", "nadozen", 4, 0, 2048, 0, 2560),
    ]


def draw(rng):
    def between(lo, hi):  # evenly over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["gemv", "sample"] + ["steps", "prompt", "steps", "prompt", "turn"] * 2)
    if kind == "gemv":
        return {"kind": "gemv", "type": rng.choice(sorted(TYPES)), "rows": between(300, 30000), "cols": 256 * between(4, 56)}
    if kind == "sample":
        return {"kind": "sample", "vocab": between(1000, 262144), "top_k": rng.choice([0, 1, 20, 40, 100, 1000]), "top_p": rng.choice([0.8, 0.9, 0.95, 1.0]),
                "temperature": rng.choice([0.5, 0.8, 1.0]), "penalty": rng.choice([1.0, 1.1])}
    design = rng.choice(sorted(GGUF) + ["tovasun", "nadozen"])
    width = rng.choice(sorted(FOLDER)) if design not in GGUF else 0
    layers = rng.choice([2, 4]) if width else rng.randint(4, 12)
    past, rows, steps = 0, 0, 0
    if kind == "steps" and design != "nadozen":
        past, steps = between(16, 20000 if not width else 2500), rng.randint(4, 12)
    elif kind == "prompt":
        past, rows = 0 if design == "nadozen" or rng.random() < 0.6 else between(16, 2000), between(5, 3000)
    else:
        rows, steps = between(5, 400), rng.randint(8, 24)
    return {k: v for k, v in _model("", design, layers, past, rows, steps, width).items() if k != "name"}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


# ---- GGUF super-blocks --------------------------------------------------------------------------------------------------------
def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _half(values):
    return values.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def _blocks(g, qtype, n, std):
    """n blocks of weights with mean 0 and deviation about `std`."""
    b = _bytes(g, n, BLOCK[qtype][1])
    size = std * (0.5 + torch.rand(n, device="cuda", generator=g)) / 1.04
    if qtype in (Q4_K, Q5_K):  # scales of 32 .. 63; the mins put a block's middle at 0
        levels = 16 if qtype == Q4_K else 32
        d = (size / (48.4 * levels / 3.4641)).to(torch.float16)
        s = torch.randint(32, 64, (n, 8), dtype=torch.uint8, device="cuda", generator=g)
        b[:, 0:2], b[:, 2:4] = _half(d), _half(d.float() * (levels - 1) / 2)
        b[:, 4:8] = (s[:, :4] & 63) | ((s[:, 4:] >> 4) << 6)
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = (s[:, 4:] & 15) | ((s[:, 4:] & 15) << 4)
    elif qtype == Q6_K:
        s = torch.randint(24, 61, (n, 16), dtype=torch.int8, device="cuda", generator=g)
        b[:, 192:208], b[:, 208:210] = s.view(torch.uint8), _half(size / (43.3 * 18.5))
    else:
        b[:, 0:2] = _half(size / (73.9 if qtype == Q8_0 else 9.23))
    return b


def _dequant(qtype, b):
    """[n, block bytes] -> [n, values of a block] in 64 bits."""
    n = b.shape[0]

    def half(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()
    if qtype in (Q4_K, Q5_K):
        p = b[:, 4:16]
        sc = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, -128:].reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if qtype == Q5_K:
            q = q + torch.stack([(b[:, 16:48] >> i) & 1 for i in range(8)], 1) * 16
        return ((half(0) * sc)[:, :, None] * q.double() - (half(2) * mn)[:, :, None]).reshape(n, 256)
    if qtype == Q6_K:
        lo, hi = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        four = torch.cat([lo & 15, lo >> 4], 2)
        two = torch.cat([(hi >> (2 * i)) & 3 for i in range(4)], 2)
        q = (four | (two << 4)).double() - 32
        sc = b[:, 192:208].view(torch.int8).double().reshape(n, 2, 4, 2).repeat_interleave(16, dim=3)
        return (half(208).reshape(n, 1, 1, 1) * sc * q).reshape(n, 256)
    if qtype == Q8_0:
        return half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    bits = torch.stack([(b[:, 2 + i // 8] >> (i % 8)) & 1 for i in range(32)], 1) * 16
    return half(0) * ((torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], 1) + bits).double() - 16)


def _file_types(layer, n):
    """What a Q4_K_M file holds: attn_v and ffn_down in Q6_K in the first and last eighth of the layers and in every third between."""
    more = layer < n // 8 or layer >= 7 * n // 8 or (layer - n // 8) % 3 == 2
    return {m: Q6_K if more and m in ("v", "down") else Q4_K for m in MATRICES}


def _gguf_inputs(case, seed):
    """Everything a decoder of this case is made from, on the GPU.  A matrix is a stretch of one pool of blocks, from a place of its own."""
    g, cfg = _generator(seed), dict(GGUF[case["design"]], n_layers=case["layers"])
    H, hd, I, V = cfg["hidden"], cfg["head_dim"], cfg["inter"], cfg["vocab"]
    qd, kvd, gemma = cfg["n_heads"] * hd, cfg["n_kv_heads"] * hd, "swa_window" in cfg
    shape = {"q": (qd, H), "k": (kvd, H), "v": (kvd, H), "o": (H, qd), "gate": (I, H), "up": (I, H), "down": (H, I)}
    largest, spare = I * H // 256, 1 << 16
    pool = {t: _blocks(g, t, largest + spare, H ** -0.5) for t in (Q4_K, Q6_K)}
    place = np.random.RandomState(seed % (1 << 31))

    def near(n, mean, spread=0.1):
        return mean * (1 + spread * torch.randn(n, device="cuda", generator=g))
    layers, caches = [], []
    for i in range(case["layers"]):
        L = {}
        for m, t in _file_types(i, case["layers"]).items():
            at = int(place.randint(spare))
            L[m] = (t, at, shape[m])
        qk = case["design"] in QK_NORM
        L["attn_norm"], L["ffn_norm"] = near(H, 1.0 if qk else 1.5), near(H, 1.0)
        L["q_norm"], L["k_norm"] = (near(hd, 1.5), near(hd, 1.5)) if qk else (None, None)
        if case["design"] == "qwen25_7b":
            L["q_bias"], L["k_bias"], L["v_bias"] = near(qd, 0.0), near(kvd, 0.0), near(kvd, 0.0)
            for b in ("q_bias", "k_bias", "v_bias"):
                L[b] = 0.5 * torch.randn(L[b].shape, device="cuda", generator=g)
        if gemma:
            L["post_attn_norm"], L["post_ffn_norm"] = near(H, 0.5), near(H, 0.5)
        layers.append(L)
        caches.append([(1.5 * torch.randn(case["past"], kvd, device="cuda", generator=g)).half(),
                       torch.randn(case["past"], kvd, device="cuda", generator=g).half()])
    table = _blocks(g, Q6_K, V * (H // 256), 8 * H ** -0.5 if gemma else 8.0)
    tokens = [int(t) for t in torch.randint(0, V, (max(1, case["rows"]),), generator=g, device="cuda").cpu()]
    return cfg, pool, layers, caches, table, near(H, 1.0), tokens


def _matrix(pool, entry):
    t, at, (rows, cols) = entry
    return t, pool[t][at:at + rows * cols // 256].reshape(rows, -1)


class _View:
    """A buffer of the decoder as a tensor, which keeps the decoder."""

    def __init__(self, owner, pointer, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (pointer, False), "version": 2}


def _ready(m, case, tokens):
    """What a program keeps: the decoder, where its logits lie, the prompt."""
    logits = torch.as_tensor(_View(m, m.L.ptm_decode_logits(m.h), m.cfg["vocab"]), device="cuda")
    return {"model": m, "case": case, "tokens": tokens, "logits": logits}


def _prepare_gguf(case, seed):
    from prometorch_amd.decode import Decoder
    cfg, pool, layers, caches, table, out_norm, tokens = _gguf_inputs(case, seed)
    host = {t: p.cpu().numpy() for t, p in pool.items()}

    def array(x):
        if isinstance(x, tuple):
            t, at, (rows, cols) = x
            return t, host[t][at:at + rows * cols // 256].reshape(rows, -1)
        return None if x is None else x.cpu().numpy()
    head = {"lm_head": table.cpu().numpy().reshape(cfg["vocab"], -1), "out_norm": out_norm.cpu().numpy()}
    m = Decoder(cfg, [{k: array(x) for k, x in L.items()} for L in layers], head, max_seq=case["past"] + case["rows"] + case["steps"] + 8)
    for i, (k, v) in enumerate(caches):
        m.k_cache[i][:case["past"]], m.v_cache[i][:case["past"]] = k, v
    if case["rows"]:
        from prometorch_amd._lib import check
        check(m.L.ptm_decode_reserve_prefill(m.h, case["rows"]), "reserve_prefill")
    return _ready(m, case, tokens)


# ---- model folders ------------------------------------------------------------------------------------------------------------
def _folder_config(case):
    s, W = FOLDER[case["width"]], case["width"]
    layers = []
    for i in range(case["layers"] // 2):
        mlp = {"kind": "dense", "ff": s["ff"]}
        if case["design"] == "tovasun":
            lat = {"heads": s["heads"], "dim": s["dim"], "rot_dim": s["rot"], "kv_rank": s["rank"], "vdim": s["dim"], "scale": 2 * (s["dim"] + s["rot"]) ** -0.5,
                   "mask": {"size": 1024}, "rot": {"base": 10000.0, "dims": s["rot"], "scaling": {"factor": 4.0, "fast": 32.0, "slow": 1.0, "original": 4096}}}
            att = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"], "scale": 2 * s["dim"] ** -0.5, "softcap": 30.0,
                   "mask": {"size": 4096, "keep_first": 4}, "rot": {"base": 10000.0, "dims": s["dim"] // 2}}
            layers += [{"type": "latent_attention", "mixer": lat, "mlp": mlp}, {"type": "attention", "mixer": att, "mlp": mlp}]
        else:
            left = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"], "scale": 2 * s["dim"] ** -0.5, "mask": {"size": 4096}}
            right = {"heads": W // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
            layers += [{"type": "wkv", "mixer": {"heads": W // 64, "dim": 64}, "rank": 64, "mlp": mlp},
                       {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 0.7, "right_scale": 0.7}, "mlp": mlp}]
    cfg = {"architecture": case["design"].capitalize(), "layers": layers, "norm": {"eps": 1e-6}, "vocab": FOLDER_VOCAB, "width": W}
    return dict(cfg, token_side={"dim": 256}) if case["design"] == "tovasun" else dict(cfg, streams=4, logit_scale=1.0)


def _folder_inputs(case, seed):
    """Configuration, name -> bfloat16 tensor on the GPU, and the tokens in the cache and of the prompt.  Norms scatter around 1,
    matrices keep the scale of their input, decays reach from a few tokens to a few hundred."""
    from prometorch_amd.testing import folder_writer
    g, cfg, out = _generator(seed), _folder_config(case), {}
    for name, shape in folder_writer.tensor_shapes(cfg).items():
        a, last = torch.randn(shape, device="cuda", generator=g), name.rsplit(".", 1)[-1]
        if last in folder_writer.NADOZEN_SPREAD:
            a = folder_writer.NADOZEN_SPREAD[last](a)
        elif ".hc" in name:
            n = shape[0]
            a = 0.9 * torch.eye(n, device="cuda") + 0.1 / n * a if last == "mix" else (1 + 0.3 * a) / (n if last == "in" else 1.0)
        elif ".mu." in name:
            a = 0.5 + 0.3 * a
        elif len(shape) == 1:
            a = 1 + 0.1 * a
        elif "embed" not in name:
            a = a * shape[1] ** -0.5
        out[name] = a.to(torch.bfloat16)
    out["head"] = out["embed"]
    tokens = [int(t) for t in torch.randint(0, FOLDER_VOCAB, (case["past"] + max(1, case["rows"]),), generator=g, device="cuda").cpu()]
    return cfg, out, tokens


def _prepare_folder(case, seed):
    from prometorch_amd import _lib, model
    from prometorch_amd.testing import folder_writer
    cfg, weights, tokens = _folder_inputs(case, seed)
    where = tempfile.mkdtemp(prefix="model_", dir="/dev/shm" if os.access("/dev/shm", os.W_OK) else None)
    try:
        with open(os.path.join(where, "config.json"), "w") as f:
            json.dump(cfg, f)
        folder_writer.write_safetensors(os.path.join(where, "model.safetensors"), {n: a.view(torch.int16).cpu().numpy().view(np.uint16) for n, a in weights.items()})
        m = model.load(where, max_seq=case["past"] + case["rows"] + case["steps"] + 8)
    finally:
        shutil.rmtree(where)
    if case["rows"]:
        _lib.check(m.L.ptm_decode_reserve_prefill(m.h, case["rows"]), "reserve_prefill")
    if case["past"]:
        m.prefill(tokens[:case["past"]])
    return _ready(m, case, tokens[case["past"]:])


# ---- one pass -----------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    g = _generator(seed)
    if case["kind"] == "model":
        return (_prepare_folder if case["width"] else _prepare_gguf)(case, seed)
    if case["kind"] == "gemv":
        t, N, K = TYPES[case["type"]], case["rows"], case["cols"]
        n, size = BLOCK[t]
        return {"case": case, "w": _blocks(g, t, N * K // n, K ** -0.5).reshape(N, K // n * size), "x": torch.randn(K, device="cuda", generator=g),
                "y": torch.empty(N, device="cuda")}
    from prometorch_amd import ops
    V = case["vocab"]
    counts = (torch.rand(V, device="cuda", generator=g) < 0.001).to(torch.int32)
    return {"case": case, "logits": 3 * torch.randn(V, device="cuda", generator=g), "counts": counts, "u": torch.rand(1, device="cuda", generator=g),
            "ws": torch.zeros(ops.sampler_workspace_bytes(), dtype=torch.uint8, device="cuda"), "token": torch.zeros(1, dtype=torch.int64, device="cuda")}


def run(state):
    case = state["case"]
    if case["kind"] == "model":
        m, tokens, out = state["model"], state["tokens"], []
        m.set_past_len(case["past"])
        if case["rows"]:
            out.append(m.prefill(tokens))
        for _ in range(case["steps"]):
            out.append(m.step(out[-1] if out else tokens[0]))
        last = {} if case["width"] else {"k": m.k_cache[-1], "v": m.v_cache[-1]}
        return {"tokens": np.array(out), "logits": state["logits"], **last}
    from prometorch_amd import ops
    if case["kind"] == "gemv":
        ops.quant_gemv(TYPES[case["type"]], state["w"], state["x"], state["y"], case["cols"], case["rows"], state["w"].shape[1])
        return state["y"]
    ops.sample_token(state["logits"], case["vocab"], state["counts"], case["temperature"], case["top_k"], case["top_p"], case["penalty"], state["u"],
                     state["ws"], state["token"])
    return state["token"]


# ---- bytes and operations -----------------------------------------------------------------------------------------------------
def _folder_sizes(case):
    """(weight values without the tables, of them in matrices, values of one token's state or cache row, by layer kind)"""
    from prometorch_amd.testing import folder_writer
    cfg = _folder_config(case)
    shapes = {n: s for n, s in folder_writer.tensor_shapes(cfg).items() if n not in ("embed", "side.embed", "head")}
    return cfg, sum(math.prod(s) for s in shapes.values()), sum(math.prod(s) for s in shapes.values() if len(s) == 2)


def work(case):
    if case["kind"] == "gemv":
        n, size = BLOCK[TYPES[case["type"]]]
        return {"bytes": case["rows"] * case["cols"] // n * size + 4 * (case["rows"] + case["cols"]), "flops": 2 * case["rows"] * case["cols"]}
    if case["kind"] == "sample":
        return {"bytes": 8 * case["vocab"] + 8, "flops": 8 * case["vocab"]}
    past, rows, steps = case["past"], case["rows"], case["steps"]

    def seen(window, lo, hi):  # keys seen by the positions lo .. hi - 1, added up
        full = max(0, min(hi, window) - lo)
        return full * (2 * lo + full + 1) // 2 + (hi - lo - full) * window
    byte, flop = 0, 0
    if case["width"]:
        cfg, values, params = _folder_sizes(case)
        weights, head, kinds = 2 * values, FOLDER_VOCAB * case["width"], []
        for L in cfg["layers"]:
            m = L["mixer"]
            a = m.get("left", m)
            if L["type"] == "wkv":
                kinds.append((0, 0, 0, m["heads"] * m["dim"] * m["dim"]))
            elif L["type"] == "latent_attention":
                kinds.append((m["mask"]["size"], m["kv_rank"] + m["rot_dim"], m["heads"] * (2 * m["dim"] + m["rot_dim"]), 0))
            else:
                state = m["right"]["heads"] * m["right"]["vdim"] * m["right"]["state"] if "right" in m else 0
                kinds.append((a["mask"]["size"], (1 if "right" in m else 2) * a["kv_heads"] * a["dim"], 2 * a["heads"] * a["dim"], state))
        head_bytes = 2 * head
    else:
        cfg, params, weights, kinds = GGUF[case["design"]], 0, 0, []
        H, hd, I = cfg["hidden"], cfg["head_dim"], cfg["inter"]
        qd, kvd = cfg["n_heads"] * hd, cfg["n_kv_heads"] * hd
        for i in range(case["layers"]):
            for m, t in _file_types(i, case["layers"]).items():
                n = {"q": qd * H, "k": kvd * H, "v": kvd * H, "o": H * qd}.get(m, I * H)
                params += n
                weights += n // 256 * BLOCK[t][1]
            local = "swa_window" in cfg and (i + 1) % cfg["swa_pattern"]
            kinds.append((cfg["swa_window"] if local else 1 << 30, 2 * kvd, 2 * qd, 0))
        head = cfg["vocab"] * H
        head_bytes = head // 256 * 210
    passes = (1 if rows else 0) + steps
    byte += passes * (weights + head_bytes + 4 * (cfg["vocab"]))
    flop += 2 * (rows + steps) * params + 2 * passes * head
    for window, row, per_key, state in kinds:
        for lo, hi in ([(past, past + rows)] if rows else []) + [(past + rows + i, past + rows + i + 1) for i in range(steps)]:
            byte += 2 * row * (min(hi, window + hi - lo) + hi - lo) + 8 * state
            flop += 2 * per_key * seen(window, lo, hi) + 4 * state * (hi - lo)
    return {"bytes": byte, "flops": flop}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    if case["kind"] == "gemv":  # products of 32-bit activations; Q4_K: of activations rounded to 8 bits, alike in any order of the sums
        return {"rel": 1e-5, "max": 1e-4}
    # rounded to 8 bits (GGUF) or bfloat16, activations leave logits 0.003 to 0.013 off the 64-bit ones, and two ways of adding up as far apart
    return {"rel": 0.02 if case["width"] else 0.03, "max": 0.3}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------------------
def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, first, window, keep=0, cap=0.0, sink=None):
    """q [n, H, d] at positions first .., k and v [positions, G, .] from 0 on; a head at a time, rows in pieces."""
    n, H, _ = q.shape
    per, out = H // k.shape[1], torch.empty(q.shape[0], H, v.shape[-1], dtype=torch.float64, device="cuda")
    for h in range(H):
        kh, vh = k[:, h // per].contiguous(), v[:, h // per].contiguous()
        for lo in range(0, n, 1024):
            rows = torch.arange(lo, min(lo + 1024, n), device="cuda")
            i, j = first + rows[:, None], torch.arange(len(kh), device="cuda")[None, :]
            s = (q[rows, h] @ kh.T) * scale
            s = cap * torch.tanh(s / cap) if cap else s
            s = s.masked_fill(~((j <= i) & ((i - j < window) | (j < keep))), -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(len(rows), 1)], 1)
            out[rows, h] = torch.softmax(s, 1)[:, :len(kh)] @ vh
    return out


def _turn(x, first, freq, amplitude=1.0, halves=False):
    """Rotation of [n, heads, d]: pairs (2i, 2i + 1), or (i, i + d / 2), of the first 2 * len(freq) values."""
    d = 2 * len(freq)
    a = (first + torch.arange(len(x), dtype=torch.float64, device="cuda"))[:, None, None] * freq
    c, s = torch.cos(a) * amplitude, torch.sin(a) * amplitude
    u, v = (x[..., :d // 2], x[..., d // 2:d]) if halves else (x[..., 0:d:2], x[..., 1:d:2])
    y = torch.cat([u * c - v * s, v * c + u * s], -1) if halves else torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)
    return torch.cat([y, x[..., d:]], -1)


def _frequencies(base, d):
    return base ** (-torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d)


def _all_tokens(case, tokens):
    """The prompt and the tokens that are fed after it: the greedy token is the last one again."""
    return (tokens if case["rows"] else []) + [tokens[-1]] * case["steps"]


def _exact_gguf(case, seed):
    cfg, pool, layers, caches, table, out_norm, tokens = _gguf_inputs(case, seed)
    H, hd, nh, nkv, eps, past = cfg["hidden"], cfg["head_dim"], cfg["n_heads"], cfg["n_kv_heads"], cfg["eps"], case["past"]
    fed = torch.tensor(_all_tokens(case, tokens), device="cuda")
    x = _dequant(Q6_K, table.reshape(cfg["vocab"], -1)[fed].reshape(-1, 210)).reshape(len(fed), H)
    x = x * H ** 0.5 if cfg.get("scale_embeddings") else x
    n = len(fed)

    def times(y, L, m):
        t, w = _matrix(pool, L[m])
        y = y @ _dequant(t, w.reshape(-1, BLOCK[t][1])).reshape(w.shape[0], -1).T
        return y + L[m + "_bias"] if m + "_bias" in L else y
    for i, L in enumerate(layers):
        L = {k: v.double() if isinstance(v, torch.Tensor) else v for k, v in L.items()}
        local = "swa_window" in cfg and (i + 1) % cfg["swa_pattern"] != 0
        h = _rms(x, eps) * L["attn_norm"]
        q, k, v = (times(h, L, m).reshape(n, -1, hd) for m in "qkv")
        if L["q_norm"] is not None:
            q, k = _rms(q, eps) * L["q_norm"], _rms(k, eps) * L["k_norm"]
        freq = _frequencies(cfg["rope_swa_base"] if local else cfg["rope_base"], hd) / (1.0 if local else cfg.get("rope_scale", 1.0))
        q, k = (_turn(y, past, freq, halves=not cfg.get("rope_interleaved")) for y in (q, k))
        k, v = (torch.cat([c.double().reshape(past, nkv, hd), y]) for c, y in zip(caches[i], (k, v)))
        caches[i] = None
        o = times(_attend(q, k, v, hd ** -0.5, past, cfg["swa_window"] if local else 1 << 30).reshape(n, -1), L, "o")
        x = x + (_rms(o, eps) * L["post_attn_norm"] if "post_attn_norm" in L else o)
        h = _rms(x, eps) * L["ffn_norm"]
        gate = times(h, L, "gate")
        gate = torch.nn.functional.gelu(gate, approximate="tanh") if cfg.get("ffn_gelu") else torch.nn.functional.silu(gate)
        o = times(gate * times(h, L, "up"), L, "down")
        x = x + (_rms(o, eps) * L["post_ffn_norm"] if "post_ffn_norm" in L else o)
    y = _rms(x[-1], eps) * out_norm.double()
    rows = table.reshape(cfg["vocab"], -1).split(16384)
    logits = torch.cat([_dequant(Q6_K, r.reshape(-1, 210)).reshape(len(r), H) @ y for r in rows])
    pad = torch.zeros(8, nkv * hd, dtype=torch.float64, device="cuda")
    return {"tokens": None, "logits": logits, "k": torch.cat([k.reshape(-1, nkv * hd), pad]), "v": torch.cat([v.reshape(-1, nkv * hd), pad])}


def _exact_tovasun(cfg, w, tokens):
    eps, n = cfg["norm"]["eps"], len(tokens)
    x = w["embed"][tokens]
    for i, L in enumerate(cfg["layers"]):
        p, m = "l%d." % i, L["mixer"]
        z, H, window = p + "mix.", m["heads"], m["mask"]["size"]
        h, rot = _rms(x, eps) * w[p + "norm1"], m["rot"]
        freq, amp = _frequencies(rot["base"], rot["dims"]), 1.0
        if "scaling" in rot:  # YaRN
            s = rot["scaling"]
            lo, hi = (rot["dims"] * math.log(s["original"] / (2 * math.pi * t)) / (2 * math.log(rot["base"])) for t in (s["fast"], s["slow"]))
            lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), rot["dims"] - 1)
            ramp = ((torch.arange(len(freq), device="cuda") - lo).double() / max(hi - lo, 0.001)).clamp(0, 1)
            freq, amp = freq * (1 - ramp) + freq / s["factor"] * ramp, 0.1 * math.log(s["factor"]) + 1
        if L["type"] == "attention":
            q, k = (_turn((_rms(h @ w[z + c].T, eps) * w[z + c + ".norm"]).reshape(n, -1, m["dim"]), 0, freq, amp) for c in "qk")
            v = (h @ w[z + "v"].T).reshape(n, -1, m["vdim"])
        else:
            q, down = (h @ w[z + "q"].T).reshape(n, H, -1), h @ w[z + "dkv"].T
            c = _rms(down[:, :m["kv_rank"]], eps) * w[z + "dkv.norm"]
            q = torch.cat([q[..., :m["dim"]], _turn(q[..., m["dim"]:], 0, freq, amp)], -1)
            k = _turn(down[:, None, m["kv_rank"]:], 0, freq, amp).expand(n, H, m["rot_dim"])
            k, v = torch.cat([(c @ w[z + "uk"].T).reshape(n, H, -1), k], -1), (c @ w[z + "uv"].T).reshape(n, H, -1)
        o = _attend(q, k, v, m["scale"], 0, window, m["mask"].get("keep_first", 0), m.get("softcap", 0.0))
        x = x + _rms(o.reshape(n, -1) @ w[z + "o"].T, eps) * w[p + "norm1b"]
        h = torch.relu((_rms(x, eps) * w[p + "norm2"]) @ w[p + "mlp.up"].T).square() @ w[p + "mlp.down"].T
        x = x + _rms(h, eps) * w[p + "norm2b"]
        d = cfg["token_side"]["dim"]
        e = torch.nn.functional.gelu(x @ w[p + "side.gate"].T, approximate="tanh") * w["side.embed"][tokens][:, i * d:(i + 1) * d]
        x = x + _rms(e @ w[p + "side.proj"].T, eps) * w[p + "side.norm"]
    return (_rms(x[-1], eps) * w["final.norm"]) @ w["head"].T


def _scan(decay, keys, values, reads, bonus=None):
    """Matrix states [heads, keys, values] over the tokens: state = decay * state + key x value, read by `reads` - before the token is
    added and with `bonus` times it, or after it."""
    state, out = torch.zeros(values.shape[1], keys.shape[2], values.shape[2], dtype=torch.float64, device="cuda"), []
    for d, k, v, r in zip(decay, keys, values, reads):
        new = k[..., None] * v[:, None, :]
        seen = state + bonus[..., None] * new if bonus is not None else None
        state = d[..., None] * state + new
        out.append(((seen if bonus is not None else state) * r[..., None]).sum(1))
    return torch.stack(out)


def _exact_nadozen(cfg, w, tokens):
    eps, n, W, silu = cfg["norm"]["eps"], len(tokens), cfg["width"], torch.nn.functional.silu

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, (W,), w[name], w[name + ".b"], eps)
    c = torch.arange(W, device="cuda")
    angle = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * 10000.0 ** (-(c - c % 2).double() / W)
    x = (w["embed"][tokens] + torch.where(c % 2 == 0, torch.sin(angle), torch.cos(angle))).expand(cfg["streams"], n, W)

    def mix(x, p, branch):
        y = branch(torch.tensordot(w[p + "in"], x, 1))
        return torch.tensordot(w[p + "mix"].T, x, 1) + w[p + "out"][:, None, None] * y

    def wkv(h, z, m):
        H, d = m["heads"], m["dim"]
        back = torch.cat([torch.zeros_like(h[:1]), h[:-1]]) - h
        r, k, v, g, dec = (h + back * w[z + "mu." + s] for s in "rkvgw")
        r, k, v = ((y @ w[z + s].T).reshape(n, H, d) for y, s in ((r, "r"), (k, "k"), (v, "v")))
        dec = torch.exp(-torch.exp(torch.tanh(dec @ w[z + "w1"].T) @ w[z + "w2"].T + w[z + "w0"])).reshape(n, H, d)
        o = _rms(_scan(dec, k, v, r, w[z + "u"]), eps).reshape(n, -1)
        return (o * w[z + "norm"] * silu(g @ w[z + "g"].T)) @ w[z + "o"].T

    def parallel(h, z, m):
        l, r = m["left"], m["right"]
        y, q = z + "left.", z + "right."
        raw = (h @ w[y + "k"].T).reshape(n, -1, l["dim"])
        query = _rms((h @ w[y + "q"].T).reshape(n, -1, l["dim"]), eps) * w[y + "q.norm"]
        o = _attend(query, _rms(raw, eps) * w[y + "k.norm"], raw, l["scale"], 0, l["mask"]["size"], sink=w[y + "sink"]).reshape(n, -1)
        left = (o * torch.sigmoid(h @ w[y + "g"].T)) @ w[y + "o"].T
        H, v, N = r["heads"], r["vdim"], r["state"]
        gate, xbc, dt = (h @ w[q + "in"].T).split([H * v, H * v + 2 * N, H], 1)
        xbc = torch.nn.functional.pad(xbc.T, (r["conv"] - 1, 0))
        xbc = silu(sum(xbc[:, i:i + n] * w[q + "conv"][:, i:i + 1] for i in range(r["conv"])).T + w[q + "conv.b"])
        xs, B, C = xbc[:, :H * v].reshape(n, H, v), xbc[:, H * v:H * v + N], xbc[:, H * v + N:]
        dt = torch.nn.functional.softplus(dt + w[q + "dt_bias"])
        decay = torch.exp(-torch.exp(w[q + "A_log"]) * dt)[..., None]
        o = _scan(decay, dt[..., None] * B[:, None, :], xs, C[:, None, :].expand(n, H, N)) + w[q + "D"][:, None] * xs
        o = _rms(o.reshape(n, -1) * silu(gate), eps) * w[q + "norm"]
        return m["left_scale"] * left + m["right_scale"] * (o @ w[q + "o"].T)
    for i, L in enumerate(cfg["layers"]):
        p = "l%d." % i
        mixer = wkv if L["type"] == "wkv" else parallel
        x = mix(x, p + "hc1.", lambda u: mixer(norm(u, p + "norm1"), p + "mix.", L["mixer"]))
        x = mix(x, p + "hc2.", lambda u: (silu((u := norm(u, p + "norm2")) @ w[p + "mlp.gate"].T) * (u @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T)
    return norm(x.sum(0)[-1:], "final.norm")[0] @ w["head"].T * cfg["logit_scale"]


def exact(case, seed):
    if case["kind"] == "sample":
        return None
    if case["kind"] == "gemv":
        s, t = prepare(case, seed), TYPES[case["type"]]
        return _dequant(t, s["w"].reshape(-1, BLOCK[t][1])).reshape(case["rows"], -1) @ s["x"].double()
    if not case["width"]:
        return _exact_gguf(case, seed)
    cfg, weights, tokens = _folder_inputs(case, seed)
    fed = tokens[:case["past"]] + _all_tokens(case, tokens[case["past"]:])
    w = {k: v.double() for k, v in weights.items()}
    return {"tokens": None, "logits": (_exact_tovasun if case["design"] == "tovasun" else _exact_nadozen)(cfg, w, torch.tensor(fed, device="cuda"))}
