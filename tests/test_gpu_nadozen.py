"""GPU: Nadozen models through the framework's decoder against the plain oracle - mechanism by mechanism, layer by layer, whole
prompts, portions, token by token, states used again, window edges, sinks, long contexts, generation - and the attention kernel's
sinks and gates by themselves."""
import ctypes as C

import numpy as np
import pytest

from folder_helpers import errors, portions
from nadozen_models import MODELS, model, parallel, random_model, variant, wkv
from oracle import nadozen_oracle as N
from prometorch_amd import _lib, model as registry, ops
from prometorch_amd.testing import folder_writer as fw

pytestmark = pytest.mark.gpu
# rms error of a position's logits over their deviation: (worst, 97th percentile, mean)
LIMITS = {"float32": (2e-4, 5e-5, 2e-5), "bfloat16": (0.2, 0.06, 0.02)}


def assert_close(got, want, precision, what=""):
    e = errors(got, want)
    worst, most, mean = LIMITS[precision]
    assert e.max() < worst and np.quantile(e, 0.97) < most and e.mean() < mean, (what, e.max(), np.quantile(e, 0.97), e.mean(), int(e.argmax()))


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    """name -> (folder, cfg, weights, tokens, oracle logits at every position), made once."""
    cache = {}

    def get(name, n=150, seed=13):
        if name not in cache:
            cfg = MODELS[name]
            w = fw.random_weights(cfg, seed)
            path = fw.write_model_folder(str(tmp_path_factory.mktemp(name)), cfg, w)
            tokens = np.random.default_rng(seed).integers(0, cfg["vocab"], n).tolist()
            cache[name] = (path, cfg, w, tokens, N.logits(tokens, w, cfg))
        return cache[name]
    return get


# ---- models -----------------------------------------------------------------------------------------
@pytest.mark.parametrize("precision", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", sorted(MODELS))
def test_prompt_portions_and_decode(dev, built, name, precision):
    path, cfg, w, tokens, want = built(name)
    m = registry.load(path, max_seq=160, precision=precision)
    assert m.layer_runs == len(cfg["layers"]) and m.cfg["vocab"] == cfg["vocab"]
    for sizes in ([len(tokens)], [2], [1], [7, 1, 1, 3, 2, 64, 5, 1, 31], [64], [66, 1], [1, 149]):
        assert_close(portions(m, tokens, sizes), want, precision, (name, sizes))
    m.close()


@pytest.mark.parametrize("seed", range(24))
def test_random_designs(dev, tmp_path, seed):
    cfg = random_model(seed)
    w = fw.random_weights(cfg, seed + 200)
    tokens = np.random.default_rng(seed).integers(0, cfg["vocab"], 170).tolist()
    want = N.logits(tokens, w, cfg)
    path = fw.write_model_folder(str(tmp_path / "m"), cfg, w)
    for precision in ("float32", "bfloat16"):
        m = registry.load(path, max_seq=171, precision=precision)
        for sizes in ([170], [97, 2, 1, 1, 1, 33, 1], [1]):
            assert_close(portions(m, tokens, sizes), want, precision, (seed, precision, sizes))
        m.close()


@pytest.mark.parametrize("name", sorted(MODELS))
def test_layers_one_by_one(dev, built, name):
    """Sum of the streams after every layer, prompt pass and decode step, in 32-bit."""
    path, cfg, w, tokens, _ = built(name)
    tokens = tokens[:40]
    want = N.residuals(tokens, w, cfg)
    m = registry.load(path, max_seq=64, precision="float32")
    scale = want.std(axis=(1, 2), keepdims=True)
    assert (np.abs(m.prefill_trace(tokens) - want) / scale).max() < 2e-4
    m.set_past_len(0)
    for i, t in enumerate(tokens):
        _, trace = m.step_trace(t)
        assert (np.abs(trace[:, 1] - want[:, i]) / scale[:, 0]).max() < 2e-4, i
    m.close()


# ---- mechanisms by themselves ---------------------------------------------------------------------------
def silent(*names):
    """Weights of the named matrices set to zero: what they carry is out of the model."""
    def change(w):
        for n in names:
            w[n] = np.zeros_like(w[n])
    return change


def loud_keys(w):
    """No decay to speak of, so that the first token still shows hundreds of tokens later."""
    w["l0.mix.w0"] = np.full_like(w["l0.mix.w0"], -9.0)
    w["l0.mix.w2"] = np.zeros_like(w["l0.mix.w2"])


def long_memory(w):
    w["l0.mix.right.dt_bias"] = np.full_like(w["l0.mix.right.dt_bias"], -4.0)
    w["l0.mix.right.A_log"] = np.full_like(w["l0.mix.right.A_log"], -4.0)


ONE_LAYER = parallel(4, 2, 24, 20, (4, 12, 20, 2, 4, 2))
MECHANISMS = {
    # embedding, sinusoid, final norm and head: the only layer writes nothing
    "embedding": ([wkv(2, 8, 4)], 1, silent("l0.mix.o")),
    # blends of the streams without any branch
    "streams": ([wkv(2, 8, 4), wkv(2, 8, 4)], 3, silent("l0.mix.o", "l1.mix.o")),
    "feed_forward": ([wkv(2, 8, 4, ff=43)], 1, silent("l0.mix.o")),
    "wkv": ([wkv(3, 24, 10)], 1, None),
    "wkv_undecayed": ([wkv(3, 24, 10)], 2, loud_keys),
    # no key, no value from the state: only the current token's bonus
    "wkv_bonus": ([wkv(3, 24, 10)], 1, lambda w: w.update({"l0.mix.w0": np.full_like(w["l0.mix.w0"], 6.0)})),
    "attention": ([ONE_LAYER], 1, silent("l0.mix.right.o")),
    "attention_one_gate": ([ONE_LAYER], 1, silent("l0.mix.right.o", "l0.mix.left.g")),
    "state_space": ([ONE_LAYER], 1, silent("l0.mix.left.o")),
    "state_space_long": ([ONE_LAYER], 1, lambda w: (silent("l0.mix.left.o")(w), long_memory(w))),
    # state without decay per step and without the skip
    "state_space_no_skip": ([ONE_LAYER], 1, silent("l0.mix.left.o", "l0.mix.right.D")),
    "shared": ([ONE_LAYER, 0, 0], 2, None),
}


@pytest.mark.parametrize("name", sorted(MECHANISMS))
def test_mechanism(dev, tmp_path, name):
    layers, streams, change = MECHANISMS[name]
    cfg = model(layers, 50, 70, streams)
    w = fw.random_weights(cfg, 31)
    if change:
        change(w)
        w = {k: fw.from_bf16(fw.to_bf16(v)) for k, v in w.items()}
    tokens = np.random.default_rng(3).integers(0, 70, 260).tolist()
    want = N.logits(tokens, w, cfg)
    path = fw.write_model_folder(str(tmp_path / "m"), cfg, w)
    for precision in ("float32", "bfloat16"):
        m = registry.load(path, max_seq=261, precision=precision)
        for sizes in ([260], [130, 1], [1], [17, 2, 3]):
            assert_close(portions(m, tokens, sizes), want, precision, (name, precision, sizes))
        m.close()


def standing_key(window, width=64):
    """One attention layer in which token 1 looks for token 0 and nothing else stands out: the queries read the input with its
    halves swapped, and token 1 is token 0 with its halves swapped."""
    cfg = model([parallel(2, 1, 32, window, (1, 8, 4, 1, 2, 1), sharp=2.0)], width, 40, 1)
    w = fw.random_weights(cfg, 5)
    w["embed"] = fw.from_bf16(fw.to_bf16(w["embed"] * 8.0))
    w["embed"][1] = np.roll(w["embed"][0], width // 2)
    w["l0.norm1"], w["l0.norm1.b"] = np.ones(width, np.float32), np.zeros(width, np.float32)
    k = np.roll(w["l0.mix.left.k"], width // 2, axis=1)
    w["l0.mix.left.q"] = np.concatenate([k, k])
    w["l0.mix.left.q.norm"] = w["l0.mix.left.k.norm"] = np.ones(32, np.float32)
    w["l0.mix.left.o"] = w["l0.mix.left.o"] * 32.0
    return cfg, w


@pytest.mark.parametrize("window", [3, 64, 65, 100, 128])
def test_keys_at_the_window_edge(dev, tmp_path, window):
    """A key that takes most of the softmax, the window's last position or one further back, at several places relative to
    tiles and portions, in prompts and decoded."""
    cfg, w = standing_key(window)
    path = fw.write_model_folder(str(tmp_path / "m"), cfg, w)
    rng = np.random.default_rng(window)
    for precision in ("float32", "bfloat16"):
        m = registry.load(path, max_seq=400, precision=precision)
        for at in (0, 1, 62, 63, 64, 129):
            tokens = rng.integers(2, 40, at + window + 6)
            tokens[at] = 0
            tokens[at + window - 1:at + window + 1] = 1  # the first still sees token 0, the second does not
            tokens = tokens.tolist()
            want = N.logits(tokens, w, cfg)
            near = [N.logits(tokens, w, variant(cfg, 0, d)) for d in (1, -1)]
            inside, outside = at + window - 1, at + window
            assert errors(near[1], want)[inside] > 0.4 and errors(near[0], want)[outside] > 0.4
            for sizes in ([len(tokens)], [at + window - 1, 1], [at + window, 2], [5]):
                assert_close(portions(m, tokens, sizes)[-9:], want[-9:], precision, (window, at, sizes))
        m.close()


@pytest.mark.parametrize("precision", ["float32", "bfloat16"])
def test_window_neighbours(dev, built, precision):
    path, cfg, w, tokens, want = built("odd")
    m = registry.load(path, max_seq=160, precision=precision)
    for sizes in ([150], [1], [9]):
        got = portions(m, tokens, sizes)
        mine = errors(got, want)[50:].mean()
        for delta in (1, -1):
            other = errors(got, N.logits(tokens, w, variant(cfg, 1, delta)))[50:].mean()
            assert other > (1000 if precision == "float32" else 5) * mine, (delta, other, mine)
    m.close()


@pytest.mark.parametrize("sink", [-30.0, 4.0, 30.0])
def test_sinks(dev, tmp_path, sink):
    """From no weight at all to nearly all of it; also where the window holds the first token only."""
    cfg = model([parallel(3, 1, 16, 5, (2, 4, 3, 1, 2, 1))], 30, 31, 1)
    w = fw.random_weights(cfg, 8)
    w["l0.mix.left.sink"] = np.array([sink, 0.0, -sink], np.float32)
    w["l0.mix.left.o"] = fw.from_bf16(fw.to_bf16(w["l0.mix.left.o"] * 4.0))
    tokens = np.random.default_rng(1).integers(0, 31, 40).tolist()
    want = N.logits(tokens, w, cfg)
    path = fw.write_model_folder(str(tmp_path / "m"), cfg, w)
    for precision in ("float32", "bfloat16"):
        m = registry.load(path, max_seq=41, precision=precision)
        for sizes in ([40], [1]):
            assert_close(portions(m, tokens, sizes), want, precision, sizes)
        m.close()


# ---- state over time ----------------------------------------------------------------------------------
@pytest.mark.parametrize("precision", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["odd", "whole"])
def test_state_is_used_again(dev, built, precision, name):
    """A second request over the first one's caches and states, shorter and longer, gives what a fresh model gives."""
    path, cfg, w, tokens, want = built(name)
    m = registry.load(path, max_seq=160, precision=precision)
    portions(m, tokens[::-1], [150])
    a = portions(m, tokens[:30], [12, 1, 1, 16])
    portions(m, tokens[::-1], [70, 1])
    b = portions(m, tokens, [100, 1])
    c = portions(m, tokens, [1, 2, 1])
    m.close()
    fresh = registry.load(path, max_seq=160, precision=precision)
    assert np.array_equal(a, portions(fresh, tokens[:30], [12, 1, 1, 16]))
    assert np.array_equal(b, portions(fresh, tokens, [100, 1]))
    assert np.array_equal(c, portions(fresh, tokens, [1, 2, 1]))
    assert_close(b, want, precision)
    fresh.close()


def test_state_does_not_go_back(dev, built):
    """Recurrent state starts over or goes on; a place in between is refused and leaves everything as it is."""
    path, cfg, w, tokens, want = built("odd")
    m = registry.load(path, max_seq=160, precision="float32")
    m.prefill(tokens[:20])
    for place in (19, 1, 21):
        with pytest.raises(_lib.PtmError):
            m.set_past_len(place)
    m.set_past_len(20)
    m.step(tokens[20])
    assert errors(m.logits()[None], want[20:21])[0] < LIMITS["float32"][0]
    m.close()


@pytest.mark.parametrize("precision", ["float32", "bfloat16"])
def test_eager_steps_equal_graph_steps(dev, built, precision):
    path, cfg, w, tokens, _ = built("odd")
    a = registry.load(path, max_seq=160, precision=precision, use_graph=True)
    b = registry.load(path, max_seq=160, precision=precision, use_graph=False)
    ya, yb = portions(a, tokens[:60], [20, 1]), portions(b, tokens[:60], [20, 1])
    assert np.array_equal(ya, yb)
    assert a.L.ptm_decode_graph_state(a.h, 0) == 1 and b.L.ptm_decode_graph_state(b.h, 0) == 0
    a.close()
    b.close()


def test_long_prompts_and_decoding(dev, tmp_path):
    """Prompts of several chunks and hundreds of decoded tokens, with states that forget slowly."""
    cfg = model([wkv(2, 12, 4), parallel(2, 1, 12, 300, (2, 8, 6, 1, 4, 1)), 0], 24, 40, 2)
    w = fw.random_weights(cfg, 17)
    loud_keys(w)
    w = {k: fw.from_bf16(fw.to_bf16(v)) for k, v in w.items()}
    tokens = np.random.default_rng(5).integers(0, 40, 2900).tolist()
    want = N.logits(tokens, w, cfg)
    path = fw.write_model_folder(str(tmp_path / "m"), cfg, w)
    for precision in ("float32", "bfloat16"):
        m = registry.load(path, max_seq=2900, precision=precision)
        got = [m.prefill_logits(tokens[:2300], range(2200, 2300))]
        for t in tokens[2300:]:
            m.step(t)
            got.append(m.logits()[None])
        assert_close(np.concatenate(got), want[2200:], precision)
        m.set_past_len(0)
        assert_close(m.prefill_logits(tokens, range(2880, 2900), chunk_rows=700), want[2880:], precision)
        m.close()


# ---- generation ---------------------------------------------------------------------------------------
@pytest.mark.parametrize("precision", ["float32", "bfloat16"])
def test_greedy_generation(dev, built, precision):
    """Greedy tokens through prefill + greedy and through generate(); every token is the oracle's best on that very text, or within
    rounding of it.  A stop token inside a run leaves the state where the text ends."""
    path, cfg, w, tokens, _ = built("odd")
    prompt, n = tokens[:23], 60
    m = registry.load(path, max_seq=160, precision=precision)
    first = m.prefill(prompt)
    out = [first] + m.greedy(first, n - 1)
    m.set_past_len(0)
    kw = dict(temperature=0.0, top_k=1, top_p=1.0)
    assert m.generate(prompt, [0.5] * n, **kw) == out
    lg = N.logits(prompt + out, w, cfg)
    lg, after = lg[len(prompt) - 1:-1], lg[len(prompt):]
    gap = (lg.max(axis=1) - lg[np.arange(n), out]) / lg.std()
    assert gap.max() < LIMITS[precision][0], gap.max()
    if precision == "float32":
        assert gap.max() == 0.0
    for stop in sorted(set(out), key=out.index)[1::4]:
        cut = out.index(stop)
        m.set_past_len(0)
        assert m.generate(prompt, [0.5] * n, stop_ids=[stop], **kw) == out[:cut]
        m.step(stop)  # the text goes on behind the stop token
        assert errors(m.logits()[None], after[cut:cut + 1])[0] < LIMITS[precision][0], cut
    m.close()


def test_command_line(dev, built, capsys):
    """Token ids in, the same greedy ids out as through the Python interface."""
    from prometorch_amd.__main__ import main
    path, cfg, w, tokens, _ = built("whole")
    m = registry.load(path, max_seq=64)
    want = m.generate(tokens[:9], [0.0] * 12, temperature=0.0, top_k=1, top_p=1.0)
    m.close()
    args = ["generate", "--model", path, "--tokens", ",".join(map(str, tokens[:9])), "--max-new", "12", "--temperature", "0"]
    assert main(args) == 0
    assert capsys.readouterr().out.split() == [str(t) for t in want]


def test_sampled_generation(dev, built):
    """The same draws give the same tokens again, picked from the logits a stepped run reads back."""
    path, cfg, w, tokens, _ = built("odd")
    m = registry.load(path, max_seq=160, precision="bfloat16")
    u = ops.mt19937_uniforms(7, 0, 30)
    kw = dict(temperature=0.8, top_k=12, top_p=0.9)
    a = m.generate(tokens[:10], u, **kw)
    m.set_past_len(0)
    assert m.generate(tokens[:10], u, **kw) == a and len(set(a)) > 3
    m.set_past_len(0)
    m.prefill(tokens[:9])
    t = tokens[9]
    for i in range(30):
        m.step(t)
        lg = m.logits().astype(np.float64) / kw["temperature"]
        top = np.argsort(-lg, kind="stable")[:12]
        p = np.exp(lg[top] - lg[top].max())
        p /= p.sum()
        assert a[i] in top[:int((np.cumsum(p) < 0.9).sum()) + 1], i
        t = a[i]
    m.close()


def test_folder_errors_on_load(dev, built, tmp_path):
    path, cfg, w, _, _ = built("odd")
    for name in ("l0.mix.mu.w", "l1.mix.left.sink", "l1.mix.right.conv.b", "l1.hc2.mix", "l3.norm1.b", "final.norm.b", "l0.mix.w1"):
        with pytest.raises(_lib.PtmError) as e:
            registry.load(fw.write_model_folder(str(tmp_path / "missing"), cfg, {k: v for k, v in w.items() if k != name}), max_seq=16)
        assert e.value.code == -10, name
    for name in ("l0.mix.w2", "l1.mix.right.in", "l0.mix.u", "l1.hc1.in"):
        with pytest.raises(_lib.PtmError) as e:
            registry.load(fw.write_model_folder(str(tmp_path / "shape"), cfg, dict(w, **{name: w[name][:-1]})), max_seq=16)
        assert e.value.code == -2, name
    m = registry.load(path, max_seq=16)
    with pytest.raises(_lib.PtmError):
        m.prefill([0] * 17)          # past the cache
    m.close()


# ---- attention kernel: sinks, output gate, scale ------------------------------------------------------------
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("case", [(5, 4, 2, 16, 0, 0), (70, 3, 1, 64, 20, 130), (130, 2, 2, 120, 64, 5), (33, 6, 3, 200, 7, 64), (9, 2, 1, 272, 4, 3)])
def test_attention_rows_sink_and_gate(dev, case, fp32):
    """rows, heads, kv heads, size, window, position of row 0; three values per head are outside the gate's columns."""
    import torch
    rows, H, G, d, window, pos0 = case
    rng = np.random.default_rng(sum(case))
    n = pos0 + rows
    rnd = (lambda *s: rng.standard_normal(s, np.float32)) if fp32 else (lambda *s: fw.from_bf16(fw.to_bf16(rng.standard_normal(s, np.float32))))
    q, k, v = rnd(rows, H, d), rnd(n, G, d), rnd(n, G, d)
    gate = rng.standard_normal((rows, H, d - 3), np.float32)
    sink = rng.standard_normal(H).astype(np.float32) * 2 + 1
    scale, see = 2.0 / np.sqrt(d), N.visible(n, {"size": window} if window else None)[pos0:]
    want = np.zeros((rows, H, d))
    for h in range(H):
        g = h // (H // G)
        s = np.where(see, q[:, h].astype(np.float64) @ k[:, g].T.astype(np.float64) * scale, -np.inf)
        want[:, h] = N.sink_softmax(s, float(sink[h])) @ v[:, g] * 0.7
        want[:, h, :d - 3] *= N.sigmoid(gate[:, h].astype(np.float64))
    put = lambda a: torch.from_numpy(a if fp32 else fw.to_bf16(a).view(np.int16)).cuda()
    Q, K, V = put(q), put(k), put(v)
    O = torch.zeros((rows, H, d), dtype=torch.float32 if fp32 else torch.bfloat16, device="cuda")
    S, Gt = torch.from_numpy(sink).cuda(), torch.from_numpy(gate).cuda()
    a = _lib.AttentionArgs(Q=Q.data_ptr(), K1=K.data_ptr(), V=V.data_ptr(), O=O.data_ptr(), q_row=H * d, k1_row=G * d, k1_head=d,
                           v_row=G * d, v_head=d, o_row=H * d, rows=rows, heads=H, kv_heads=G, dim1=d, vdim=d, window=window, pos0=pos0,
                           scale=scale, fp32=int(fp32), sink=S.data_ptr(), gate=Gt.data_ptr(), gate_row=H * (d - 3), gate_head=d - 3,
                           out_scale=0.7)
    _lib.check(_lib.load().ptm_attention_rows(C.byref(a), None), "attention_rows")
    torch.cuda.synchronize()
    err = np.abs(O.float().cpu().numpy() - want)
    assert err.max() < (2e-5 if fp32 else 2.5e-2), err.max()


# workgroups of one round of the chip, of two with long row blocks beside short ones (257 .. 512), of more; heads off 8 and off the size classes; a scale
# that is negative or zero, capped scores, scores that move the softmax's reference by more and by less than 2^8, gates off 16 bytes
@pytest.mark.parametrize("rows,heads,kv_heads,dim,scale,cap,loud,shift", [
    (130, 4, 2, 64, -1.0, 0.0, 1, 0), (40, 2, 1, 40, 0.0, 0.0, 1, 0), (40, 2, 2, 128, 0.0, 5.0, 1, 1), (150, 3, 1, 104, 1.0, 9.0, 1, 2), (150, 3, 1, 104, -1.0, 9.0, 4, 0),
    (257, 2, 1, 128, 1.0, 0.0, 8, 0), (257, 2, 1, 200, 1.0, 0.0, 24, 1), (255, 64, 4, 16, 1.0, 0.0, 3, 0), (257, 128, 4, 32, 1.0, 0.0, 3, 1), (512, 128, 4, 16, 1.0, 20.0, 3, 0),
    (516, 128, 4, 16, -1.0, 0.0, 1, 3)])
def test_prompt_attention_forms(dev, rows, heads, kv_heads, dim, scale, cap, loud, shift):
    """Against 64 bits.  Values and gates are at most some 5 * 0.7; what is stored is off by 2^-9 of that, the weights by 2^-16."""
    import torch
    pos0, window = 11, 200
    rng = np.random.default_rng(rows + heads + dim)
    n = pos0 + rows
    rnd = lambda *s: fw.from_bf16(fw.to_bf16(rng.standard_normal(s, np.float32)))
    q, k, v = rnd(rows, heads, dim), rnd(n, kv_heads, dim), rnd(n, kv_heads, dim)
    k = fw.from_bf16(fw.to_bf16(k * np.where(np.arange(n) % 64 == 37, loud, 1).astype(np.float32)[:, None, None]))
    gate = rng.standard_normal(rows * heads * (dim - shift) + 4).astype(np.float32)
    sink = rng.standard_normal(heads).astype(np.float32)
    scale, see = scale * 2.0 / np.sqrt(dim), N.visible(n, {"size": window})[pos0:]
    want = np.zeros((rows, heads, dim))
    for h in range(heads):
        g = h // (heads // kv_heads)
        s = q[:, h].astype(np.float64) @ k[:, g].T.astype(np.float64) * scale
        s = np.where(see, cap * np.tanh(s / cap) if cap else s, -np.inf)
        want[:, h] = N.sink_softmax(s, float(sink[h])) @ v[:, g] * 0.7
    gates = gate[shift:shift + rows * heads * (dim - shift)].reshape(rows, heads, dim - shift)
    want[:, :, :dim - shift] *= N.sigmoid(gates.astype(np.float64))
    put = lambda a: torch.from_numpy(fw.to_bf16(a).view(np.int16)).cuda()
    Q, K, V = put(q), put(k), put(v)
    O = torch.zeros((rows, heads, dim), dtype=torch.bfloat16, device="cuda")
    S, Gt = torch.from_numpy(sink).cuda(), torch.from_numpy(gate).cuda()
    a = _lib.AttentionArgs(Q=Q.data_ptr(), K1=K.data_ptr(), V=V.data_ptr(), O=O.data_ptr(), q_row=heads * dim, k1_row=kv_heads * dim, k1_head=dim, v_row=kv_heads * dim,
                           v_head=dim, o_row=heads * dim, rows=rows, heads=heads, kv_heads=kv_heads, dim1=dim, vdim=dim, window=window, pos0=pos0, scale=scale, softcap=cap,
                           fp32=0, sink=S.data_ptr(), gate=Gt.data_ptr() + 4 * shift, gate_row=heads * (dim - shift), gate_head=dim - shift, out_scale=0.7)
    _lib.check(_lib.load().ptm_attention_rows(C.byref(a), None), "attention_rows")
    torch.cuda.synchronize()
    err = np.abs(O.float().cpu().numpy() - want)
    assert err.max() < 1e-2, err.max()


@pytest.mark.parametrize("dim,vdim,cap", [(64, 64, 0.0), (128, 64, 0.0), (128, 128, 0.0), (192, 128, 0.0), (256, 256, 0.0), (128, 128, 50.0)])
@pytest.mark.parametrize("part", ["weights", "gate"])
def test_prompt_attention_rounds_like_64_bits(dev, dim, vdim, cap, part):
    """The share of values that are not the nearest bfloat16 number to the 64-bit result.  Borders are 2^-7 of the power of two below apart and a value is up to
    twice that power: relative errors of e take 256 e of the values past one.
    weights: a score of 2^7 to 2^8 times the weight of the first comes in a later tile.  Its own weight is 1, which has no rounding; what the first weighs,
    2^-7, is rounded at 2^-17, and five operations at 2^-24: e < 4e-7, 1e-4 of the values.  Measured against another score than the largest it is itself off by
    up to 2^-17, and 2e-4 to 3e-4 differed.
    gate: one visible key, so that the gate is all that is computed: 1 / (1 + e^-z) in 32 bits, z down to -80, and two products: e < 4e-7 again.  With z
    times log2(e) rounded in front of the exponential, 3e-6 at z = -80, 1.35e-4 to 1.9e-4 differed."""
    import torch
    rows, heads, pos0 = 260, 4, 200
    rng = np.random.default_rng(dim + vdim)
    n = pos0 + rows
    rnd = lambda *s: fw.from_bf16(fw.to_bf16(rng.standard_normal(s, np.float32)))
    gates = np.zeros((rows, heads, vdim), np.float32)
    if part == "weights":
        q, k = np.zeros((rows, heads, dim), np.float32), np.zeros((n, 1, dim), np.float32)
        q[..., 0], q[..., 1] = 1, fw.from_bf16(fw.to_bf16(rng.random((rows, heads), np.float32)))
        k[:, 0, 0] = -120
        k[0, 0, 0], k[150, 0, :2] = 0, (5, 0.4375)
    else:
        q, k = rnd(rows, heads, dim), rnd(n, 1, dim)
        gates = (-80 * rng.random((rows, heads, vdim))).astype(np.float32)
    v = rnd(n, 1, vdim)
    see = N.visible(n, {"size": 1} if part == "gate" else None)[pos0:]
    s = np.einsum("rhd,nd->hrn", q.astype(np.float64), k[:, 0].astype(np.float64))
    s = np.where(see, cap * np.tanh(s / cap) if cap else s, -np.inf)
    p = np.exp(s - s.max(2, keepdims=True))
    want = np.einsum("hrn,nv->rhv", p / p.sum(2, keepdims=True), v[:, 0].astype(np.float64)) / (1 + np.exp(-gates.astype(np.float64)) if part == "gate" else 1)
    put = lambda a: torch.from_numpy(fw.to_bf16(a).view(np.int16)).cuda()
    Q, K, V, G = put(q), put(k), put(v), torch.from_numpy(gates).cuda()
    O = torch.zeros((rows, heads, vdim), dtype=torch.bfloat16, device="cuda")
    a = _lib.AttentionArgs(Q=Q.data_ptr(), K1=K.data_ptr(), V=V.data_ptr(), O=O.data_ptr(), q_row=heads * dim, k1_row=dim, k1_head=dim, v_row=vdim, v_head=vdim,
                           o_row=heads * vdim, rows=rows, heads=heads, kv_heads=1, dim1=dim, vdim=vdim, window=1 if part == "gate" else 0, pos0=pos0, scale=1.0, softcap=cap,
                           fp32=0, gate=G.data_ptr() if part == "gate" else None, gate_row=heads * vdim, gate_head=vdim if part == "gate" else 0)
    _lib.check(_lib.load().ptm_attention_rows(C.byref(a), None), "attention_rows")
    torch.cuda.synchronize()
    differ = (O.cpu() != torch.from_numpy(want).to(torch.bfloat16)).double().mean().item()
    print("differ: %.2e" % differ, flush=True)
    assert differ <= 1e-4


# ---- products with the gated epilogue are reached through the models; shapes around their tile edges -------------
@pytest.mark.parametrize("ff", [1, 15, 16, 17, 64, 100, 257])
def test_feed_forward_sizes(dev, tmp_path, ff):
    cfg = model([wkv(1, 8, 3, ff=ff)], 40, 33, 1)
    w = fw.random_weights(cfg, ff)
    silent("l0.mix.o")(w)
    w["l0.mlp.down"] = fw.from_bf16(fw.to_bf16(w["l0.mlp.down"] * 3.0))
    tokens = np.random.default_rng(ff).integers(0, 33, 140).tolist()
    want = N.logits(tokens, w, cfg)
    path = fw.write_model_folder(str(tmp_path / "m"), cfg, w)
    for precision in ("float32", "bfloat16"):
        m = registry.load(path, max_seq=141, precision=precision)
        for sizes in ([140], [50, 20, 1]):
            assert_close(portions(m, tokens, sizes), want, precision, (ff, sizes))
        m.close()


@pytest.mark.parametrize("width,ff", [(3600, 20), (4096, 4100), (1800, 4200)])
def test_decoding_at_large_widths(dev, tmp_path, width, ff):
    """Decode products whose waves have whole rings of 8 chunks behind the streams' sums: one row a wave, two, and a ragged last one."""
    cfg = model([wkv(2, 8, 4, ff=ff), parallel(2, 1, 16, 9, (2, 4, 7, 1, 2, 2), ff=ff)], width, 33, 2)
    w = fw.random_weights(cfg, width + ff)
    tokens = np.random.default_rng(ff).integers(0, 33, 6).tolist()
    want = N.logits(tokens, w, cfg)
    path = fw.write_model_folder(str(tmp_path / "m"), cfg, w)
    for precision in ("float32", "bfloat16"):
        m = registry.load(path, max_seq=8, precision=precision)
        assert_close(portions(m, tokens, [1]), want, precision, (width, ff))
        m.close()


# ---- the scan over 16 tokens at a time ------------------------------------------------------------------
def ssm_reference(w, proj, m, pos0, ring, S):
    """Token by token in 64 bits: (y * silu(z) before the norm's row kernel, normed), state."""
    import torch
    H, V, n, G, taps = m
    inner, ch = H * V, H * V + 2 * G * n
    conv, cb, dtb, neg_a, D, norm = [t.double() for t in w]
    p = proj.double()
    past = [ring[(pos0 - taps + 1 + j) % taps].double() if pos0 - taps + 1 + j >= 0 else torch.zeros(ch, device="cuda", dtype=torch.float64) for j in range(taps - 1)]
    x = torch.cat([torch.stack(past)] * (taps > 1) + [p[:, inner:inner + ch]])
    c = torch.nn.functional.silu(sum(x[j:j + len(p)] * conv[:, j] for j in range(taps)) + cb)
    dt = torch.nn.functional.softplus(p[:, inner + ch:] + dtb)
    out = []
    for t in range(len(p)):
        xt, B, C = c[t, :inner].reshape(H, V), *(c[t, inner + i * G * n:inner + (i + 1) * G * n].reshape(G, n).repeat_interleave(H // G, 0) for i in (0, 1))
        S = torch.exp(neg_a * dt[t])[:, None, None] * S + dt[t][:, None, None] * xt[:, :, None] * B[:, None, :]
        y = (S * C[:, None, :]).sum(2) + D[:, None] * xt
        y = y.reshape(-1) * torch.nn.functional.silu(p[t, :inner])
        out.append(y / (y.pow(2).mean() + 1e-6).sqrt() * norm)
    return torch.stack(out), S


# every number of key tiles a wave has, states and columns off the tiles, groups, more rows than tiles in flight, tokens off 16, many heads of one group and of
# two (two heads a wave, the last by itself)
@pytest.mark.parametrize("heads,vdim,state,groups,taps,rows", [(2, 16, 64, 1, 4, 16), (3, 5, 20, 1, 2, 15), (4, 64, 128, 1, 4, 97), (4, 33, 100, 2, 3, 130), (2, 17, 200, 1, 4, 49),
                                                               (2, 16, 256, 2, 4, 17), (2, 20, 300, 1, 4, 70), (1, 64, 512, 1, 6, 33), (18, 8, 16, 2, 4, 1),
                                                               (40, 9, 9, 40, 4, 33), (6, 1, 1, 6, 4, 40),
                                                               (65, 4, 8, 1, 4, 1030), (66, 3, 70, 2, 2, 1030)])
@pytest.mark.parametrize("pos0", [0, 21])
def test_state_space_scan(dev, heads, vdim, state, groups, taps, rows, pos0):
    """One call against the recurrence in 64 bits.  A sum of up to 512 products, 16 decays deep, is off by some 1e-6 of its terms; a first value that is
    infinite reaches no token before its own."""
    import torch
    from gemm_helpers import harness
    h = harness()
    for f in ("ssm_scratch", "ssm_state_floats"):
        getattr(h, f).restype = C.c_int64
    g = torch.Generator(device="cuda").manual_seed(rows + state)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)
    inner, ch = heads * vdim, heads * vdim + 2 * groups * state
    w = [rand(ch, taps) * taps ** -0.5, 0.1 * rand(ch), rand(heads) - 2, -torch.exp(0.8 * rand(heads)), rand(heads), 1 + 0.1 * rand(inner)]
    proj, ring = rand(rows, inner + ch + heads), rand(taps, ch)
    kp = h.ssm_state_floats(1, state, 1)
    S0 = torch.zeros(heads, vdim, kp, device="cuda")
    S0[:, :, :state] = rand(heads, vdim, state)

    def run(proj):
        S, r, out = S0.clone(), ring.clone(), torch.empty(rows, inner, device="cuda")
        scratch = [torch.full((h.ssm_scratch(heads, vdim, state, groups, rows, i),), float("nan"), device="cuda") for i in range(4)]
        ptrs = lambda ts: (C.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
        assert h.ssm_run((C.c_int * 5)(heads, vdim, state, groups, taps), ptrs(w), C.c_void_p(proj.data_ptr()), rows, C.c_int64(pos0), C.c_void_p(r.data_ptr()),
                         C.c_void_p(S.data_ptr()), ptrs(scratch), C.c_void_p(out.data_ptr()), None) == 0
        torch.cuda.synchronize()
        return out, S, r

    out, S, r = run(proj)
    want, want_S = ssm_reference(w, proj, (heads, vdim, state, groups, taps), pos0, ring, (S0[:, :, :state] if pos0 else 0 * S0[:, :, :state]).double())
    for a, b in ((out, want), (S[:, :, :state], want_S)):
        assert float((a.double() - b).abs().max() / b.pow(2).mean().sqrt()) < 3e-5
    assert (S[:, :, state:] == 0).all()
    for j in range(min(taps, rows)):
        assert torch.equal(r[(pos0 + rows - 1 - j) % taps], proj[rows - 1 - j, inner:inner + ch])
    if rows > 9:
        loud = proj.clone()
        loud[9, inner] = float("inf")
        assert torch.equal(run(loud)[0][:9], out[:9])
    # a last token's x and B that are infinite leave the states that they enter infinite, and all others alone
    for at, where in ((0, (0, 0)), (inner, (slice(heads // groups), slice(None), 0))):
        loud, mask = proj.clone(), torch.zeros(heads, vdim, state, dtype=torch.bool, device="cuda")
        loud[-1, inner + at], mask[where] = float("inf") * float(w[0][at, -1].sign()), True
        got = run(loud)[1][:, :, :state]
        assert torch.equal(got.isinf(), mask) and not got.isnan().any(), at


# every number of key tiles a wave has, dims off 4 and off the tiles, tokens off 16, one head and many; decays next to 1, next to 0 and 0
@pytest.mark.parametrize("heads,dim,rows", [(2, 64, 16), (3, 5, 15), (1, 1, 2), (4, 62, 97), (3, 100, 130), (40, 64, 33), (2, 200, 49), (1, 300, 70), (1, 512, 17), (2, 128, 1)])
@pytest.mark.parametrize("pos0", [0, 21])
def test_wkv_scan(dev, heads, dim, rows, pos0):
    """One call against the recurrence in 64 bits.  A sum of up to 512 products, 16 decays deep, is off by some 1e-6 of its terms; a value that is
    infinite reaches no token before its own."""
    import torch
    from gemm_helpers import harness
    h = harness()
    for f in ("wkv_scratch", "ssm_state_floats"):
        getattr(h, f).restype = C.c_int64
    gen = torch.Generator(device="cuda").manual_seed(rows + dim)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    proj = rand(rows, 5, heads, dim)
    proj[:, 4] = torch.exp(-torch.exp(3 * rand(rows, heads, dim)))
    proj[rows // 2, 4, 0] = 0.0
    u, norm, last = rand(heads, dim), 1 + 0.1 * rand(heads, dim), rand(64)
    kp = h.ssm_state_floats(1, dim, 1)
    S0 = torch.zeros(heads, dim, kp, device="cuda")
    S0[:, :, :dim] = rand(heads, dim, dim)

    def run(proj):
        S, out, shift = S0.clone(), torch.empty(rows, heads, dim, device="cuda"), torch.zeros(2, 64, device="cuda")
        scratch = [torch.full((h.wkv_scratch(heads, dim, rows, i),), float("nan"), device="cuda") for i in range(2)]
        p = lambda t: C.c_void_p(t.data_ptr())
        assert h.wkv_run(heads, dim, p(proj), p(u), p(norm), rows, C.c_int64(pos0), p(S), (C.c_void_p * 2)(*[t.data_ptr() for t in scratch]), p(last), p(shift), p(out), None) == 0
        torch.cuda.synchronize()
        return out, S, shift

    out, S, shift = run(proj)
    r, k, v, g, w = proj.double().unbind(1)
    want, want_S = [], (S0[:, :, :dim] if pos0 else 0 * S0[:, :, :dim]).double()  # [head][column][key]
    for t in range(rows):
        kv = v[t, :, :, None] * k[t, :, None, :]
        o = ((want_S + u.double()[:, None, :] * kv) * r[t, :, None, :]).sum(2)
        want_S = w[t, :, None, :] * want_S + kv
        want.append(o / (o.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * norm.double() * torch.nn.functional.silu(g[t]))
    for a, b in ((out, torch.stack(want)), (S[:, :, :dim], want_S)):
        assert float((a.double() - b).abs().max() / b.pow(2).mean().sqrt()) < 3e-5
    assert (S[:, :, dim:] == 0).all() and torch.equal(shift[(pos0 + rows - 1) % 2], last)
    if rows > 9:
        for part in (0, 1, 2):
            loud = proj.clone()
            loud[9, part, 0, 0] = float("inf")
            assert torch.equal(run(loud)[0][:9], out[:9])
    for part, where in ((2, (0, 0)), (1, (0, slice(None), 0))):  # a last token's v and k that are infinite
        loud, mask = proj.clone(), torch.zeros(heads, dim, dim, dtype=torch.bool, device="cuda")
        loud[-1, part, 0, 0], mask[where] = float("inf"), True
        got = run(loud)[1][:, :, :dim]
        assert torch.equal(got.isinf(), mask) and not got.isnan().any(), part
