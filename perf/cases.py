"""The calls that a program built on this library makes, with their sizes.

Each case is one pass through the package's public entry points (the Sampler
class over the C ABI): the single-row call that replaces the reference's
sampler, the batched and decode-loop sampling calls, the speech_head
projection, the T3 transformer's decode step and prompt pass, and a whole
decode loop.  `listed()` gives the fixed ones, `draw()` more of the same
ranges.  Inputs are synthetic (seeded, made on the GPU): logits as the
workloads module makes them, matrices as random blocks of the GGUF formats.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"

# GPT-2 medium T3 Turbo (the model the library's tests and bench run)
N_LAYER, N_EMBD, N_HEAD, HEAD_DIM = 24, 1024, 16, 64
V_TURBO, V_LLAMA = 6563, 8194
WTYPES = {"f16": 1, "q4_0": 2, "q5_0": 6, "q8_0": 8}
BLOCK_BYTES = {"f16": 64, "q4_0": 18, "q5_0": 22, "q8_0": 34}
# block scales that give weights of standard deviation about 0.02
BLOCK_SCALE = {"q4_0": 4.3e-3, "q5_0": 2.2e-3, "q8_0": 2.7e-4}
EPS = 1e-5


def _package():
    """chatterbox.cpp_amd (a dotted directory name: loaded by path)."""
    if "cbx_amd" not in sys.modules:
        d = os.path.join(_ROOT, "chatterbox.cpp_amd")
        spec = importlib.util.spec_from_file_location(
            "cbx_amd", os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["cbx_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["cbx_amd"]


_handle = []


def _sampler():
    """The one handle that a serving program keeps for all its calls."""
    if not _handle:
        _handle.append(_package().Sampler(device=0, max_vocab=32768, max_history=8192))
    return _handle[0]


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # the reference's call shape: one row of host logits in, a token out
        # (the drop-in body of sample_next_token_ex, PCIe included)
        dict(name="row", kind="row", vocab=V_TURBO, history=256, top_k=1000, cfg=False),
        # a throughput run: 256 streams, many steps' logits already there
        dict(name="batch_256x256", kind="batch", streams=256, steps=256, vocab=V_TURBO,
             history=1000),
        # the serving loop over given logits: one launch per step, the
        # streams' state on the device
        dict(name="decode_256", kind="decode", streams=256, steps=16, vocab=V_TURBO, history=1000),
        # classifier-free guidance with top-k off (the Llama T3's vocabulary)
        dict(name="cfg_48", kind="cfg", streams=48, vocab=V_LLAMA, history=700, top_k=0),
        # a large masked vocabulary, forced stops among the rows
        dict(name="masked_1024", kind="masked", streams=1024, vocab=32768, history=512),
        # the speech_head of a guided batch: 128 projected rows
        dict(name="head_q4_0_64cfg", kind="head", rows=64, cfg=True, vocab=V_TURBO, wtype="q4_0"),
        # the speech_head of a few streams
        dict(name="head_q8_0_7", kind="head", rows=7, cfg=False, vocab=V_TURBO, wtype="q8_0"),
        # a whole decode loop of one stream: T3 step, head and sampler, the
        # ids fed back on the device
        dict(name="loop_1", kind="loop", streams=1, steps=4, position=300, n_ctx=1024,
             wtype="q4_0"),
        # one T3 decode step: a few streams, and a full serving batch
        dict(name="step_q8_0_6", kind="step", streams=6, position=280, n_ctx=768, wtype="q8_0"),
        dict(name="step_64", kind="step", streams=64, position=256, n_ctx=512, wtype="q4_0"),
        # the prompt pass: one stream's prompt (the time to its first token),
        # and a serving batch's ragged prompts in one call
        dict(name="prompt_1x251", kind="prompt", streams=1, shortest=251, longest=251, start=0,
             n_ctx=512, wtype="q4_0"),
        dict(name="prompt_64x256", kind="prompt", streams=64, shortest=129, longest=383, start=0,
             n_ctx=512, wtype="q4_0"),
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["row", "batch", "decode", "cfg", "masked", "head", "head", "loop", "step",
                       "step", "step", "prompt", "prompt", "prompt"])
    vocab = rng.choice([V_TURBO, V_TURBO, V_LLAMA, rng.randint(3000, 8400)])
    wtype = rng.choice(["q4_0", "q4_0", "f16", "q5_0", "q8_0"])
    if kind == "row":
        return dict(kind="row", vocab=vocab, history=rng.randint(0, 1000),
                    top_k=rng.choice([50, 250, 1000]), cfg=rng.random() < 0.3)
    if kind == "batch":
        streams = _log(rng, 16, 1024)
        return dict(kind="batch", streams=streams, steps=max(1, _log(rng, 1024, 65536) // streams),
                    vocab=vocab, history=rng.randint(100, 1000))
    if kind == "decode":
        return dict(kind="decode", streams=_log(rng, 1, 512), steps=rng.randint(4, 16),
                    vocab=vocab, history=rng.randint(32, 1000))
    if kind == "cfg":
        return dict(kind="cfg", streams=_log(rng, 1, 128), vocab=vocab,
                    history=rng.randint(0, 1000), top_k=rng.choice([0, 0, 1000]))
    if kind == "masked":
        return dict(kind="masked", streams=_log(rng, 64, 1024), vocab=_log(rng, 9000, 32768),
                    history=rng.randint(16, 512))
    if kind == "head":
        return dict(kind="head", rows=_log(rng, 1, 256), cfg=rng.random() < 0.5,
                    vocab=rng.choice([V_TURBO, rng.randint(3000, 8400)]), wtype=wtype)
    if kind == "loop":
        streams = _log(rng, 1, 32)
        position = rng.randint(40, 1000)
        return dict(kind="loop", streams=streams, steps=rng.randint(1, 4), position=position,
                    n_ctx=1024, wtype=wtype)
    if kind == "step":
        streams = _log(rng, 1, 96)
        position = _log(rng, 30, min(1500, 32000 // streams))
        return dict(kind="step", streams=streams, position=position,
                    n_ctx=position + rng.randint(20, 120), wtype=wtype)
    streams = _log(rng, 1, 48)
    longest = _log(rng, 24, min(700, 14000 // streams))
    start = rng.choice([0, 0, 0, rng.randint(1, 100)])
    return dict(kind="prompt", streams=streams, shortest=max(1, longest - rng.randint(0, longest // 2)),
                longest=longest, start=start, n_ctx=start + longest + rng.randint(1, 200), wtype=wtype)


# ----------------------------------------------------------------- the inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _logits(g, rows, vocab, sigma=3.0):
    """N(0, sigma) with five spikes a row at heights U[6, 12]."""
    x = torch.randn((rows, vocab), generator=g, device=DEV)
    x *= sigma
    at = torch.randint(0, vocab, (rows, 5), generator=g, device=DEV)
    up = torch.rand((rows, 5), generator=g, device=DEV) * 6.0 + 6.0
    x.scatter_reduce_(1, at, up, "amax")  # the same result where two spikes meet
    return x


def _ids(g, shape, vocab):
    return torch.randint(0, vocab, shape, generator=g, device=DEV, dtype=torch.int32)


def _params(seed, streams, **fixed):
    """Per-stream knobs as the batched workload draws them, or fixed ones."""
    rng = np.random.default_rng(seed)
    ks = rng.choice([50, 250, 1000], size=streams)
    ts = rng.uniform(0.5, 1.2, size=streams)
    base = dict(top_p=0.9, repeat_penalty=1.2, min_p=0.0, cfg_weight=0.0)
    return _package().params_tensor(
        [dict(base, top_k=int(ks[i]), temp=float(ts[i]), **fixed) if not fixed
         else dict(base, **fixed) for i in range(streams)], device=DEV)


def _matrix(g, n_out, n_in, wtype):
    """Random rows of a GGUF matrix as the bytes a loaded file holds."""
    blocks = n_out * n_in // 32
    if wtype == "f16":
        w = torch.randn((n_out, n_in), generator=g, device=DEV) * 0.02
        return w.to(torch.float16).view(torch.uint8).reshape(-1)
    b = torch.randint(0, 256, (blocks, BLOCK_BYTES[wtype]), generator=g, device=DEV,
                      dtype=torch.uint8)
    d = BLOCK_SCALE[wtype] * (0.7 + 0.6 * torch.rand((blocks, 1), generator=g, device=DEV))
    b[:, :2] = d.to(torch.float16).view(torch.uint8)
    return b.reshape(-1)


def _values(w, n_out, n_in, wtype):
    """The values of _matrix's bytes, in 64 bits."""
    if wtype == "f16":
        return w.view(torch.float16).reshape(n_out, n_in).double()
    b = w.reshape(-1, BLOCK_BYTES[wtype])
    d = b[:, :2].contiguous().view(torch.float16).double()
    if wtype == "q8_0":
        q = b[:, 2:].contiguous().view(torch.int8).double()
    else:
        n = b[:, -16:]
        q = torch.cat([n & 15, n >> 4], 1).int()
        if wtype == "q5_0":
            bit = torch.arange(32, device=w.device)
            high = (b[:, 2:6].int()[:, bit // 8] >> (bit % 8)) & 1
            q = q + (high << 4)
        q = (q - (16 if wtype == "q5_0" else 8)).double()
    return (q * d).reshape(n_out, n_in)


_SHAPES = (("attn_w", 3, 1), ("attn_proj_w", 1, 1), ("fc_w", 4, 1), ("fc_proj_w", 1, 4))


def _model(g, wtype, n_pos):
    """A Turbo-shaped T3 with random weights, as load_t3_gguf would leave it."""
    n = N_EMBD

    def vec(k, base=0.0, sd=0.05):
        return torch.randn(k, generator=g, device=DEV) * sd + base

    layers = []
    for _ in range(N_LAYER):
        one = {key: _matrix(g, o * n, i * n, wtype) for key, o, i in _SHAPES}
        one.update(ln_1_g=vec(n, 1.0), ln_1_b=vec(n), attn_b=vec(3 * n, 0.0, 0.02),
                   attn_proj_b=vec(n, 0.0, 0.02), ln_2_g=vec(n, 1.0), ln_2_b=vec(n),
                   fc_b=vec(4 * n, 0.0, 0.02), fc_proj_b=vec(n, 0.0, 0.02))
        layers.append(one)
    wpe = torch.randn((n_pos, n), generator=g, device=DEV) * 0.1
    emb = torch.randn((V_TURBO, n), generator=g, device=DEV) * 0.5
    weights = dict(layers=layers, wpe=wpe, emb=emb, ln_f_g=vec(n, 1.0), ln_f_b=vec(n), wtype=wtype)
    model = _package().Sampler.t3_model(layers, wpe, emb, weights["ln_f_g"], weights["ln_f_b"],
                                        wtype=WTYPES[wtype], n_head=N_HEAD, eps=EPS)
    return model, weights


def _caches(g, streams, n_ctx, filled):
    """Keys and values of [0, filled) as earlier calls left them."""
    def one():
        c = torch.zeros((streams, N_LAYER, N_HEAD, n_ctx, HEAD_DIM), device=DEV)
        if filled:
            c[:, :, :, :filled].normal_(0.0, 0.6, generator=g)
        return c
    return one(), one()


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = dict(case=case, sampler=_sampler(), seed=seed)
    if kind == "row":
        rng = np.random.default_rng(seed)
        V = case["vocab"]
        s["logits"] = (rng.standard_normal(V) * 3.0).astype(np.float32)
        s["logits"][rng.choice(V, size=5, replace=False)] = 12.0
        s["uncond"] = (s["logits"] + rng.standard_normal(V).astype(np.float32)
                       if case["cfg"] else None)
        s["history"] = rng.integers(0, V, size=case["history"]).astype(np.int32)
        s["params"] = _package().Params(top_k=case["top_k"], top_p=0.95, temp=0.8,
                                        repeat_penalty=1.2, min_p=0.05,
                                        cfg_weight=0.5 if case["cfg"] else 0.0)
        s["u"] = float(rng.random())
    elif kind == "batch":
        B, T, V = case["streams"], case["steps"], case["vocab"]
        s["logits"] = _logits(g, B * T, V)
        s["history"] = _ids(g, (B, case["history"]), V)
        s["history_len"] = _ids(g, (B,), case["history"] + 1)
        s["params"] = _params(seed, B)
        s["tokens"] = torch.empty(B * T, dtype=torch.int32, device=DEV)
        s["info"] = torch.zeros(B * T, dtype=torch.int32, device=DEV)
    elif kind == "decode":
        B, T, V = case["streams"], case["steps"], case["vocab"]
        s["logits"] = _logits(g, T * B, V).reshape(T, B, V)
        s["history"] = _ids(g, (B, case["history"] + T + 1), V)
        begin = torch.zeros((2, B), dtype=torch.int32, device=DEV)  # every stream running,
        begin[1] = _ids(g, (B,), case["history"] + 1)               # its history's length
        s["begin"], s["now"] = begin, begin.clone()
        s["next"] = torch.empty(B, dtype=torch.int32, device=DEV)
        s["decode"] = _package().Sampler.decode_state(s["now"][0], s["history"], s["now"][1],
                                                      next_token=s["next"])
        s["params"] = _params(seed, B)
        s["tokens"] = torch.empty((T, B), dtype=torch.int32, device=DEV)
    elif kind == "cfg":
        B, V = case["streams"], case["vocab"]
        s["logits"] = _logits(g, B, V)
        s["uncond"] = s["logits"] + torch.randn((B, V), generator=g, device=DEV)
        s["history"] = _ids(g, (B, max(1, case["history"])), V)
        s["history_len"] = _ids(g, (B,), case["history"] + 1)
        s["params"] = _params(seed, B, top_k=case["top_k"], top_p=0.95, temp=0.8, min_p=0.05,
                              cfg_weight=0.5)
        s["tokens"] = torch.empty(B, dtype=torch.int32, device=DEV)
        s["info"] = torch.zeros(B, dtype=torch.int32, device=DEV)
    elif kind == "masked":
        B, V = case["streams"], case["vocab"]
        W = (V + 31) // 32
        s["logits"] = torch.randn((B, V), generator=g, device=DEV) * 4.0
        bits = torch.rand((B, W, 32), generator=g, device=DEV) < 0.2
        bits[:, (V - 1) // 32, (V - 1) % 32] = True
        word = (bits.long() << torch.arange(32, device=DEV)).sum(-1)
        s["allowed"] = torch.where(word >= 2**31, word - 2**32, word).to(torch.int32).contiguous()
        s["force"] = (torch.rand(B, generator=g, device=DEV) < 1.0 / 16).to(torch.uint8)
        s["history"] = _ids(g, (B, case["history"]), V)
        s["history_len"] = torch.full((B,), case["history"], dtype=torch.int32, device=DEV)
        s["params"] = _params(seed, B, top_k=50, temp=0.8, repeat_penalty=1.3, min_p=0.02)
        s["tokens"] = torch.empty(B, dtype=torch.int32, device=DEV)
        s["info"] = torch.zeros(B, dtype=torch.int32, device=DEV)
    elif kind == "head":
        R, V, n = case["rows"], case["vocab"], N_EMBD
        s["weights"] = _matrix(g, V, n, case["wtype"])
        s["bias"] = torch.randn(V, generator=g, device=DEV) * 0.1
        sets = 2 if case["cfg"] else 1
        s["hidden"] = [torch.randn((R, n), generator=g, device=DEV) for _ in range(sets)]
        s["logits"] = [torch.empty((R, V), device=DEV) for _ in range(sets)]
        s["head"] = _package().Sampler.head(
            s["weights"], WTYPES[case["wtype"]], n, s["hidden"][0], s["logits"][0], bias=s["bias"],
            hidden_uncond=s["hidden"][1] if case["cfg"] else None,
            logits_uncond=s["logits"][1] if case["cfg"] else None)
    elif kind in ("step", "loop"):
        B, p, n = case["streams"], case["position"], N_EMBD
        s["model"], s["weights"] = _model(g, case["wtype"], case["n_ctx"])
        s["k"], s["v"] = _caches(g, B, case["n_ctx"], p + 1)
        # streams of a serving batch stand at positions of their own
        s["positions"] = torch.randint(max(1, p - p // 8), p + 1, (B,), generator=g, device=DEV,
                                       dtype=torch.int32)
        s["hidden"] = torch.empty((B, n), device=DEV)
        s["tokens"] = _ids(g, (B,), V_TURBO)
        if kind == "loop":
            T, V = case["steps"], V_TURBO
            s["head_w"] = _matrix(g, V, n, case["wtype"])
            s["head_b"] = torch.randn(V, generator=g, device=DEV) * 0.1
            s["logits"] = [torch.empty((B, V), device=DEV) for _ in range(T)]
            s["heads"] = [_package().Sampler.head(s["head_w"], WTYPES[case["wtype"]], n,
                                                  s["hidden"], x, bias=s["head_b"])
                          for x in s["logits"]]
            s["history"] = _ids(g, (B, p + T + 1), V)
            # rows: state, history length, position, the next id to feed
            s["begin"] = torch.stack([torch.zeros_like(s["positions"]), s["positions"],
                                      s["positions"], s["tokens"]])
            s["now"] = s["begin"].clone()
            s["decode"] = _package().Sampler.decode_state(s["now"][0], s["history"], s["now"][1],
                                                          next_token=s["now"][3])
            s["params"] = _params(seed, B, top_k=1000, top_p=0.95, temp=0.8)
            s["out"] = torch.empty((T, B), dtype=torch.int32, device=DEV)
    elif kind == "prompt":
        B, n, first = case["streams"], N_EMBD, case["start"]
        # the prompts' lengths belong to the case: outputs keep their shapes
        lens = np.random.default_rng([B, case["longest"]]).integers(
            case["shortest"], case["longest"] + 1, size=B)
        s["model"], s["weights"] = _model(g, case["wtype"], case["n_ctx"])
        s["k"], s["v"] = _caches(g, B, case["n_ctx"], first)
        s["lens"] = [int(x) for x in lens]
        s["slots"] = torch.from_numpy(np.repeat(np.arange(B, dtype=np.int32), lens)).to(DEV)
        s["positions"] = torch.from_numpy(np.concatenate(
            [np.arange(first, first + x, dtype=np.int32) for x in lens])).to(DEV)
        rows = int(lens.sum())
        s["inputs"] = torch.randn((rows, n), generator=g, device=DEV) * 0.5
        s["hidden"] = torch.empty((rows, n), device=DEV)
    else:
        raise ValueError(kind)
    return s


# ------------------------------------------------------------------- one pass


def run(s):
    case, smp = s["case"], s["sampler"]
    kind = case["kind"]
    if kind == "row":
        return smp.sample_row(s["logits"], s["history"], s["params"], s["u"],
                              logits_uncond=s["uncond"])
    if kind == "batch":
        smp.sample_batch(s["logits"], s["params"], s["tokens"], n_steps=case["steps"],
                         history=s["history"], history_len=s["history_len"], info=s["info"],
                         seed=s["seed"], max_survivors=1000, stop_token=case["vocab"] - 1)
        return s["tokens"], s["info"]
    if kind == "decode":
        s["now"].copy_(s["begin"])
        for t in range(case["steps"]):
            smp.decode_step(s["logits"][t], s["params"], s["tokens"][t], s["decode"],
                            seed=s["seed"], step0=t, stop_token=case["vocab"] - 1)
        return s["tokens"], s["now"], s["history"], s["next"]
    if kind == "cfg":
        smp.sample_batch(s["logits"], s["params"], s["tokens"], logits_uncond=s["uncond"],
                         history=s["history"], history_len=s["history_len"], info=s["info"],
                         seed=s["seed"], max_survivors=case["top_k"],
                         stop_token=case["vocab"] - 1)
        return s["tokens"], s["info"]
    if kind == "masked":
        smp.sample_batch(s["logits"], s["params"], s["tokens"], history=s["history"],
                         history_len=s["history_len"], allowed=s["allowed"],
                         force_stop=s["force"], stop_token=case["vocab"] - 1, info=s["info"],
                         seed=s["seed"], max_survivors=50)
        return s["tokens"], s["info"]
    if kind == "head":
        smp.head_logits(s["head"], case["rows"], case["vocab"], case["vocab"])
        return s["logits"]
    if kind == "step":
        positions = s["positions"].clone()
        smp.t3_step(s["model"], positions, s["k"], s["v"], s["hidden"], tokens=s["tokens"])
        return s["hidden"], positions, s["k"], s["v"]
    if kind == "loop":
        now = s["now"]
        now.copy_(s["begin"])
        for t in range(case["steps"]):
            smp.t3_step(s["model"], now[2], s["k"], s["v"], s["hidden"], tokens=now[3],
                        state=now[0])
            smp.decode_step(s["logits"][t], s["params"], s["out"][t], s["decode"],
                            head=s["heads"][t], seed=s["seed"], step0=t, stop_token=V_TURBO - 1)
        return s["logits"], s["out"], now, s["history"], s["hidden"], s["k"], s["v"]
    smp.t3_prefill(s["model"], s["slots"], s["positions"], s["k"], s["v"], s["hidden"],
                   inputs=s["inputs"])
    return s["hidden"], s["k"], s["v"]


# ------------------------------------------------- what a pass cannot do without


def _t3_work(rows, mean_keys, cached_keys, wtype, rows_out):
    """`rows` rows through the layers, each over `mean_keys` keys, with
    `cached_keys` keys in all read from the caches."""
    n = N_EMBD
    return dict(bytes=N_LAYER * (12 * n * n // 32 * BLOCK_BYTES[wtype]
                                 + 2 * n * 4 * (cached_keys + rows)) + rows_out * n * 4 * 2,
                flops=N_LAYER * rows * (2.0 * 12 * n * n + 4.0 * n * mean_keys))


def _head_work(rows, vocab, wtype):
    return dict(bytes=vocab * N_EMBD // 32 * BLOCK_BYTES[wtype] + rows * 4 * (N_EMBD + vocab)
                + 4 * vocab, flops=2.0 * rows * vocab * N_EMBD)


def work(case):
    kind = case["kind"]
    if kind == "row":
        return dict(bytes=case["vocab"] * 4 * (2 if case["cfg"] else 1) + 4 * case["history"] + 40,
                    flops=0.0)
    if kind in ("batch", "decode"):
        rows = case["streams"] * case["steps"]
        return dict(bytes=rows * (4 * case["vocab"] + 2 * case["history"] + 32), flops=0.0)
    if kind == "cfg":
        return dict(bytes=case["streams"] * (8 * case["vocab"] + 2 * case["history"] + 32),
                    flops=0.0)
    if kind == "masked":
        return dict(bytes=case["streams"] * (4 * case["vocab"] + case["vocab"] // 8
                                             + 4 * case["history"] + 33), flops=0.0)
    if kind == "head":
        return _head_work(case["rows"] * (2 if case["cfg"] else 1), case["vocab"], case["wtype"])
    if kind in ("step", "loop"):
        B, p = case["streams"], case["position"]
        mean = (max(1, p - p // 8) + p) / 2 + 1
        w = _t3_work(B, mean, int(B * mean), case["wtype"], B)
        if kind == "step":
            return w
        h, T = _head_work(B, V_TURBO, case["wtype"]), case["steps"]
        return dict(bytes=T * (w["bytes"] + h["bytes"] + B * 4 * (V_TURBO + p)),
                    flops=T * (w["flops"] + h["flops"]))
    mean = (case["shortest"] + case["longest"]) / 2
    rows = int(case["streams"] * mean)
    return _t3_work(rows, case["start"] + (mean + 1) / 2, case["streams"] * case["start"],
                    case["wtype"], rows)


def tolerance(case):
    """Tokens, flags and state are whole numbers and stay the same.  The
    projection and the transformer compute in 32 bits: about four times the
    distance that a 64-bit computation shows."""
    kind = case["kind"]
    if kind in ("row", "batch", "decode", "cfg", "masked"):
        return "exact"
    if kind == "head":
        return dict(rel=6e-7)
    return dict(rel=1e-5)


# -------------------------------------------------------- the same in 64 bits


def _norm(x, gain, bias):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + EPS) * gain.double() + bias.double()


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * x * (1.0 + 0.044715 * x * x)))


def _layers(w, x, attend):
    """The transformer over rows x; attend(layer, q, k, v) gives the heads."""
    n = N_EMBD
    for i, one in enumerate(w["layers"]):
        def product(rows, key, bias, n_out, n_in):
            return rows @ _values(one[key], n_out, n_in, w["wtype"]).t() + one[bias].double()
        u = _norm(x, one["ln_1_g"], one["ln_1_b"])
        q, k, v = product(u, "attn_w", "attn_b", 3 * n, n).reshape(-1, 3, N_HEAD, HEAD_DIM).unbind(1)
        x = x + product(attend(i, q, k, v).reshape(-1, n), "attn_proj_w", "attn_proj_b", n, n)
        u = _norm(x, one["ln_2_g"], one["ln_2_b"])
        x = x + product(_gelu(product(u, "fc_w", "fc_b", 4 * n, n)), "fc_proj_w", "fc_proj_b",
                        n, 4 * n)
    return _norm(x, w["ln_f_g"], w["ln_f_b"])


def _step64(s):
    """One decode step of the state's streams: hidden rows and caches."""
    w, at = s["weights"], s["positions"].long()
    kc, vc = s["k"].double(), s["v"].double()
    row = torch.arange(at.numel(), device=DEV)
    seen = torch.arange(kc.shape[3], device=DEV)[None, None, :] <= at[:, None, None]

    def attend(i, q, k, v):
        kc[row, i, :, at], vc[row, i, :, at] = k, v
        a = (kc[:, i] * q[:, :, None]).sum(-1) / math.sqrt(HEAD_DIM)
        a = torch.softmax(a.masked_fill(~seen, -math.inf), -1)
        return (a[..., None] * vc[:, i]).sum(2)

    x = w["emb"][s["tokens"].long()].double() + w["wpe"][at].double()
    return _layers(w, x, attend), kc, vc


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("head", "step", "loop", "prompt"):
        return None  # tokens and flags: whole numbers
    s = prepare(case, seed)
    if kind == "head":
        w = _values(s["weights"], case["vocab"], N_EMBD, case["wtype"])
        return [h.double() @ w.t() + s["bias"].double() for h in s["hidden"]]
    if kind == "step":
        hidden, kc, vc = _step64(s)
        return hidden, None, kc, vc
    if kind == "loop":  # later steps stand on sampled ids: the first step's logits
        hidden = _step64(s)[0]
        w = _values(s["head_w"], V_TURBO, N_EMBD, case["wtype"])
        first = hidden @ w.t() + s["head_b"].double()
        return [first] + [None] * (case["steps"] - 1), None, None, None, None, None, None
    kc, vc, first = s["k"].double(), s["v"].double(), case["start"]

    def attend(i, q, k, v):
        out, r = torch.empty_like(q), 0
        for b, T in enumerate(s["lens"]):
            kc[b, i, :, first:first + T] = k[r:r + T].transpose(0, 1)
            vc[b, i, :, first:first + T] = v[r:r + T].transpose(0, 1)
            K, W = kc[b, i, :, :first + T], vc[b, i, :, :first + T]
            a = torch.matmul(q[r:r + T].transpose(0, 1), K.transpose(1, 2).contiguous())
            late = torch.ones((T, first + T), dtype=torch.bool, device=DEV).triu(first + 1)
            a = torch.softmax((a / math.sqrt(HEAD_DIM)).masked_fill(late, -math.inf), -1)
            out[r:r + T] = torch.matmul(a, W).transpose(0, 1)
            r += T
        return out

    return _layers(s["weights"], s["inputs"].double(), attend), kc, vc
