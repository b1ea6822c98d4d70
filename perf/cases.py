"""Performance cases: the calls a text-to-speech service makes of this library.

A request's prompt is prefilled, its frames are decoded (alone or batched with
other requests over the paged KV pool), the flow head turns each decoded frame
into a latent, and the audio decoder turns latents into 24 kHz PCM. Each case is
one such call, or the short run of calls that belongs together, through the
public C ABI. Weights stand for a trained checkpoint's: N(0, 0.04) rounded to the
pack's formats (Q8_0 blocks or bf16), LayerNorm gains near 1, which keeps the
stack as well conditioned as a trained one is.

  listed()   the cases that are reported by name
  draw(rng)  one more case of the same ranges
  prepare / run / work / tolerance / exact   see each function
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WIDTH, HEADS, FFN, LAYERS, DROPIN_LAYERS = 512, 8, 2048, 12, 9
HEAD_BLOCKS, FRAME_SAMPLES, MIMI_ROWS, WINDOW = 6, 1920, 16, 250
THETA, TEMPERATURE = 10000.0, 0.7
WEIGHT_SEED = 2026  # the checkpoint: one for all requests

P_F32, P_I32 = ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_int32)
P_SZ = ctypes.POINTER(ctypes.c_size_t)


def _package():
    if "speech_mac_amd" not in sys.modules:
        home = os.path.join(ROOT, "speech-mac_amd")
        spec = importlib.util.spec_from_file_location(
            "speech_mac_amd", os.path.join(home, "__init__.py"), submodule_search_locations=[home])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["speech_mac_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["speech_mac_amd"]


def _lib():
    lib = _package().load()
    _check(lib.pgpu_device_init(), lib)
    return lib


def _check(ok, lib):
    if not ok:
        raise RuntimeError(_package().last_error(lib) or "the call was refused")


def _f32(a):
    return a.ctypes.data_as(P_F32)


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # One Q8_0 projection of one frame (the MLP's second): the smallest device call.
        {"name": "matvec_b1", "kind": "matvec", "rows": 512, "columns": 2048, "batch": 1},
        # A whole request through the single-stream API on host buffers: an odd-sized
        # prompt, then frames one at a time.
        {"name": "request_211", "kind": "request", "prompt": 211, "frames": 16},
        # A lightly loaded server whose checkpoint was not quantized.
        {"name": "decode_b12_bf16", "kind": "decode", "streams": 12, "low": 1, "high": 2048,
         "q8": False, "frames": 4},
        # The headline: 64 requests somewhere in their lives.
        {"name": "decode_b64", "kind": "decode", "streams": 64, "low": 1, "high": 2048, "q8": True,
         "frames": 4},
        # A full server with long contexts.
        {"name": "decode_b256", "kind": "decode", "streams": 256, "low": 256, "high": 8187,
         "q8": True, "frames": 4},
        # Prompts of newly admitted requests: a few that continue a prefix already held, ragged,
        # and a full admission round.
        {"name": "prefill_3_ragged", "kind": "prefill", "streams": 3, "low": 37, "high": 300,
         "prefix": 200},
        {"name": "prefill_16x256", "kind": "prefill", "streams": 16, "low": 256, "high": 256,
         "prefix": 0},
        # After the decode step: output norm, flow head, EOS logit, next input.
        {"name": "head_b1", "kind": "head", "streams": 1},
        {"name": "head_b64", "kind": "head", "streams": 64},
        # Speech as it is played (a frame per call), a second of it, and a long utterance at once.
        {"name": "pcm_stream_8", "kind": "pcm", "frames": 8, "chunk": 1},
        {"name": "pcm_13", "kind": "pcm", "frames": 13, "chunk": 13},
        {"name": "pcm_250", "kind": "pcm", "frames": 250, "chunk": 250},
    ]


def _between(rng, low, high):
    """A whole number in [low, high], even over its logarithm."""
    return min(high, max(low, int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(("matvec", "request", "decode", "decode", "prefill", "prefill", "head",
                       "pcm", "pcm"))
    if kind == "matvec":
        rows, columns = rng.choice(((2048, 512), (512, 2048), (1536, 512), (512, 512)))
        return {"kind": kind, "rows": rows, "columns": columns, "batch": _between(rng, 2, 64)}
    if kind == "request":
        return {"kind": kind, "prompt": _between(rng, 24, 600), "frames": _between(rng, 4, 32)}
    if kind == "decode":
        high = _between(rng, 64, 6000)
        return {"kind": kind, "streams": _between(rng, 1, 256), "low": rng.randint(1, high // 4),
                "high": high, "q8": rng.random() < 0.75, "frames": 4}
    if kind == "prefill":
        high = _between(rng, 24, 400)
        return {"kind": kind, "streams": _between(rng, 1, 16), "low": rng.randint(8, high),
                "high": high, "prefix": rng.choice((0, 0, rng.randint(1, 700)))}
    if kind == "head":
        return {"kind": kind, "streams": _between(rng, 2, 256)}
    frames = _between(rng, 3, 400)
    return {"kind": kind, "frames": frames, "chunk": max(-(-frames // 16), _between(rng, 1, frames))}


# ---------------------------------------------------------------- checkpoints


def _bf16(x):
    """fp32 -> the nearest bf16, as bits."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _value(bits):
    """What a stored weight means, in 64 bits: bf16 bits, or Q8_0 blocks [rows][columns / 32]."""
    if bits.dtype == np.uint16:
        return (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    scale = bits["scale_bits"].view(np.float16).astype(np.float64)
    return (scale[..., None] * bits["values"]).reshape(bits.shape[0], -1)


def _q8(w):
    """fp32 [rows][columns] -> Q8_0 blocks: each 32 weights share the scale max/127, in fp16."""
    blocks = np.empty((w.shape[0], w.shape[1] // 32), _package().Q8_BLOCK)
    w = w.reshape(w.shape[0], -1, 32)
    scale = (np.abs(w).max(-1) / 127).astype(np.float16)
    blocks["scale_bits"] = scale.view(np.uint16)
    q = np.rint(w / scale[..., None].astype(np.float32))
    blocks["values"] = np.clip(q, -127, 127).astype(np.int8)
    return blocks


def _flow_weights(layers, q8):
    rng = np.random.default_rng(WEIGHT_SEED)
    out = []
    for _ in range(layers):
        layer = {}
        for name, rows, cols in (("qkv", 3 * WIDTH, WIDTH), ("out", WIDTH, WIDTH),
                                 ("mlp_in", FFN, WIDTH), ("mlp_out", WIDTH, FFN)):
            w = rng.standard_normal((rows, cols), np.float32) * np.float32(0.04)
            layer[name] = _q8(w) if q8 else _bf16(w)
        for n in ("norm1", "norm2"):
            layer[n + "_weight"] = _bf16(1 + 0.1 * rng.standard_normal(WIDTH))
            layer[n + "_bias"] = _bf16(0.1 * rng.standard_normal(WIDTH))
        out.append(layer)
    return out


def _head_weights():
    rng = np.random.default_rng(WEIGHT_SEED + 1)
    shapes = {"input_weight": (WIDTH, 32), "cond_weight": (WIDTH, WIDTH),
              "final_ada_weight": (2 * WIDTH, WIDTH), "final_weight": (32, WIDTH)}
    for i in range(2):
        shapes[f"time_weight_{i}_0"], shapes[f"time_weight_{i}_1"] = (WIDTH, 256), (WIDTH, WIDTH)
        shapes[f"time_freqs_{i}"], shapes[f"time_alpha_{i}"] = (128,), (WIDTH,)
    for b in range(HEAD_BLOCKS):
        shapes[f"block_ada_weight_{b}"] = (3 * WIDTH, WIDTH)
        shapes[f"block_norm_weight_{b}"] = (WIDTH,)
        for j in range(2):
            shapes[f"block_mlp_weight_{b}_{j}"] = (WIDTH, WIDTH)
    for name in list(shapes):
        if "_weight" in name:
            shapes[name.replace("_weight", "_bias")] = shapes[name][:1]
    out = {}
    for name, shape in shapes.items():
        if "freqs" in name:
            v = rng.uniform(0.001, 1.0, shape)
        elif "alpha" in name or "norm_weight" in name:
            v = 1 + 0.1 * rng.standard_normal(shape)
        else:
            v = rng.standard_normal(shape) * (0.05 if "bias" in name else 0.04)
        out[name] = _bf16(v)
    out["eos_weight"] = _bf16(rng.standard_normal((1, WIDTH)) * 0.05)
    out["eos_bias"] = _bf16(rng.standard_normal(1) * 0.05)
    out["norm_weight"] = _bf16(1 + 0.1 * rng.standard_normal(WIDTH))
    out["norm_bias"] = _bf16(0.1 * rng.standard_normal(WIDTH))
    out["embed"] = _bf16(rng.standard_normal((WIDTH, 32)) * 0.1)
    return out


# The audio decoder's convolutions: weight shape ([out, in, k], or [in, out, k] where it
# upsamples), stride.
CONVS = [((512, 512, 7), 1),
         ((512, 256, 12), 6), ((128, 256, 3), 1), ((256, 128, 1), 1),
         ((256, 128, 10), 5), ((64, 128, 3), 1), ((128, 64, 1), 1),
         ((128, 64, 8), 4), ((32, 64, 3), 1), ((64, 32, 1), 1),
         ((1, 64, 3), 1)]
MIMI = [("qkv", (3 * WIDTH, WIDTH)), ("out", (WIDTH, WIDTH)), ("mlp_in", (FFN, WIDTH)),
        ("mlp_out", (WIDTH, FFN)), ("norm1_weight", (WIDTH,)), ("norm1_bias", (WIDTH,)),
        ("norm2_weight", (WIDTH,)), ("norm2_bias", (WIDTH,)), ("scale1", (WIDTH,)),
        ("scale2", (WIDTH,))]


def _audio_weights():
    """Gains that keep activations near 1 through every stage."""
    rng = np.random.default_rng(WEIGHT_SEED + 2)
    out = {"projection": _bf16(0.3 * rng.standard_normal((WIDTH, 32))),
           "upsample": _bf16(0.3 * rng.standard_normal((WIDTH, 32)))}
    for layer in range(2):
        for name, shape in MIMI:
            v = rng.standard_normal(shape)
            if len(shape) == 2:
                v = v * shape[1] ** -0.5
            elif name in ("norm1_weight", "norm2_weight"):
                v = 1 + 0.1 * v
            else:
                v = v * (0.3 if "scale" in name else 0.1)
            out[f"{layer}.{name}"] = _bf16(v)
    for i, (shape, stride) in enumerate(CONVS):
        cin, cout = (shape[0], shape[1]) if stride > 1 else (shape[1], shape[0])
        out[f"conv{i}"] = _bf16(rng.standard_normal(shape) * (cin * shape[2] / stride) ** -0.5)
        out[f"bias{i}"] = _bf16(0.05 * rng.standard_normal(cout))
    return out


_kept = {}  # what a program loads once: device weights by checkpoint


def _once(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _flow_model(q8):
    def make():
        lib, views, model = _lib(), _package().Views(), ctypes.c_void_p()
        layers = views.layers([{k: v.reshape(-1) if v.dtype != np.uint16 else v
                                for k, v in d.items()} for d in _flow_weights(LAYERS, q8)])
        _check(lib.phonon_flow_model_create(layers, LAYERS, ctypes.byref(model)), lib)
        return model
    return _once(("flow", q8), make)


def _dropin_weights():
    def make():
        lib, views = _lib(), _package().Views()
        layers = views.layers([{k: v.reshape(-1) if v.dtype != np.uint16 else v
                                for k, v in d.items()} for d in _flow_weights(DROPIN_LAYERS, True)])
        _check(lib.phonon_flow_prepare_weights(layers, DROPIN_LAYERS), lib)
        return views, layers
    return _once("dropin", make)[1]


def _head_views():
    def make():
        views, w = _package().Views(), _head_weights()
        one = {k: views.bf16(w[k], w[k].shape) for k in
               ("eos_weight", "eos_bias", "norm_weight", "norm_bias", "embed")}
        return views, views.flow_head(w), one
    return _once("head", make)[1:]


def _pcm_model():
    def make():
        pkg, lib, w = _package(), _lib(), _audio_weights()
        views, mimi, model = pkg.Views(), pkg.PhononMimiModel(), ctypes.c_void_p()
        mimi.config, mimi.stride = lib.phonon_mimi_config(), MIMI_ROWS
        mimi.projection = views.bf16(w["projection"], (WIDTH, 32, 1))
        mimi.upsample = views.bf16(w["upsample"], (WIDTH, 1, 32))
        for layer in range(2):
            for f, (name, shape) in enumerate(MIMI):
                mimi.layers[layer][f] = views.bf16(w[f"{layer}.{name}"], shape)
        convs = (ctypes.c_void_p * 11)()
        for i, (shape, stride) in enumerate(CONVS):
            conv, b = ctypes.c_void_p(), w[f"bias{i}"]
            _check(lib.phonon_conv_model_create(
                ctypes.byref(views.bf16(w[f"conv{i}"], shape)), ctypes.byref(views.bf16(b, b.shape)),
                stride, int(stride > 1), ctypes.byref(conv)), lib)
            convs[i] = conv
        _check(lib.phonon_pcm_model_from_parts(ctypes.byref(mimi), convs, ctypes.byref(model)), lib)
        return views, mimi, model
    return _once("pcm", make)[2]


# ------------------------------------------------------------------- requests


class _State:
    """What a program holds for a case, given back when it is dropped."""

    def __init__(self, case):
        self.case, self.lib, self.closers = case, _lib(), []

    def own(self, handle, destroy):
        self.closers.append((handle, destroy))
        return handle

    def view(self, rows):
        """The cache's own rows as an array, which keeps what holds them alive."""
        shape = (DROPIN_LAYERS, self.cache.capacity, WIDTH)
        held = (ctypes.c_float * math.prod(shape)).from_address(
            ctypes.addressof(rows.contents))
        held.state = self
        return np.frombuffer(held, np.float32).reshape(shape)

    def __del__(self):
        for handle, destroy in reversed(self.closers):
            destroy(handle)


def _serving_stream():
    """One HIP stream that the program runs its device calls on, as a server does."""
    return _once("stream", torch.cuda.Stream).cuda_stream


def _normal(seed, *shape, scale=1.0):
    g = torch.Generator("cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda") * scale


def _host_normal(seed, *shape):
    return np.random.default_rng(seed).standard_normal(shape, np.float32)


def _contexts(case):
    """Per stream: positions held before the pass, and positions a prefill adds."""
    n, low, high, prefix = (case.get(k, 0) for k in ("streams", "low", "high", "prefix"))
    rng = np.random.default_rng([n, low, high, prefix])
    if case["kind"] == "decode":
        return rng.integers(low, high + 1, n), np.zeros(n, np.int64)
    held = rng.integers(0, prefix + 1, n) if prefix else np.zeros(n, np.int64)
    return held, rng.integers(low, high + 1, n)


def _tables(case, seed):
    """Shuffled block tables, each stream with the blocks it needs: (tables, pool blocks)."""
    held, added = _contexts(case)
    need = -(-(held + added + case.get("frames", 0)) // 16)
    ids = np.random.default_rng(seed).permutation(int(need.sum())).astype(np.int32)
    tables = np.zeros((len(need), int(need.max())), np.int32)
    at = 0
    for s, k in enumerate(need):
        tables[s, :k] = ids[at: at + k]
        at += k
    return tables, len(ids)


def _layer_kv(seed, layer, blocks):
    """K and V of one layer's blocks: [block][head][K, V][16 positions][64]."""
    return _normal(seed * 64 + layer, blocks, HEADS, 2, 16, 64)


def _open_batch(state, seed, slots):
    """Pool with its contexts, and a batch bound to the model."""
    case, lib = state.case, state.lib
    tables, blocks = _tables(case, seed)
    pool, batch = ctypes.c_void_p(), ctypes.c_void_p()
    _check(lib.phonon_kv_pool_create(LAYERS, blocks, ctypes.byref(pool)), lib)
    state.own(pool, lib.phonon_kv_pool_destroy)
    ids = np.zeros(blocks, np.int32)
    _check(lib.phonon_kv_pool_alloc(pool, blocks, ids.ctypes.data_as(P_I32)), lib)
    view = _package().PgpuPagedKv()
    _check(lib.phonon_kv_pool_view(pool, ctypes.byref(view)), lib)
    for layer in range(LAYERS):
        kv = _layer_kv(seed, layer, blocks)
        _check(lib.pgpu_copy_d2d(None, view.base + 4 * layer * view.layer_stride, kv.data_ptr(),
                                 kv.numel() * 4), lib)
    model = _flow_model(case.get("q8", True))
    _check(lib.phonon_flow_batch_create(model, pool, slots, 16 * tables.shape[1],
                                        ctypes.byref(batch)), lib)
    state.own(batch, lib.phonon_flow_batch_destroy)
    state.batch, state.tables = batch, tables
    state.held, state.added = (a.astype(np.uintp) for a in _contexts(case))
    torch.cuda.synchronize()


def prepare(case, seed):
    """Inputs, contexts and handles of a request, from the seed alone; the checkpoint on the
    device is the program's and is made once."""
    s = _State(case)
    lib, kind = s.lib, case["kind"]
    if kind == "matvec":
        rows, cols, batch = case["rows"], case["columns"], case["batch"]
        w = _once(("matvec", rows, cols), lambda: _matvec_weights(rows, cols))
        handle = ctypes.c_void_p()
        _check(lib.phonon_q8_device_create(w.ctypes.data, rows, cols, 1, ctypes.byref(handle)), lib)
        s.matrix = s.own(handle, lib.phonon_q8_device_destroy)
        s.x, s.y = _normal(seed, batch, cols), torch.zeros(batch, rows, device="cuda")
        s.stream = _serving_stream()
    elif kind == "request":
        s.weights = _dropin_weights()
        s.cache = _package().PhononKvCache()
        _check(lib.phonon_kv_cache_init(ctypes.byref(s.cache), case["prompt"] + case["frames"]), lib)
        s.own(ctypes.byref(s.cache), lib.phonon_kv_cache_destroy)
        s.x = _host_normal(seed, case["prompt"] + case["frames"], WIDTH)
    elif kind == "decode":
        _open_batch(s, seed, case["streams"])
        s.x = _normal(seed + 5, case["streams"], WIDTH)
        s.rows = [torch.empty_like(s.x) for _ in range(2)]
        s.stream = lib.phonon_flow_batch_stream(s.batch)
    elif kind == "prefill":
        _, added = _contexts(case)
        _open_batch(s, seed, int(added.sum()))
        s.x = _normal(seed + 5, int(added.sum()), WIDTH)
        s.y = torch.empty_like(s.x)
    elif kind == "head":
        n = case["streams"]
        head, one = _head_views()
        s.head = ctypes.c_void_p()
        _check(lib.phonon_flow_head_device_create(
            ctypes.byref(head), ctypes.byref(one["eos_weight"]), ctypes.byref(one["eos_bias"]), n,
            ctypes.byref(s.head)), lib)
        s.own(s.head, lib.phonon_flow_head_device_destroy)
        _check(lib.phonon_flow_head_device_set_frame(
            s.head, ctypes.byref(one["norm_weight"]), ctypes.byref(one["norm_bias"]),
            ctypes.byref(one["embed"])), lib)
        _check(lib.phonon_flow_head_device_set_stream(s.head, _serving_stream()), lib)
        s.decoded, s.cond = _normal(seed, n, WIDTH, scale=3.0), _normal(seed + 1, n, WIDTH)
        s.noise = _normal(seed + 2, n, 32)
        s.out = [torch.empty(n, 32, device="cuda"), torch.empty(n, device="cuda"),
                 torch.empty(n, WIDTH, device="cuda")]
    else:
        handle = ctypes.c_void_p()
        _check(lib.phonon_pcm_state_create(_pcm_model(), ctypes.byref(handle)), lib)
        s.pcm = s.own(handle, lib.phonon_pcm_state_destroy)
        s.x = _host_normal(seed, case["frames"], 32)
        s.y = np.zeros(case["frames"] * FRAME_SAMPLES, np.float32)
    torch.cuda.synchronize()
    return s


def _matvec_weights(rows, cols):
    rng = np.random.default_rng(WEIGHT_SEED + 3)
    return _q8(rng.standard_normal((rows, cols), np.float32) * np.float32(0.04))


def run(s):
    """One pass. Decode and prefill end with the status check that makes their rows valid; the
    matvec and the head are enqueued, as between other device work."""
    case, lib = s.case, s.lib
    kind = case["kind"]
    if kind == "matvec":
        _check(lib.phonon_q8_device_matvec(s.matrix, 0, s.x.data_ptr(), s.y.data_ptr(),
                                           case["batch"], s.stream), lib)
        return s.y
    if kind == "request":
        prompt, frames, cache = case["prompt"], case["frames"], ctypes.byref(s.cache)
        out = np.empty((1 + frames, WIDTH), np.float32)
        lib.phonon_kv_cache_reset(cache)
        _check(lib.phonon_flow_stack_prefill(s.weights, cache, _f32(s.x), prompt, THETA,
                                             _f32(out[0])), lib)
        for i in range(frames):
            _check(lib.phonon_flow_stack_step(s.weights, cache, prompt + i, _f32(s.x[prompt + i]),
                                              THETA, _f32(out[1 + i])), lib)
        return out, s.view(s.cache.keys), s.view(s.cache.values)
    if kind == "decode":
        a, b = s.rows
        _check(lib.phonon_flow_batch_set_streams(
            s.batch, case["streams"], s.held.ctypes.data_as(P_SZ), s.tables.ctypes.data_as(P_I32),
            s.tables.shape[1]), lib)
        _check(lib.pgpu_copy_d2d(s.stream, a.data_ptr(), s.x.data_ptr(), s.x.numel() * 4), lib)
        for _ in range(case["frames"]):
            _check(lib.phonon_flow_batch_step_device(s.batch, a.data_ptr(), THETA, b.data_ptr()),
                   lib)
            a, b = b, a
        _check(lib.phonon_flow_batch_sync(s.batch), lib)
        return a, b  # the rows of the last frame and of the one before it
    if kind == "prefill":
        _check(lib.phonon_flow_batch_prefill_device(
            s.batch, case["streams"], s.held.ctypes.data_as(P_SZ), s.added.ctypes.data_as(P_SZ),
            s.tables.ctypes.data_as(P_I32), s.tables.shape[1], s.x.data_ptr(), THETA,
            s.y.data_ptr()), lib)
        _check(lib.phonon_flow_batch_sync(s.batch), lib)
        return s.y
    if kind == "head":
        latents, eos, following = s.out
        _check(lib.phonon_flow_head_device_frame(
            s.head, case["streams"], s.decoded.data_ptr(), s.cond.data_ptr(), s.noise.data_ptr(),
            TEMPERATURE, latents.data_ptr(), eos.data_ptr(), following.data_ptr()), lib)
        return s.out
    lib.phonon_pcm_state_reset(s.pcm)
    frames, chunk = case["frames"], case["chunk"]
    for f in range(0, frames, chunk):
        n = min(chunk, frames - f)
        y = s.y[f * FRAME_SAMPLES: (f + n) * FRAME_SAMPLES]
        _check(lib.phonon_pcm_process(s.pcm, _f32(s.x[f:]), n, _f32(y), y.size, None, 0), lib)
    return s.y


# ------------------------------------------------------------- work, tolerance


def _pair_sum(first, count):
    """Keys attended by `count` positions from `first` on."""
    return count * first + count * (count + 1) // 2


def work(case):
    """Each weight and each key and value read once a step, rows in and out, and the products."""
    kind = case["kind"]
    per_layer = 4 * WIDTH * WIDTH + 2 * WIDTH * FFN
    if kind == "matvec":
        rows, cols, batch = case["rows"], case["columns"], case["batch"]
        return {"bytes": rows * cols * 34 / 32 + 4 * batch * (rows + cols),
                "flops": 2 * rows * cols * batch}
    if kind == "request":
        p, f = case["prompt"], case["frames"]
        keys = _pair_sum(0, p + f)
        return {"bytes": DROPIN_LAYERS * ((1 + f) * per_layer * 34 / 32 + 4096 * _pair_sum(p, f) +
                                          4096 * (p + f)) + 2048 * (p + 2 * f + 1),
                "flops": DROPIN_LAYERS * (2 * per_layer * (p + f) + 4 * WIDTH * keys)}
    if kind == "decode":
        n, f = case["streams"], case["frames"]
        keys = sum(_pair_sum(int(c), f) for c in _contexts(case)[0])
        weight = per_layer * (34 / 32 if case["q8"] else 2)
        return {"bytes": LAYERS * (f * weight + 4096 * keys + 4096 * n * f) + 4096 * n * f,
                "flops": LAYERS * (2 * per_layer * n * f + 4 * WIDTH * keys)}
    if kind == "prefill":
        held, added = _contexts(case)
        rows, keys = int(added.sum()), sum(_pair_sum(int(p), int(c)) for p, c in zip(held, added))
        return {"bytes": LAYERS * (per_layer * 34 / 32 + 4096 * (int(held.sum()) + rows)) +
                4096 * rows,
                "flops": LAYERS * (2 * per_layer * rows + 4 * WIDTH * keys)}
    if kind == "head":
        n = case["streams"]
        weights = (64 * WIDTH + WIDTH * WIDTH + (3 * HEAD_BLOCKS + 2 + 2 * HEAD_BLOCKS) *
                   WIDTH * WIDTH + 32 * WIDTH + WIDTH)
        return {"bytes": 2 * weights + 4 * n * (3 * WIDTH + 65), "flops": 2 * weights * n}
    f = case["frames"]
    held = sum(min(t + 1, WINDOW) for t in range(min(MIMI_ROWS * f, WINDOW)))
    held += max(0, MIMI_ROWS * f - WINDOW) * WINDOW
    weights, flops = 2 * per_layer + 64 * WIDTH, 2 * f * MIMI_ROWS * 2 * per_layer
    positions = f * MIMI_ROWS
    for shape, stride in CONVS:
        weights += math.prod(shape)
        flops += 2 * positions * math.prod(shape)
        positions *= stride
    calls = -(-f // case["chunk"])
    return {"bytes": 2 * weights * calls + 4 * f * (32 + FRAME_SAMPLES),
            "flops": flops + 2 * f * 64 * WIDTH + 2 * 4 * WIDTH * held}


def tolerance(case):
    """Sums in 32 bits, whose order another implementation may change: the outputs are 1e-7 (a
    projection) to 6e-7 (the head, the stack, the decoder's stages) off 64 bits, and as far from
    each other with their sums in another order. The prefill's default takes activations at 22
    significant bits: 5e-6 to 1e-5 off, and as far from its exact mode; a request's rows and
    keys follow from it."""
    return {"rel": 4e-5 if case["kind"] in ("prefill", "request") else 1e-5}


# ----------------------------------------------------------------- in 64 bits


def _norm(x, w, b, eps):
    m = x.mean(-1, keepdim=True)
    y = (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w + b


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))


def _silu(x):
    return x / (1 + torch.exp(-x))


def _rope(x, positions):
    """Interleaved pairs of [rows][512], their phases position * frequency as fp32 has them (the
    checkpoint's convention)."""
    expo = (np.arange(32, dtype=np.float32) * 2) / np.float32(64)
    freq = np.float32(1) / np.power(np.float64(THETA), expo.astype(np.float64)).astype(np.float32)
    phase = np.asarray(positions, np.float32)[:, None] * freq[None, :]
    phase = torch.tensor(phase.astype(np.float64), device=x.device)[:, None, :]
    c, s = torch.cos(phase), torch.sin(phase)
    h = x.view(x.shape[0], HEADS, 32, 2)
    return torch.stack([h[..., 0] * c - h[..., 1] * s, h[..., 0] * s + h[..., 1] * c],
                       -1).reshape(x.shape)


def _attend(q, k, v, mask=None):
    """[queries][8][64] over [keys][8][64]; mask [queries][keys] True where it may look."""
    score = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0).contiguous()) / 8
    if mask is not None:
        score = score.masked_fill(~mask, -math.inf)
    p = torch.softmax(score, -1)
    return torch.matmul(p, v.transpose(0, 1).contiguous()).transpose(0, 1).reshape(q.shape[0], WIDTH)


def _device64(weights):
    return [{k: torch.tensor(_value(v), device="cuda") for k, v in d.items()} for d in weights]


def _flow_exact(layers, x, counts, positions, kv):
    """Rows x of streams with counts[s] rows each at positions[s].. through the layers; kv[layer][s]
    holds (K, V) [positions][8][64] and grows by the rows' own."""
    for at, w in enumerate(layers):
        qkv = _norm(x, w["norm1_weight"], w["norm1_bias"], 1e-5) @ w["qkv"].T
        row = np.concatenate([p + np.arange(c) for p, c in zip(positions, counts)])
        q = _rope(qkv[:, :WIDTH].contiguous(), row).view(-1, HEADS, 64)
        k = _rope(qkv[:, WIDTH: 2 * WIDTH].contiguous(), row).view(-1, HEADS, 64)
        v = qkv[:, 2 * WIDTH:].reshape(-1, HEADS, 64)
        got, o = [], 0
        for s, c in enumerate(counts):
            ks, vs = (torch.cat([a, b[o: o + c]]) for a, b in zip(kv(at, s), (k, v)))
            kv(at, s, (ks, vs))
            p = int(positions[s])
            may = torch.arange(p + c, device="cuda")[None, :] <= p + torch.arange(
                c, device="cuda")[:, None]
            got.append(_attend(q[o: o + c], ks, vs, None if c == 1 else may))
            o += c
        x = x + torch.cat(got) @ w["out"].T
        h = _gelu(_norm(x, w["norm2_weight"], w["norm2_bias"], 1e-5) @ w["mlp_in"].T)
        x = x + h @ w["mlp_out"].T
    return x


class _Contexts:
    """K and V by (layer, stream), in 64 bits when asked for: the pool's blocks plus what the
    frames since then added."""

    def __init__(self, case, seed):
        self.tables, blocks = _tables(case, seed)
        self.held, _ = _contexts(case)
        self.kv = [_layer_kv(seed, layer, blocks) for layer in range(LAYERS)]
        self.more = {}

    def __call__(self, layer, s, grown=None):
        n = int(self.held[s])
        if grown is not None:
            self.more[layer, s] = tuple(a[n:].clone() for a in grown)
            return None
        ids = torch.tensor(self.tables[s, : -(-n // 16)], device="cuda", dtype=torch.int64)
        kv = self.kv[layer][ids].double().permute(2, 0, 3, 1, 4).reshape(2, -1, HEADS, 64)
        more = self.more.get((layer, s))
        return tuple(torch.cat([kv[i, :n], more[i]]) if more else kv[i, :n] for i in range(2))


def exact(case, seed):
    """What run() returns, in 64 bits."""
    kind = case["kind"]
    if kind == "matvec":
        w = torch.tensor(_value(_matvec_weights(case["rows"], case["columns"])), device="cuda")
        return _normal(seed, case["batch"], case["columns"]).double() @ w.T
    if kind == "request":
        return _exact_request(case, seed)
    if kind == "decode":
        layers, contexts = _device64(_flow_weights(LAYERS, case["q8"])), _Contexts(case, seed)
        x, n, before = _normal(seed + 5, case["streams"], WIDTH).double(), case["streams"], None
        for f in range(case["frames"]):
            before, x = x, _flow_exact(layers, x, [1] * n, contexts.held + f, contexts)
        return x, before
    if kind == "prefill":
        layers, contexts = _device64(_flow_weights(LAYERS, True)), _Contexts(case, seed)
        _, added = _contexts(case)
        x = _normal(seed + 5, int(added.sum()), WIDTH).double()
        return _flow_exact(layers, x, [int(c) for c in added], contexts.held, contexts)
    if kind == "head":
        return _exact_head(case, seed)
    return _exact_pcm(case, seed)


def _exact_request(case, seed):
    layers, prompt, frames = _device64(_flow_weights(DROPIN_LAYERS, True)), case["prompt"], \
        case["frames"]
    x = torch.tensor(_host_normal(seed, prompt + frames, WIDTH), device="cuda").double()
    held = {}

    def kv(layer, s, grown=None):
        if grown is not None:
            held[layer] = grown
        return held.get(layer) or (torch.empty(0, HEADS, 64, device="cuda").double(),) * 2

    y = _flow_exact(layers, x, [prompt + frames], [0], kv)
    keys, values = (torch.stack([held[i][j] for i in range(DROPIN_LAYERS)]).reshape(
        DROPIN_LAYERS, prompt + frames, WIDTH) for j in range(2))
    return y[prompt - 1:], keys, values


def _exact_head(case, seed):
    n = case["streams"]
    w = {k: torch.tensor(_value(v), device="cuda") for k, v in _head_weights().items()}
    decoded = _normal(seed, n, WIDTH, scale=3.0).double()
    cond, noise = _normal(seed + 1, n, WIDTH).double(), _normal(seed + 2, n, 32).double()
    state = _norm(decoded, w["norm_weight"], w["norm_bias"], 1e-5)

    def affine(name, x):
        return x @ w[name].T + w[name.replace("_weight", "_bias")]

    def time(i, value):
        phase = value * w[f"time_freqs_{i}"]
        h = _silu(affine(f"time_weight_{i}_0", torch.cat([torch.cos(phase), torch.sin(phase)])))
        h = affine(f"time_weight_{i}_1", h)
        return w[f"time_alpha_{i}"] * h / torch.sqrt((h ** 2).mean() + 1e-5)

    noise = noise * math.sqrt(TEMPERATURE)
    x = affine("input_weight", noise)
    y = _silu(affine("cond_weight", state) + 0.5 * (time(0, 0.0) + time(1, 1.0)))
    for b in range(HEAD_BLOCKS):
        shift, scale, gate = affine(f"block_ada_weight_{b}", y).split(WIDTH, -1)
        h = _norm(x, w[f"block_norm_weight_{b}"], w[f"block_norm_bias_{b}"], 1e-6)
        h = _silu(affine(f"block_mlp_weight_{b}_0", h * (1 + scale) + shift))
        x = x + gate * affine(f"block_mlp_weight_{b}_1", h)
    shift, scale = affine("final_ada_weight", y).split(WIDTH, -1)
    latents = noise + affine("final_weight", _norm(x, None, None, 1e-6) * (1 + scale) + shift)
    return [latents, affine("eos_weight", state)[:, 0], latents @ w["embed"].T + cond]


def _exact_pcm(case, seed):
    w = {k: torch.tensor(_value(v), device="cuda") for k, v in _audio_weights().items()}
    frames = case["frames"]
    latents = torch.tensor(_host_normal(seed, frames, 32), device="cuda").double()
    cur = latents @ w["projection"].T
    prev = torch.cat([torch.zeros_like(cur[:1]), cur[:-1]])
    up = w["upsample"].T
    x = (prev[:, None] * up[MIMI_ROWS:] + cur[:, None] * up[:MIMI_ROWS]).reshape(-1, WIDTH)
    at = torch.arange(len(x), device="cuda")
    may = (at[None, :] <= at[:, None]) & (at[None, :] > at[:, None] - WINDOW)
    for i in range(2):
        qkv = _norm(x, w[f"{i}.norm1_weight"], w[f"{i}.norm1_bias"], 1e-5) @ w[f"{i}.qkv"].T
        q, k = (_rope(qkv[:, j * WIDTH: (j + 1) * WIDTH].contiguous(), np.arange(len(x)))
                .view(-1, HEADS, 64) for j in range(2))
        a = _attend(q, k, qkv[:, 2 * WIDTH:].reshape(-1, HEADS, 64), may)
        x = x + w[f"{i}.scale1"] * (a @ w[f"{i}.out"].T)
        h = _norm(x, w[f"{i}.norm2_weight"], w[f"{i}.norm2_bias"], 1e-5)
        x = x + w[f"{i}.scale2"] * (_gelu(h @ w[f"{i}.mlp_in"].T) @ w[f"{i}.mlp_out"].T)

    def elu(v):
        return torch.where(v <= 0, torch.expm1(v), v)

    def conv(i, v):
        shape, stride = CONVS[i]
        weight, bias = w[f"conv{i}"], w[f"bias{i}"]
        taps = 2 if stride > 1 else shape[2]
        past = torch.cat([torch.zeros_like(v[:1]).expand(taps - 1, -1), v])
        if stride > 1:  # position t stride + k: row t by tap k, row t - 1 by tap stride + k
            parts = [past[1:] @ weight[:, :, k] + past[:-1] @ weight[:, :, stride + k] + bias
                     for k in range(stride)]
            return torch.stack(parts, 1).reshape(len(v) * stride, -1)
        return sum(past[j: j + len(v)] @ weight[:, :, j].T for j in range(taps)) + bias

    x = conv(0, x)
    for stage in range(3):
        x = conv(1 + 3 * stage, elu(x))
        x = x + conv(3 + 3 * stage, elu(conv(2 + 3 * stage, elu(x))))
    return conv(10, elu(x))[:, 0]
