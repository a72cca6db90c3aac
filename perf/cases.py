"""The work that is timed: calls of the library's C entry points as a text-to-speech program makes them, over the
range of sizes such a program meets.

`listed()` names twelve of them, `draw()` gives others of the same ranges.  A case's weights are random values of
the model's shapes, uploaded once per process and the same for every case and seed (a program loads one
checkpoint); what the seed decides is the call's own input: hidden states, prompt embeddings, noise, codes, rows.
The library holds one key/value cache per process, so the rows that a decode step or a continued prompt finds
there are the same for every seed, too: `prepare` writes them, positions 0 up to the call's own, every time.
"""
import ctypes
import importlib
import importlib.util
import os
import sys
import weakref

import numpy as np
import torch

DIM, Q_DIM, KV_DIM, FFN, LAYERS, AC_LAYERS = 3072, 4096, 1024, 9216, 26, 3
LATENT, CODES, SEM_ROWS, EULER = 36, 37, 8320, 7
CACHE = 8192                               # rows of the key/value cache: the size the C program allocates
AUDIO_ROWS = 8194 + LATENT * 23            # audio-code embedding table: semantic codes, then 36 books of 23
LAYER_ELEMS = DIM * (Q_DIM + 2 * KV_DIM) + Q_DIM * DIM + 3 * DIM * FFN
SAMPLES = 1920                             # waveform samples per codec frame


def _package():
    """The Python mirror of the C ABI (its folder's name is no identifier)."""
    name = "voxtral_tts_c_amd"
    if name not in sys.modules:
        folder = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "voxtral-tts.c_amd")
        if os.path.isdir("voxtral-tts.c_amd"):
            folder = os.path.abspath("voxtral-tts.c_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---- the cases ---------------------------------------------------------------------------------

def listed():
    return [
        # the kernel-level product at batch 1 (9216 x 3072 is a gate projection): the smallest call, a few us
        {"name": "linear_1row", "kind": "linear", "rows": 1, "n": 9216, "k": 3072},
        # one backbone step early in an utterance (64-token prompt, a few frames in)
        {"name": "decode_pos81", "kind": "decode", "pos": 81},
        # and near the end of the longest one (2000 frames)
        {"name": "decode_pos1999", "kind": "decode", "pos": 1999},
        # one frame of the flow-matching transformer: semantic head, 7 guided Euler steps, quantisation
        {"name": "acoustic_frame", "kind": "acoustic"},
        # one whole turn of the generation loop, the call that is made for every 80 ms of audio
        {"name": "frame_pos301", "kind": "frame", "pos": 301},
        # prompts: a few words without a long voice sample, a usual one (voice rows + a sentence), the benchmark's
        # 512 tokens, and a long ragged one (long voice sample + a page of text)
        {"name": "prefill_37", "kind": "prefill", "rows": 37, "start": 0},
        {"name": "prefill_226", "kind": "prefill", "rows": 226, "start": 0},
        {"name": "prefill_512", "kind": "prefill", "rows": 512, "start": 0},
        {"name": "prefill_1531", "kind": "prefill", "rows": 1531, "start": 0},
        # codes -> waveform: two words (21 frames), a 40-word paragraph (212), a page (80 s of audio)
        {"name": "codec_21", "kind": "codec", "frames": 21},
        {"name": "codec_212", "kind": "codec", "frames": 212},
        {"name": "codec_1003", "kind": "codec", "frames": 1003},
    ]


# (out, in) of the matrices a program multiplies with: the projections of a layer, the semantic head, the 36-wide
# projections of the acoustic latent, the output head over the vocabulary
MATRICES = [(9216, 3072), (3072, 9216), (4096, 3072), (1024, 3072), (3072, 4096), (8320, 3072), (3072, 36), (36, 3072),
            (131072, 3072)]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["linear", "decode", "frame", "prefill", "prefill", "codec", "codec"])
    if kind == "linear":
        n, k = rng.choice(MATRICES)
        return {"kind": "linear", "rows": _log(rng, 1, 300), "n": n, "k": k}
    if kind == "decode":
        return {"kind": "decode", "pos": _log(rng, 9, CACHE - 1)}
    if kind == "frame":
        return {"kind": "frame", "pos": _log(rng, 9, 2300)}
    if kind == "prefill":
        rows = _log(rng, 6, 1400)
        start = 0 if rng.random() < 0.7 else _log(rng, 5, 600)      # a prompt continued behind cached rows
        return {"kind": "prefill", "rows": rows, "start": start}
    return {"kind": "codec", "frames": _log(rng, 2, 1000)}


# ---- what a program has in hand ----------------------------------------------------------------

_up = {}                                   # what this process has uploaded: the handle of a program


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(shape, seed, std=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=_gen(seed), device="cuda") * std).to(dtype)


def _gain(n, seed):
    """RMSNorm gains: positive, about 1."""
    return torch.randn(n, generator=_gen(seed), device="cuda").abs() * 0.5 + 0.75


def _lib():
    if "lib" not in _up:
        lib = _package().lib()
        assert lib.tts_hip_init(CACHE) == 0, lib.tts_hip_last_error()
        _up["lib"] = lib
        _up["errors"] = lib.tts_hip_error_count()
    return _up["lib"]


def _check():
    _package().check_errors(_up["errors"])


def _layer(seed):
    """One layer's weights in host memory, as a checkpoint's mapping holds them."""
    w = [_normal(s, seed * 16 + i, 0.02, torch.bfloat16).cpu() for i, s in enumerate(
        ((Q_DIM, DIM), (KV_DIM, DIM), (KV_DIM, DIM), (DIM, Q_DIM), (FFN, DIM), (DIM, FFN), (FFN, DIM)))]
    a, f = _gain(DIM, seed * 16 + 8).cpu(), _gain(DIM, seed * 16 + 9).cpu()
    p = [t.data_ptr() for t in w]
    return _package().HostLayer(p[0], p[1], p[2], p[3], a.data_ptr(), p[4], p[5], p[6], f.data_ptr()), (w, a, f)


def _backbone():
    lib = _lib()
    if "backbone" not in _up:
        for i in range(LAYERS):
            src, keep = _layer(100 + i)
            assert lib.tts_hip_upload_llm_layer(i, ctypes.byref(src)) == 0, lib.tts_hip_last_error()
            del keep
        norm = _gain(DIM, 99).cpu()
        assert lib.tts_hip_upload_llm_norm(norm.data_ptr()) == 0, lib.tts_hip_last_error()
        _up["backbone"] = True
    return lib


def _acoustic():
    lib = _lib()
    if "acoustic" not in _up:
        P = _package()
        inv = np.zeros(DIM // 2, np.float32)
        lib.tts_hip_default_time_inv_freq(inv.ctypes.data, DIM // 2)
        bf = torch.bfloat16
        t = {"input_proj_bf16": _normal((DIM, LATENT), 901, 0.2, bf), "time_proj_bf16": _normal((DIM, DIM), 902, 0.02, bf),
             "llm_proj_bf16": _normal((DIM, DIM), 903, 0.02, bf), "semantic_out_bf16": _normal((SEM_ROWS, DIM), 904, 0.02, bf),
             "semantic_out_bias": _normal(SEM_ROWS, 905, 0.1), "acoustic_out_bf16": _normal((LATENT, DIM), 906, 0.02, bf),
             "norm": _gain(DIM, 907)}
        t = {name: v.cpu() for name, v in t.items()}
        table = _normal((AUDIO_ROWS, DIM), 908, 0.05, bf).cpu()
        offsets = np.zeros(CODES, np.int32)
        offsets[1:] = 8194 + 23 * np.arange(LATENT)
        layers = [_layer(950 + i) for i in range(AC_LAYERS)]
        h = P.HostAcoustic()
        h.time_inv_freq = inv.ctypes.data
        for name, v in t.items():
            setattr(h, name, v.data_ptr())
        for i, (src, _) in enumerate(layers):
            h.layers[i] = src
        assert lib.tts_hip_upload_acoustic_weights(ctypes.addressof(h)) == 0, lib.tts_hip_last_error()
        assert lib.tts_hip_upload_audio_embeddings(table.data_ptr(), AUDIO_ROWS, offsets.ctypes.data) == 0, lib.tts_hip_last_error()
        _up["acoustic"] = True
    return lib


def _codec():
    lib = _lib()
    if "codec" not in _up:
        P = _package()
        synth = importlib.import_module(P.__name__ + ".synth")
        weights = synth.CodecWeights(3)
        struct = weights.struct()
        assert lib.tts_hip_upload_codec_weights(ctypes.addressof(struct)) == 0, lib.tts_hip_last_error()
        libc = ctypes.CDLL(None)
        libc.free.argtypes = [ctypes.c_void_p]
        _up["codec"] = weights
        _up["free"] = libc.free
    return lib


class _View:
    """Device memory that belongs to the library, as torch sees it."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 3}


def _cache():
    """The library's K and V caches, [26, CACHE, 1024] each."""
    if "cache" not in _up:
        c = _package().ctx()
        _up["cache"] = tuple(torch.as_tensor(_View(p, (LAYERS, CACHE, KV_DIM)), device="cuda")
                             for p in (c.kv_cache_k_gpu, c.kv_cache_v_gpu))
    return _up["cache"]


def _conversation(rows):
    """Cached rows 0 .. rows - 1 of every layer, as earlier calls left them: k and v ~N(0,1)."""
    if rows > 0:
        for which, c in enumerate(_cache()):
            g = _gen(7 + which)
            for l in range(LAYERS):
                c[l, :rows].copy_(torch.randn((rows, KV_DIM), generator=g, device="cuda"))


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    torch.cuda.synchronize()
    if kind == "linear":
        s["lib"] = _lib()
        s["rows"], s["n"], s["k"] = case["rows"], case["n"], case["k"]
        s["w"] = _normal((s["n"], s["k"]), 5, 0.02, torch.bfloat16)
        s["x"] = _normal((s["rows"], s["k"]), seed)
        s["y"] = torch.empty((s["rows"], s["n"]), device="cuda")
    elif kind == "decode":
        s["lib"] = _backbone()
        s["pos"] = case["pos"]
        _conversation(s["pos"])
        s["x"] = _normal(DIM, seed)
        s["y"] = torch.empty(DIM, device="cuda")
        s["kv"] = [c[:, s["pos"]] for c in _cache()]
    elif kind == "acoustic":
        s["lib"] = _acoustic()
        g = np.random.default_rng(seed)
        s["h"] = g.standard_normal(DIM, dtype=np.float32)
        s["x0"] = g.standard_normal(LATENT, dtype=np.float32)
        s["codes"], s["x"] = np.zeros(CODES, np.int32), np.zeros(LATENT, np.float32)
    elif kind == "frame":
        _backbone()
        s["lib"] = _acoustic()
        s["pos"] = case["pos"]
        _conversation(s["pos"])
        s["embed"] = _normal(DIM, seed, 0.3)              # 37 rows of N(0, 0.05)
        s["x0"] = np.random.default_rng(seed).standard_normal(LATENT, dtype=np.float32)
        s["codes"] = np.zeros(CODES, np.int32)
        s["kv"] = [c[:, s["pos"]] for c in _cache()]
    elif kind == "prefill":
        s["lib"] = _backbone()
        s["rows"], s["start"] = case["rows"], case["start"]
        _conversation(s["start"])
        s["embeds"] = np.random.default_rng(seed).standard_normal((s["rows"], DIM), dtype=np.float32)
        s["kv"] = [c[:, s["start"]:s["start"] + s["rows"]] for c in _cache()]
    else:
        s["lib"] = _codec()
        s["frames"] = case["frames"]
        s["codes"] = _up["codec"].random_codes(s["frames"], seed)
        s["free"] = _up["free"]
    torch.cuda.synchronize()
    _check()
    return s


# ---- one call ----------------------------------------------------------------------------------

def run(s):
    kind, lib = s["kind"], s["lib"]
    if kind == "linear":
        lib.tts_hip_linear_bf16(s["y"].data_ptr(), s["x"].data_ptr(), None, s["rows"], s["k"], s["n"], s["w"].data_ptr())
        return s["y"]
    if kind == "decode":
        lib.tts_hip_llm_forward_device(s["y"].data_ptr(), s["x"].data_ptr(), s["pos"])
        return {"hidden": s["y"], "k": s["kv"][0], "v": s["kv"][1]}
    if kind == "acoustic":
        lib.tts_hip_acoustic_frame(s["codes"].ctypes.data, s["h"].ctypes.data, s["x0"].ctypes.data, s["x"].ctypes.data)
        return {"codes": s["codes"], "latent": s["x"]}
    if kind == "frame":
        # the embedding of the frame's codes comes back in place of the input: called again, the next frame's input
        lib.tts_hip_generate_frame(s["codes"].ctypes.data, s["embed"].data_ptr(), s["x0"].ctypes.data, s["pos"])
        return {"codes": s["codes"], "embed": s["embed"], "k": s["kv"][0], "v": s["kv"][1]}
    if kind == "prefill":
        lib.tts_hip_llm_prefill(s["embeds"].ctypes.data, s["rows"], s["start"])
        return {"k": s["kv"][0], "v": s["kv"][1]}
    out, n = ctypes.POINTER(ctypes.c_float)(), ctypes.c_int(0)
    lib.tts_hip_codec_decode(s["codes"].ctypes.data, s["frames"], ctypes.byref(out), ctypes.byref(n))
    wave = np.ctypeslib.as_array(out, shape=(n.value,))           # the caller owns it and frees it
    weakref.finalize(wave, s["free"], ctypes.cast(out, ctypes.c_void_p).value)
    return wave


# ---- what a call cannot do without -------------------------------------------------------------

def _decode_work(pos):
    row = 2 * KV_DIM * 4
    return {"bytes": LAYERS * (2 * LAYER_ELEMS + 2 * DIM * 4 + (pos + 1) * row) + 3 * DIM * 4,
            "flops": LAYERS * (2 * LAYER_ELEMS + 4 * Q_DIM * (pos + 1))}


def _acoustic_work():
    per_step = AC_LAYERS * LAYER_ELEMS + 2 * DIM * LATENT
    once = SEM_ROWS * DIM + DIM * DIM
    return {"bytes": 2 * (EULER * per_step + once), "flops": 2 * (EULER * 6 * per_step + once)}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        r, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": 2 * n * k + 4 * r * (n + k), "flops": 2 * r * n * k}
    if kind == "decode":
        return _decode_work(case["pos"])
    if kind == "acoustic":
        return _acoustic_work()
    if kind == "frame":
        d, a = _decode_work(case["pos"]), _acoustic_work()
        return {"bytes": d["bytes"] + a["bytes"] + 2 * CODES * DIM, "flops": d["flops"] + a["flops"]}
    if kind == "prefill":
        # what comes out is K and V of every layer: behind the last layer's k|v nothing is needed
        r, st = case["rows"], case["start"]
        elems = (LAYERS - 1) * LAYER_ELEMS + 2 * KV_DIM * DIM
        keys = r * st + r * (r + 1) // 2
        return {"bytes": 2 * elems + 4 * r * DIM + LAYERS * 2 * KV_DIM * 4 * r + (LAYERS - 1) * 2 * KV_DIM * 4 * st,
                "flops": 2 * r * elems + (LAYERS - 1) * 4 * Q_DIM * keys}
    # codec: 8 layers of 4 attention matrices and 3 of 1024 x 4096, two of them at each of 1, 2, 4, 8 x the frames,
    # an input convolution (292 -> 1024, 3 taps), three transposed ones (1024 -> 1024, 4 taps), an output one (7 taps)
    f = case["frames"]
    layer = 4 * 1024 * 1024 + 3 * 1024 * 4096
    up = 4 * 1024 * 1024
    first, last = 3 * 292 * 1024, 7 * 1024 * 240
    return {"bytes": 4 * (8 * layer + 3 * up + first + last) + 4 * f * (CODES + SAMPLES),
            "flops": 2 * f * (2 * layer * 15 + up * 7 + first + 8 * last)}


def tolerance(case):
    """About four times what two correct summation orders differ by, measured: a product against its sum in float64,
    decode steps on two grids and against the sequential CPU sum, prefills against the same rows one decode step at a
    time, the codec against the sequential CPU sum."""
    kind = case["kind"]
    if kind == "linear":
        # fp32 sums up to 7 rows (2e-7), activations of 16 mantissa bits from 8 on (2.5e-6, largest 1.2e-5)
        return {"rel": 1e-6, "max": 5e-6} if case["rows"] < 8 else {"rel": 1e-5, "max": 5e-5}
    if kind == "decode":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "acoustic":
        return {"rel": 4e-5, "max": 4e-4, "differ": 0.01}       # codes: a latent on a quantiser's edge
    if kind == "frame":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.01}
    if kind == "prefill":
        return {"rel": 1e-4, "max": 9e-4}                       # 2.7e-5, 2.2e-4
    return {"rel": 1.5e-5, "max": 1e-4}                         # 3.7e-6, 1.6e-5
