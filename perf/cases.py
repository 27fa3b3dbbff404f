"""The work that a user of this library has it do, as cases that can be timed and compared.

Every case goes through the public entry points (tsr_hip.Device over the C ABI, and tsr_llama.LlamaDecoder),
at sizes of the benchmark, the tests and the models that the repository names (a Llama-3-8B architecture, a
Qwen2.5-0.5B shaped FFN), or at generic ones:

  mul_mat       GGML_OP_MUL_MAT on a Q8_0 / Q4_K weight: one decode row (replayed from a captured graph over
                the weights of several layers, as a decode token is), short ubatches of a few rows, and
                prefill ubatches; with the residual addend, the fused RMS_NORM or the SWIGLU epilogue
  fa_decode     FLASH_ATTN_EXT of one query row over a q8_0 cache with a device-resident plan, over the caches
                of several layers (captured, as above)
  fa_rows       FLASH_ATTN_EXT of a causal ubatch behind a history
  layer_decode  the launches of one Llama decoder layer for one token, replayed from a captured graph
  layer_prefill one Llama decoder layer over a ubatch of prompt tokens
  model_decode  LlamaDecoder: one token by graph replay, its logits read back (a host-side sampler)
  model_prefill LlamaDecoder: a prompt prefilled, the logits of its last token read back

Outputs are the ops' whole result buffers. Results of the single ops depend on f32 summation order only (the
quantization of the activations is elementwise and part of the op's definition).
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "tesseract-npu_amd"))

import tsr_hip as H  # noqa: E402
import tsr_llama as LL  # noqa: E402
import tsr_synth as S  # noqa: E402

_FMT = {"q8_0": H.FMT_Q8_0, "q4_k": H.FMT_Q4_K}
_CTX = []


def _dev():
    """The one library context that a program holds."""
    if not _CTX:
        _CTX.append(H.Device(0))
    return _CTX[0]


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # one decode row of a small model's FFN up matrix (the Qwen2.5-0.5B shape) over 8 layers: latency
        {"name": "decode_q80_4864x896", "kind": "mul_mat", "fmt": "q8_0", "N": 4864, "K": 896, "T": 1, "opt": "none",
         "layers": 8},
        # one decode row of the Llama-3-8B FFN down matrix with the residual, over 4 layers
        {"name": "decode_q4k_4096x14336", "kind": "mul_mat", "fmt": "q4_k", "N": 4096, "K": 14336, "T": 1, "opt": "add",
         "layers": 4},
        # the Llama-3-8B Q|K|V rows for 8 tokens with the fused norm: several sequences decoded together, a
        # short draft verified, the tail of a prompt
        {"name": "rows8_q4k_norm_6144x4096", "kind": "mul_mat", "fmt": "q4_k", "N": 6144, "K": 4096, "T": 8,
         "opt": "norm", "layers": 1},
        # a short prompt (100 tokens, ragged) through a Q4_K projection with the residual
        {"name": "prompt100_q4k_4096x4096", "kind": "mul_mat", "fmt": "q4_k", "N": 4096, "K": 4096, "T": 100,
         "opt": "add", "layers": 1},
        # the benchmark's prefill: 512 tokens, Q8_0
        {"name": "prefill512_q80_4096x4096", "kind": "mul_mat", "fmt": "q8_0", "N": 4096, "K": 4096, "T": 512,
         "opt": "none", "layers": 1},
        # the largest product: the Llama-3-8B gate|up rows with SWIGLU over a ubatch of 512
        {"name": "prefill512_q4k_glu_28672", "kind": "mul_mat", "fmt": "q4_k", "N": 28672, "K": 4096, "T": 512,
         "opt": "glu", "layers": 1},
        # decode attention at 8192 cells over 4 layers' caches (the benchmark's attention workload)
        {"name": "fa_decode_8192", "kind": "fa_decode", "cells": 8192, "n_head": 32, "n_head_kv": 8, "D": 128,
         "layers": 4},
        # causal attention of a 512-token ubatch behind 1536 cells
        {"name": "fa_rows512_hist1536", "kind": "fa_rows", "T": 512, "hist": 1536, "n_head": 32, "n_head_kv": 8,
         "D": 128},
        # one Llama-3-8B decoder layer, one token at context 4096
        {"name": "layer_decode_8b_4096", "kind": "layer_decode", "n_embd": 4096, "n_ff": 14336, "n_head": 32,
         "n_head_kv": 8, "D": 128, "pos": 4100},
        # one Llama-3-8B decoder layer over a ragged ubatch of 300 tokens behind 700 cells
        {"name": "layer_prefill_8b_300", "kind": "layer_prefill", "n_embd": 4096, "n_ff": 14336, "n_head": 32,
         "n_head_kv": 8, "D": 128, "T": 300, "hist": 700},
        # a whole small Q4_K model, one token at a time with the logits on the host
        {"name": "model_decode_4x2048", "kind": "model_decode", "n_layer": 4, "n_embd": 2048, "n_ff": 5632,
         "n_head": 32, "n_head_kv": 8, "D": 64, "n_vocab": 8192, "fmt": "q4_k", "pos": 1200},
        # the same model's prompt prefill, 333 tokens in ubatches of 256 (the second one ragged)
        {"name": "model_prefill_4x2048", "kind": "model_prefill", "n_layer": 4, "n_embd": 2048, "n_ff": 5632,
         "n_head": 32, "n_head_kv": 8, "D": 64, "n_vocab": 8192, "fmt": "q4_k", "T": 333, "ubatch": 256},
    ]


_HEADS = [(32, 8, 128), (32, 8, 64), (16, 8, 128), (14, 2, 64), (8, 1, 128), (8, 4, 256)]   # n_head, n_head_kv, D
_MOST = 512.0 * 28672 * 4096        # multiply-adds of the largest listed product


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mul_mat"] * 6 + ["fa_decode"] * 2 + ["fa_rows"] * 2 + ["layer_decode", "layer_prefill"])
    if kind == "mul_mat":
        fmt = rng.choice(["q8_0", "q4_k"])
        T = 1 if rng.random() < 0.25 else _log(rng, 2, 512)
        opt = rng.choice(["none", "add", "norm", "glu"])
        bs = 32 if fmt == "q8_0" else 256
        # the norm inside the product is the matvec kernels' (a ubatch of 16 or more runs its own RMS_NORM);
        # so is Q8_0's SWIGLU
        if T >= 16 and (opt == "norm" or (opt == "glu" and fmt == "q8_0")):
            opt = "none"
        K = bs * max(1, _log(rng, 512, 8192 if opt == "norm" else 14336) // bs)
        N = _log(rng, 512, 28672)
        if opt == "glu":
            N += N & 1
        while float(T) * N * K > _MOST:
            N = (N // 4) * 2
        layers = 8 if T == 1 and N * K < (16 << 20) else 4 if T == 1 else 1
        return {"kind": kind, "fmt": fmt, "N": N, "K": K, "T": T, "opt": opt, "layers": layers}
    if kind == "fa_decode":
        nh, nkv, D = rng.choice(_HEADS)
        return {"kind": kind, "cells": _log(rng, 64, 16384), "n_head": nh, "n_head_kv": nkv, "D": D, "layers": 4}
    if kind == "fa_rows":
        nh, nkv, D = rng.choice(_HEADS)
        T = _log(rng, 2, 512)
        hist = 0 if rng.random() < 0.3 else _log(rng, 16, 3584)
        return {"kind": kind, "T": T, "hist": hist, "n_head": nh, "n_head_kv": nkv, "D": D}
    nh, nkv, D = rng.choice([(32, 8, 128), (32, 8, 64), (16, 8, 128)])
    c = {"kind": kind, "n_embd": nh * D, "n_ff": 256 * rng.randint(2 * nh * D // 256, 7 * nh * D // 512), "n_head": nh,
         "n_head_kv": nkv, "D": D}
    if kind == "layer_decode":
        c["pos"] = _log(rng, 64, 8192)
    else:
        c["T"] = _log(rng, 4, 400)
        c["hist"] = 0 if rng.random() < 0.3 else _log(rng, 16, 2048)
    return c


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _wseed(seed, *what):
    return S.seed_of(f"cases-{seed}", "/".join(map(str, what)))


def _blocks(fmt, N, K, seed, *what):
    """A random-init weight (normal, std 0.02) as ggml blocks."""
    return S.quant_rows(_FMT[fmt], _wseed(seed, *what), N, K, 0.02)


def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(_wseed(seed, what) & 0x7FFFFFFFFFFFFFFF)


def _randn(seed, what, *shape):
    return torch.randn(*shape, generator=_gen(seed, what), device="cuda", dtype=torch.float32)


def _act(seed, what, T, K):
    """Hidden-state rows: normal values with a few channels several times larger than the rest."""
    x = _randn(seed, what, T, K)
    x[:, ::61] *= 6.0
    return x


def _norm_w(seed, what, K):
    return 1.0 + 0.1 * _randn(seed, what, K)


def _empty(*shape):
    return torch.empty(*shape, device="cuda", dtype=torch.float32)


def _ptr(t):
    return t.data_ptr()


def _cache(d, seed, what, cells, kv_size, E):
    """A K and a V cache whose cells [0, cells) hold quantized rows."""
    out = []
    idx = torch.arange(max(cells, 1), device="cuda", dtype=torch.int64)
    for which, name in ((H.KV_K, "k"), (H.KV_V, "v")):
        kv = d.kv(E, kv_size)
        if cells:
            rows = _randn(seed, f"{what}.{name}", cells, E)
            torch.cuda.synchronize()
            d.kv_set_rows(kv, which, _ptr(rows), cells, E, _ptr(idx))
            d.sync()
        out.append(kv)
    return out


def _capture(d, fn):
    """fn's launches as a graph (run once first, as a program's first token is)."""
    fn()
    d.sync()
    d.graph_begin()
    try:
        fn()
    finally:
        g = d.graph_end()
    return g


def _model_cfg(c, seed):
    return LL.LlamaConfig(f"cases-{seed}", c["n_layer"], c["n_embd"], c["n_ff"], c["n_head"], c["n_head_kv"], c["D"],
                          c["n_vocab"], wfmt=_FMT[c["fmt"]], ofmt=_FMT[c["fmt"]])


def _tokens(c, seed, n):
    return np.random.default_rng(_wseed(seed, "tokens") & 0xFFFFFFFF).integers(0, c["n_vocab"], n).astype(np.int32)


def _n_kv(end):
    return (end + 255) // 256 * 256


def prepare(case, seed):
    d, c, kind = _dev(), case, case["kind"]
    st = {"case": c, "d": d}
    if kind == "mul_mat":
        fmt, N, K, T = c["fmt"], c["N"], c["K"], c["T"]
        No = N // 2 if c["opt"] == "glu" else N
        st["w"] = [d.weight(_FMT[fmt], _blocks(fmt, N, K, seed, "w", i), N, K) for i in range(c["layers"])]
        st["x"] = [_act(seed, f"x{i}", T, K) for i in range(c["layers"])]
        st["y"] = [_empty(T, No) for _ in range(c["layers"])]
        st["add"] = [_randn(seed, f"add{i}", T, No) for i in range(c["layers"])] if c["opt"] == "add" else None
        st["nw"] = _norm_w(seed, "nw", K) if c["opt"] == "norm" else None
    elif kind == "fa_decode":
        nh, nkv, D, cells = c["n_head"], c["n_head_kv"], c["D"], c["cells"]
        st["kv"] = [_cache(d, seed, f"kv{i}", cells, _n_kv(cells), nkv * D) for i in range(c["layers"])]
        st["q"] = [_randn(seed, f"q{i}", nh * D) for i in range(c["layers"])]
        st["out"] = [_empty(nh * D) for _ in range(c["layers"])]
        st["plan"] = d.fa_plan(D, nh, nkv, 1, _n_kv(cells))
        st["plan"].set(LL.msum_decode(cells - 1, _n_kv(cells)), [[cells - 1, cells]])
    elif kind == "fa_rows":
        nh, nkv, D, T, hist = c["n_head"], c["n_head_kv"], c["D"], c["T"], c["hist"]
        st["kc"], st["vc"] = _cache(d, seed, "kv", hist + T, _n_kv(hist + T), nkv * D)
        st["q"] = _randn(seed, "q", T, nh * D)
        st["out"] = _empty(T, nh * D)
        st["msum"] = LL.msum_causal(hist, T, _n_kv(hist + T))
        st["runs"] = np.array([[hist, hist + T]], np.uint32)
    elif kind in ("layer_decode", "layer_prefill"):
        nh, nkv, D, n, ff = c["n_head"], c["n_head_kv"], c["D"], c["n_embd"], c["n_ff"]
        T, hist = (1, c["pos"]) if kind == "layer_decode" else (c["T"], c["hist"])
        nq, E = nh * D, nkv * D
        for name, N, K in (("wqkv", nq + 2 * E, n), ("wo", n, nq), ("wgu", 2 * ff, n), ("wd", n, ff)):
            st[name] = d.weight(H.FMT_Q4_K, _blocks("q4_k", N, K, seed, name), N, K)
        st["kc"], st["vc"] = _cache(d, seed, "kv", hist, _n_kv(hist + T), E)
        st["x"], st["an"], st["fn"] = _act(seed, "x", T, n), _norm_w(seed, "an", n), _norm_w(seed, "fn", n)
        st["xn"], st["hn"], st["qkv"], st["att"] = _empty(T, n), _empty(T, n), _empty(T, nq + 2 * E), _empty(T, nq)
        st["h"], st["glu"], st["y"], st["tab"] = _empty(T, n), _empty(T, ff), _empty(T, n), _empty(D)
        st["pos"] = torch.arange(hist, hist + T, device="cuda", dtype=torch.int32)
        st["cell"] = torch.arange(hist, hist + T, device="cuda", dtype=torch.int64)
        st["msum"] = LL.msum_causal(hist, T, _n_kv(hist + T))
        st["runs"] = np.array([[hist, hist + T]], np.uint32)
        if kind == "layer_decode":
            st["plan"] = d.fa_plan(D, nh, nkv, 1, _n_kv(hist + 1))
            st["plan"].set(st["msum"], st["runs"])
    else:
        cfg = _model_cfg(c, seed)
        w = LL.SyntheticWeights(cfg)
        kv_size = _n_kv(c["pos"] + 8 if kind == "model_decode" else c["T"])
        st["m"] = LL.LlamaDecoder(d, cfg, w, kv_size)
        if kind == "model_decode":
            st["m"].prefill_history(w, c["pos"])
            st["token"] = int(_tokens(c, seed, 1)[0])
        else:
            st["tokens"] = _tokens(c, seed, c["T"])
    torch.cuda.synchronize()
    if kind == "mul_mat" and c["T"] == 1:
        st["graph"] = _capture(d, lambda: _mul_mats(st))
    elif kind == "fa_decode":
        st["graph"] = _capture(d, lambda: _fa_decodes(st))
    elif kind == "layer_decode":
        st["graph"] = _capture(d, lambda: _layer_decode(st))
    return st


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def _mul_mats(st):
    d, c = st["d"], st["case"]
    T, K, N = c["T"], c["K"], c["N"]
    for i in range(c["layers"]):
        w, x, y = st["w"][i], _ptr(st["x"][i]), _ptr(st["y"][i])
        if c["opt"] == "norm":
            d.mul_mat_norm(w, x, T, K, 1e-5, _ptr(st["nw"]), y, N)
        elif c["opt"] == "glu":
            d.mul_mat(w, x, T, K, y, N // 2, flags=H.MM_GLU)
        elif c["opt"] == "add":
            d.mul_mat(w, x, T, K, y, N, add=_ptr(st["add"][i]), add_stride=N)
        else:
            d.mul_mat(w, x, T, K, y, N)


def _fa_decodes(st):
    d, c = st["d"], st["case"]
    nq = c["n_head"] * c["D"]
    for i in range(c["layers"]):
        kc, vc = st["kv"][i]
        d.flash_attn_plan(st["plan"], _ptr(st["q"][i]), nq, kc, vc, 1.0 / math.sqrt(c["D"]), _ptr(st["out"][i]), nq)


def _layer_decode(st):
    d, c = st["d"], st["case"]
    n, ff, D, nq = c["n_embd"], c["n_ff"], c["D"], c["n_head"] * c["D"]
    d.rope_table(_ptr(st["pos"]), D, 500000.0, _ptr(st["tab"]))
    d.attn_qkv_plan_rope_tab(st["plan"], st["wqkv"], _ptr(st["x"]), 1e-5, _ptr(st["an"]), _ptr(st["qkv"]), st["kc"],
                             st["vc"], 1.0 / math.sqrt(D), D, H.ROPE_NORMAL, _ptr(st["tab"]), _ptr(st["cell"]),
                             _ptr(st["att"]), nq)
    d.mul_mat(st["wo"], _ptr(st["att"]), 1, nq, _ptr(st["h"]), n, add=_ptr(st["x"]), add_stride=n)
    d.mul_mat_norm(st["wgu"], _ptr(st["h"]), 1, n, 1e-5, _ptr(st["fn"]), _ptr(st["glu"]), ff, flags=H.MM_GLU)
    d.mul_mat(st["wd"], _ptr(st["glu"]), 1, ff, _ptr(st["y"]), n, add=_ptr(st["h"]), add_stride=n)


def _layer_prefill(st):
    """The op list of LlamaDecoder's prefill ubatch for one layer."""
    d, c = st["d"], st["case"]
    n, ff, D, nq, T = c["n_embd"], c["n_ff"], c["D"], c["n_head"] * c["D"], c["T"]
    w3 = nq + 2 * c["n_head_kv"] * D
    if T >= 16:
        d.rms_norm(_ptr(st["x"]), n, T, n, 1e-5, _ptr(st["xn"]), n, w=_ptr(st["an"]), w_stride=n)
        d.mul_mat(st["wqkv"], _ptr(st["xn"]), T, n, _ptr(st["qkv"]), w3)
    else:
        d.mul_mat_norm(st["wqkv"], _ptr(st["x"]), T, n, 1e-5, _ptr(st["an"]), _ptr(st["qkv"]), w3)
    d.rope_kv(_ptr(st["qkv"]), T, w3, D, c["n_head"], c["n_head_kv"], D, H.ROPE_NORMAL, _ptr(st["pos"]), 500000.0,
              st["kc"], st["vc"], _ptr(st["cell"]))
    d.flash_attn(_ptr(st["qkv"]), T, w3, st["kc"], st["vc"], D, c["n_head"], c["n_head_kv"], 1.0 / math.sqrt(D),
                 st["msum"], _ptr(st["att"]), nq, new_runs=st["runs"])
    d.mul_mat(st["wo"], _ptr(st["att"]), T, nq, _ptr(st["h"]), n, add=_ptr(st["x"]), add_stride=n)
    if T >= 16:
        d.rms_norm(_ptr(st["h"]), n, T, n, 1e-5, _ptr(st["hn"]), n, w=_ptr(st["fn"]), w_stride=n)
        d.mul_mat(st["wgu"], _ptr(st["hn"]), T, n, _ptr(st["glu"]), ff, flags=H.MM_GLU)
    else:
        d.mul_mat_norm(st["wgu"], _ptr(st["h"]), T, n, 1e-5, _ptr(st["fn"]), _ptr(st["glu"]), ff, flags=H.MM_GLU)
    d.mul_mat(st["wd"], _ptr(st["glu"]), T, ff, _ptr(st["y"]), n, add=_ptr(st["h"]), add_stride=n)


def run(state):
    st, c = state, state["case"]
    kind = c["kind"]
    if kind == "mul_mat":
        if "graph" in st:
            st["graph"].launch()
        else:
            _mul_mats(st)
        return st["y"]
    if kind == "fa_decode":
        st["graph"].launch()
        return st["out"]
    if kind == "fa_rows":
        nq = c["n_head"] * c["D"]
        st["d"].flash_attn(_ptr(st["q"]), c["T"], nq, st["kc"], st["vc"], c["D"], c["n_head"], c["n_head_kv"],
                           1.0 / math.sqrt(c["D"]), st["msum"], _ptr(st["out"]), nq, new_runs=st["runs"])
        return st["out"]
    if kind == "layer_decode":
        st["graph"].launch()
        return {k: st[k] for k in ("qkv", "att", "h", "glu", "y")}
    if kind == "layer_prefill":
        _layer_prefill(st)
        return {k: st[k] for k in ("qkv", "att", "h", "glu", "y")}
    if kind == "model_decode":
        st["m"].step_graph(st["token"], c["pos"])
    else:
        st["m"].prefill(st["tokens"], 0, c["ubatch"])
    return st["m"].read_logits()


# ---------------------------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------------------------
def _wbytes(fmt, N, K):
    return N * (K // 32 * 34 if fmt == "q8_0" else K // 256 * 144)


def _layer_work(c, T, hist, fmt="q4_k"):
    n, ff, nq, E = c["n_embd"], c["n_ff"], c["n_head"] * c["D"], c["n_head_kv"] * c["D"]
    mm = ((nq + 2 * E, n), (n, nq), (2 * ff, n), (n, ff))
    pairs = T * hist + T * (T + 1) / 2.0
    b = sum(_wbytes(fmt, N, K) for N, K in mm) + 2 * (hist + T) * E // 32 * 34
    f = sum(2.0 * T * N * K for N, K in mm) + 4.0 * pairs * nq
    return b, f


def work(case):
    c, kind = case, case["kind"]
    if kind == "mul_mat":
        N, K, T = c["N"], c["K"], c["T"]
        No = N // 2 if c["opt"] == "glu" else N
        b = _wbytes(c["fmt"], N, K) + 4 * T * (K + No * (2 if c["opt"] == "add" else 1)) + (4 * K if c["opt"] == "norm" else 0)
        return {"bytes": c["layers"] * b, "flops": c["layers"] * 2.0 * T * N * K}
    if kind in ("fa_decode", "fa_rows"):
        T, hist, L = (1, c["cells"] - 1, c["layers"]) if kind == "fa_decode" else (c["T"], c["hist"], 1)
        nq, E = c["n_head"] * c["D"], c["n_head_kv"] * c["D"]
        pairs = T * hist + T * (T + 1) / 2.0
        return {"bytes": L * (2 * (hist + T) * E // 32 * 34 + 8 * T * nq), "flops": L * 4.0 * pairs * nq}
    if kind in ("layer_decode", "layer_prefill"):
        T, hist = (1, c["pos"]) if kind == "layer_decode" else (c["T"], c["hist"])
        b, f = _layer_work(c, T, hist)
        nq, E = c["n_head"] * c["D"], c["n_head_kv"] * c["D"]
        return {"bytes": b + 4 * T * (3 * c["n_embd"] + 2 * nq + 2 * E + c["n_ff"]), "flops": f}
    T, hist = (1, c["pos"]) if kind == "model_decode" else (c["T"], 0)
    b, f = _layer_work(c, T, hist, c["fmt"])
    return {"bytes": c["n_layer"] * b + _wbytes(c["fmt"], c["n_vocab"], c["n_embd"]) + 4 * (T * c["n_embd"] + c["n_vocab"]),
            "flops": c["n_layer"] * f + 2.0 * c["n_vocab"] * c["n_embd"]}


def tolerance(case):
    """About four times what exact() measures (rel): the products and the attention are f32 sums of exactly
    quantized operands; a norm in front of the quantization turns its last-bit differences into single steps
    of the int8 activations, and a layer's or a model's products see those of all the ops before them."""
    kind = case["kind"]
    if kind == "mul_mat":
        return {"rel": 3e-4, "max": 1e-1} if case["opt"] == "norm" else {"rel": 1e-6, "max": 1e-4}
    if kind in ("fa_decode", "fa_rows"):
        return {"rel": 1e-6, "max": 1e-4}
    return {"rel": 3e-2, "max": 5e-1}


# ---------------------------------------------------------------------------------------------
# the results in 64 bits: operands quantized by the ops' rule (f32), every sum in f64
# ---------------------------------------------------------------------------------------------
def _qact32(x):
    """QACT A32: blocks of 32, d = amax / 127, quants rounded half away, the scale rounded to fp16."""
    b = x.float().cpu().reshape(x.shape[0], -1, 32)
    dd = b.abs().amax(2) / 127.0
    inv = torch.where(dd != 0, 1.0 / torch.where(dd != 0, dd, torch.ones_like(dd)), torch.zeros_like(dd))
    v = b * inv[:, :, None]
    t = torch.trunc(v)
    q = (t + torch.where((v - t).abs() >= 0.5, torch.sign(v), torch.zeros_like(v))).clamp(-128, 127)
    return (q.double() * dd.half().double()[:, :, None]).reshape(x.shape).cuda()


def _qact256(x):
    """QACT A256: blocks of 256, iscale = -127 / (the first value of the largest magnitude), quants rounded half
    to even, d = 1 / iscale."""
    b = x.float().cpu().reshape(x.shape[0], -1, 256)
    top = torch.gather(b, 2, b.abs().argmax(2, keepdim=True))
    one = torch.ones_like(top)
    isc = torch.where(top != 0, torch.div(-127.0 * one, torch.where(top != 0, top, one)), torch.zeros_like(top))
    q = torch.round(isc * b).clamp(-128, 127)
    dd = torch.where(isc != 0, 1.0 / torch.where(isc != 0, isc, one), torch.zeros_like(isc))
    return (q.double() * dd.double()).reshape(x.shape).cuda()


def _dequant(fmt, blocks, K):
    """ggml blocks -> f64 [N, K]."""
    b = torch.from_numpy(blocks).cuda()
    if fmt == "q8_0":
        b = b.reshape(-1, K // 32, 34)
        sc = b[:, :, 0:2].contiguous().view(torch.float16).double()
        return (b[:, :, 2:].contiguous().view(torch.int8).double() * sc).reshape(-1, K)
    b = b.reshape(-1, 144)
    sm = b[:, 0:4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = b[:, 16:].reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
    return (q * (sm[:, 0:1] * sc)[:, :, None] - (sm[:, 1:2] * mn)[:, :, None]).reshape(-1, K)


def _mm64(fmt, blocks, x, K):
    xq = _qact32(x) if fmt == "q8_0" else _qact256(x)
    return xq @ _dequant(fmt, blocks, K).T.contiguous()


def _rms64(x, w, eps=1e-5):
    x = x.double()
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * w.double()


def _glu64(y):
    g, u = y[:, 0::2], y[:, 1::2]
    return g / (1.0 + torch.exp(-g)) * u


def _rope64(x, n_heads, D, pos, base):
    """ROPE, mode NORMAL (pairs 2i, 2i + 1)."""
    i = torch.arange(D // 2, device="cuda", dtype=torch.float64)
    th = pos.double()[:, None] * torch.pow(torch.tensor(base, dtype=torch.float64, device="cuda"), -2.0 * i / D)
    c, s = torch.cos(th)[:, None, :], torch.sin(th)[:, None, :]
    v = x.double().reshape(x.shape[0], n_heads, D // 2, 2)
    return torch.stack([v[..., 0] * c - v[..., 1] * s, v[..., 0] * s + v[..., 1] * c], 3).reshape(x.shape)


def _attn64(q, k, v, n_head, n_head_kv, D, hist):
    """Causal attention of the rows of q behind hist cells; k, v [cells, E] already quantized (f64)."""
    T, G = q.shape[0], n_head // n_head_kv
    qq = _qact32(q)
    out = torch.empty(T, n_head * D, device="cuda", dtype=torch.float64)
    dead = torch.arange(k.shape[0], device="cuda")[None, :] > hist + torch.arange(T, device="cuda")[:, None]
    for h in range(n_head):
        kk, vv = k[:, h // G * D:(h // G + 1) * D], v[:, h // G * D:(h // G + 1) * D]
        s = qq[:, h * D:(h + 1) * D] @ kk.T.contiguous() / math.sqrt(D)
        out[:, h * D:(h + 1) * D] = torch.softmax(s.masked_fill(dead, -math.inf), 1) @ vv
    return out


def _layer64(x, kh, vh, w, c, hist, fmt="q4_k", base=500000.0):
    """One layer; w: {"wqkv", "wo", "wgu", "wd"} ggml blocks and the norms; kh, vh: the history rows (f32)."""
    n, ff, D, nh, nkv = c["n_embd"], c["n_ff"], c["D"], c["n_head"], c["n_head_kv"]
    nq, E, T = nh * D, nkv * D, x.shape[0]
    qkv = _mm64(fmt, w["wqkv"], _rms64(x, w["an"]), n)
    pos = torch.arange(hist, hist + T, device="cuda")
    rot = _rope64(qkv[:, :nq + E].contiguous(), nh + nkv, D, pos, base)
    k = _qact32(torch.cat([kh, rot[:, nq:].float()]))
    v = _qact32(torch.cat([vh, qkv[:, nq + E:].float()]))
    att = _attn64(rot[:, :nq].contiguous(), k, v, nh, nkv, D, hist)
    h = _mm64(fmt, w["wo"], att, nq) + x.double()
    glu = _glu64(_mm64(fmt, w["wgu"], _rms64(h, w["fn"]), n))
    y = _mm64(fmt, w["wd"], glu, ff) + h
    return {"qkv": qkv, "rot": torch.cat([rot, qkv[:, nq + E:]], 1), "att": att, "h": h, "glu": glu, "y": y}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "mul_mat":
        out = []
        for i in range(c["layers"]):
            x = _act(seed, f"x{i}", c["T"], c["K"])
            if c["opt"] == "norm":
                x = _rms64(x, _norm_w(seed, "nw", c["K"]))
            y = _mm64(c["fmt"], _blocks(c["fmt"], c["N"], c["K"], seed, "w", i), x, c["K"])
            if c["opt"] == "add":
                y = y + _randn(seed, f"add{i}", c["T"], c["N"]).double()
            out.append(_glu64(y) if c["opt"] == "glu" else y)
        return out
    if kind in ("fa_decode", "fa_rows"):
        nh, nkv, D = c["n_head"], c["n_head_kv"], c["D"]
        out = []
        for i in range(c.get("layers", 1)):
            tag = f"kv{i}" if kind == "fa_decode" else "kv"
            cells = c["cells"] if kind == "fa_decode" else c["hist"] + c["T"]
            k, v = (_qact32(_randn(seed, f"{tag}.{s}", cells, nkv * D)) for s in "kv")
            if kind == "fa_rows":
                return _attn64(_randn(seed, "q", c["T"], nh * D), k, v, nh, nkv, D, c["hist"])
            out.append(_attn64(_randn(seed, f"q{i}", nh * D)[None], k, v, nh, nkv, D, cells - 1)[0])
        return out
    if kind in ("layer_decode", "layer_prefill"):
        n, ff, D = c["n_embd"], c["n_ff"], c["D"]
        nq, E = c["n_head"] * D, c["n_head_kv"] * D
        T, hist = (1, c["pos"]) if kind == "layer_decode" else (c["T"], c["hist"])
        w = {name: _blocks("q4_k", N, K, seed, name)
             for name, N, K in (("wqkv", nq + 2 * E, n), ("wo", n, nq), ("wgu", 2 * ff, n), ("wd", n, ff))}
        w["an"], w["fn"] = _norm_w(seed, "an", n), _norm_w(seed, "fn", n)
        kh, vh = ((_randn(seed, f"kv.{s}", hist, E) if hist else _empty(0, E)) for s in "kv")
        r = _layer64(_act(seed, "x", T, n), kh, vh, w, c, hist)
        if kind == "layer_prefill":                                   # rope_kv rotates the rows in place
            r["qkv"] = r["rot"]
        del r["rot"]
        return r
    cfg = _model_cfg(c, seed)
    sw = LL.SyntheticWeights(cfg)
    T, hist = (1, c["pos"]) if kind == "model_decode" else (c["T"], 0)
    x = torch.from_numpy(sw.embedding()[_tokens(c, seed, T)]).cuda()
    for il in range(cfg.n_layer):
        t = {name.split(".")[2]: sw.quant(name, N, K, cfg.wfmt) for name, N, K in LL.layer_tensors(cfg, il)}
        w = {"wqkv": np.concatenate([t["attn_q"], t["attn_k"], t["attn_v"]]), "wo": t["attn_output"], "wd": t["ffn_down"],
             "wgu": np.stack([t["ffn_gate"], t["ffn_up"]], 1).reshape(2 * cfg.n_ff, -1)}
        for k, name in (("an", "attn_norm"), ("fn", "ffn_norm")):
            w[k] = torch.from_numpy(sw.norm(f"blk.{il}.{name}.weight")).cuda()
        kh, vh = (torch.from_numpy(sw.kv_history(il, i, hist)).cuda() if hist else _empty(0, cfg.E) for i in (0, 1))
        x = _layer64(x, kh, vh, w, c, hist, c["fmt"])["y"]
    x = _rms64(x[-1:], torch.from_numpy(sw.norm("output_norm.weight")).cuda())
    return _mm64(c["fmt"], sw.quant("output.weight", cfg.n_vocab, cfg.n_embd, cfg.ofmt), x, cfg.n_embd)[0]
