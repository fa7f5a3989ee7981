"""The work a user of this backend has it do, as cases that can be timed and
checked: the decode and prefill calls of include/dsv4_gpu.h through the
package's binding, over the shapes of DeepSeek-V4-scale models.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  inputs, weights and handles, on the GPU
  run(state)           one pass; returns its outputs
  work(case)           bytes and operations a pass cannot do without
  tolerance(case)      how far another correct implementation may be off
  exact(case, seed)    the outputs in 64 bits, plain torch

Weights and activations have the benchmark's distributions: e4m3 codes
uniform over the finite ones with block scales 2^-8..2^-4, e2m1 nibbles
uniform with E8M0 scales 2^-6..2^2, bf16 weights N(0, 0.02), activations
N(0, 1).
"""
import ctypes
import importlib.util
import itertools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda:0"
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
LIMIT = 10.0                     # the model's swiglu limit
EPS = 1e-6

# Resident matrices are keyed by their host address, so a host matrix that
# was uploaded stays allocated while the process lives.
_kept = []
# Every prepared MoE or attention state takes a layer of its own.
_moe_layer = itertools.count()
_attn_layer = itertools.count()
_pkg = None


def backend():
    """The package's binding, its library loaded and the device up."""
    global _pkg
    if _pkg is None:
        if "dsv4_amd" not in sys.modules:
            spec = importlib.util.spec_from_file_location(
                "dsv4_amd", os.path.join(ROOT, "deepseek-v4-in-c_amd", "__init__.py"))
            mod = importlib.util.module_from_spec(spec)
            sys.modules["dsv4_amd"] = mod
            spec.loader.exec_module(mod)
        sys.modules["dsv4_amd"].init()
        _pkg = sys.modules["dsv4_amd"]
    return _pkg


# ---------------------------------------------------------------- cases
def listed():
    return [
        # One token through a mid-size trunk matrix with fp32 block scales:
        # a small decode GEMV, where latency counts.
        dict(name="fp8_decode_4096x4096", op="fp8", rows=4096, cols=4096, scales="f32", nt=1),
        # One token through the query up-projection, E8M0 scales.
        dict(name="fp8_decode_24576x1536", op="fp8", rows=24576, cols=1536, scales="e8m0", nt=1),
        # A full prefill batch through a square trunk matrix.
        dict(name="fp8_prefill_7168x7168_64", op="fp8", rows=7168, cols=7168, scales="e8m0",
             nt=64),
        # The ragged end of a prompt through the query down-projection.
        dict(name="fp8_prefill_1536x7168_13", op="fp8", rows=1536, cols=7168, scales="f32",
             nt=13),
        # The decode loop's head: logits over the vocabulary, then the pick.
        dict(name="head_decode_129280x7168", op="head", rows=129280, cols=7168),
        # A prefill batch through a layer's BF16 compressor projection.
        dict(name="bf16_prefill_1024x4096_48", op="bf16", rows=1024, cols=4096, nt=48),
        # A prefill batch through one expert's gate matrix, reached through
        # the matmul dispatch rather than the fused routed pass.
        dict(name="fp4_prefill_2048x7168_24", op="fp4", rows=2048, cols=7168, nt=24),
        # One token through 8 of 256 routed experts.
        dict(name="moe_decode_8of256", op="moe", hidden=7168, inter=2048, experts=256, topk=8,
             nt=1),
        # A full prefill batch through the routed experts.
        dict(name="moe_prefill_64_8of256", op="moe", hidden=7168, inter=2048, experts=256,
             topk=8, nt=64),
        # One sparse-attention decode step over a long context.
        dict(name="mla_decode_32768_top2048", op="mla", n=32768, k=2048, iheads=16, idim=128,
             keys="fp8", heads=64, dqk=576, dv=512, kv="bf16"),
        # One token through a compressed (ratio 4) attention block at 2200
        # positions, where the indexer selects among the compressed rows.
        dict(name="attn_csa_2200", op="attn", ratio=4, pos=2200),
        # A short prefill chunk through the matmul dispatch from host
        # buffers, as the C program calls it for a shared expert.
        dict(name="host_mmq_n_2048x4096_16", op="host", rows=2048, cols=4096, nt=16),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    op = rng.choice(["fp8", "fp8", "bf16", "fp4", "moe", "mla", "attn", "host"])
    nt = 1 if rng.random() < 0.35 else rng.randint(2, 64)
    if op in ("fp8", "bf16", "fp4", "host"):
        rmax, cmax, step = dict(fp8=(32768, 16384, 16), bf16=(16384, 8192, 8),
                                fp4=(8192, 8192, 32), host=(8192, 8192, 16))[op]
        rows, cols = _log(rng, 64, rmax), _log(rng, 512, cmax, step)
        # at most 2^33 multiply-adds in a pass, 2^31 but for FP8
        nt = max(1, min(nt, (1 << (33 if op == "fp8" else 31)) // (rows * cols)))
        c = dict(op=op, rows=rows, cols=cols, nt=nt)
        if op == "fp8":
            c["scales"] = rng.choice(["f32", "e8m0"])
        return c
    if op == "moe":
        # models' expert shapes are multiples of 512; others are taken too
        whole = rng.random() < 0.75
        experts = rng.choice([8, 16, 64, 256])
        return dict(op=op, hidden=_log(rng, 512, 7168, 512 if whole else 32),
                    inter=_log(rng, 512, 2048, 512 if whole else 32), experts=experts,
                    topk=rng.randint(1, min(8, experts)), nt=nt if whole else min(nt, 8))
    if op == "mla":
        n = _log(rng, 64, 65536)
        return dict(op=op, n=n, k=min(n, _log(rng, 32, 2048)), iheads=rng.choice([16, 64]),
                    idim=128, keys=rng.choice(["fp8", "bf16", "f32"]),
                    heads=rng.choice([16, 64, 128]), dqk=576, dv=512,
                    kv=rng.choice(["bf16", "f32"]))
    return dict(op="attn", ratio=rng.choice([4, 128]), pos=_log(rng, 16, 4500))


# ------------------------------------------------------------- the inputs
def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + salt)
    return g


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * scale


def _ints(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=dtype)


def _fp8(g, rows, cols, scales="e8m0"):
    """e4m3 codes over the finite ones, and the 128x128 block scales."""
    w = _ints(g, 0, 254, (rows, cols), torch.uint8)
    w += (w >= 127).to(torch.uint8)
    grid = ((rows + 127) // 128, (cols + 127) // 128)
    e = _ints(g, -8, -3, grid, torch.int32)
    if scales == "e8m0":
        return w, (127 + e).to(torch.uint8)
    return w, torch.exp2(e.float() + torch.rand(grid, generator=g, device=DEV))


def _fp4(g, rows, cols):
    """Packed e2m1 nibbles and the E8M0 scale of each 1x32 block."""
    w = _ints(g, 0, 256, (rows, cols // 2), torch.uint8)
    s = (127 + _ints(g, -6, 3, (rows, cols // 32), torch.int32)).to(torch.uint8)
    return w, s


def _bf16(g, rows, cols):
    return _normal(g, rows, cols, scale=0.02).to(torch.bfloat16)


def _row_cache(g, n, d, fmt):
    """n rows of width d in a KV format: (data, row scales or None)."""
    v = _normal(g, n, d, scale=1.0 / math.sqrt(d))
    if fmt == "f32":
        return v, None
    if fmt == "bf16":
        return v.to(torch.bfloat16), None
    s = torch.exp2(torch.ceil(torch.log2(v.abs().amax(1) / 448.0)))
    return (v / s[:, None]).to(torch.float8_e4m3fn).view(torch.uint8), s


def _routes(g, nt, experts, topk):
    """Each token's experts and their softmax weights."""
    z = _normal(g, nt, experts)
    v, i = torch.topk(z, topk, dim=1)
    return i.to(torch.int32).contiguous(), torch.softmax(v, 1).contiguous()


def _stream():
    return torch.cuda.current_stream().cuda_stream or None


_KV = {"f32": 0, "bf16": 1, "fp8": 2}


def _inputs(case, seed):
    """The tensors of a case but for the attention block's."""
    op, nt = case["op"], case.get("nt", 1)
    g = _gen(seed, 1)
    if op in ("fp8", "host"):
        w, s = _fp8(g, case["rows"], case["cols"], case.get("scales", "e8m0"))
        return dict(w=w, s=s, x=_normal(g, nt, case["cols"]))
    if op in ("bf16", "head"):
        return dict(w=_bf16(g, case["rows"], case["cols"]), x=_normal(g, nt, case["cols"]))
    if op == "fp4":
        w, s = _fp4(g, case["rows"], case["cols"])
        return dict(w=w, s=s, x=_normal(g, nt, case["cols"]))
    if op == "moe":
        E, h, i = case["experts"], case["hidden"], case["inter"]
        w1, s1 = _fp4(g, E * i, h)
        w3, s3 = _fp4(g, E * i, h)
        w2, s2 = _fp4(g, E * h, i)
        idx, wt = _routes(g, nt, E, case["topk"])
        return dict(w1=w1, s1=s1, w3=w3, s3=s3, w2=w2, s2=s2, idx=idx, wt=wt,
                    x=_normal(g, nt, h))
    kd, ks = _row_cache(g, case["n"], case["idim"], case["keys"])
    kv, _ = _row_cache(g, case["n"], case["dqk"], case["kv"])
    return dict(keys=kd, kscale=ks, kv=kv, qi=_normal(g, case["iheads"], case["idim"]),
                wi=_normal(g, case["iheads"]), q=_normal(g, case["heads"], case["dqk"]),
                sink=_normal(g, case["heads"]))


# The attention block's shapes: hidden 4096, 64 heads of 512, window 128.
A = dict(hidden=4096, ql=1024, H=64, hd=512, rd=64, win=128, ol=1024, og=8, ih=64, idd=128,
         topk=512)


def _attn_inputs(case, seed):
    g = _gen(seed, 2)
    ratio, coff = case["ratio"], 2 if case["ratio"] == 4 else 1
    hd, hid = A["hd"], A["hidden"]
    t = dict(wq_a=_fp8(g, A["ql"], hid), wq_b=_fp8(g, A["H"] * hd, A["ql"]),
             wkv=_fp8(g, hd, hid), wo_a=_fp8(g, A["og"] * A["ol"], A["H"] * hd // A["og"]),
             wo_b=_fp8(g, hid, A["og"] * A["ol"]),
             comp_wkv=_bf16(g, coff * hd, hid), comp_wgate=_bf16(g, coff * hd, hid))
    if ratio == 4:
        t.update(idx_wq_b=_fp8(g, A["ih"] * A["idd"], A["ql"]), idx_wproj=_bf16(g, A["ih"], hid))
    t.update(q_norm=1 + _normal(g, A["ql"], scale=0.1), kv_norm=1 + _normal(g, hd, scale=0.1),
             comp_norm=1 + _normal(g, hd, scale=0.1), sink=_normal(g, A["H"]),
             comp_ape=_normal(g, ratio, coff * hd, scale=0.5))
    t["x"] = _normal(g, case["pos"] + 1, hid, scale=0.5)
    return t


def _rope(n):
    th = np.arange(n)[:, None] / (160000.0 ** (np.arange(A["rd"] // 2) * 2.0 / A["rd"]))[None, :]
    return np.cos(th).astype(np.float32), np.sin(th).astype(np.float32)


# Positions past the prepared one that a state's passes decode before its
# sequence starts over.
AHEAD = 8192


def _attn_bind(case, t):
    """Make the layer resident, bind it, and decode up to the position."""
    D = backend()
    L = D.lib()
    keep = []

    def host(v):
        a = v.cpu()
        a = a.view(torch.int16).numpy() if a.dtype == torch.bfloat16 else a.numpy()
        keep.append(a)
        return a

    def mat(v):
        if isinstance(v, tuple):
            w, s = host(v[0]), host(v[1])
            m = D.DSV4QMat(w.ctypes.data, s.ctypes.data, D.WFP8, w.shape[0], w.shape[1], 128, 128)
        else:
            w = host(v)
            m = D.DSV4QMat(w.ctypes.data, None, D.WBF16, w.shape[0], w.shape[1], 0, 0)
        if L.dsv4_gpu_upload(ctypes.byref(m)) != 0:
            raise RuntimeError("upload failed")
        return m

    w = D.AttnW()
    for name in ("wq_a", "wq_b", "wkv", "wo_a", "wo_b", "comp_wkv", "comp_wgate", "idx_wq_b",
                 "idx_wproj"):
        if name in t:
            setattr(w, name, mat(t[name]))
    for name in ("q_norm", "kv_norm", "sink", "comp_norm", "comp_ape"):
        setattr(w, name, host(t[name]).ctypes.data)
    npos = case["pos"] + AHEAD
    cs, sn = _rope(npos)
    keep.extend([cs, sn])
    w.rope_cos, w.rope_sin = cs.ctypes.data, sn.ctypes.data
    idx = case["ratio"] == 4
    c = D.AttnCfg(hidden=A["hidden"], q_lora=A["ql"], n_heads=A["H"], head_dim=A["hd"],
                  rope_dim=A["rd"], window=A["win"], ratio=case["ratio"],
                  idx_heads=A["ih"] if idx else 0, idx_dim=A["idd"], idx_topk=A["topk"],
                  o_groups=A["og"], o_lora=A["ol"], max_pos=npos, rms_eps=EPS)
    layer = next(_attn_layer)
    if L.dsv4_gpu_attn_bind(layer, ctypes.byref(c), ctypes.byref(w)) != 0:
        raise RuntimeError("attn_bind failed")
    _kept.append(keep)
    return layer, npos


def prepare(case, seed):
    D = backend()
    L = D.lib()
    op, nt = case["op"], case.get("nt", 1)
    f32 = dict(device=DEV, dtype=torch.float32)
    if op == "attn":
        t = _attn_inputs(case, seed)
        layer, npos = _attn_bind(case, t)
        s = dict(op=op, L=L, layer=layer, x=t["x"], out=torch.empty(A["hidden"], **f32),
                 at=case["pos"], start=case["pos"], end=npos, st=_stream())
        for p in range(case["pos"]):
            if L.dsv4_gpu_attn_step_d(s["out"].data_ptr(), t["x"][p].data_ptr(), layer, p,
                                      s["st"]) != 0:
                raise RuntimeError("attn_step failed")
        return s
    s = _inputs(case, seed)
    s.update(op=op, L=L, st=_stream(), nt=nt)
    if op in ("fp8", "bf16", "fp4", "head"):
        s["y"] = torch.empty(nt, case["rows"], **f32)
        s.update(rows=case["rows"], cols=case["cols"])
        s["sf"] = 1 if case.get("scales") == "f32" else 0
        s["tok"] = torch.zeros(1, device=DEV, dtype=torch.int32)
    elif op == "host":
        w, sc = s["w"].cpu().numpy(), s["s"].cpu().numpy()
        m = D.qmat(w, sc)
        if L.dsv4_gpu_upload(ctypes.byref(m)) != 0:
            raise RuntimeError("upload failed")
        _kept.append((w, sc))
        s = dict(op=op, D=D, m=m, nt=nt, x=s["x"].cpu().numpy())
    elif op == "moe":
        E, h, i = case["experts"], case["hidden"], case["inter"]
        layer = next(_moe_layer)

        def q(w, sc, e, rows, cols):
            return D.DSV4QMat(w.data_ptr() + e * rows * cols // 2,
                              sc.data_ptr() + e * rows * cols // 32, D.WFP4, rows, cols, 1, 32)
        for e in range(E):
            ew = D.DSV4ExpertW(q(s["w1"], s["s1"], e, i, h), q(s["w3"], s["s3"], e, i, h),
                               q(s["w2"], s["s2"], e, h, i))
            if L.dsv4_gpu_bind_expert_d(layer, e, ctypes.byref(ew)) != 0:
                raise RuntimeError("bind_expert failed")
        s.update(layer=layer, hidden=h, inter=i, topk=case["topk"], out=torch.empty(nt, h, **f32))
    else:
        s.update({k: v for k, v in case.items() if k not in ("keys", "kv", "op")})
        s["kfmt"], s["vfmt"] = _KV[case["keys"]], _KV[case["kv"]]
        s["o"] = torch.empty(case["heads"], case["dv"], **f32)
        s["sel"] = torch.zeros(case["k"], device=DEV, dtype=torch.int32)
    return s


# ----------------------------------------------------------------- a pass
def run(s):
    op = s["op"]
    if op == "host":
        return s["D"].mmq_n(s["m"], s["x"])
    L, st = s["L"], s["st"]
    if op in ("fp8", "bf16", "fp4", "head"):
        y, x, w = s["y"].data_ptr(), s["x"].data_ptr(), s["w"].data_ptr()
        rows, cols, nt = s["rows"], s["cols"], s["nt"]
        if op == "fp8":
            sc = s["s"].data_ptr()
            rc = (L.dsv4_gpu_fp8_gemv_d(y, x, w, sc, s["sf"], rows, cols, st) if nt == 1 else
                  L.dsv4_gpu_fp8_gemv_n_d(y, x, w, sc, s["sf"], rows, cols, nt, st))
        elif op == "fp4":
            sc = s["s"].data_ptr()
            rc = (L.dsv4_gpu_fp4_gemv_d(y, x, w, sc, rows, cols, 1, 32, st) if nt == 1 else
                  L.dsv4_gpu_fp4_gemv_n_d(y, x, w, sc, rows, cols, 1, 32, nt, st))
        else:
            rc = (L.dsv4_gpu_bf16_gemv_d(y, x, w, rows, cols, st) if nt == 1 else
                  L.dsv4_gpu_bf16_gemv_n_d(y, x, w, rows, cols, nt, st))
        out = s["y"]
        if op == "head":
            rc |= L.dsv4_gpu_argmax_d(s["tok"].data_ptr(), y, rows, st)
            out = (s["y"], s["tok"])
    elif op == "moe":
        a = (s["idx"].data_ptr(), s["wt"].data_ptr())
        b = (s["topk"], s["hidden"], s["inter"], LIMIT, st)
        o, x = s["out"].data_ptr(), s["x"].data_ptr()
        rc = (L.dsv4_gpu_moe_fp4_d(o, x, s["layer"], *a, *b) if s["nt"] == 1 else
              L.dsv4_gpu_moe_fp4_n_d(o, x, s["layer"], *a, s["nt"], *b))
        out = s["out"]
    elif op == "mla":
        ks = s["kscale"]
        rc = L.dsv4_gpu_mla_decode_d(
            s["o"].data_ptr(), s["sel"].data_ptr(), s["qi"].data_ptr(), s["wi"].data_ptr(),
            s["iheads"], s["idim"], s["keys"].data_ptr(),
            None if ks is None else ks.data_ptr(), s["kfmt"], s["idim"], s["n"], s["k"],
            s["q"].data_ptr(), s["kv"].data_ptr(), s["vfmt"], s["dqk"], s["n"],
            s["sink"].data_ptr(), s["heads"], s["dqk"], s["dv"], 1.0 / math.sqrt(s["dqk"]), st)
        out = (s["o"], s["sel"])
    else:
        if s["at"] == s["end"]:                 # the sequence is full: a new one
            if L.dsv4_gpu_attn_reset(s["layer"]) != 0:
                raise RuntimeError("attn_reset failed")
            s["at"] = 0
        p = s["at"]
        rc = L.dsv4_gpu_attn_step_d(s["out"].data_ptr(), s["x"][p % s["x"].shape[0]].data_ptr(),
                                    s["layer"], p, st)
        s["at"] = p + 1
        out = s["out"]
    if rc != 0:
        raise RuntimeError("%s: the call was refused" % op)
    return out


# ------------------------------------------------- bytes, operations, limits
def _mm(rows, cols, nt, wbits, sbytes):
    return (rows * cols * wbits // 8 + sbytes + 4 * nt * (rows + cols), 2 * rows * cols * nt)


def _blocks(rows, cols):
    return -(-rows // 128) * -(-cols // 128)


def work(case):
    op, nt = case["op"], case.get("nt", 1)
    if op in ("fp8", "host"):
        r, c = case["rows"], case["cols"]
        b, f = _mm(r, c, nt, 8, _blocks(r, c) * (4 if case.get("scales") == "f32" else 1))
    elif op in ("bf16", "head"):
        b, f = _mm(case["rows"], case["cols"], nt, 16, 0)
    elif op == "fp4":
        r, c = case["rows"], case["cols"]
        b, f = _mm(r, c, nt, 4, r * c // 32)
    elif op == "moe":
        h, i, E, k = case["hidden"], case["inter"], case["experts"], case["topk"]
        one = 3 * h * i * 17 // 32              # nibbles and scales of an expert
        distinct = E * (1 - (1 - k / E) ** nt)  # independent tokens
        b, f = distinct * one + 8 * nt * h, 6 * h * i * k * nt
    elif op == "mla":
        es = {"fp8": 1, "bf16": 2, "f32": 4}
        n, k, h = case["n"], case["k"], case["heads"]
        b = n * (case["idim"] * es[case["keys"]] + (4 if case["keys"] == "fp8" else 0)) + \
            k * case["dqk"] * es[case["kv"]] + 4 * h * (case["dqk"] + case["dv"]) + 4 * k
        f = 2 * n * case["iheads"] * case["idim"] + 2 * k * h * (case["dqk"] + case["dv"])
    else:
        coff, hd, hid, ql = 2 if case["ratio"] == 4 else 1, A["hd"], A["hidden"], A["ql"]
        comp = case["pos"] // case["ratio"]
        sel = case["ratio"] == 4 and comp > A["topk"]
        w8 = ql * hid + A["H"] * hd * ql + hd * hid + A["ol"] * A["H"] * hd + hid * A["og"] * A["ol"]
        w16 = 2 * coff * hd * hid
        if sel:
            w8 += A["ih"] * A["idd"] * ql
            w16 += A["ih"] * hid
        rows = min(case["pos"] + 1, A["win"]) + (min(comp, A["topk"]) if sel else comp)
        b = w8 + 2 * w16 + 4 * rows * hd + (4 * comp * A["idd"] if sel else 0) + 8 * hid
        f = 2 * (w8 + w16) + 4 * rows * A["H"] * hd
    return dict(bytes=float(b), flops=float(f))


def tolerance(case):
    """f32 accumulation in another order: about four times the distance
    between the results and their 64-bit values."""
    return dict(rel=dict(moe=5e-6, attn=2e-6, mla=1e-6).get(case["op"], 5e-7))


# --------------------------------------------------------------- in 64 bits
def _scaled(w, grid, br, bc):
    """w times its block scales, both f64."""
    r, c = w.shape
    return w * grid.repeat_interleave(br, 0)[:r].repeat_interleave(bc, 1)[:, :c]


def _e8m0(s):
    return torch.exp2(s.double() - 127.0)


def _deq8(w, s):
    f = w.view(torch.float8_e4m3fn).float().double()
    return _scaled(f, _e8m0(s) if s.dtype == torch.uint8 else s.double(), 128, 128)


def _deq4(w, s):
    tab = torch.tensor(E2M1 + tuple(-v for v in E2M1), device=DEV, dtype=torch.float64)
    n = torch.stack((w & 15, w >> 4), 2).reshape(w.shape[0], -1)
    return _scaled(tab[n.int()], _e8m0(s), 1, 32)


def _attend(q, kv, sink, scale, dv):
    """softmax over rows and a sink that takes part in the denominator only."""
    z = (q @ kv.T) * scale
    m = torch.maximum(z.max(1).values, sink)
    e = torch.exp(z - m[:, None])
    return (e @ kv[:, :dv]) / (e.sum(1) + torch.exp(sink - m))[:, None]


def _exact_moe(t, case):
    h, i, nt = case["hidden"], case["inter"], case["nt"]
    out = torch.zeros(nt, h, device=DEV, dtype=torch.float64)
    x, idx, wt = t["x"].double(), t["idx"].long(), t["wt"].double()
    for e in idx.unique().tolist():
        tok, k = torch.nonzero(idx == e, as_tuple=True)
        a, b = slice(e * i, (e + 1) * i), slice(e * h, (e + 1) * h)
        g = x[tok] @ _deq4(t["w1"][a], t["s1"][a]).T
        u = x[tok] @ _deq4(t["w3"][a], t["s3"][a]).T
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        y = (g * torch.sigmoid(g) * u) @ _deq4(t["w2"][b], t["s2"][b]).T
        out.index_add_(0, tok, y * wt[tok, k][:, None])
    return out


def _select(qi, keys, wi, k):
    """The indexer's choice: scores, largest first, ties to the lower index."""
    dots = torch.relu(qi @ keys.T)
    sc = (wi @ dots).float() * (torch.rsqrt(torch.tensor(float(qi.shape[1]), device=DEV)) *
                                torch.rsqrt(torch.tensor(float(qi.shape[0]), device=DEV)))
    return torch.sort(sc, descending=True, stable=True).indices[:k]


def _rms(v, w=None):
    v = v / torch.sqrt((v * v).mean(-1, keepdim=True) + EPS)
    return v if w is None else v * w


def _rotate(v, pos, inverse=False):
    """RoPE of the last rd elements, interleaved pairs; pos per row or one."""
    cs, sn = _rope(int(pos.max()) + 1)
    c = torch.from_numpy(cs).to(DEV).double()[pos]
    s = torch.from_numpy(sn).to(DEV).double()[pos] * (-1.0 if inverse else 1.0)
    out = v.clone()
    re, im = v[..., -A["rd"]::2], v[..., -A["rd"] + 1::2]
    out[..., -A["rd"]::2] = re * c - im * s
    out[..., -A["rd"] + 1::2] = re * s + im * c
    return out


def _exact_attn(case, seed):
    t = _attn_inputs(case, seed)
    t = {k: _deq8(*v) if isinstance(v, tuple) else v.double() for k, v in t.items()}
    P, ratio, hd, win = case["pos"], case["ratio"], A["hd"], A["win"]
    X, x = t["x"], t["x"][P]
    at = torch.tensor(P, device=DEV)
    lo = max(0, P + 1 - win)
    ring = torch.arange(lo, P + 1, device=DEV)
    rows = [_rotate(_rms(X[lo:] @ t["wkv"].T, t["kv_norm"]), ring)]
    n = (P + 1) // ratio
    qr = _rms(t["wq_a"] @ x, t["q_norm"])
    if n:
        kv = (X[:n * ratio] @ t["comp_wkv"].T).view(n, ratio, -1)
        sc = (X[:n * ratio] @ t["comp_wgate"].T).view(n, ratio, -1) + t["comp_ape"]
        if ratio == 4:           # the window before's first halves, this one's second
            none = torch.full_like(sc[:1, :, :hd], -math.inf)
            sc = torch.cat((torch.cat((none, sc[:-1, :, :hd])), sc[:, :, hd:]), 1)
            kv = torch.cat((torch.cat((torch.zeros_like(none), kv[:-1, :, :hd])), kv[:, :, hd:]), 1)
        pooled = (torch.softmax(sc, 1) * kv).sum(1)
        comp = _rotate(_rms(pooled, t["comp_norm"]), torch.arange(n, device=DEV) * ratio)
        if ratio == 4 and n > A["topk"]:
            qi = _rotate((t["idx_wq_b"] @ qr).view(A["ih"], A["idd"]), at)
            keys = comp.reshape(-1)[:n * A["idd"]].view(n, A["idd"])   # idx_dim stride
            comp = comp[_select(qi, keys, t["idx_wproj"] @ x, A["topk"])]
        rows.append(comp)
    q = _rotate(_rms((t["wq_b"] @ qr).view(A["H"], hd)), at)
    o = _attend(q, torch.cat(rows), t["sink"], 1.0 / math.sqrt(hd), hd)
    o = _rotate(o, at, inverse=True).view(A["og"], -1, 1)
    return t["wo_b"] @ torch.bmm(t["wo_a"].view(A["og"], A["ol"], -1), o).reshape(-1)


def exact(case, seed):
    backend()
    op = case["op"]
    if op == "attn":
        return _exact_attn(case, seed)
    t = _inputs(case, seed)
    if op == "moe":
        return _exact_moe(t, case)
    if op == "mla":
        keys = t["keys"].view(torch.float8_e4m3fn).float().double() * t["kscale"][:, None].double() \
            if case["keys"] == "fp8" else t["keys"].double()
        sel = _select(t["qi"].double(), keys, t["wi"].double(), case["k"])
        o = _attend(t["q"].double(), t["kv"][sel].double(), t["sink"].double(),
                    1.0 / math.sqrt(case["dqk"]), case["dv"])
        return o, None
    x = t["x"].double()
    if op in ("bf16", "head"):
        y = torch.cat([x @ w.double().T for w in t["w"].split(16384)], 1)
        return (y, None) if op == "head" else y
    y = x @ (_deq4 if op == "fp4" else _deq8)(t["w"], t["s"]).T
    return y.cpu().numpy() if op == "host" else y
