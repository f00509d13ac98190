"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values; `kind` says which public entry points it calls:

  step    Runner.step: forward, backward and Adam of a decoder (gradients and loss come back)
  linear  one linear layer: y = x W^T, dx = dy W, dW = dy^T x
  mlp_up  the gate/up projection with SwiGLU (forward)
  attn    flash attention forward and backward
  head    cut cross-entropy over the vocabulary, forward and backward
  lora    a LoRA linear layer, forward and backward
  norm    RMSNorm forward and backward

`form` is the operand form: "fp32" (the reference's precision and the default of every entry
point), "mixed" (fp32 in memory, bf16 products: precision = bf16 of the fp32 entry points) or
"bf16" (operands resident in bf16, fp32 sums and results).
"""
from __future__ import annotations

import ctypes
import functools
import math
import struct
import tempfile

import torch

F32, BF16 = torch.float32, torch.bfloat16


# ── the cases ────────────────────────────────────────────────────────────

def _step(name, **kw):
    c = dict(kind="step", name=name, eps=1e-6, theta=1e6, qk_norm=True, tied=False, n_seqs=1)
    c.update(kw)
    return c


def listed():
    return [
        # The smallest training step in use: a 2-layer decoder in the reference's precision on
        # one 128-token sequence.  Launches and latency count.
        _step("step_2l_fp32", form="fp32", layers=2, dim=256, heads=4, kv_heads=2, head_dim=64,
              ff=768, vocab=4096, n_pos=128, theta=1e6),
        # The headline step's widths, batch (4 sequences of 512 tokens) and tied 152k vocabulary in
        # bf16 operands, with 4 of its 28 layers: enough of them that layers and head weigh alike.
        _step("step_4l_bf16", form="bf16", layers=4, dim=1024, heads=16, kv_heads=8,
              head_dim=128, ff=3072, vocab=151936, n_pos=512, n_seqs=4, tied=True),
        # One linear layer of a 16-token fine-tune step, the reference's own run length.
        dict(kind="linear", name="linear_fp32_16", form="fp32", t=16, n=1024, k=3072),
        # The largest linear layer: gate or up of a long-context full fine-tune.
        dict(kind="linear", name="linear_bf16_8192", form="bf16", t=8192, n=12288, k=4096),
        # The gate/up projection and SwiGLU of one layer of the headline step.
        dict(kind="mlp_up", name="mlp_up_bf16_2048", form="bf16", t=2048, n=3072, k=1024),
        # Attention of a batch of four 2048-token sequences, grouped queries 2:1.
        dict(kind="attn", name="attn_bf16_2048", form="bf16", b=4, n=2048, heads=16, kv_heads=8,
             head_dim=128, causal=True),
        # Attention over an odd number of tokens (a document as long as it is), groups 4:1.
        dict(kind="attn", name="attn_bf16_1001", form="bf16", b=2, n=1001, heads=32, kv_heads=8,
             head_dim=128, causal=True),
        # Attention of a short fine-tune window in the reference's precision.
        dict(kind="attn", name="attn_fp32_100", form="fp32", b=1, n=100, heads=16, kv_heads=8,
             head_dim=128, causal=True),
        # The loss head of the headline step through the standalone entry points.
        dict(kind="head", name="head_mixed_2048", form="mixed", t=2048, vocab=151936, dim=1024,
             z_loss=0.0, smoothing=0.0),
        # The loss head of a short step over an odd vocabulary (a tokenizer with a few added
        # tokens), with both of its regularisers.
        dict(kind="head", name="head_fp32_127", form="fp32", t=127, vocab=32003, dim=768,
             z_loss=1e-4, smoothing=0.1),
        # A rank-16 adapter on a 2560-wide projection, as in a LoRA fine-tune of 2048 tokens.
        dict(kind="lora", name="lora_mixed_2048", form="mixed", t=2048, n=2560, k=2560, r=16),
        # The norm of one layer of the headline step, both directions, gain gradient included.
        dict(kind="norm", name="norm_2048", form="fp32", t=2048, dim=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly multiples of 64, some of 8, a few odd."""
    w = _log(rng, lo, hi)
    u = rng.random()
    g = 64 if u < 0.7 else 8 if u < 0.9 else 1
    return max(lo, (w + g // 2) // g * g)


_CAP = {"fp32": 3e11, "mixed": 6e11, "bf16": 2.4e12}  # FLOP of a drawn layer


def draw(rng):
    kind = rng.choices(["linear", "mlp_up", "attn", "head", "lora", "norm", "step"],
                       [3, 1, 3, 2, 1, 1, 1])[0]
    while True:
        if kind in ("linear", "mlp_up", "lora"):
            form = rng.choice({"linear": ["fp32", "mixed", "bf16", "bf16"],
                               "mlp_up": ["fp32", "bf16"], "lora": ["fp32", "mixed"]}[kind])
            c = dict(kind=kind, form=form, t=_log(rng, 16, 8192), n=_width(rng, 256, 12288),
                     k=_width(rng, 256, 12288))
            if kind == "lora":
                c["r"] = rng.choice([4, 8, 16, 32, 64])
        elif kind == "attn":
            form = rng.choice(["fp32", "bf16", "bf16"])
            kv = rng.choice([2, 4, 8])
            n = _log(rng, 16, 4096 if form == "bf16" else 1024)
            if rng.random() < 0.5:
                n = max(16, (n + 32) // 64 * 64)
            c = dict(kind=kind, form=form, b=rng.choice([1, 1, 2, 4]), n=n,
                     heads=kv * rng.choice([1, 2, 4]), kv_heads=kv,
                     head_dim=rng.choice([64, 128, 128]), causal=rng.random() < 0.85)
        elif kind == "head":
            reg = rng.random() < 0.3
            c = dict(kind=kind, form=rng.choice(["fp32", "mixed"]), t=_log(rng, 16, 4096),
                     vocab=_log(rng, 4096, 151936), dim=_width(rng, 256, 2560),
                     z_loss=1e-4 if reg else 0.0, smoothing=0.1 if reg else 0.0)
            if rng.random() < 0.6:
                c["vocab"] = (c["vocab"] + 63) // 64 * 64
        elif kind == "norm":
            c = dict(kind=kind, form="fp32", t=_log(rng, 16, 16384), dim=_width(rng, 64, 4096))
        else:
            kv = rng.choice([2, 4])
            c = _step("", form=rng.choice(["fp32", "bf16"]), layers=rng.randint(1, 3),
                      dim=rng.choice([128, 256, 512]), heads=kv * rng.choice([1, 2]), kv_heads=kv,
                      head_dim=rng.choice([64, 128]), ff=64 * rng.randint(4, 24),
                      vocab=_log(rng, 1000, 16384), n_pos=_log(rng, 16, 512),
                      n_seqs=rng.choice([1, 1, 2, 4]), qk_norm=rng.random() < 0.7,
                      tied=rng.random() < 0.5)
            del c["name"]
        if work(c)["flops"] <= _CAP[c["form"]]:
            return c


# ── what a pass cannot do without ────────────────────────────────────────

def _causal_pairs(n, causal):
    return n * (n + 1) / 2 if causal else float(n) * n


def work(c):
    kind, e = c["kind"], 2 if c["form"] == "bf16" else 4
    if kind == "linear":
        t, n, k = c["t"], c["n"], c["k"]
        return {"bytes": e * (t * k + n * k + t * n) + 4 * (t * n + t * k + n * k),
                "flops": 6.0 * t * n * k}
    if kind == "mlp_up":
        t, f, k = c["t"], c["n"], c["k"]
        return {"bytes": e * (t * k + 2 * f * k) + 4 * t * 2 * f + e * t * f,
                "flops": 4.0 * t * f * k}
    if kind == "attn":
        q, kv = c["b"] * c["n"] * c["heads"] * c["head_dim"], c["b"] * c["n"] * c["kv_heads"] * c["head_dim"]
        pairs = c["b"] * c["heads"] * _causal_pairs(c["n"], c["causal"])
        # in: q, k, v, dO; out: O, LSE, dQ, dK, dV
        return {"bytes": e * (2 * q + 2 * kv) + 4 * (2 * q + 2 * kv + c["b"] * c["n"] * c["heads"]),
                "flops": 14.0 * pairs * c["head_dim"]}
    if kind == "head":
        t, v, d = c["t"], c["vocab"], c["dim"]
        return {"bytes": 4.0 * (2 * t * d + 2 * v * d + 3 * t), "flops": 6.0 * t * v * d}
    if kind == "lora":
        t, n, k, r = c["t"], c["n"], c["k"], c["r"]
        return {"bytes": 4.0 * (2 * t * k + 2 * t * n + n * k + 2 * r * (n + k) + t * r),
                "flops": 4.0 * t * n * k + 6.0 * t * r * (n + k)}
    if kind == "norm":
        return {"bytes": 4.0 * (4 * c["t"] * c["dim"] + 2 * c["dim"]), "flops": 16.0 * c["t"] * c["dim"]}
    t, d, f, v = c["n_pos"] * c["n_seqs"], c["dim"], c["ff"], c["vocab"]
    qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    mats = c["layers"] * (d * (qd + 2 * kvd) + qd * d + 3 * d * f)
    params = mats + (1 if c["tied"] else 2) * v * d
    attn = 14.0 * c["layers"] * c["heads"] * c["head_dim"] * c["n_seqs"] * _causal_pairs(c["n_pos"], True)
    # Adam reads param, gradient and both moments and writes param and moments
    return {"bytes": 28.0 * params, "flops": 6.0 * t * mats + 6.0 * t * v * d + attn}


# ── the library beside torch ─────────────────────────────────────────────

@functools.lru_cache(None)
def _load():
    """The framework's library in a process that has torch in it already.

    torch brings its own HIP runtime, and where that is older than the one the library was linked
    with, the loader refuses the library for the one newer symbol that it names, hipStreamGetId
    (a process that loads the library first runs both on the newer runtime).  There, a private copy
    is loaded in which that reference is hipStreamIsCapturing's: the same arguments, and it writes
    0, one identity for all streams, which holds here because every call uses one stream."""
    from valkyr_amd import _lib, lib

    try:
        return lib()
    except OSError:
        with open(_lib.LIB_PATH, "rb") as f:
            b = bytearray(f.read())
    shoff, = struct.unpack_from("<Q", b, 40)
    sections = {}
    for i in range(struct.unpack_from("<H", b, 60)[0]):
        kind, off, size = (struct.unpack_from("<IIQQQQ", b, shoff + 64 * i)[k] for k in (1, 4, 5))
        sections.setdefault(kind, (off, size))  # the first string table is .dynstr
    (sym, size), (text, _), (ver, _), (need, _) = (sections[k] for k in (11, 3, 0x6FFFFFFF, 0x6FFFFFFE))
    at = {}
    for i in range(size // 24):
        name = text + struct.unpack_from("<I", b, sym + 24 * i)[0]
        at[bytes(b[name:b.index(0, name)]).decode()] = i
    new, old = at["hipStreamGetId"], at["hipStreamIsCapturing"]
    dropped, = struct.unpack_from("<H", b, ver + 2 * new)
    b[sym + 24 * new:sym + 24 * new + 4] = b[sym + 24 * old:sym + 24 * old + 4]
    b[ver + 2 * new:ver + 2 * new + 2] = b[ver + 2 * old:ver + 2 * old + 2]
    while True:  # the version it asked for becomes one that may be missing
        _, count, _, aux, step = struct.unpack_from("<HHIII", b, need)
        entry = need + aux
        for _ in range(count):
            _, flags, index, _, more = struct.unpack_from("<IHHII", b, entry)
            if index == dropped:
                struct.pack_into("<H", b, entry + 4, flags | 2)
            entry += more
        if not step:
            break
        need += step
    with tempfile.NamedTemporaryFile(suffix=".so") as f:
        f.write(b)
        f.flush()
        path, _lib.LIB_PATH = _lib.LIB_PATH, f.name
        try:
            return lib()
        finally:
            _lib.LIB_PATH = path


# ── inputs ───────────────────────────────────────────────────────────────

class _Stream:
    """torch's current stream, as the entry points take one."""

    @property
    def handle(self):
        return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _normal(g, shape, std=1.0, dtype=F32):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _new(*shape, dtype=F32):
    return torch.empty(shape, device="cuda", dtype=dtype)


class _DeviceArray:
    """A runner's device array as torch takes it (no copy); the tensor made of it keeps this object,
    and so the runner that owns the memory."""

    def __init__(self, owner, addr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (addr, False),
                                         "version": 2}


def _step_weights(c, g):
    """The weights of a small decoder, on the host, as Runner takes them."""
    d, f, v = c["dim"], c["ff"], c["vocab"]
    qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]

    def mat(*shape):
        return _normal(g, shape, 0.02).cpu().numpy()

    def gain(n):
        return (1.0 + _normal(g, (n,), 0.02)).cpu().numpy()

    layers = []
    for _ in range(c["layers"]):
        w = dict(w_n1=gain(d), w_q=mat(qd, d), w_k=mat(kvd, d), w_v=mat(kvd, d), w_o=mat(d, qd),
                 w_n2=gain(d), w_gate=mat(f, d), w_up=mat(f, d), w_down=mat(d, f))
        if c["qk_norm"]:
            w.update(w_q_norm=gain(c["head_dim"]), w_k_norm=gain(c["head_dim"]))
        layers.append(w)
    out = dict(embed=mat(v, d), final_norm=gain(d), layers=layers)
    if not c["tied"]:
        out["lm_head"] = mat(v, d)
    return out


def _small(c):
    return work(c)["bytes"] < 2e9


def _step_ids(c, g):
    t = c["n_pos"] * c["n_seqs"]
    ids = torch.randint(0, c["vocab"], (2, t), generator=g, device="cuda").cpu().numpy().astype("uint32")
    return ids[0], ids[1]


def _inputs(c, seed):
    """The numbers a case starts from, made from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = BF16 if c["form"] == "bf16" else F32
    kind = c["kind"]
    if kind == "linear":
        return dict(x=_normal(g, (c["t"], c["k"]), 1.0, dt), w=_normal(g, (c["n"], c["k"]), 0.02, dt),
                    dy=_normal(g, (c["t"], c["n"]), 0.1, dt))
    if kind == "mlp_up":
        return dict(x=_normal(g, (c["t"], c["k"]), 1.0, dt), w=_normal(g, (2 * c["n"], c["k"]), 0.02, dt))
    if kind == "attn":
        q, kv = (c["b"] * c["n"], c["heads"], c["head_dim"]), (c["b"] * c["n"], c["kv_heads"], c["head_dim"])
        return dict(q=_normal(g, q, 1.0, dt), k=_normal(g, kv, 1.0, dt), v=_normal(g, kv, 1.0, dt),
                    dout=_normal(g, q, 0.1, dt))
    if kind == "head":
        return dict(h=_normal(g, (c["t"], c["dim"])), w=_normal(g, (c["vocab"], c["dim"]), 0.02),
                    ids=torch.randint(0, c["vocab"], (c["t"],), generator=g, device="cuda", dtype=torch.int32))
    if kind == "lora":
        return dict(x=_normal(g, (c["t"], c["k"])), w=_normal(g, (c["n"], c["k"]), 0.02),
                    a=_normal(g, (c["r"], c["k"]), 0.02), b=_normal(g, (c["n"], c["r"]), 0.02),
                    dy=_normal(g, (c["t"], c["n"]), 0.1))
    if kind == "norm":
        return dict(x=_normal(g, (c["t"], c["dim"])), w=1.0 + _normal(g, (c["dim"],), 0.02),
                    dy=_normal(g, (c["t"], c["dim"]), 0.1))
    ids, targets = _step_ids(c, g)
    return dict(ids=ids, targets=targets, weights=_step_weights(c, g) if _small(c) else None)


def _grad_views(r, c):
    """Views of the runner's gradients: one for each run of neighbours within the embedding, the
    head and final norm, and each layer."""
    from valkyr_amd import runner as R

    per_layer = range(11) if c["qk_norm"] else range(9)
    groups = [[(-1, R.EMBED)], [(-1, R.FINAL_NORM)]] + ([] if c["tied"] else [[(-1, R.LM_HEAD)]])
    groups += [[(l, w) for w in per_layer] for l in range(c["layers"])]
    views = []
    for group in groups:
        spans = sorted(r.device_ptr(R.GRAD, l, w) for l, w in group)
        runs = [list(spans[0])]
        for p, n in spans[1:]:
            if runs[-1][0] + 4 * runs[-1][1] == p:
                runs[-1][1] += n
            else:
                runs.append([p, n])
        views += [torch.as_tensor(_DeviceArray(r, p, n), device="cuda") for p, n in runs]
    return views


def prepare(case, seed):
    from valkyr_amd import Runner, make_config
    from valkyr_amd import kernels as K

    _load()
    c, s = case, _inputs(case, seed)
    kind, st = c["kind"], _Stream()
    prec = 0 if c["form"] == "fp32" else 1
    s.update(case=c, stream=st, prec=prec, K=K)
    if kind == "linear":
        s.update(y=_new(c["t"], c["n"]), dx=_new(c["t"], c["k"]), dw=_new(c["n"], c["k"]))
    elif kind == "mlp_up":
        s.update(gu=_new(c["t"], 2 * c["n"]),
                 gated=_new(c["t"], c["n"], dtype=BF16 if c["form"] == "bf16" else F32))
    elif kind == "attn":
        t, h, kv, hd = c["b"] * c["n"], c["heads"], c["kv_heads"], c["head_dim"]
        p = K.attn_params(c["n"], c["n"], h, kv, hd, c["causal"], c["b"], K.BF16 if prec else K.F32)
        s.update(p=p, o=_new(t, h, hd), lse=_new(t, h), d=_new(t, h), dq=_new(t, h, hd),
                 dk=_new(t, kv, hd), dv=_new(t, kv, hd), o16=_new(t, h, hd, dtype=BF16) if prec else None,
                 ws=torch.empty(max(16, K.fa_backward_workspace_bytes(p)), device="cuda", dtype=torch.uint8))
    elif kind == "head":
        s.update(p=K.cce_params(c["t"], c["vocab"], c["dim"], c["z_loss"], c["smoothing"], prec),
                 lse=_new(c["t"]), rows=_new(c["t"]), mean=_new(1), dh=_new(c["t"], c["dim"]),
                 dw=_new(c["vocab"], c["dim"]))
    elif kind == "lora":
        s.update(y=_new(c["t"], c["n"]), inter=_new(c["t"], c["r"]), dx=_new(c["t"], c["k"]),
                 da=_new(c["r"], c["k"]), db=_new(c["n"], c["r"]))
    elif kind == "norm":
        s.update(y=_new(c["t"], c["dim"]), dx=_new(c["t"], c["dim"]), dw=_new(c["dim"]))
    else:
        cfg = make_config(dim=c["dim"], n_heads=c["heads"], n_kv_heads=c["kv_heads"],
                          head_dim=c["head_dim"], ff_dim=c["ff"], n_pos=c["n_pos"], n_seqs=c["n_seqs"],
                          n_layers=c["layers"], vocab_size=c["vocab"], rms_eps=c["eps"], causal=1,
                          rotary_dim=c["head_dim"], rope_theta=c["theta"], qk_norm=int(c["qk_norm"]),
                          lr=1e-4, tied_embeddings=int(c["tied"]), precision=prec)
        r = Runner(cfg, s.pop("weights"))
        if not _small(c):
            r.init_random(seed=seed, std=0.02)
        s.update(runner=r, grads=_grad_views(r, c))
    return s


def run(s):
    c, K, st = s["case"], s["K"], s["stream"]
    kind, prec = c["kind"], s["prec"]
    if kind == "step":
        r = s["runner"]
        r.step(s["ids"], s["targets"])
        return {"loss": r.last_loss(), "grads": s["grads"]}
    ptr = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    if kind == "linear":
        t, n, k = c["t"], c["n"], c["k"]
        if c["form"] == "bf16":
            K.matmul_nt_bf16(ptr["x"], ptr["w"], ptr["y"], t, n, k, stream=st)
            K.linear_backward_dx_bf16(ptr["dy"], ptr["w"], ptr["dx"], t, n, k, stream=st)
            K.linear_backward_dw_bf16(ptr["dy"], ptr["x"], ptr["dw"], t, n, k, stream=st)
        else:
            K.matmul_nt(ptr["x"], ptr["w"], ptr["y"], t, n, k, prec, stream=st)
            K.linear_backward_dx(ptr["dy"], ptr["w"], ptr["dx"], t, n, k, prec, stream=st)
            K.linear_backward_dw(ptr["dy"], ptr["x"], ptr["dw"], t, n, k, prec, stream=st)
        return [s["y"], s["dx"], s["dw"]]
    if kind == "mlp_up":
        f = K.gate_up_swiglu_bf16 if c["form"] == "bf16" else K.gate_up_swiglu
        f(ptr["x"], ptr["w"], ptr["gu"], ptr["gated"], c["t"], c["n"], c["k"], stream=st)
        return [s["gu"], s["gated"]]
    if kind == "attn":
        p, io = s["p"], [ptr[k] for k in ("q", "k", "v")]
        out = [ptr[k] for k in ("dq", "dk", "dv")]
        K.fa_forward(p, *io, ptr["o"], ptr["lse"], stream=st)
        if prec:
            K.cast_f32_to_bf16(ptr["o"], ptr["o16"], s["o"].numel(), stream=st)
            K.fa_backward_from_o(p, *io, ptr["o16"], ptr["dout"], ptr["lse"], ptr["d"], *out,
                                 workspace=ptr["ws"], stream=st)
        else:
            K.fa_bw_d(p, ptr["o"], ptr["dout"], ptr["d"], stream=st)
            K.fa_backward(p, *io, ptr["dout"], ptr["lse"], ptr["d"], *out, workspace=ptr["ws"], stream=st)
        return [s["o"], s["lse"], s["dq"], s["dk"], s["dv"]]
    if kind == "head":
        p = s["p"]
        K.cce_forward(p, ptr["h"], ptr["w"], ptr["ids"], ptr["lse"], ptr["rows"], ptr["mean"], stream=st)
        K.cce_backward(p, ptr["h"], ptr["w"], ptr["ids"], ptr["lse"], ptr["dh"], ptr["dw"], stream=st)
        return [s["lse"], s["rows"], s["mean"], s["dh"], s["dw"]]
    if kind == "lora":
        dims = (c["t"], c["n"], c["k"], c["r"], 2.0, prec)
        K.lora_forward(ptr["x"], ptr["w"], ptr["a"], ptr["b"], ptr["y"], ptr["inter"], *dims, stream=st)
        K.lora_backward(ptr["dy"], ptr["x"], ptr["w"], ptr["a"], ptr["b"], ptr["inter"], ptr["dx"],
                        ptr["da"], ptr["db"], *dims, stream=st)
        return [s["y"], s["inter"], s["dx"], s["da"], s["db"]]
    K.rmsnorm_forward(ptr["x"], ptr["w"], ptr["y"], c["t"], c["dim"], 1e-6, stream=st)
    K.rmsnorm_backward(ptr["dy"], ptr["x"], ptr["w"], ptr["dx"], ptr["dw"], c["t"], c["dim"], 1e-6, stream=st)
    return [s["y"], s["dx"], s["dw"]]


# About four times the error against `exact` that was measured over the ranges.  The sums of fp32
# and of bf16-operand products are fp32 (the head's dh is one over the whole vocabulary); "mixed"
# rounds operands to bf16; attention in bf16 rounds P and dS, and the bf16 gated activation is
# itself stored in 16 bits.  In the bf16 step a change of 1e-6 in one gain moves the gradients
# by 0.005 to 0.009, and they are 0.015 from those of fp32 operands.
def tolerance(c):
    kind, form = c["kind"], c["form"]
    if kind == "step" and form == "bf16":
        return {"rel": 3e-2}
    if form == "mixed" or (form == "bf16" and kind in ("attn", "mlp_up")):
        return {"rel": 1e-2}
    return {"rel": 3e-5 if kind == "head" else 1e-5}


# ── the same in 64 bits ──────────────────────────────────────────────────

def _rms64(x, w, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _attend64(q, k, v, causal):
    """[b, n, h, hd] each; returns O and the log-sum-exp."""
    n, g = q.shape[1], q.shape[2] // k.shape[2]
    k, v = k.repeat_interleave(g, 2), v.repeat_interleave(g, 2)
    s = torch.matmul(q.transpose(1, 2), k.permute(0, 2, 3, 1).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    lse = torch.logsumexp(s, -1)
    o = torch.matmul(torch.exp(s - lse[..., None]), v.transpose(1, 2).contiguous())
    return o.transpose(1, 2), lse.transpose(1, 2)


def _decoder_grads64(c, s):
    """Loss and gradients of the decoder, in the layout of run()'s views."""
    w = s["weights"]
    up = lambda a: torch.tensor(a, device="cuda", dtype=torch.float64, requires_grad=True)  # noqa: E731
    embed, final = up(w["embed"]), up(w["final_norm"])
    head = embed if c["tied"] else up(w["lm_head"])
    layers = [{k: up(a) for k, a in lw.items()} for lw in w["layers"]]
    b, n, hd = c["n_seqs"], c["n_pos"], c["head_dim"]
    ids = torch.tensor(s["ids"].astype("int64"), device="cuda")
    targets = torch.tensor(s["targets"].astype("int64"), device="cuda")
    j = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    ang = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * c["theta"] ** (-2.0 * j / hd)
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]

    def rope(x):
        p, q = x.split(hd // 2, -1)
        return torch.cat([p * cos - q * sin, p * sin + q * cos], -1)

    x = embed[ids]
    for lw in layers:
        h = _rms64(x, lw["w_n1"], c["eps"])
        q, k, v = ((h @ lw[m].T).view(b, n, -1, hd) for m in ("w_q", "w_k", "w_v"))
        if c["qk_norm"]:
            q, k = _rms64(q, lw["w_q_norm"], c["eps"]), _rms64(k, lw["w_k_norm"], c["eps"])
        o = _attend64(rope(q), rope(k), v, True)[0].reshape(b * n, -1)
        x = x + o @ lw["w_o"].T
        h = _rms64(x, lw["w_n2"], c["eps"])
        x = x + (torch.nn.functional.silu(h @ lw["w_gate"].T) * (h @ lw["w_up"].T)) @ lw["w_down"].T
    logits = _rms64(x, final, c["eps"]) @ head.T
    loss = torch.nn.functional.cross_entropy(logits, targets)
    loss.backward()
    return loss, embed, final, head, layers


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "step":
        if not _small(c):
            return None
        s = _inputs(c, seed)
        loss, embed, final, head, layers = _decoder_grads64(c, s)
        order = ["w_n1", "w_q", "w_k", "w_v", "w_o", "w_n2", "w_gate", "w_up", "w_down"]
        order += ["w_q_norm", "w_k_norm"] if c["qk_norm"] else []
        groups = [[embed], [final]] + ([] if c["tied"] else [[head]])
        groups += [[lw[k] for k in order] for lw in layers]
        # neighbours are returned as one view where every tensor is whole 256-byte blocks
        return {"loss": float(loss.detach()), "grads": [torch.cat([t.grad.reshape(-1) for t in g]) for g in groups]}
    with torch.no_grad():
        s = {k: v.double() if isinstance(v, torch.Tensor) and v.is_floating_point() else v
             for k, v in _inputs(c, seed).items()}
        if kind == "linear":
            return [s["x"] @ s["w"].T, s["dy"] @ s["w"], s["dy"].T @ s["x"]]
        if kind == "mlp_up":
            gu = s["x"] @ s["w"].T
            return [gu, torch.nn.functional.silu(gu[:, :c["n"]]) * gu[:, c["n"]:]]
        if kind == "attn":
            b, n, g = c["b"], c["n"], c["heads"] // c["kv_heads"]
            parts = []
            for i in range(b):  # one sequence at a time: the scores are in 64 bits
                q, k, v, do = (s[m].view(b, n, -1, c["head_dim"])[i:i + 1] for m in ("q", "k", "v", "dout"))
                with torch.enable_grad():
                    q, k, v = (t.clone().requires_grad_() for t in (q, k, v))
                    o, lse = _attend64(q, k, v, c["causal"])
                    grads = torch.autograd.grad(o, (q, k, v), do)
                parts.append([t.detach()[0] for t in (o, lse, *grads)])
            return [torch.cat(p) for p in zip(*parts)]
        if kind == "head":
            t = torch.arange(c["t"], device="cuda")
            ids, z = s["ids"].long(), s["h"] @ s["w"].T
            lse = torch.logsumexp(z, 1)
            rows = lse - (1 - c["smoothing"]) * z[t, ids] - c["smoothing"] * z.mean(1) + c["z_loss"] * lse * lse
            dz = torch.exp(z - lse[:, None]) * (1 + 2 * c["z_loss"] * lse)[:, None] - c["smoothing"] / c["vocab"]
            dz[t, ids] -= 1 - c["smoothing"]
            dz /= c["t"]
            return [lse, rows, rows.mean()[None], dz @ s["w"], dz.T @ s["h"]]
        if kind == "lora":
            inter, dyb = s["x"] @ s["a"].T, s["dy"] @ s["b"]
            return [s["x"] @ s["w"].T + 2.0 * inter @ s["b"].T, inter, s["dy"] @ s["w"] + 2.0 * dyb @ s["a"],
                    2.0 * dyb.T @ s["x"], 2.0 * s["dy"].T @ inter]
        r = torch.rsqrt((s["x"] * s["x"]).mean(1, keepdim=True) + 1e-6)
        xh, gy = s["x"] * r, s["dy"] * s["w"]
        return [xh * s["w"], r * (gy - xh * (gy * xh).mean(1, keepdim=True)), (s["dy"] * xh).sum(0)]
