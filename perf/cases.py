"""The work that a user of this library has it do, as timed cases.

Four paths, each through the entry points a program calls:

* ``mv``    -- one packed batch-1 matvec (``DeviceOps.matvec_packed``), the
  call a decode step makes per weight matrix;
* ``token`` -- every weight matrix of one decode step, layer after layer
  (``matvec2_packed`` for q|k with v, ``matvec_packed`` for the rest), the
  stream the benchmark times;
* ``mm``    -- a packed product of several vectors (``DeviceOps.matmul_packed``,
  or with ``host`` the drop-in ABI over host buffers, ``LLMGpu.matmul``):
  batched decode lanes at 2 to 64 vectors, a prompt above that;
* ``moe``   -- one mixture-of-experts layer: router and grouped experts
  (``DeviceOps.route`` and ``moe_experts_packed``) for one token, for decode
  lanes and for a prompt.

Weights follow the benchmark recipe (random codes, f16 scales |N(0, 2e-3)|);
activations are N(0, 1), as behind an RMS norm.  Weights are packed once in
``prepare``, as a program does at load time.
"""
import math

import torch

import aspida_amd as aa
from aspida_amd import synth

KIND = {name: k for k, name in aa.KIND_NAMES.items()}


MOE_LAYER = {"dim": 2048, "inter": 768, "experts": 128, "top_k": 8, "gu_kind": "Q4_K", "down_kind": "Q6_K",
             "gated": True}


def listed():
    return [
        # The attention output projection of a 4096-wide decoder, one token:
        # the smallest call a decode step makes.
        {"name": "mv_q4k_4096x4096", "path": "mv", "kind": "Q4_K", "out": 4096, "in": 4096},
        # An FFN up projection in the 3-bit format, one token.
        {"name": "mv_q3k_14336x4096", "path": "mv", "kind": "Q3_K", "out": 14336, "in": 4096},
        # One token of the Llama-3-8B Q4_K_M weight stream (32 layers and the head).
        {"name": "token_8b_q4km", "path": "token", "hidden": 4096, "kv": 1024, "ffn": 14336, "vocab": 128256,
         "layers": 32},
        # Eight decode lanes on the FFN up projection.
        {"name": "mm_q4k_14336x4096_b8", "path": "mm", "kind": "Q4_K", "out": 14336, "in": 4096, "batch": 8,
         "host": False},
        # Sixteen decode lanes on a 5-bit model's FFN up projection.
        {"name": "mm_q5k_14336x4096_b16", "path": "mm", "kind": "Q5_K", "out": 14336, "in": 4096, "batch": 16,
         "host": False},
        # A batch of 64 on the FFN down projection, which Q4_K_M keeps in Q6_K.
        {"name": "mm_q6k_4096x14336_b64", "path": "mm", "kind": "Q6_K", "out": 4096, "in": 14336, "batch": 64,
         "host": False},
        # A 512-token prompt chunk through the stacked gate|up projection.
        {"name": "mm_q4k_28672x4096_b512", "path": "mm", "kind": "Q4_K", "out": 28672, "in": 4096, "batch": 512,
         "host": False},
        # A prompt of odd length on a matrix whose rows do not fill a tile.
        {"name": "mm_q6k_5001x3584_b333", "path": "mm", "kind": "Q6_K", "out": 5001, "in": 3584, "batch": 333,
         "host": False},
        # The drop-in ABI as the host program calls it for a prompt: host
        # buffers in and out, 32 vectors (the host's own batch limit).
        {"name": "host_mm_q4k_4096x4096_b32", "path": "mm", "kind": "Q4_K", "out": 4096, "in": 4096, "batch": 32,
         "host": True},
        # The Qwen3-MoE layer (128 experts and a shared one, top 8): one
        # token, 32 decode lanes, a prompt chunk of 1024.
        {"name": "moe_t1", "path": "moe", "tokens": 1, **MOE_LAYER},
        {"name": "moe_t32", "path": "moe", "tokens": 32, **MOE_LAYER},
        {"name": "moe_t1024", "path": "moe", "tokens": 1024, **MOE_LAYER},
    ]


# Products of the listed range stay below the gate|up prompt chunk.
MM_MAX = 28672 * 4096 * 512


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["mv", "mv", "mm", "mm", "mm", "mm", "mm", "host", "moe", "moe", "moe", "token"])
    if path == "mv":
        return {"path": "mv", "kind": rng.choice(sorted(KIND)), "out": _log_int(rng, 1024, 65536),
                "in": 256 * _log_int(rng, 4, 64)}
    if path == "mm":
        c = {"path": "mm", "kind": rng.choice(sorted(KIND)), "out": _log_int(rng, 1024, 28672),
             "in": 256 * _log_int(rng, 4, 64), "batch": _log_int(rng, 2, 1024), "host": False}
        c["batch"] = max(2, min(c["batch"], MM_MAX // (c["out"] * c["in"])))
        return c
    if path == "host":
        return {"path": "mm", "kind": rng.choice(sorted(KIND)), "out": _log_int(rng, 1024, 14336),
                "in": 256 * _log_int(rng, 4, 32), "batch": rng.randint(1, 64), "host": True}
    if path == "token":
        hidden = 256 * rng.randint(8, 16)
        return {"path": "token", "hidden": hidden, "kv": rng.choice([512, 1024]), "ffn": 256 * rng.randint(20, 56),
                "vocab": rng.randint(32000, 128256), "layers": rng.randint(4, 32)}
    n_exp = rng.choice([16, 32, 60, 64, 128])
    gu, down = rng.choice([("Q4_K", "Q6_K"), ("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q6_K", "Q6_K"), ("Q5_K", "Q6_K"),
                           ("Q8_0", "Q8_0")])
    return {"path": "moe", "tokens": _log_int(rng, 1, 1024), "dim": 256 * rng.randint(4, 8),
            "inter": 256 * rng.randint(1, 3), "experts": n_exp, "top_k": rng.randint(2, 8), "gu_kind": gu,
            "down_kind": down, "gated": rng.random() < 0.75}


# ---- inputs ----------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _sp():
    return torch.cuda.current_stream().cuda_stream


def _raw(kind, out, inp, g, n=1):
    """n ggml matrices [out][inp] of random super-blocks, uint8 on the device."""
    return synth.blocks_torch(kind, n * out * (inp // 256), generator=g)


def _packed(dev, kind, out, inp, g, n=1):
    src = _raw(kind, out, inp, g, n)
    dst = torch.empty(n * dev.packed_bytes(kind, inp, out), dtype=torch.uint8, device="cuda")
    if n == 1:
        dev.pack(kind, src.data_ptr(), inp, out, dst.data_ptr(), _sp())
    else:
        dev.pack_experts(kind, src.data_ptr(), src.numel() // n, inp, out, n, dst.data_ptr(), _sp())
    return dst


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", dtype=torch.float32, generator=g)


def _out(*shape, dtype=torch.float32):
    return torch.empty(*shape, device="cuda", dtype=dtype)


def _token_mats(c):
    """(kind, out, in) of a token's matrices: per layer q|k and v (which share
    a launch), o, gate|up and down, then the head."""
    h, q4, q6 = c["hidden"], KIND["Q4_K"], KIND["Q6_K"]
    layer = [(q4, h + c["kv"], h), (q6, c["kv"], h), (q4, h, h), (q4, 2 * c["ffn"], h), (q6, h, c["ffn"])]
    return layer * c["layers"] + [(q6, c["vocab"], h)]


class HostWeight:
    """A host weight and its HBM mirror, dropped with the object."""

    def __init__(self, gpu, data):
        self.gpu, self.data = gpu, data

    def __del__(self):
        self.gpu.free_weight(self.data)


def prepare(case, seed):
    g = _generator(seed)
    dev = aa.DeviceOps()
    st = {"case": case, "dev": dev}
    path = case["path"]
    if path == "mv":
        kind, out, inp = KIND[case["kind"]], case["out"], case["in"]
        st.update(kind=kind, w=_packed(dev, kind, out, inp, g), x=_randn(g, inp), y=_out(out))
    elif path == "token":
        st["x"] = {n: _randn(g, n) for n in sorted({case["hidden"], case["ffn"]})}
        # Every launch's output is its own part of one buffer.
        mats = _token_mats(case)
        st["y"] = _out(sum(o for _, o, _ in mats))
        parts = st["y"].split([o for _, o, _ in mats])
        st["mats"] = [(k, _packed(dev, k, o, i, g), o, i, y) for (k, o, i), y in zip(mats, parts)]
    elif path == "mm":
        kind, out, inp, batch = KIND[case["kind"]], case["out"], case["in"], case["batch"]
        st["kind"] = kind
        if case["host"]:
            st["gpu"] = aa.LLMGpu()
            st["w"] = HostWeight(st["gpu"], _raw(kind, out, inp, g).cpu().numpy())
            st["x"] = _randn(g, batch, inp).cpu().numpy()
        else:
            st.update(w=_packed(dev, kind, out, inp, g), x=_randn(g, batch, inp), y=_out(batch, out))
    else:
        T, d, i, n, k = (case[f] for f in ("tokens", "dim", "inter", "experts", "top_k"))
        gu, dn = KIND[case["gu_kind"]], KIND[case["down_kind"]]
        st.update(gu=gu, dn=dn, router=_randn(g, n, d) * 0.02, sgi=_randn(g, d) * 0.02,
                  gate=_packed(dev, gu, i, d, g, n), up=_packed(dev, gu, i, d, g, n),
                  down=_packed(dev, dn, d, i, g, n), shg=_packed(dev, gu, i, d, g), shu=_packed(dev, gu, i, d, g),
                  shd=_packed(dev, dn, d, i, g), x=_randn(g, T, d), logits=_out(T, n),
                  idx=_out(T, k, dtype=torch.int32), tw=_out(T, k), y=_out(T, d),
                  work=_out(dev.moe_packed_work_bytes(T, d, i, k), dtype=torch.uint8))
    return st


def _matvec(dev, mat, x, sp):
    k, w, o, i, y = mat
    dev.matvec_packed(k, w.data_ptr(), i, o, x[i].data_ptr(), y.data_ptr(), sp)


def run(st):
    c, dev, sp = st["case"], st["dev"], _sp()
    if c["path"] == "mv":
        dev.matvec_packed(st["kind"], st["w"].data_ptr(), c["in"], c["out"], st["x"].data_ptr(), st["y"].data_ptr(),
                          sp)
        return st["y"]
    if c["path"] == "token":
        mats = iter(st["mats"])
        for _ in range(c["layers"]):
            (ka, wa, oa, inp, ya), (kb, wb, ob, _, yb) = next(mats), next(mats)
            dev.matvec2_packed(ka, wa.data_ptr(), oa, ya.data_ptr(), kb, wb.data_ptr(), ob, yb.data_ptr(), inp,
                               st["x"][inp].data_ptr(), sp)
            for _ in range(3):
                _matvec(dev, next(mats), st["x"], sp)
        _matvec(dev, next(mats), st["x"], sp)
        return st["y"]
    if c["path"] == "mm":
        if c["host"]:
            return st["gpu"].matmul(st["w"].data, st["kind"], c["in"], c["out"], st["x"])
        dev.matmul_packed(st["kind"], st["w"].data_ptr(), c["in"], c["out"], c["batch"], st["x"].data_ptr(),
                          st["y"].data_ptr(), sp)
        return st["y"]
    T, d, i, n, k = (c[f] for f in ("tokens", "dim", "inter", "experts", "top_k"))
    p = {f: st[f].data_ptr() for f in ("router", "sgi", "gate", "up", "down", "shg", "shu", "shd", "x", "logits",
                                       "idx", "tw", "y", "work")}
    dev.route(p["router"], n, d, T, k, p["x"], p["logits"], p["idx"], p["tw"], sp)
    dev.moe_experts_packed(p["x"], T, d, k, i, n, p["idx"], p["tw"], p["gate"], p["up"], st["gu"], p["down"],
                           st["dn"], p["shg"], p["shu"], p["shd"], p["sgi"] if c["gated"] else 0, p["work"],
                           p["y"], sp)
    return [st["logits"], st["idx"], st["tw"], st["y"]]


# ---- what a pass cannot do without -----------------------------------------

def work(case):
    path = case["path"]
    if path in ("mv", "mm"):
        o, i, b = case["out"], case["in"], case.get("batch", 1)
        return {"bytes": aa.weight_bytes(KIND[case["kind"]], i, o) + 4 * b * (i + o), "flops": 2 * b * i * o}
    if path == "token":
        mats = _token_mats(case)
        return {"bytes": sum(aa.weight_bytes(k, i, o) + 4 * o for k, o, i in mats) +
                4 * (case["hidden"] + case["ffn"]), "flops": sum(2 * i * o for _, o, i in mats)}
    T, d, i, n, k = (case[f] for f in ("tokens", "dim", "inter", "experts", "top_k"))
    expert = 2 * aa.weight_bytes(KIND[case["gu_kind"]], d, i) + aa.weight_bytes(KIND[case["down_kind"]], i, d)
    # Distinct experts that T independent choices of k out of n reach on average.
    distinct = n * (1.0 - (1.0 - k / n) ** T)
    return {"bytes": int((distinct + 1) * expert + 4 * n * d + 4 * T * (2 * d + n + 2 * k)),
            "flops": 2 * T * (n * d + (k + 1) * 3 * d * i)}


def tolerance(case):
    # About four times the error measured against 64 bits.  Up to four vectors
    # run on the batch-1 kernels, whose matrix-core sums span quarters of a
    # super-block: 1e-5 for the 2- and 3-bit formats (their scale and min terms
    # cancel most), 2e-6 for the others.  Larger batches: 5e-7.  The MoE layer
    # chains two products, SwiGLU and the softmax weights: 2.4e-6.
    if case["path"] == "moe":
        return {"rel": 1e-5, "differ": 2e-3}
    if case["path"] == "mm" and case["batch"] > 4:
        return {"rel": 2e-6}
    return {"rel": 4e-5 if case.get("kind") in ("Q2_K", "Q3_K") else 1e-5}


# ---- the same in 64 bits ---------------------------------------------------

def _f16(b):
    """f64 of little-endian f16 bytes [..., 2]; Inf and NaN patterns read as 0."""
    v = b.contiguous().view(torch.float16).squeeze(-1).double()
    return torch.where(torch.isfinite(v), v, torch.zeros_like(v))


def _scale_min(sc):
    """The eight 6-bit (scale, min) pairs of Q4_K's and Q5_K's 12 bytes."""
    lo, mid, hi = sc[:, 0:4].int(), sc[:, 4:8].int(), sc[:, 8:12].int()
    s = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    m = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return s.double(), m.double()


def _decode(kind, b):
    """f64 [n][256] of super-block bytes [n][block]."""
    n = b.shape[0]
    name = aa.KIND_NAMES[kind]
    if name in ("Q4_K", "Q5_K"):
        s, m = _scale_min(b[:, 4:16])
        qs = b[:, -128:].int().view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32)
        if name == "Q5_K":
            sh = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 8, 1)
            q = q + (((b[:, 16:48].int().view(n, 1, 32) >> sh) & 1) << 4)
        w = _f16(b[:, 0:2]).view(n, 1, 1) * s.unsqueeze(2) * q - _f16(b[:, 2:4]).view(n, 1, 1) * m.unsqueeze(2)
    elif name == "Q6_K":
        ql, qh = b[:, 0:128].int().view(n, 2, 2, 32), b[:, 128:192].int().view(n, 2, 1, 32)
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int32).view(1, 1, 4, 1)
        q = torch.cat([ql & 15, ql >> 4], 2) + (((qh >> sh) & 3) << 4) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(n, 16, 1)
        w = _f16(b[:, 208:210]).view(n, 1, 1) * sc * q.reshape(n, 16, 16)
    elif name in ("Q3_K", "Q2_K"):
        q0 = 32 if name == "Q3_K" else 16
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int32).view(1, 1, 4, 1)
        q = ((b[:, q0:q0 + 64].int().view(n, 2, 1, 32) >> sh) & 3).view(n, 8, 32)
        if name == "Q3_K":
            bit = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 8, 1)
            q = q + 4 * ((b[:, 0:32].int().view(n, 1, 32) >> bit) & 1) - 4
            s = b[:, 96:108].int()
            lo = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
            hi = torch.cat([(s[:, 8:12] >> (2 * j)) & 3 for j in range(4)], 1)
            w = _f16(b[:, 108:110]).view(n, 1, 1) * (lo + 16 * hi - 32).double().view(n, 16, 1) * q.reshape(n, 16, 16)
        else:
            s = b[:, 0:16].int().view(n, 16, 1)
            w = _f16(b[:, 80:82]).view(n, 1, 1) * (s & 15) * q.reshape(n, 16, 16) - \
                _f16(b[:, 82:84]).view(n, 1, 1) * (s >> 4)
    else:
        blk = b.view(n, 8, 34)
        w = _f16(blk[:, :, 0:2]).unsqueeze(2) * blk[:, :, 2:].contiguous().view(torch.int8).double()
    return w.reshape(n, 256)


def _product(kind, raw, out, inp, x):
    """f64 x [b][inp] times the transpose of ggml bytes raw [out][inp]."""
    blocks = raw.view(out, inp // 256, aa.BLOCK_BYTES[kind])
    y = torch.empty(x.shape[0], out, dtype=torch.float64, device=x.device)
    step = max(1, (1 << 25) // inp)
    for r in range(0, out, step):
        part = blocks[r:r + step]
        w = _decode(kind, part.reshape(-1, part.shape[2])).view(part.shape[0], inp)
        y[:, r:r + step] = x @ w.t()
    return y


def _moe_exact(case, g):
    T, d, i, n, k = (case[f] for f in ("tokens", "dim", "inter", "experts", "top_k"))
    gu, dn = KIND[case["gu_kind"]], KIND[case["down_kind"]]
    router, sgi = (_randn(g, n, d) * 0.02).double(), (_randn(g, d) * 0.02).double()
    gate, up, down = _raw(gu, i, d, g, n), _raw(gu, i, d, g, n), _raw(dn, d, i, g, n)
    shared = _raw(gu, i, d, g), _raw(gu, i, d, g), _raw(dn, d, i, g)
    x = _randn(g, T, d).double()

    def ffn(wg, wu, wd, rows):
        a = _product(gu, wg, i, d, rows)
        h = a * torch.sigmoid(a) * _product(gu, wu, i, d, rows)
        return _product(dn, wd, d, i, h)

    logits = x @ router.t()
    p = torch.softmax(logits, 1)
    tw, idx = torch.sort(p, dim=1, descending=True, stable=True)
    tw, idx = tw[:, :k], idx[:, :k]
    tw = tw / tw.sum(1, keepdim=True)
    y = ffn(*shared, x)
    if case["gated"]:
        y = y * torch.sigmoid(x @ sgi).unsqueeze(1)
    gate, up, down = (t.view(n, -1) for t in (gate, up, down))
    for e in range(n):
        t, slot = torch.nonzero(idx == e, as_tuple=True)
        if t.numel():
            y[t] += tw[t, slot].unsqueeze(1) * ffn(gate[e], up[e], down[e], x[t])
    return [logits, None, tw, y]


def exact(case, seed):
    g = _generator(seed)
    if case["path"] == "mv":
        kind = KIND[case["kind"]]
        w = _raw(kind, case["out"], case["in"], g)
        return _product(kind, w, case["out"], case["in"], _randn(g, 1, case["in"]).double())[0]
    if case["path"] == "token":
        x = {n: _randn(g, 1, n).double() for n in sorted({case["hidden"], case["ffn"]})}
        return torch.cat([_product(k, _raw(k, o, i, g), o, i, x[i])[0] for k, o, i in _token_mats(case)])
    if case["path"] == "mm":
        kind = KIND[case["kind"]]
        w = _raw(kind, case["out"], case["in"], g)
        y = _product(kind, w, case["out"], case["in"], _randn(g, case["batch"], case["in"]).double())
        return y.cpu().numpy() if case["host"] else y
    return _moe_exact(case, g)
