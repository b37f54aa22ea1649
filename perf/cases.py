"""The work that programs on this library have it do, as measurable cases.

A case is one pass of one path through the public Python interface (`t2h`):

- cond:    the conditioning rows of a forward: timestep embedding, its MLP, the
           adaLN linear and a block's six chunks (1 to 16 rows: all launches);
- linear:  a plain projection (the cross attention's k/v of the image tokens);
- qkv:     the qkv projection with the attention epilogue and head-major pack;
- mlp:     LN + modulate, the MLP's first linear with GELU, its second with the
           gated residual join;
- out:     an attention's out projection joined to an f32 residual stream of a
           ragged sparse batch;
- glue:    the per-token work of one cross block around its attention and MLP
           chains (three norms, three joins), dense or sparse;
- chain:   LN + modulate, QK RMSNorm + RoPE, GELU + bias and the gated residual
           over one sparse batch, each on rows of its own;
- pack:    the attention epilogue and pack over an existing packed qkv;
- sampler: one classifier-free-guidance Euler step, with or without rescale.

The token counts are those of the sparse-structure grid (16^3 = 4,096 tokens),
the structured latent (2,369), the ragged 64^3 pair (39,804) and the 128^3 shell
(201,436), and anything between for drawn cases. Widths are the two the
configurations and tests use: 1536 (12 heads of 128) and 1024 (16 heads of 64),
with an MLP of four times the width.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "trellis2-mojo_amd"))

from t2h import block, nn, ops, sparse  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
HEADS = {1536: (12, 128), 1024: (16, 64)}
EPS = 1e-6
SIGMA_MIN = 1e-5
FREQ_DIM = 256          # width of the sinusoidal timestep embedding
FULL = 201_436          # tokens of the 128^3 shell


def listed():
    return [
        # one generation's conditioning: a single timestep row through weights of 34 MB
        dict(name="cond_b1", path="cond", rows=1, width=1536, dtype="f16"),
        # k/v of the 1,029 image tokens for one cross attention (an odd row count)
        dict(name="kv_1029", path="linear", rows=1029, width=1024, outs=3072, dtype="f16"),
        # the structured-latent DiT's qkv at its token count, reference k layout
        dict(name="qkv_2369", path="qkv", rows=2369, width=1536, dtype="bf16", grid=64, kt=True),
        # ... and at the 128^3 shell's, with k in the layout an MFMA attention reads
        dict(name="qkv_201k", path="qkv", rows=FULL, width=1536, dtype="f16", grid=128, kt=False),
        # the MLP half of a structured-latent block
        dict(name="mlp_2369", path="mlp", rows=2369, width=1536, dtype="f16", batch=1),
        # ... and of the largest sparse batch: the most work of any case
        dict(name="mlp_201k", path="mlp", rows=FULL, width=1536, dtype="bf16", batch=1),
        # out projection of a ragged batch of two onto the f32 residual stream
        dict(name="out_39804", path="out", rows=39_804, width=1536, dtype="f16", batch=2),
        # glue of the dense sparse-structure block, f32 as the reference runs it
        dict(name="glue_dense_4096", path="glue", rows=4096, width=1536, dtype="f32", batch=1, sparse=False),
        # glue of a sparse block over a ragged batch of two
        dict(name="glue_39804", path="glue", rows=39_804, width=1536, dtype="f16", batch=2, sparse=True),
        # the per-token chain over the whole shell (the benchmark's workload, out of place)
        dict(name="chain_201k", path="chain", rows=FULL, width=1536, dtype="f16", grid=128),
        # epilogue + pack of a qkv that another program's GEMM left packed
        dict(name="pack_39804", path="pack", rows=39_804, width=1536, dtype="f16", grid=64, kt=True),
        # one guided, rescaled step over the whole shell's latent
        dict(name="sampler_201k", path="sampler", rows=FULL, channels=32, batch=1, rescale=0.7, dtype="f32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["cond", "linear", "qkv", "mlp", "out", "glue", "chain", "pack", "sampler"])
    width = rng.choice([1536, 1536, 1024])
    half = rng.choice(["f16", "bf16"])
    if path == "cond":
        return dict(path=path, rows=rng.randint(1, 16), width=width, dtype=half)
    if path == "linear":
        return dict(path=path, rows=_log_int(rng, 64, 60_000), width=width, outs=width * rng.choice([1, 2, 3, 4]),
                    dtype=half)
    if path in ("qkv", "pack"):
        rows = _log_int(rng, 600, 150_000)
        dt = half if path == "qkv" else rng.choice(["f16", "bf16", "f32"])
        return dict(path=path, rows=rows, width=width, dtype=dt, grid=64 if rows <= 40_000 else 128,
                    kt=rng.random() < 0.5)
    if path == "mlp":
        return dict(path=path, rows=_log_int(rng, 600, 150_000), width=width, dtype=half, batch=rng.randint(1, 4))
    if path == "out":
        return dict(path=path, rows=_log_int(rng, 600, 150_000), width=width, dtype=half, batch=rng.randint(1, 4))
    if path == "glue":
        b = rng.randint(1, 4)
        dense = rng.random() < 0.4
        rows = b * _log_int(rng, 300, 10_000) if dense else _log_int(rng, 600, 150_000)
        return dict(path=path, rows=rows, width=width, dtype=rng.choice(["f16", "bf16", "f32"]), batch=b,
                    sparse=not dense)
    if path == "chain":
        rows = _log_int(rng, 600, 150_000)
        return dict(path=path, rows=rows, width=width, dtype=half, grid=64 if rows <= 40_000 else 128)
    return dict(path="sampler", rows=_log_int(rng, 600, FULL), channels=rng.choice([8, 32]), batch=rng.randint(1, 4),
                rescale=rng.choice([0.0, 0.7]), dtype="f32")


# ---- inputs, from the seed alone -------------------------------------------
class _Make:
    def __init__(self, seed: int):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dev = torch.device("cuda")

    def randn(self, shape, std=1.0, mean=0.0, dtype=torch.float32):
        return torch.randn(shape, generator=self.g, device=self.dev).mul_(std).add_(mean).to(dtype)

    def rows(self, n, c, dtype, std=1.0):
        """Token rows whose channels differ in scale, as a residual stream's do."""
        spread = torch.exp(0.3 * torch.randn((c,), generator=self.g, device=self.dev))
        return (torch.randn((n, c), generator=self.g, device=self.dev) * (spread * std)).to(dtype)

    def weight(self, n, k, dtype):
        return self.randn((n, k), std=k ** -0.5, dtype=dtype)

    def shell(self, n, res):
        """n voxels of a rough sphere shell on a res^3 grid, as (0, x, y, z) in
        lexicographic order (the order the sparse stage lists them in)."""
        ax = torch.arange(res, device=self.dev, dtype=torch.float32) - (res - 1) / 2
        d = (ax.view(-1, 1, 1) ** 2 + ax.view(1, -1, 1) ** 2 + ax.view(1, 1, -1) ** 2).sqrt().flatten()
        d = (d - 0.39 * res).abs() + 1.5 * torch.rand(d.shape, generator=self.g, device=self.dev)
        idx = torch.topk(d, n, largest=False).indices.sort().values
        out = torch.zeros((n, 4), dtype=torch.int32, device=self.dev)
        out[:, 1], out[:, 2], out[:, 3] = idx // (res * res), idx // res % res, idx % res
        return out

    def split(self, n, b):
        """Uneven token offsets of b batches over n rows (host list)."""
        share = torch.rand((b,), generator=self.g, device=self.dev).add_(0.5).cpu().tolist()
        cuts = [0]
        for i in range(b - 1):
            cuts.append(cuts[-1] + int(n * share[i] / sum(share)))
        return cuts + [n]


def _up(n, m):
    return (n + m - 1) // m * m


def _inputs(case, seed):
    mk = _Make(seed)
    path, rows = case["path"], case["rows"]
    dt = DTYPES[case["dtype"]]
    c = case.get("width", 0)
    h, d = HEADS.get(c, (0, 0))
    s = {"case": case}
    if path == "cond":
        s.update(t=torch.rand((rows,), generator=mk.g, device=mk.dev) * 1000.0,
                 w0=mk.weight(c, FREQ_DIM, dt), b0=mk.randn((c,), 0.02),
                 w2=mk.weight(c, c, dt), b2=mk.randn((c,), 0.02),
                 wm=mk.weight(6 * c, c, dt), bm=mk.randn((6 * c,), 0.02), share=mk.randn((6 * c,), 0.1))
    elif path == "linear":
        s.update(x=mk.rows(rows, c, dt), w=mk.weight(case["outs"], c, dt), b=mk.randn((case["outs"],), 0.02))
    elif path == "qkv":
        s.update(x=mk.rows(rows, c, dt), w=mk.weight(3 * c, c, dt), b=mk.randn((3 * c,), 0.02),
                 gq=mk.randn((h, d), 0.02, 1.0), gk=mk.randn((h, d), 0.02, 1.0), coords=mk.shell(rows, case["grid"]))
    elif path == "mlp":
        b = case["batch"]
        s.update(x=mk.rows(rows, c, dt), shift=mk.randn((b, c), 0.1), scale=mk.randn((b, c), 0.1),
                 gate=mk.randn((b, c), 0.3), w1=mk.weight(4 * c, c, dt), b1=mk.randn((4 * c,), 0.02),
                 w2=mk.weight(c, 4 * c, dt), b2=mk.randn((c,), 0.02), cuts=mk.split(rows, b))
    elif path == "out":
        b = case["batch"]
        s.update(x=mk.rows(rows, c, dt, 0.5), w=mk.weight(c, c, dt), b=mk.randn((c,), 0.02),
                 gate=mk.randn((b, c), 0.3), res=mk.rows(rows, c, torch.float32), cuts=mk.split(rows, b))
    elif path == "glue":
        b = case["batch"]
        s.update(x=mk.rows(rows, c, dt), h=[mk.rows(rows, c, dt, 0.5) for _ in range(3)],
                 w=mk.randn((c,), 0.02, 1.0), b=mk.randn((c,), 0.02), share=mk.randn((6 * c,), 0.1),
                 mod=mk.randn((b, 6 * c), 0.1), cuts=mk.split(rows, b))
    elif path == "chain":
        s.update(x=mk.rows(rows, c, dt), y=mk.rows(rows, c, dt, 0.5), q=mk.rows(rows, c, dt).view(rows, h, d),
                 k=mk.rows(rows, c, dt).view(rows, h, d), u=mk.rows(rows, 4 * c, dt), bias=mk.randn((4 * c,), 0.02),
                 shift=mk.randn((c,), 0.1), scale=mk.randn((c,), 0.1), gate=mk.randn((c,), 0.3),
                 gq=mk.randn((h, d), 0.02, 1.0), gk=mk.randn((h, d), 0.02, 1.0), coords=mk.shell(rows, case["grid"]))
    elif path == "pack":
        s.update(qkv=mk.rows(rows, 3 * c, dt), gq=mk.randn((h, d), 0.02, 1.0), gk=mk.randn((h, d), 0.02, 1.0),
                 coords=mk.shell(rows, case["grid"]))
    else:
        shape = (rows, case["channels"])
        pos = mk.randn(shape)
        s.update(x=mk.randn(shape), pos=pos, neg=pos + 0.3 * mk.randn(shape), cuts=mk.split(rows, case["batch"]))
    return s


def _batch_offsets(cuts):
    return torch.tensor(cuts, dtype=torch.int64, device="cuda")


def _ragged_coords(cuts):
    """Coordinates that only tell the batches apart (the glue reads no positions)."""
    n = cuts[-1]
    co = torch.zeros((n, 4), dtype=torch.int32, device="cuda")
    r = torch.arange(n, device="cuda")
    for b in range(len(cuts) - 1):
        co[cuts[b]:cuts[b + 1], 0] = b
    co[:, 1], co[:, 2], co[:, 3] = r // 4096 % 64, r // 64 % 64, r % 64
    return co


def prepare(case, seed):
    s = _inputs(case, seed)
    path = case["path"]
    if path == "cond":
        s["mod"] = sparse.Modulation(modulation=s["share"])
    elif path in ("qkv", "chain", "pack"):
        _, d = HEADS[case["width"]]
        s["freqs"] = nn.rope_freqs(d)
        s["pad"] = _up(case["rows"], 64)
    elif path in ("mlp", "out"):
        s["offsets"] = _batch_offsets(s["cuts"])
    elif path == "glue":
        s["block"] = block.ModulatedCrossBlock(case["width"], s["w"], s["b"], modulation=s["share"], eps=EPS)
        if case["sparse"]:
            s["xs"] = sparse.SparseTensor(s["x"], _ragged_coords(s["cuts"]), case["batch"])
        else:
            s["xs"] = s["x"].view(case["batch"], -1, case["width"])
    elif path == "sampler":
        n = len(s["cuts"])
        s["ws"] = torch.empty(ops.flow_euler_workspace(case["rows"], case["channels"], n), dtype=torch.uint8,
                              device="cuda")
    return s


# ---- one pass ----------------------------------------------------------------
T_NOW, T_NEXT, GUIDANCE = 0.8, 0.72, 5.0


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "cond":
        e = ops.timestep_embedding(s["t"], FREQ_DIM, dtype=DTYPES[case["dtype"]])
        e = ops.linear(e, s["w0"], s["b0"], act=ops.ACT_SILU)
        e = ops.linear(e, s["w2"], s["b2"], act=ops.ACT_SILU)
        m = ops.linear(e, s["wm"], s["bm"], out_dtype=torch.float32)
        return s["mod"].chunks(m, case["width"])
    if path == "linear":
        return ops.linear(s["x"], s["w"], s["b"])
    if path == "qkv":
        h, _ = HEADS[case["width"]]
        return ops.qkv_linear_pack(s["x"], s["w"], h, bias=s["b"], gamma_q=s["gq"], gamma_k=s["gk"], mp=s["pad"],
                                   lp=s["pad"], freqs=s["freqs"], coords=s["coords"], k_transposed=case["kt"])
    if path == "mlp":
        y = ops.ln_modulate(s["x"], EPS, shift=s["shift"], scale=s["scale"], offsets=s["offsets"])
        y = ops.linear(y, s["w1"], s["b1"], act=ops.ACT_GELU_TANH)
        return ops.linear_gate_residual(y, s["w2"], s["x"], bias=s["b2"], gate=s["gate"], offsets=s["offsets"])
    if path == "out":
        return ops.linear_gate_residual(s["x"], s["w"], s["res"], bias=s["b"], gate=s["gate"], offsets=s["offsets"])
    if path == "glue":
        seen = []

        def chain(i):
            def call(y):
                seen.append(y)
                return s["h"][i]
            return call
        out = s["block"].forward(s["xs"], s["mod"], chain(0), chain(1), chain(2))
        return [*seen, out.feats if case["sparse"] else out]
    if path == "chain":
        a = ops.ln_modulate(s["x"], EPS, shift=s["shift"], scale=s["scale"])
        q, k = ops.qk_rmsnorm_rope(q=s["q"], k=s["k"], gamma_q=s["gq"], gamma_k=s["gk"], freqs=s["freqs"],
                                   coords=s["coords"])
        u = ops.activation(s["u"], ops.ACT_GELU_TANH, bias=s["bias"])
        return [a, q, k, u, ops.gate_residual(s["x"], s["y"], gate=s["gate"])]
    if path == "pack":
        h, d = HEADS[case["width"]]
        q, k, v = s["qkv"].view(case["rows"], 3, h, d).unbind(1)
        return ops.attn_pack(q=q, k=k, v=v, mp=s["pad"], lp=s["pad"], gamma_q=s["gq"], gamma_k=s["gk"],
                             freqs=s["freqs"], coords=s["coords"], k_transposed=case["kt"])
    return ops.flow_euler_step(s["x"], s["pos"], T_NOW, T_NEXT, SIGMA_MIN, v_neg=s["neg"], guidance_strength=GUIDANCE,
                               guidance_rescale=case["rescale"], seg_offsets=s["cuts"], workspace=s["ws"])


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    t, c, e = case["rows"], case.get("width", 0), SIZE[case["dtype"]]
    path = case["path"]
    if path == "cond":
        w = FREQ_DIM * c + c * c + 6 * c * c
        return {"bytes": e * w + 4 * t * 6 * c, "flops": 2 * t * w}
    if path == "linear":
        n = case["outs"]
        return {"bytes": e * (t * c + n * c + t * n), "flops": 2 * t * n * c}
    if path == "qkv":
        return {"bytes": e * (t * c + 3 * c * c + 3 * _up(t, 64) * c) + 16 * t, "flops": 6 * t * c * c}
    if path == "mlp":
        return {"bytes": e * (2 * t * c + 8 * c * c), "flops": 16 * t * c * c}
    if path == "out":
        return {"bytes": e * (t * c + c * c) + 8 * t * c, "flops": 2 * t * c * c}
    if path == "glue":      # four inputs, four outputs
        return {"bytes": 8 * e * t * c, "flops": 40 * t * c}
    if path == "chain":     # x once, y, q, k, u in; a, q, k, u, x out
        return {"bytes": e * t * 16 * c + 16 * t, "flops": 150 * t * c}
    if path == "pack":
        return {"bytes": e * 3 * c * (t + _up(t, 64)) + 16 * t, "flops": 30 * t * c}
    return {"bytes": 5 * e * t * case["channels"], "flops": 30 * t * case["channels"]}


# Largest errors measured against exact() over the listed and 40 drawn cases, in
# units of one rounding to the storage type (the relative 2-norm of it), as
# (rel, max): the tolerance is four times them. out and sampler are f32; an f32
# pack shows the rotation angles' own rounding.
ROUNDING = {"f32": 4.5e-8, "f16": 2.1e-4, "bf16": 1.7e-3}
SEEN = {"cond": (1.7, 6.0), "linear": (1.0, 2.4), "qkv": (1.0, 2.4), "mlp": (1.05, 5.5), "out": (1.1, 30.0),
        "glue": (1.9, 10.0), "chain": (1.0, 2.4), "pack": (1.0, 2.4), "sampler": (2.0, 15.0)}


def tolerance(case):
    u = ROUNDING["f32" if case["path"] in ("out", "sampler") else case["dtype"]]
    rel, top = (3.0, 120.0) if case["path"] == "pack" and case["dtype"] == "f32" else SEEN[case["path"]]
    return {"rel": 4 * rel * u, "max": 4 * top * u}


# ---- the same in 64 bits ------------------------------------------------------
def _ln(x, w1, b):
    m = x.mean(-1, keepdim=True)
    v = (x - m).square_().mean(-1, keepdim=True)
    return (x - m) / (v + EPS).sqrt() * w1 + b


def _gelu_tanh(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _silu(x):
    return x / (1 + torch.exp(-x))


def _angles(coords, d):
    """[T, D/2] rotation angles: axis-major slots, unused slots 0."""
    fd = d // 2 // 3
    freqs = torch.from_numpy((np.float32(1.0) / np.power(np.float32(10000.0), np.arange(fd, dtype=np.float32)
                                                         / np.float32(fd))).astype(np.float64)).cuda()
    a = torch.zeros((coords.shape[0], d // 2), dtype=torch.float64, device="cuda")
    a[:, :3 * fd] = (coords[:, 1:].double().unsqueeze(-1) * freqs).flatten(1)
    return a


def _rms_rope(x, gamma, ang):
    """x [T, H, D]"""
    d = x.shape[-1]
    x = x * x.square().sum(-1, keepdim=True).clamp_min(1e-24).rsqrt() * (gamma.double() * math.sqrt(d))
    c, sn = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)
    re, im = x[..., 0::2], x[..., 1::2]
    return torch.stack((re * c - im * sn, re * sn + im * c), -1).flatten(-2)


def _head_major(x, pad, scale=1.0, transposed=False):
    t, h, d = x.shape
    if transposed:
        out = torch.zeros((h, d, pad), dtype=torch.float64, device="cuda")
        out[:, :, :t] = x.permute(1, 2, 0)
    else:
        out = torch.zeros((h, pad, d), dtype=torch.float64, device="cuda")
        out[:, :t] = x.permute(1, 0, 2)
    return out.mul_(scale)


def _attention_operands(case, s, qkv):
    h, d = HEADS[case["width"]]
    pad = _up(case["rows"], 64)
    ang = _angles(s["coords"], d)
    q, k, v = (y.reshape(-1, h, d) for y in qkv.chunk(3, 1))
    return [_head_major(_rms_rope(q, s["gq"], ang), pad, 1 / math.sqrt(d)),
            _head_major(_rms_rope(k, s["gk"], ang), pad, transposed=case["kt"]), _head_major(v, pad)]


def exact(case, seed):
    s = _inputs(case, seed)
    path, c = case["path"], case.get("width", 0)

    def spread(p):          # [B, C] parameter rows -> one per token
        cuts = s["cuts"]
        if case.get("sparse") is False:
            n = case["rows"] // case["batch"]
            cuts = [b * n for b in range(case["batch"] + 1)]
        return torch.repeat_interleave(p.double(), torch.tensor(cuts, device="cuda").diff(), 0)

    def lin(x, w, b):
        return x.double() @ w.double().T + b.double()
    if path == "cond":
        half = FREQ_DIM // 2
        f = torch.exp(-math.log(10000.0) * torch.arange(half, dtype=torch.float64, device="cuda") / half)
        a = s["t"].double().unsqueeze(1) * f
        e = torch.cat([a.cos(), a.sin()], 1)
        e = _silu(lin(_silu(lin(e, s["w0"], s["b0"])), s["w2"], s["b2"]))
        return list((lin(e, s["wm"], s["bm"]) + s["share"].double()).chunk(6, 1))
    if path == "linear":
        return lin(s["x"], s["w"], s["b"])
    if path == "qkv":
        return _attention_operands(case, s, lin(s["x"], s["w"], s["b"]))
    if path == "mlp":
        y = _ln(s["x"].double(), 1 + spread(s["scale"]), spread(s["shift"]))
        y = _gelu_tanh(lin(y, s["w1"], s["b1"]))
        return s["x"].double() + lin(y, s["w2"], s["b2"]) * spread(s["gate"])
    if path == "out":
        return s["res"].double() + lin(s["x"], s["w"], s["b"]) * spread(s["gate"])
    if path == "glue":
        sh1, sc1, g1, sh3, sc3, g3 = (spread(p) for p in (s["mod"] + s["share"]).chunk(6, 1))
        x = s["x"].double()
        outs = [_ln(x, 1 + sc1, sh1)]
        x = x + s["h"][0].double() * g1
        outs.append(_ln(x, s["w"].double(), s["b"].double()))
        x = x + s["h"][1].double()
        outs.append(_ln(x, 1 + sc3, sh3))
        x = x + s["h"][2].double() * g3
        return [*outs, x] if case["sparse"] else [*outs, x.view(case["batch"], -1, c)]
    if path == "chain":
        _, d = HEADS[c]
        ang = _angles(s["coords"], d)
        return [_ln(s["x"].double(), 1 + s["scale"].double(), s["shift"].double()),
                _rms_rope(s["q"].double(), s["gq"], ang), _rms_rope(s["k"].double(), s["gk"], ang),
                _gelu_tanh(s["u"].double() + s["bias"].double()),
                s["x"].double() + s["y"].double() * s["gate"].double()]
    if path == "pack":
        return _attention_operands(case, s, s["qkv"].double())
    x, pos, neg = (s[n].double() for n in ("x", "pos", "neg"))
    a, cc = 1.0 - SIGMA_MIN, SIGMA_MIN + (1.0 - SIGMA_MIN) * T_NOW
    v = pos * GUIDANCE + neg * (1.0 - GUIDANCE)
    if case["rescale"] > 0.0:
        x0p, x0c = a * x - cc * pos, a * x - cc * v
        for lo, hi in zip(s["cuts"], s["cuts"][1:]):
            r = x0p[lo:hi].std(correction=0) / x0c[lo:hi].std(correction=0)
            x0c[lo:hi] *= case["rescale"] * r + (1.0 - case["rescale"])
        v = (a * x - x0c) / cc
    return x - (T_NOW - T_NEXT) * v, a * x - cc * v
