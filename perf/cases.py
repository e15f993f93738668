"""The measured workloads of the encode path: what a program that quantises a model's
Linears has this package do, one kind per public entry point.

=========  ===============================================================================
kind       one pass
=========  ===============================================================================
linear     a whole small Linear: calibration tokens -> Hessian -> transform -> factor ->
           rotation -> GPTQ of its two row classes (a k_proj or an MoE expert)
hessian    ``HessianStats`` of one input over its calibration batches, then its transform
           to the stored basis (once per distinct input of a model)
factor     ``inverse_factor`` of one transformed Hessian (once per distinct input)
experts    ``inverse_factors_batched`` of an MoE projection's experts
gptq       ``encode_jobs_gptq`` of one tensor's row classes given the factor (once per
           tensor), optionally with the activation ordering and the compensated weights
refine     ``refine_groups`` sweeps over a tensor's GPTQ codes (once per tensor)
qad        one training step's decode of a fake-quantised Linear, forward and backward
=========  ===============================================================================

Inputs follow the calibration recipe of the benchmark: unit normal tokens with 1 % of the
channels twenty times larger, weights N(0, 0.02^2), rows split between INT2/B32, INT4/B64
and INT8/B64 ladders, order-16 rotation of every column group.
"""

import math
from types import SimpleNamespace

import torch

from hi2_amd.encode import encode_rows
from hi2_amd.format import fwht_groups
from hi2_amd.hessian import (GptqJob, HessianStats, encode_jobs_gptq, inverse_factor,
                             inverse_factors_batched)
from hi2_amd.qad_kernel import original, stored
from hi2_amd.refine import refine_groups

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
DAMP = 0.01
GROUP = 16


def listed():
    return [
        # an expert-sized Linear end to end: latency and launches
        dict(name="linear_1024", kind="linear", n=1024, k=1024, t=4096, int2=0.3),
        # the widest input of an 8B block (down_proj), bf16 tokens in one batch
        dict(name="hessian_14336_bf16", kind="hessian", k=14336, t=8192, batches=1,
             dtype="bf16", scale=False),
        # a half-precision model: ragged batches, smoothing vector
        dict(name="hessian_2560_f16", kind="hessian", k=2560, t=1777, batches=3,
             dtype="f16", scale=True),
        # single-precision activations of an attention input
        dict(name="hessian_4096_f32", kind="hessian", k=4096, t=2048, batches=2,
             dtype="f32", scale=False),
        # an attention or MLP input's factor, and the widest one
        dict(name="factor_4096", kind="factor", k=4096, t=8192),
        dict(name="factor_14336", kind="factor", k=14336, t=8192),
        # the experts of an MoE down projection
        dict(name="experts_32x1024", kind="experts", e=32, k=1024, t=2048),
        # k_proj / v_proj of an 8B block: few rows
        dict(name="gptq_1024x4096", kind="gptq", n=1024, k=4096, int2=0.3, int8=0.0,
             act_order=False, comp=False),
        # down_proj of an 8B block
        dict(name="gptq_4096x14336", kind="gptq", n=4096, k=14336, int2=0.3, int8=0.0,
             act_order=False, comp=False),
        # gate_proj of a 4B block with activation ordering, the compensated weights kept
        # as a training start
        dict(name="gptq_9216x2560_order", kind="gptq", n=9216, k=2560, int2=0.0, int8=0.03,
             act_order=True, comp=True),
        # q_proj of an 8B block, the default two sweeps
        dict(name="refine_4096x4096", kind="refine", n=4096, k=4096, int2=0.3, passes=2),
        # the same tensor in training: latents in step units, rotation and smoothing
        dict(name="qad_4096x4096", kind="qad", n=4096, k=4096, int2=0.3, unit=True,
             basis=True),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _mult(x, m):
    return max(m, int(x) // m * m)


def draw(rng):
    kind = rng.choice(["linear", "hessian", "hessian", "hessian", "factor", "factor", "experts",
                       "gptq", "gptq", "gptq", "refine", "qad"])
    if kind == "linear":
        k = _mult(_log(rng, 256, 2048), 64)
        return dict(kind=kind, n=int(_log(rng, 64, 4096)), k=k,
                    t=int(k * rng.uniform(3.0, 6.0)), int2=round(rng.uniform(0.1, 0.5), 2))
    if kind == "hessian":
        dtype = rng.choice(["bf16", "f16", "f32"])
        k = _mult(_log(rng, 256, 14336 if dtype == "bf16" else 9216), 16)
        return dict(kind=kind, k=k, t=int(_log(rng, 64, 4096)), batches=rng.randint(1, 2),
                    dtype=dtype, scale=rng.random() < 0.5)
    if kind == "factor":
        k = _mult(_log(rng, 256, 12288), 16)
        return dict(kind=kind, k=k, t=int(k * rng.uniform(0.6, 3.0)) if k > 8192 else 2 * k + 5)
    if kind == "experts":
        k = _mult(_log(rng, 256, 2048), 16)
        return dict(kind=kind, e=rng.randint(2, max(2, int(32 * 2 ** 20 / (k * k)))), k=k, t=2 * k)
    if kind in ("gptq", "refine"):
        k = _mult(_log(rng, 256, 14336 if kind == "gptq" else 6144), 64)
        work = (4096.0 if kind == "gptq" else 2048.0) * 14336 ** (2 if kind == "gptq" else 1) * (
            1 if kind == "gptq" else 4096)
        n = int(_log(rng, 16, max(17, min(16384, work / k ** 2))))
        if kind == "refine":
            return dict(kind=kind, n=n, k=k, int2=round(rng.uniform(0.0, 0.5), 2),
                        passes=rng.randint(1, 3))
        return dict(kind=kind, n=n, k=k, int2=round(rng.uniform(0.0, 0.5), 2),
                    int8=rng.choice([0.0, 0.03, 0.2]), act_order=rng.random() < 0.25,
                    comp=rng.random() < 0.4)
    k = _mult(_log(rng, 256, 14336), 64)
    return dict(kind="qad", n=int(_log(rng, 64, 4096.0 * 14336 / k)), k=k,
                int2=round(rng.uniform(0.0, 0.5), 2), unit=rng.random() < 0.7,
                basis=rng.random() < 0.7)


# ---- inputs -------------------------------------------------------------------------------
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1) + salt)


def _tokens(t, k, g, dtype=torch.float32):
    x = torch.randn(t, k, generator=g, device=DEV)
    x[:, torch.randperm(k, generator=g, device=DEV)[: -(-k // 100)]] *= 20.0
    return x.to(dtype)


def _h16(dtype):
    h = torch.ones(1, 1, dtype=dtype, device=DEV)
    for _ in range(4):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / 4.0


def _rotate(x):
    """``x`` with every 16-column group rotated (x [rows, k])."""
    return (x.reshape(x.shape[0], -1, GROUP) @ _h16(x.dtype)).reshape(x.shape)


def _hessian64(t, k, g):
    """The transformed mean Hessian of rotated tokens, float64."""
    x = _rotate(_tokens(t, k, g).double())
    return x.T @ x / t


def _factor64(hs):
    """Upper U with ``U^T U = (hs + DAMP mean(diag) I)^-1``, float64: J inv(chol(J A J)) J."""
    a = hs.clone()
    a.diagonal().add_(DAMP * a.diagonal().mean())
    low = torch.linalg.cholesky(a.flip(0, 1))
    del a
    eye = torch.eye(hs.shape[0], dtype=hs.dtype, device=hs.device)
    return torch.linalg.solve_triangular(low, eye, upper=False).flip(0, 1).contiguous()


def _classes(n, g, int2, int8=0.0):
    """The allocation: ``[(row indices, nbits, block)]``, a random choice of rows each."""
    p = torch.randperm(n, generator=g, device=DEV)
    n2, n8 = int(round(int2 * n)), int(round(int8 * n))
    parts = [(p[:n2], 2, 32), (p[n2:n2 + n8], 8, 64), (p[n2 + n8:], 4, 64)]
    return [(r.sort().values, nb, b) for r, nb, b in parts if r.numel()]


def _weights(n, k, g):
    return torch.randn(n, k, generator=g, device=DEV) * 0.02


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind == "linear":
        k = case["k"]
        return SimpleNamespace(
            kind=kind, k=k, x=_tokens(case["t"], k, g, torch.bfloat16),
            w=_weights(case["n"], k, g), had=torch.ones(k // GROUP, dtype=torch.uint8, device=DEV),
            classes=_classes(case["n"], g, case["int2"]))
    if kind == "hessian":
        k = case["k"]
        scale = None
        if case["scale"]:
            scale = torch.empty(k, device=DEV).uniform_(0.5, 2.0, generator=g).half()
        had = (torch.rand(k // GROUP, generator=g, device=DEV) < 0.9).to(torch.uint8)
        xs = [_tokens(case["t"], k, g, DTYPES[case["dtype"]]) for _ in range(case["batches"])]
        return SimpleNamespace(kind=kind, k=k, xs=xs, scale=scale, had=had)
    if kind == "factor":
        return SimpleNamespace(kind=kind, hs=_hessian64(case["t"], case["k"], g).float())
    if kind == "experts":
        hs = torch.stack([_hessian64(case["t"], case["k"], g).float() for _ in range(case["e"])])
        return SimpleNamespace(kind=kind, hs=hs)
    if kind in ("gptq", "refine"):
        n, k = case["n"], case["k"]
        hs = _hessian64(max(2 * k, 1024) if k <= 4096 else 8192, k, g)
        d, perm = hs.diagonal().float().contiguous(), None
        if case.get("act_order"):
            perm = torch.argsort(d, descending=True, stable=True)
            u = _factor64(hs[perm][:, perm]).float()
        else:
            u = _factor64(hs).float()
        w = _weights(n, k, g)
        jobs = [GptqJob(w[r], d, u, nb, b, perm)
                for r, nb, b in _classes(n, g, case["int2"], case.get("int8", 0.0))]
        if kind == "gptq":
            return SimpleNamespace(kind=kind, jobs=jobs, comp=case["comp"])
        encs = encode_jobs_gptq(jobs)
        return SimpleNamespace(
            kind=kind, hs=hs.float(), passes=case["passes"],
            groups=[(j.w, e, j.nbits, j.block) for j, e in zip(jobs, encs)])
    # qad: the latents start at the weights, in units of their block's step when unit
    n, k = case["n"], case["k"]
    w = _weights(n, k, g)
    d = torch.ones(k, device=DEV)
    unit = torch.ones(n, k, device=DEV)
    groups, params = [], []
    for rows, nb, b in _classes(n, g, case["int2"]):
        e = encode_rows(w[rows], d, nb, b)
        step = e.params[..., 1].float() * e.consts[:, 2:3].float()
        unit[rows] = step.clamp_min(1e-6).repeat_interleave(b, dim=1)
        # bytes between integers, as the optimiser leaves them
        lo_u, st_u = (e.params[..., i].float()
                      + (torch.rand(e.params.shape[:2], generator=g, device=DEV) - 0.5) * 0.8
                      for i in (0, 1))
        lo_u.requires_grad_()
        st_u.requires_grad_()
        groups.append(SimpleNamespace(rows=rows, consts=e.consts.contiguous(), nbits=nb, block=b,
                                      lo_u=lo_u, step_u=st_u))
        params += [lo_u, st_u]
    if not case["unit"]:
        unit = torch.ones(0, device=DEV)
    latent = (w / unit if case["unit"] else w).requires_grad_()
    had = torch.ones(k // GROUP, dtype=torch.uint8, device=DEV)
    scale = torch.empty(k, device=DEV).uniform_(0.5, 2.0, generator=g).half()
    fq = SimpleNamespace(latent=latent, unit=unit, groups=groups, had=had, col_scale=scale,
                         has_had=True, has_scale=True)
    grad = torch.randn(n, k, generator=g, device=DEV) * 1e-3
    return SimpleNamespace(kind="qad", fq=fq, basis=case["basis"], leaves=[latent] + params,
                           grad=grad)


# ---- one pass -----------------------------------------------------------------------------
def _encoded(encs):
    return [[e.codes, e.params, e.consts, e.sse] + ([] if e.comp is None else [e.comp])
            for e in encs]


def run(st):
    if st.kind == "linear":
        stats = HessianStats(st.k)
        stats.update(st.x)
        hs = stats.transformed(None, st.had)
        u = inverse_factor(hs, DAMP)
        d = hs.diagonal()
        wt = fwht_groups(st.w, st.had)
        encs = encode_jobs_gptq([GptqJob(wt[r], d, u, nb, b) for r, nb, b in st.classes])
        return {"u": u, "encoded": _encoded(encs)}
    if st.kind == "hessian":
        stats = HessianStats(st.k)
        for x in st.xs:
            stats.update(x)
        return stats.transformed(st.scale, st.had)
    if st.kind == "factor":
        return inverse_factor(st.hs, DAMP)
    if st.kind == "experts":
        return inverse_factors_batched(st.hs, DAMP)
    if st.kind == "gptq":
        return _encoded(encode_jobs_gptq(st.jobs, comp=st.comp))
    if st.kind == "refine":
        return refine_groups(st.groups, st.hs, st.passes)
    w = original(st.fq) if st.basis else stored(st.fq, True)
    return [w.detach()] + list(torch.autograd.grad(w, st.leaves, st.grad))


# ---- what a pass cannot do without ---------------------------------------------------------
def work(case):
    kind, k = case["kind"], case["k"]
    if kind == "linear":
        n, t = case["n"], case["t"]
        return {"bytes": 2.0 * t * k + 4.0 * n * k + 1.0 * n * k,
                "flops": 1.0 * t * k * k + 2.0 * k ** 3 / 3 + 1.0 * n * k * k}
    if kind == "hessian":
        t = case["t"] * case["batches"]
        return {"bytes": (4 if case["dtype"] == "f32" else 2) * 1.0 * t * k + 4.0 * k * k,
                "flops": 1.0 * t * k * k}
    if kind == "factor":
        return {"bytes": 8.0 * k * k, "flops": 2.0 * k ** 3 / 3}
    if kind == "experts":
        e = case["e"]
        return {"bytes": 8.0 * e * k * k, "flops": 2.0 * e * k ** 3 / 3}
    n = case["n"]
    if kind == "gptq":
        return {"bytes": (5.0 + (4.0 if case["comp"] else 0.0)) * n * k + 2.0 * k * k,
                "flops": 1.0 * n * k * k}
    if kind == "refine":  # the gradient, then each sweep's updates (the last one forward only)
        return {"bytes": 6.0 * n * k + 4.0 * k * k,
                "flops": 2.0 * n * k * k * (1.0 + case["passes"] - 0.5)}
    # forward reads latent and unit and writes the weights; backward reads the gradient,
    # latent and unit and writes the latent's gradient
    per = 6 * 4 if case["unit"] else 4 * 4
    return {"bytes": float(per) * n * k, "flops": 20.0 * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        # a rounding or ladder decision on a tie takes a row another way (under 0.2 % of
        # the codes with three or more tokens per column); u as for a factor
        return {"rel": 5e-3, "max": 0.2, "differ": 8e-3}
    if kind == "hessian":  # 32-bit sums over the tokens: up to 1.4e-6 off 64 bits
        return {"rel": 6e-6, "max": 2.4e-4}
    if kind in ("factor", "experts"):
        # fp32 arithmetic on a matrix whose condition only the damping bounds when it has
        # fewer tokens than columns: 1.4e-4 off 64 bits there, 5e-6 to 7e-6 with two per column
        return {"rel": 6e-4, "max": 2.4e-2} if case["t"] < 2 * case["k"] else {
            "rel": 2e-5, "max": 4e-3}
    if kind in ("gptq", "refine"):
        return "exact"  # every decision is defined by the stored fp32 operation order
    return {"rel": 1e-6, "max": 1e-4}  # block sums of at most 64 terms: 2.3e-7 off 64 bits


# ---- the same in 64 bits -------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind == "linear":
        x = _rotate(st.x.double())
        # the codes and everything that follows them are decisions of fp32 roundings
        return {"u": _factor64(x.T @ x / case["t"]), "encoded": None}
    if kind == "hessian":
        k = case["k"]
        s = torch.zeros(k, k, dtype=torch.float64, device=DEV)
        for x in st.xs:
            xd = x.double()
            s.addmm_(xd.T, xd)
        s /= float(case["t"] * case["batches"])
        if st.scale is not None:
            inv = 1.0 / st.scale.double()
            s *= inv[:, None]
            s *= inv[None, :]
        flags = st.had.bool().repeat_interleave(GROUP)
        s = torch.where(flags[None, :], _rotate(s), s)
        return torch.where(flags[:, None], _rotate(s.T).T, s)
    if kind == "factor":
        return _factor64(st.hs.double())
    if kind == "experts":
        return torch.stack([_factor64(h.double()) for h in st.hs])
    if kind in ("gptq", "refine"):
        return None  # rounding decisions: no 64-bit value
    return _qad64(st)


def _qad64(st):
    fq = st.fq
    latent = fq.latent.detach()
    v = latent * fq.unit if fq.unit.numel() else latent
    out = torch.empty_like(latent, dtype=torch.float64)
    grad = st.grad.double()
    if st.basis:
        grad = _rotate(grad / fq.col_scale.double())
    g_lat = torch.empty_like(out)
    per = []
    for gr in fq.groups:
        b, n = gr.block, gr.rows.numel()
        c = gr.consts.double()
        lb = gr.lo_u.detach().round().clamp(0, 255).double()
        sb = gr.step_u.detach().round().clamp(0, 255).double()
        lo = (lb * c[:, 1:2] + c[:, 0:1]).float().half().double()[..., None]
        step = (sb * c[:, 2:3]).float().half().double()[..., None]
        safe = torch.where(step == 0, torch.ones_like(step), step)
        # the reference rounds the difference and the quotient to fp32 before the code
        vb = v[gr.rows].reshape(n, -1, b)
        z = ((vb - lo.float()) / safe.float()).double()
        top = float(2 ** gr.nbits - 1)
        q = torch.where(step == 0, torch.zeros_like(z), z.round().clamp(0, top))
        out[gr.rows] = (lo + q * step).float().half().double().reshape(n, -1)
        gb = grad[gr.rows].reshape(n, -1, b)
        gz = torch.where((z >= 0) & (z <= top), gb * step, torch.zeros_like(gb))
        gv = gz / safe
        g_lat[gr.rows] = gv.reshape(n, -1)
        per.append(c[:, 1:2] * (gb - gv).sum(-1))
        st_term = torch.where(step == 0, torch.zeros_like(gz), gz * z / safe)
        per.append(c[:, 2:3] * (gb * q - st_term).sum(-1))
    if fq.unit.numel():
        g_lat *= fq.unit.double()
    if st.basis:
        out = _rotate(out) / fq.col_scale.double()
    return [out, g_lat] + per
