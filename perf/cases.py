"""The workloads this package's speed is judged by.

One case is one call (or one forward and backward pair) of a public entry
point: the fused scans over whole sequences (prefill), the streaming steps
(decode), and the elementwise scan with its backward (training).  Sizes are
those of the benchmark's configurations and of the row sweep, plus ragged ones
of the same kinds; values follow ``tssm.workloads`` (normal activations,
log-uniform decay rates, exponential or log-normal time gaps).

``exact`` restates each path in float64 with plain torch.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("triton-ssm_amd"))

import tssm  # noqa: E402
from ssm_scan import ssm_backward, ssm_forward  # noqa: E402
from tssm.session import RingSession  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BYTES = {"f32": 4, "bf16": 2, "f16": 2}


def listed():
    return [
        # the headline: prefill of a multihead layer, one decay per head
        dict(name="multihead_bf16", kind="multihead", B=8, L=4096, H=16, P=64, dtype="bf16",
             disc="zoh", per_head=True, extras=False),
        # the reference's own parameter layout (decay per channel, skip weights, Euler input)
        # in fp32, resumed from a state, at sizes that fill no tile
        dict(name="multihead_f32_resume", kind="multihead", B=3, L=1111, H=12, P=32, dtype="f32",
             disc="euler", per_head=False, extras=True),
        # the smallest scan: a Mamba-1 layer over a short window, launch-bound
        dict(name="selective_small", kind="selective", B=2, L=256, D=16, N=16, dtype="f32",
             per_channel_dt=False, extras=False),
        # a Mamba-1 layer in bf16 as models use it: a step size per channel, skip weights,
        # the final state kept for decoding; a prompt length that ends inside a chunk
        dict(name="selective_bf16", kind="selective", B=4, L=2000, D=768, N=16, dtype="bf16",
             per_channel_dt=True, extras=True),
        # the whole Mamba-1 input projection (step size, B and C from x) with the scan
        dict(name="xproj_f32", kind="xproj", B=16, L=2048, D=256, N=16, R=16),
        # irregular observations: time-aware interpolation feeding the Mamba-1 scan
        dict(name="interp_scan_f32", kind="interp", B=16, T=2048, F=256, N=16, K=10, FTILE=128,
             observed=0.7),
        # one very long sequence
        dict(name="ssd_long_bf16", kind="ssd", B=1, L=262144, H=8, P=64, N=16, dtype="bf16",
             gaps="lognormal", extras=False),
        # the headline shapes with a full P x N state per head
        dict(name="ssd_n64_bf16", kind="ssd", B=8, L=4096, H=16, P=64, N=64, dtype="bf16",
             gaps="softplus", extras=False),
        # the same layer in fp32, resumed from a state, its final state kept; a ragged length
        dict(name="ssd_n64_f32", kind="ssd", B=2, L=4000, H=16, P=64, N=64, dtype="f32",
             gaps="softplus", extras=True),
        # decode: one step of 4096 streams, 4 GiB of state updated in place
        dict(name="ssd_stream", kind="stream", S=4096, H=32, P=64, N=128),
        # training: the elementwise scan forward and backward
        dict(name="elementwise_train", kind="train", B=8, L=4096, H=1024, dtype="f32"),
        # decode of irregular streams: ring insert, forward fill and state step
        dict(name="ring_step", kind="ring", S=4096, H=1024, K=10, observed=0.3),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["multihead", "multihead", "selective", "selective", "xproj", "interp",
                       "ssd", "ssd", "ssd", "stream", "train", "ring"])
    if kind == "multihead":
        H, P = rng.randint(1, 16), rng.choice([8, 16, 32, 64, 64, 128])
        B = _log(rng, 1, 8)
        return dict(kind=kind, B=B, L=_log(rng, 64, max(64, 4096 * 1024 // (H * P))), H=H, P=P,
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                    disc=rng.choice(["zoh", "euler"]), per_head=rng.random() < 0.5,
                    extras=rng.random() < 0.5)
    if kind == "selective":
        N = rng.choice([8, 16, 16, 16, 32])
        D = _log(rng, 16, 1024)
        B = _log(rng, 1, 16)
        most = (16 * 2048 * 256 * 16) // (B * D * N)
        return dict(kind=kind, B=B, L=_log(rng, min(64, most), min(32768, most)), D=D, N=N,
                    dtype=rng.choice(["f32", "bf16", "bf16"]),
                    per_channel_dt=rng.random() < 0.6, extras=rng.random() < 0.5)
    if kind == "xproj":
        return dict(kind=kind, B=_log(rng, 1, 16), L=_log(rng, 64, 2048), D=4 * rng.randint(16, 64),
                    N=rng.choice([8, 16]), R=rng.choice([16, 32, 48, 64]))
    if kind == "interp":
        return dict(kind=kind, B=_log(rng, 1, 16), T=_log(rng, 64, 2048), F=4 * rng.randint(4, 64),
                    N=rng.choice([8, 16]), K=rng.randint(3, 16), FTILE=rng.choice([64, 128]),
                    observed=rng.choice([0.01, 0.05, 0.3, 0.7]))
    if kind == "ssd":
        H, P = rng.randint(1, 16), rng.choice([32, 64, 64])
        N = rng.choice([8, 16, 32, 64, 64])
        dtype = rng.choice(["bf16", "bf16", "f16", "f32", "f32"])
        B = _log(rng, 1, 8)
        # at most the work of the headline shapes in bf16 (a quarter of it in the other types)
        most = (8 * 4096 * 16 * 64 * 64) // (B * H * P * N) // (1 if dtype == "bf16" else 4)
        return dict(kind=kind, B=B, L=_log(rng, min(64, most), min(262144, most)), H=H, P=P, N=N,
                    dtype=dtype, gaps=rng.choice(["softplus", "lognormal"]),
                    extras=rng.random() < 0.5)
    if kind == "stream":
        return dict(kind=kind, S=_log(rng, 1, 4096), H=rng.randint(1, 32), P=rng.choice([32, 64]),
                    N=rng.choice([16, 64, 128]))
    if kind == "train":
        return dict(kind=kind, B=_log(rng, 1, 8), L=_log(rng, 64, 4096), H=4 * rng.randint(8, 256),
                    dtype=rng.choice(["f32", "f32", "bf16"]))
    return dict(kind="ring", S=_log(rng, 1, 4096), H=4 * rng.randint(8, 256), K=rng.randint(3, 16),
                observed=rng.choice([0.002, 0.02, 0.3]))


# ------------------------------------------------------------------ inputs
class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device="cuda") * scale).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def exponential(self, *shape, mean=1.0):
        return torch.empty(*shape, device="cuda").exponential_(1.0 / mean, generator=self.g)


def _inputs(c, seed):
    d, k = _Draw(seed), c["kind"]
    dt_ = DTYPES[c.get("dtype", "f32")]
    if k == "multihead":
        B, L, H, P = c["B"], c["L"], c["H"], c["P"]
        a_log = d.uniform(*((H,) if c["per_head"] else (H, P)), lo=0.0, hi=math.log(16.0))
        gap = d.exponential(B, L, 1)
        s = dict(u=d.normal(B, L, H * P, dtype=dt_),
                 B=d.normal(B, L, H, P, scale=P ** -0.5, dtype=dt_),
                 C=d.normal(B, L, H, P, scale=P ** -0.5, dtype=dt_),
                 dt=torch.nn.functional.softplus(d.normal(B, L, H)) * gap, A_log=a_log,
                 D=None, h0=None)
        if c["extras"]:
            s.update(D=d.normal(H * P), h0=d.normal(B, H, P))
        return s
    if k in ("selective", "xproj"):
        B, L, D, N = c["B"], c["L"], c["D"], c["N"]
        s = dict(x=d.normal(B, L, D, dtype=dt_),
                 A_log=d.uniform(D, N, lo=math.log(0.5), hi=math.log(5.0)), D=None, h0=None)
        if k == "xproj":
            R = c["R"]
            bias = math.log(math.expm1(0.05)) + d.uniform(D, lo=-0.5, hi=0.5)
            s.update(W_x=d.normal(D, R + 2 * N, scale=D ** -0.5),
                     W_dt=d.normal(R, D, scale=0.5 * R ** -0.5), bias=bias, D=d.normal(D))
            return s
        shape = (B, L, D) if c["per_channel_dt"] else (B, L)
        s.update(dt=d.exponential(*shape, mean=0.05).clamp_(1e-3, 1.0),
                 B=d.normal(B, L, N, scale=N ** -0.5, dtype=dt_),
                 C=d.normal(B, L, N, scale=N ** -0.5, dtype=dt_))
        if c["extras"]:
            s.update(D=d.normal(D), h0=d.normal(B, D, N))
        return s
    if k == "interp":
        B, T, F, N = c["B"], c["T"], c["F"], c["N"]
        M = (d.uniform(B, T, F) < c["observed"]).float()
        return dict(V=d.normal(B, T, F) * M, M=M,
                    tau=torch.sort(d.uniform(B, T, hi=T * 100.0 / 2048), dim=1).values,
                    A_log=d.uniform(F, N, lo=math.log(0.5), hi=math.log(5.0)),
                    B=d.normal(B, T, N, scale=N ** -0.5), C=d.normal(B, T, N, scale=N ** -0.5))
    if k == "ssd":
        B, L, H, P, N = c["B"], c["L"], c["H"], c["P"], c["N"]
        if c["gaps"] == "lognormal":
            dt = torch.exp(d.normal(B, L, H) * 1.5 - 3.0)
        else:
            dt = torch.nn.functional.softplus(d.normal(B, L, H)) * d.exponential(B, L, 1)
        s = dict(x=d.normal(B, L, H, P, dtype=dt_), dt=dt,
                 A_log=d.uniform(H, hi=math.log(16.0)),
                 B=d.normal(B, L, H, N, scale=N ** -0.5, dtype=dt_),
                 C=d.normal(B, L, H, N, scale=N ** -0.5, dtype=dt_), D=None, h0=None)
        if c["extras"]:
            s.update(D=d.normal(H, P), h0=d.normal(B, H, P, N))
        return s
    if k == "stream":
        S, H, P, N = c["S"], c["H"], c["P"], c["N"]
        return dict(x=d.normal(S, H, P), dt=d.exponential(S, mean=0.1),
                    A_log=d.uniform(H, hi=math.log(16.0)),
                    B=d.normal(S, H, N, scale=N ** -0.5), C=d.normal(S, H, N, scale=N ** -0.5),
                    D=d.normal(H, P), state=d.normal(S, H, P, N))
    if k == "train":
        B, L, H = c["B"], c["L"], c["H"]
        gap = d.exponential(B, L, 1, mean=0.3)
        rate = torch.exp(d.uniform(H, lo=math.log(0.5), hi=math.log(5.0)))
        return dict(u=d.normal(B, L, H, dtype=dt_), A=torch.exp(-gap * rate).to(dt_),
                    B=(d.normal(B, L, H) * gap).to(dt_), C=d.normal(B, L, H, dtype=dt_),
                    D=d.normal(H, dtype=dt_), dY=d.normal(B, L, H, dtype=dt_))
    S, H, K = c["S"], c["H"], c["K"]
    return dict(V=d.normal(S, K + 1, H), M=(d.uniform(S, K + 1, H) < c["observed"]).float(),
                tau=torch.arange(K + 1, device="cuda", dtype=torch.float32).repeat(S, 1),
                head=torch.randint(0, K + 1, (S,), generator=d.g, device="cuda",
                                   dtype=torch.int32),
                h=d.normal(S, H), v=d.normal(S, H),
                m=(d.uniform(S, H) < c["observed"]).float(), tau_new=d.uniform(S, lo=50.0, hi=60.0),
                Abar=torch.exp(-0.3 * d.uniform(H, lo=0.5, hi=5.0)), Bbar=d.normal(H, scale=0.3),
                C=d.normal(S, H), D=d.normal(H))


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "ring":
        ring = RingSession(case["S"], case["H"], case["K"], block_h=128, device="cuda")
        ring.ring_V, ring.ring_M, ring.ring_tau = s.pop("V"), s.pop("M"), s.pop("tau")
        ring.ring_head, ring.h = s.pop("head"), s.pop("h")
        s["ring"] = ring
    s["case"] = case
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "multihead":
        return tssm.multihead_ssm_forward(s["u"], s["A_log"], s["B"], s["C"], s["dt"], s["D"],
                                          disc=c["disc"], h0=s["h0"], return_state=c["extras"])
    if k == "selective":
        return tssm.selective_scan_forward(s["x"], s["dt"], s["A_log"], s["B"], s["C"], s["D"],
                                           h0=s["h0"], return_state=c["extras"])
    if k == "xproj":
        return tssm.selective_scan_forward(s["x"], None, s["A_log"], None, None, s["D"],
                                           return_state=True,
                                           x_proj=(s["W_x"], s["W_dt"], s["bias"], 1e-3, 0.1))
    if k == "interp":
        return tssm.fused_interp_ssm_forward(s["V"], s["M"], s["tau"], s["A_log"], s["B"], s["C"],
                                             K=c["K"], FTILE=c["FTILE"], return_state=True)
    if k == "ssd":
        return tssm.ssd_scan_forward(s["x"], s["dt"], s["A_log"], s["B"], s["C"], s["D"],
                                     h0=s["h0"], return_state=c["extras"])
    if k == "stream":
        y = tssm.ssd_stream_step(s["x"], s["dt"], s["A_log"], s["B"], s["C"], s["D"], s["state"])
        return y, s["state"]
    if k == "train":
        y, h = ssm_forward(s["u"], s["A"], s["B"], s["C"], s["D"])
        return (y, h) + tuple(ssm_backward(s["u"], s["A"], s["B"], s["C"], h, s["dY"]))
    r = s["ring"]
    y = r.step(s["v"], s["m"], s["tau_new"], s["Abar"], s["Bbar"], s["C"], s["D"])
    return y, r.h, r.ring_V, r.ring_M, r.ring_tau, r.ring_head


# ------------------------------------------------------------------ cost and precision
def work(c):
    k, e = c["kind"], BYTES[c.get("dtype", "f32")]
    if k == "multihead":
        n, rows = c["B"] * c["L"] * c["H"] * c["P"], c["B"] * c["L"] * c["H"]
        state = c["B"] * c["H"] * c["P"] * 8 + c["H"] * c["P"] * 4 if c["extras"] else 0
        return dict(bytes=4 * n * e + rows * 4 + c["H"] * (1 if c["per_head"] else c["P"]) * 4
                    + state, flops=8 * n)
    if k == "selective":
        n, rows = c["B"] * c["L"] * c["D"], c["B"] * c["L"]
        state = c["B"] * c["D"] * c["N"] * 8 + c["D"] * 4 if c["extras"] else 0
        return dict(bytes=2 * n * e + (n if c["per_channel_dt"] else rows) * 4
                    + 2 * rows * c["N"] * e + c["D"] * c["N"] * 4 + state, flops=8 * n * c["N"])
    if k == "xproj":
        n, cols = c["B"] * c["L"] * c["D"], c["R"] + 2 * c["N"]
        return dict(bytes=8 * n + c["D"] * (cols + c["R"] + c["N"] + 2) * 4
                    + c["B"] * c["D"] * c["N"] * 4,
                    flops=8 * n * c["N"] + 2 * n * (cols + c["R"]))
    if k == "interp":
        n, rows = c["B"] * c["T"] * c["F"], c["B"] * c["T"]
        return dict(bytes=16 * n + rows * (4 + 8 * c["N"]) + c["F"] * c["N"] * 4
                    + c["B"] * c["F"] * c["N"] * 4, flops=8 * n * c["N"] + 3 * n)
    if k == "ssd":
        rows = c["B"] * c["L"] * c["H"]
        state = c["B"] * c["H"] * c["P"] * c["N"] * 8 + c["H"] * c["P"] * 4 if c["extras"] else 0
        return dict(bytes=rows * (2 * (c["P"] + c["N"]) * e + 4) + c["H"] * 4 + state,
                    flops=5 * rows * c["P"] * c["N"])
    if k == "stream":
        n = c["S"] * c["H"]
        return dict(bytes=n * (8 * c["P"] * c["N"] + 8 * c["P"] + 8 * c["N"]) + c["S"] * 4,
                    flops=5 * n * c["P"] * c["N"])
    if k == "train":
        n = c["B"] * c["L"] * c["H"]
        # forward: u, A, B, C in, y, h out; backward: u, A, B, C, h, dY in, four gradients out
        return dict(bytes=16 * n * e, flops=14 * n)
    n = c["S"] * c["H"]
    return dict(bytes=32 * n, flops=6 * n)


def tolerance(c):
    k, t = c["kind"], c.get("dtype", "f32")
    if t == "f32":
        return {"rel": 4e-6}
    return {"rel": 8e-3 if t == "bf16" else 1e-3}


# ------------------------------------------------------------------ float64 restatements
def _coef(dt, a, disc):
    return torch.expm1(dt * a) / a if disc == "zoh" else dt + 0 * a


def _ssd_exact(s, Q=64):
    """Chunked dual form: within a chunk sum_s exp(cum_t - cum_s) coef_s (C_t.B_s) x_s, across
    chunks the state."""
    x, dt, Bm, Cm = (s[k].double() for k in ("x", "dt", "B", "C"))
    Bsz, L, H, P = x.shape
    N, pad = Bm.shape[-1], (-L) % Q
    a = -torch.exp(s["A_log"].double())

    def cut(t):  # [B, L, H, ...] -> [B, H, chunk, Q, ...]
        t = torch.nn.functional.pad(t, (0, 0) * (t.dim() - 2) + (0, pad))
        return t.reshape(Bsz, -1, Q, *t.shape[2:]).movedim(3, 1).contiguous()

    dtc = cut(dt)
    la = dtc * a[None, :, None, None]
    coef, cum = torch.expm1(la) / a[None, :, None, None], torch.cumsum(la, -1)
    xc, bc, cc = cut(x) * coef[..., None], cut(Bm), cut(Cm)
    keep = torch.ones(Q, Q, dtype=torch.bool, device=x.device).tril()
    M = (cum[..., :, None] - cum[..., None, :]).masked_fill_(~keep, -math.inf).exp_()
    M *= torch.matmul(cc, bc.transpose(-1, -2).contiguous())
    y = torch.matmul(M, xc)
    del M
    end = torch.matmul((xc * torch.exp(cum[..., -1:] - cum)[..., None]).transpose(-1, -2)
                       .contiguous(), bc)
    h = torch.zeros(Bsz, H, P, N, dtype=torch.float64, device=x.device) if s["h0"] is None \
        else s["h0"].double()
    decay, enter = torch.exp(cum[..., -1]), torch.empty_like(end)
    for i in range(end.shape[2]):
        enter[:, :, i] = h
        h = decay[:, :, i, None, None] * h + end[:, :, i]
    y += torch.exp(cum)[..., None] * torch.matmul(cc, enter.transpose(-1, -2).contiguous())
    y = y.movedim(1, 3).reshape(Bsz, -1, H, P)[:, :L]
    if s["D"] is not None:
        y = y + s["D"].double().reshape(H, P) * x
    return y, h


def _selective_exact(x, dt, A_log, Bm, Cm, D=None, h0=None):
    x, dt, Bm, Cm, A_log = (t.double() for t in (x, dt, Bm, Cm, A_log))
    a = -torch.exp(A_log)
    if dt.dim() == 2:
        dt = dt[..., None].expand_as(x)
    h = torch.zeros(x.shape[0], *a.shape, dtype=torch.float64, device=x.device) if h0 is None \
        else h0.double()
    y = torch.empty_like(x)
    for t in range(x.shape[1]):
        em = torch.expm1(dt[:, t, :, None] * a)
        h = h + em * (h + x[:, t, :, None] * Bm[:, t, None] / a)
        y[:, t] = (h * Cm[:, t, None]).sum(-1)
    return (y if D is None else y + D.double() * x), h


def _interp_exact(V, M, tau, K, FTILE):
    V, M, tau = V.double(), M.double(), tau.double()
    Bsz, T, F = V.shape
    nt = -(-F // FTILE)
    seen = torch.nn.functional.pad(M, (0, nt * FTILE - F)).reshape(Bsz, T, nt, FTILE).sum(-1) > 0.5
    prev = torch.full((Bsz, T, nt), -1, device=V.device)
    nxt = prev.clone()
    at = torch.arange(T, device=V.device)[None, :, None]
    for k in range(min(K, T - 1), 0, -1):
        prev[:, k:] = torch.where(seen[:, :-k], (at - k)[:, k:], prev[:, k:])
        nxt[:, :-k] = torch.where(seen[:, k:], (at + k)[:, :-k], nxt[:, :-k])
    tile = torch.arange(F, device=V.device) // FTILE
    p, n = prev[..., tile], nxt[..., tile]
    wide = tau[..., None].expand_as(V)
    tp, tn = wide.gather(1, p.clamp(min=0)), wide.gather(1, n.clamp(min=0))
    w = torch.where(tn - tp > 1e-9, (wide - tp) / (tn - tp), 0.5).clamp(0.0, 1.0)
    vp, vn = V.gather(1, p.clamp(min=0)), V.gather(1, n.clamp(min=0))
    out = torch.where(n >= 0, vn, V)
    out = torch.where(p >= 0, vp, out)
    return torch.where((p >= 0) & (n >= 0), (1.0 - w) * vp + w * vn, out)


def exact(case, seed):
    s, k = _inputs(case, seed), case["kind"]
    if k == "multihead":
        H, P = case["H"], case["P"]
        Bm, C, dt = s["B"].double(), s["C"].double(), s["dt"].double()[..., None]
        u = s["u"].double().reshape(Bm.shape)
        a = -torch.exp(s["A_log"].double()).reshape(H, -1).expand(H, P)
        A, h = torch.exp(dt * a), _coef(dt, a, case["disc"]) * Bm * u
        prev = torch.zeros_like(h[:, 0]) if s["h0"] is None else s["h0"].double()
        for t in range(h.shape[1]):
            prev = h[:, t].addcmul_(A[:, t], prev)
        y = (C * h).sum(-1)
        if s["D"] is not None:
            y += (u * s["D"].double().reshape(H, P)).sum(-1)
        y = y.repeat_interleave(P, -1)
        return (y, h[:, -1]) if case["extras"] else y
    if k == "selective":
        y, h = _selective_exact(s["x"], s["dt"], s["A_log"], s["B"], s["C"], s["D"], s["h0"])
        return (y, h) if case["extras"] else y
    if k == "xproj":
        R, N = case["R"], case["N"]
        z = torch.matmul(s["x"].double(), s["W_x"].double())
        dt = torch.matmul(z[..., :R], s["W_dt"].double()) + s["bias"].double()
        dt = torch.logaddexp(dt, torch.zeros_like(dt)).clamp(1e-3, 0.1)
        return _selective_exact(s["x"], dt, s["A_log"], z[..., R:R + N], z[..., R + N:], s["D"])
    if k == "interp":
        Vhat = _interp_exact(s["V"], s["M"], s["tau"], case["K"], case["FTILE"])
        tau = s["tau"].double()
        dt = torch.diff(tau, dim=1, prepend=torch.zeros_like(tau[:, :1]))
        return (Vhat,) + _selective_exact(Vhat, dt, s["A_log"], s["B"], s["C"])
    if k == "ssd":
        y, h = _ssd_exact(s)
        return (y, h) if case["extras"] else y
    if k == "stream":
        x, Bm, C, dt = (s[n].double() for n in ("x", "B", "C", "dt"))
        la = -dt[:, None] * torch.exp(s["A_log"].double())
        coef = torch.expm1(la) / -torch.exp(s["A_log"].double())
        h = s["state"].double().mul_(torch.exp(la)[..., None, None])
        h += (coef[..., None] * x)[..., None] * Bm[:, :, None]
        y = torch.matmul(h, C[..., None])[..., 0] + s["D"].double() * x
        return y, h
    if k == "train":
        u, A, Bm, C, dY = (s[n].double() for n in ("u", "A", "B", "C", "dY"))
        h, dh = Bm * u, C * dY
        for t in range(1, h.shape[1]):
            h[:, t].addcmul_(A[:, t], h[:, t - 1])
        y = C * h + s["D"].double() * u
        if case["dtype"] != "f32":
            h_in = h.to(DTYPES[case["dtype"]]).double()   # the backward is given the stored states
        else:
            h_in = h
        for t in range(h.shape[1] - 2, -1, -1):
            dh[:, t].addcmul_(A[:, t + 1], dh[:, t + 1])
        before = torch.cat([torch.zeros_like(h[:, :1]), h_in[:, :-1]], 1)
        return y, h, Bm * dh, before * dh, u * dh, dY * h_in
    head = (s["head"].long() + 1) % (case["K"] + 1)
    rows, n = torch.arange(case["S"], device="cuda"), case["K"] + 1
    V, M, tau, H = s["V"].double(), s["M"].double(), s["tau"].double(), case["H"]
    V[rows, head], M[rows, head], tau[rows, head] = s["v"].double(), s["m"].double(), \
        s["tau_new"].double()
    nt = -(-H // 128)

    def tiles(t):
        return torch.nn.functional.pad(t, (0, nt * 128 - H)).reshape(*t.shape[:-1], nt, 128).sum(-1)

    seen, now = tiles(M) > 0.5, tiles(s["m"].double())
    slot = torch.full((case["S"], nt), -1, device="cuda")
    for j in range(n - 1, 0, -1):
        at = (head - j) % n
        slot = torch.where(seen[rows, at], at[:, None], slot)
    slot = torch.where(now < 0.5, slot, -1).repeat_interleave(128, 1)[:, :H]
    old = V.gather(1, slot.clamp(min=0)[:, None])[:, 0]
    vhat = torch.where(slot >= 0, old, s["v"].double())
    h = s["Abar"].double() * s["h"].double() + s["Bbar"].double() * vhat
    return (s["C"].double() * h + s["D"].double() * vhat, h, V, M, tau, head.to(torch.int32))
