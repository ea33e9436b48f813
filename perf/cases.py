"""Performance cases of the recurrences: what a program that uses this package has it do.

Each case is one pass through public entry points at the sizes of the
package's own configurations (gdnx_amd.workloads, bench.py, the reference
layer's defaults) or of ordinary use:

  kind          entry point                               in real use
  scan_train    gdn3.gdn3_scan forward + backward         a training step of the dense-state GDN3 recurrence
  scan_prefill  gdn3.gdn3_scan, no gradient, final state  a prompt taken in before decoding
  decode        decode_cache.DecodeStateCache.step        one served token per sequence (dense state)
  decode_gdn3   gdn3.gdn3_decode_step                     one served token per sequence (Kronecker-residual state)
  layer_train   layer.gdn3_layer_core forward + backward  a training step of the GDN3 layer's core (gates, decay and
                                                          RoPE, the recurrence with its compactions, routing and norm)
  gdn3_prefill  gdn3.gdn3_recurrent_state, no gradient    a long prompt in the Kronecker-residual regime
  kmd2_train    kmd2.scan forward + backward              a training step of the KMD-2 recurrence (a decay per channel)
  kmd2_eval     kmd2.scan, no gradient                    its evaluation
  rls_train     rls.rls_scan forward + backward           a training step of the rank-r RLS variant

Work counts, for every token and chain, the products of the recurrence itself
with its state of D x D values (read, erase, write: 6 D^2 operations forward,
twice as much again backward), and each input, output and gradient once.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from gdnx_amd import gdn3, kmd2, layer, rls
from gdnx_amd.decode_cache import DecodeStateCache

DEV = "cuda"
TAUS = (0.05, 0.02, 0.005, 0.001)      # the lanes' decay timescales
SLOW_DECAY = 0.97                      # the layer's blend of compacted factors
RANK = 4                               # Kronecker terms of the GDN3 state


def _factors(D):
    return (16, 16, 8, 8) if D == 128 else (8, 8, 8, 8)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the headline training step: four sequences of 4096 tokens, the 16-head layer with four lanes
        dict(name="scan_train_layer", kind="scan_train", B=4, T=4096, H=16, M=4, D=128, dtype="bf16"),
        # fine-tuning on one document at a time: one sequence, a length that fills no chunk
        dict(name="scan_train_one", kind="scan_train", B=1, T=1999, H=16, M=4, D=128, dtype="bf16"),
        # the small float32 model of experiments and gradient checks
        dict(name="scan_train_f32", kind="scan_train", B=1, T=256, H=2, M=1, D=64, dtype="f32"),
        # a prompt before decoding
        dict(name="scan_prefill", kind="scan_prefill", B=1, T=8190, H=16, M=4, D=128, dtype="bf16"),
        # a full serving batch: 256 sequences, 16 heads of 4 lanes x 4 decays
        dict(name="decode_batch", kind="decode", B=256, H=16, M=16, D=128, dtype="bf16"),
        # a few interactive users: the smallest call, latency and launches
        dict(name="decode_few", kind="decode", B=3, H=16, M=4, D=128, dtype="bf16"),
        # serving the reference layer's own state; the sequences are at different positions, so a sixteenth of them compacts
        dict(name="decode_gdn3", kind="decode_gdn3", B=256, H=16, M=4, D=128, P=16, every=16, dtype="bf16"),
        # a training step of the layer as the reference runs it (a compaction every 16 tokens)
        dict(name="layer_train", kind="layer_train", B=4, T=4096, H=16, M=4, D=128, P=16, every=16, dtype="bf16"),
        # long context: 32768 tokens, a compaction every 2048
        dict(name="gdn3_longctx", kind="gdn3_prefill", B=1, T=32768, H=16, M=4, D=128, P=16, every=2048, dtype="bf16"),
        # the reference's scan benchmark, training and evaluation shapes
        dict(name="kmd2_train", kind="kmd2_train", B=2, T=512, H=16, r_out=4, D=128, dtype="f32"),
        dict(name="kmd2_eval", kind="kmd2_eval", B=1, T=2048, H=16, r_out=4, D=128, dtype="f32"),
        # the RLS layer's defaults
        dict(name="rls_train", kind="rls_train", B=8, T=1024, H=16, r=1, r_out=1, D=64, dtype="f32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("scan_train", "scan_train", "scan_prefill", "decode", "decode_gdn3", "layer_train",
                       "gdn3_prefill", "kmd2_train", "kmd2_eval", "rls_train"))
    D = rng.choice((64, 128, 128))
    if kind in ("scan_train", "scan_prefill"):
        dtype = rng.choice(("bf16", "bf16", "bf16", "f32"))
        B, H, M = rng.randint(1, 4), rng.choice((2, 4, 8, 16)), rng.choice((1, 2, 4, 4))
        cap = (4 if dtype == "bf16" else 1) * 4096 * 64
        return dict(kind=kind, B=B, T=min(_log_int(rng, 64, 8192), cap // (B * H * M)), H=H, M=M, D=D, dtype=dtype)
    if kind == "decode":
        return dict(kind=kind, B=_log_int(rng, 1, 256), H=rng.choice((4, 8, 16)), M=rng.choice((1, 4, 16)), D=D,
                    dtype=rng.choice(("bf16", "f32")))
    if kind == "decode_gdn3":
        return dict(kind=kind, B=_log_int(rng, 1, 256), H=rng.choice((8, 16)), M=rng.choice((1, 4)), D=D, P=16,
                    every=rng.choice((16, 64)), dtype="bf16")
    if kind == "layer_train":
        return dict(kind=kind, B=rng.randint(1, 4), T=_log_int(rng, 64, 2048), H=rng.choice((8, 16)),
                    M=rng.choice((2, 4)), D=D, P=16, every=16, dtype="bf16")
    if kind == "gdn3_prefill":
        return dict(kind=kind, B=rng.randint(1, 2), T=_log_int(rng, 512, 16384), H=rng.choice((8, 16)), M=4, D=D,
                    P=rng.choice((16, 32)), every=rng.choice((512, 2048)), dtype="bf16")
    if kind in ("kmd2_train", "kmd2_eval"):
        return dict(kind=kind, B=rng.randint(1, 4), T=_log_int(rng, 64, 2048), H=rng.choice((4, 8, 16)),
                    r_out=rng.choice((1, 4)), D=D, dtype="f32")
    return dict(kind=kind, B=rng.randint(1, 8), T=_log_int(rng, 64, 1024), H=rng.choice((4, 8, 16)),
                r=rng.choice((1, 2, 4)), r_out=rng.choice((1, 2)), D=rng.choice((32, 64)), dtype="f32")


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _io(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


class _Draws:
    """Values of one seed, drawn on the GPU in a fixed order."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(int(seed) % (1 << 63))

    def n(self, *shape):
        return torch.randn(*shape, generator=self.gen, device=DEV)

    def unit(self, *shape):
        return F.normalize(self.n(*shape), dim=-1)

    def gate(self, *shape):
        return torch.sigmoid(self.n(*shape))


def _lane_log_decay(d, M, *lead):
    """log(1 - tau) of the lane's timescale (the four in turn) + N(0, 0.01^2)."""
    base = torch.tensor([math.log(1.0 - TAUS[m % 4]) for m in range(M)], device=DEV)
    return base + 0.01 * d.n(*lead, M)


def _tensors(case, seed):
    """The inputs of a case by name, in the types that the call takes."""
    d, kind, io = _Draws(seed), case["kind"], _io(case)
    B, T, H, M, D = (case.get(n) for n in ("B", "T", "H", "M", "D"))
    if kind in ("scan_train", "scan_prefill"):
        x = dict(q=d.unit(B, T, H, D).to(io), k=d.unit(B, T, H, D).to(io), v=d.n(B, T, H, D).to(io),
                 beta=d.gate(B, T, H, M), log_g=_lane_log_decay(d, M, B, T, H))
        if kind == "scan_train":
            x["dy"] = d.n(B, T, H, M, D).to(io)
        return x
    if kind == "decode":
        return dict(q=d.unit(B, H, D).to(io), k=d.unit(B, H, D).to(io), v=d.n(B, H, D).to(io), a_e=d.gate(B, H, M),
                    a_w=d.gate(B, H, M), log_g=_lane_log_decay(d, M, B, H).clamp(max=0.0),
                    state=d.n(B, H, M, D, D).mul_(0.02))
    if kind == "decode_gdn3":
        a_v, a_k, b_v, b_k = _factors(D)
        return dict(q=d.unit(B, H, M, D).to(io), k=d.unit(B, H, M, D).to(io), v=d.n(B, H, D).to(io),
                    b=d.gate(B, H, M, D), w=d.gate(B, H, M, D),
                    decay=_lane_log_decay(d, M, B, H).clamp(max=0.0).exp(),
                    A=0.2 * d.n(B, H, M, RANK, a_v, a_k), Bf=0.1 * d.n(B, H, M, RANK, b_v, b_k),
                    U=0.4 * d.n(B, H, M, D, case["P"]), Vb=0.9 * d.unit(B, H, M, case["P"], D).transpose(-1, -2),
                    pos=(4096 + 5 * torch.arange(B, device=DEV)).to(torch.int32))
    if kind == "layer_train":
        return dict(q=d.unit(B, T, H, D).to(io), k=d.unit(B, T, H, D).to(io), v=d.n(B, T, H, D).to(io),
                    b_proj=d.n(B, T, H, M, D).to(io), proj_a=d.n(B, T, H).to(io), w_proj=d.n(B, T, H, M, D).to(io),
                    proj_b=d.n(B, T, H).to(io), decay_proj=d.n(B, T, H, M, 4).mul_(3).to(io),
                    rates=torch.tensor(TAUS, device=DEV), router=d.n(B, T, H, M).to(io),
                    norm=0.5 + torch.rand(D, generator=d.gen, device=DEV), dout=d.n(B, T, H, D).to(io))
    if kind == "gdn3_prefill":
        return dict(q=d.unit(B, T, H, D).to(io), k=d.unit(B, T, H, D).to(io), v=d.n(B, T, H, D).to(io),
                    b=d.gate(B, T, H, M), w=d.gate(B, T, H, M),
                    decay=_lane_log_decay(d, M, B, T, H).clamp(max=0.0).exp())
    if kind in ("kmd2_train", "kmd2_eval"):
        r = case["r_out"]
        x = dict(q=d.n(B, T, H, r, D).mul_(D ** -0.5), k=d.unit(B, T, H, D), v=d.n(B, T, H, D),
                 g=torch.exp(-F.softplus(d.n(B, T, H, D) * 1.2 - 0.6)), beta_e=d.gate(B, T, H),
                 beta_w=d.gate(B, T, H), out_mix=d.n(H, r))
        if kind == "kmd2_train":
            x["dy"] = d.n(B, T, H, D)
        return x
    r, ro = case["r"], case["r_out"]
    return dict(q=d.unit(B, T, H, ro, D), K=d.unit(B, T, H, r, D), V=d.n(B, T, H, r, D), Bg=d.gate(B, T, H, r, D),
                Wg=d.gate(B, T, H, r, D), a=torch.sigmoid(0.5 * d.n(B, T, H, D) + 6.0).clamp(max=0.999),
                out_mix=d.n(H, ro), dy=d.n(B, T, H, D))


# the inputs that get a gradient, in the order of the outputs
GRADS = {
    "scan_train": ("q", "k", "v", "beta", "log_g"),
    "layer_train": ("q", "k", "v", "b_proj", "proj_a", "w_proj", "proj_b", "decay_proj", "router", "norm"),
    "kmd2_train": ("q", "k", "v", "g", "beta_e", "beta_w", "out_mix"),
    "rls_train": ("q", "K", "V", "Bg", "Wg", "a", "out_mix"),
}


def _grad_names(case):
    names = GRADS.get(case["kind"], ())
    return names[:-1] if "out_mix" in names and case["r_out"] == 1 else names


def prepare(case, seed):
    x = _tensors(case, seed)
    st = dict(case=case, x=x)
    for n in _grad_names(case):
        x[n].requires_grad_(True)
    if case["kind"] == "decode":
        # a serving loop's cache, its sequences' states in slots that are in no order
        B = case["B"]
        cache = DecodeStateCache(B, case["H"], case["M"], case["D"], device=DEV)
        slots = cache.alloc(B)
        slots = [slots[(7 * i + 3) % B] for i in range(B)] if math.gcd(7, B) == 1 else slots
        init = x.pop("state")
        for i, s in enumerate(slots):
            cache.state(s).copy_(init[i])
        st.update(cache=cache, slots=slots)
    if case["kind"] == "decode_gdn3":
        x["Vb"] = x["Vb"].contiguous()
        st["state"] = tuple(x.pop(n) for n in ("A", "Bf", "U", "Vb"))
    return st


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    wrt = [x[n] for n in _grad_names(case)]
    if kind == "scan_train":
        y = gdn3.gdn3_scan(x["q"], x["k"], x["v"], x["beta"], x["log_g"])
        return (y, *torch.autograd.grad(y, wrt, x["dy"]))
    if kind == "scan_prefill":
        with torch.no_grad():
            return gdn3.gdn3_scan(x["q"], x["k"], x["v"], x["beta"], x["log_g"], return_state=True)
    if kind == "decode":
        y = state["cache"].step(state["slots"], x["q"], x["k"], x["v"], x["a_e"], x["a_w"], x["log_g"])
        return y, state["cache"].pool
    if kind == "decode_gdn3":
        H, M, D = case["H"], case["M"], case["D"]
        v = x["v"].unsqueeze(2).expand(case["B"], H, M, D)
        with torch.no_grad():
            y = gdn3.gdn3_decode_step(x["q"], x["k"], v, x["b"], x["w"], x["decay"], state["state"], x["pos"],
                                      R=RANK, P=case["P"], factors=_factors(D), slow_decay=SLOW_DECAY,
                                      compact_every=case["every"])
            x["pos"].add_(1)
        return (y, *state["state"])
    if kind == "layer_train":
        out = layer.gdn3_layer_core(x["q"], x["k"], x["v"], x["b_proj"], x["proj_a"], x["w_proj"], x["proj_b"],
                                    x["decay_proj"], x["rates"], x["router"], x["norm"], R=RANK, P=case["P"],
                                    factors=_factors(case["D"]), slow_decay=SLOW_DECAY, compact_every=case["every"])
        return (out, *torch.autograd.grad(out, wrt, x["dout"]))
    if kind == "gdn3_prefill":
        with torch.no_grad():
            y, s, _ = gdn3.gdn3_recurrent_state(x["q"], x["k"], x["v"], x["b"], x["w"], x["decay"], R=RANK,
                                                P=case["P"], factors=_factors(case["D"]), slow_decay=SLOW_DECAY,
                                                compact_every=case["every"], return_state=True)
        return (y, *s)
    if kind in ("kmd2_train", "kmd2_eval"):
        args = [x[n] for n in ("q", "k", "v", "g", "beta_e", "beta_w")]
        mix = x["out_mix"] if case["r_out"] > 1 else None
        if kind == "kmd2_eval":
            with torch.no_grad():
                return kmd2.scan(*args, mix)
        y = kmd2.scan(*args, mix)
        return (y, *torch.autograd.grad(y, wrt, x["dy"]))
    y = rls.rls_scan(x["q"], x["K"], x["V"], x["Bg"], x["Wg"], x["a"],
                     out_mix=x["out_mix"] if case["r_out"] > 1 else None)
    return (y, *torch.autograd.grad(y, wrt, x["dy"]))


def work(case):
    kind, io = case["kind"], (2 if case["dtype"] == "bf16" else 4)
    B, T, H, D = case["B"], case.get("T", 1), case["H"], case["D"]
    M = case.get("M", 1)
    rows, chains = B * T * H, B * T * H * M
    qkv, gates = 3 * rows * D * io, 2 * chains * 4
    if kind == "scan_train":
        y = chains * D * io
        return {"bytes": 2 * qkv + 2 * gates + 2 * y, "flops": 18 * chains * D * D}
    if kind == "scan_prefill":
        return {"bytes": qkv + gates + chains * D * io + B * H * M * D * D * 4, "flops": 6 * chains * D * D}
    if kind == "decode":
        return {"bytes": qkv + 3 * chains * 4 + chains * D * io + 2 * chains * D * D * 4, "flops": 6 * chains * D * D}
    if kind == "decode_gdn3":
        a_v, a_k, b_v, b_k = _factors(D)
        P = case["P"]
        fac = RANK * (a_v * a_k + b_v * b_k)
        state = 2 * fac + 2 * P * D + (P + 1) * D      # A, B and Vb both ways, U in, one slot of it out
        flops = 2 * (2 * RANK * D * (a_k + b_v) + 4 * P * D)
        # q, k per lane, v per head, the gates per channel, y
        return {"bytes": chains * (3 * D * io + 2 * D * 4 + 4 + state * 4) + rows * D * io, "flops": chains * flops}
    if kind == "layer_train":
        # q, k, v, the projections, the router, out and their gradients; the Kronecker reads of h and q, the window
        per = rows * (3 * D + 2 * M * D + 2 + 4 * M + M + D) * io
        return {"bytes": 2 * per, "flops": 3 * chains * (2 * 4 * RANK * D * 16 + 8 * case["P"] * D)}
    if kind == "gdn3_prefill":
        return {"bytes": qkv + 3 * chains * 4 + chains * D * io,
                "flops": chains * (2 * 4 * RANK * D * 16 + 8 * case["P"] * D)}
    if kind in ("kmd2_train", "kmd2_eval"):
        per = rows * (case["r_out"] * D + 3 * D + 2) * 4
        y = rows * D * 4
        if kind == "kmd2_eval":
            return {"bytes": per + y, "flops": rows * (7 * D * D + 2 * case["r_out"] * D)}
        return {"bytes": 2 * per + 2 * y, "flops": 3 * rows * (7 * D * D + 2 * case["r_out"] * D)}
    r, ro = case["r"], case["r_out"]
    per = rows * (ro * D + 4 * r * D + D) * 4
    return {"bytes": 2 * per + 2 * rows * D * 4, "flops": 3 * rows * D * D * (1 + 6 * r + 2 * ro)}


def tolerance(case):
    """Two correct runs at the same precision, from the distance of one to the
    same in 64 bits.  bf16 operands, float32 sums: 3.4e-3 (outputs) to 6e-3
    (the decays' gradients) in a training step, 1.7e-3 in a decode step, which
    only rounds its output.  float32 throughout: 2e-7 to 6e-7, and single
    values up to 1e-4 of the root mean square in KMD-2's decay gradients, which
    are differences of large sums.  Compacted factors (gdn3_prefill): 2e-3,
    through the gaps of the singular values.  The layer's gradients of q and k
    have single values 0.3 off where a head's routed output is nearly zero
    and its norm divides by it."""
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind == "decode":
        return {"rel": 7e-3, "max": 1.6e-2} if bf16 else {"rel": 1e-6, "max": 1e-5}
    if not bf16:
        return {"rel": 3e-6, "max": 5e-4 if kind == "kmd2_train" else 5e-5}
    return {"scan_train": {"rel": 1.5e-2, "max": 0.2}, "scan_prefill": {"rel": 1.2e-2, "max": 0.1},
            "decode_gdn3": {"rel": 7e-3, "max": 1.6e-2}, "layer_train": {"rel": 1.5e-2, "max": 1.0},
            "gdn3_prefill": {"rel": 8e-3, "max": 0.2}}[kind]


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _alpha(c):
    """(1 - exp(-c)) / c, 1 at c = 0."""
    safe = torch.where(c == 0, torch.ones_like(c), c)
    return torch.where(c == 0, 1.0 - c / 2, -torch.expm1(-safe) / safe)


def _pad_tokens(x, n):
    return x if n == 0 else torch.cat([x, x.new_zeros(x.shape[0], n, *x.shape[2:])], 1)


def _dense_scan(q, k, v, beta, log_g, C=64):
    """The gated delta rule with a = alpha(beta |k|^2) beta, chunk by chunk."""
    B, T, H, D = q.shape
    M = beta.shape[-1]
    a = _alpha(beta * k.square().sum(-1, keepdim=True)) * beta
    g = log_g.clamp(max=0.0)
    n = -T % C
    q, k, v, a, g = (_pad_tokens(x, n) for x in (q, k, v, a, g))
    S = q.new_zeros(B * H * M, D, D)
    low = torch.ones(C, C, dtype=torch.bool, device=q.device).tril()
    eye = torch.eye(C, dtype=q.dtype, device=q.device)
    ys = []
    for t in range(0, T, C):
        def wide(x):        # [B,C,H,D] -> [N,C,D]
            return x[:, t:t + C].permute(0, 2, 1, 3).unsqueeze(2).expand(B, H, M, C, D).reshape(-1, C, D)

        def lane(x):        # [B,C,H,M] -> [N,C,1]
            return x[:, t:t + C].permute(0, 2, 3, 1).reshape(-1, C, 1)
        qc, kc, vc, ac, G = wide(q), wide(k), wide(v), lane(a), lane(g).cumsum(1)
        Dm = (G - G.transpose(1, 2)).masked_fill(~low, -math.inf).exp()
        L = ac * torch.bmm(kc, kc.transpose(1, 2).contiguous()) * Dm * (1 - eye)
        rhs = ac * vc - ac * G.exp() * torch.bmm(kc, S)
        R = torch.linalg.solve_triangular(eye + L, rhs, upper=False, unitriangular=True)
        y = G.exp() * torch.bmm(qc, S) + torch.bmm(torch.bmm(qc, kc.transpose(1, 2).contiguous()) * Dm, R)
        S = G[:, -1:].exp() * S + torch.bmm((kc * (G[:, -1:] - G).exp()).transpose(1, 2).contiguous(), R)
        ys.append(y)
    y = torch.cat(ys, 1)[:, :T].reshape(B, H, M, T, D).permute(0, 3, 1, 2, 4)
    return y, S.reshape(B, H, M, D, D)


def _orthonormal(Y):
    for _ in range(2):
        cols = []
        for i in range(Y.shape[-1]):
            c = Y[..., i]
            for p in cols:
                c = c - (p * c).sum(-1, keepdim=True) * p
            cols.append(c / c.norm(dim=-1, keepdim=True).clamp_min(1e-300))
        Y = torch.stack(cols, -1)
    return Y


def _compact(A, Bf, U, Vb, G):
    """The factors after a compaction: R terms of the rearranged A (x) B + U Vb^T
    by a sketched range finder (two power iterations), blended into the old ones."""
    N, R, a_v, a_k = A.shape
    b_v, b_k = Bf.shape[-2:]
    res = torch.bmm(U, Vb.transpose(1, 2).contiguous())
    res = res.reshape(N, a_v, b_v, a_k, b_k).permute(0, 1, 3, 2, 4).reshape(N, a_v * a_k, b_v * b_k)
    Rm = torch.bmm(A.reshape(N, R, -1).transpose(1, 2).contiguous(), Bf.reshape(N, R, -1)) + res
    RmT = Rm.transpose(1, 2).contiguous()
    Y = torch.bmm(Rm, G)
    for _ in range(2):
        Y = torch.bmm(Rm, torch.bmm(RmT, _orthonormal(Y)))
    Q = _orthonormal(Y)
    Bm = torch.bmm(Q.transpose(1, 2).contiguous(), Rm)
    w, E = torch.linalg.eigh(torch.bmm(Bm, Bm.transpose(1, 2).contiguous()).cpu())
    w, E = w.flip(-1)[:, :R].to(Rm.device), E.flip(-1)[:, :, :R].contiguous().to(Rm.device)
    s = w.clamp_min(0.0).sqrt()
    Vs = torch.bmm(RmT, torch.bmm(Q, E)) / s.clamp_min(1e-300)[:, None]
    at = Vs.abs().argmax(1, keepdim=True)
    sg = torch.where(Vs.gather(1, at) < 0, -1.0, 1.0).to(Vs.dtype)
    A2 = (torch.bmm(Q, E) * sg * s[:, None]).transpose(1, 2).reshape(A.shape)
    B2 = (Vs * sg).transpose(1, 2).reshape(Bf.shape)
    return SLOW_DECAY * A + (1 - SLOW_DECAY) * A2, SLOW_DECAY * Bf + (1 - SLOW_DECAY) * B2


def _sketch(N, n, q):
    gen = torch.Generator(device="cpu").manual_seed(1234)
    return torch.randn(N, n, q, generator=gen).double().to(DEV)


def _kron_matrix(A, Bf):
    N = A.shape[0]
    D = A.shape[2] * Bf.shape[2]
    return (A[:, :, :, None, :, None] * Bf[:, :, None, :, None, :]).sum(1).reshape(N, D, D)


def _kron_window_scan(q, k, v, b, w, decay, P, every):
    """The Kronecker-residual recurrence, window by window; q, k, v, b, w
    [B,T,H,M,D], decay [B,T,H,M]."""
    B, T, H, M, D = q.shape
    N = B * H * M
    a_v, a_k, b_v, b_k = _factors(D)
    q, k, h, u = (x.permute(0, 2, 3, 1, 4).reshape(N, T, D) for x in (q, k, b * k, w * v))
    alpha = _alpha((k * h).sum(-1))
    lg = decay.clamp(0.0, 1.0).log().permute(0, 2, 3, 1).reshape(N, T)
    A, Bf = q.new_zeros(N, RANK, a_v, a_k), q.new_zeros(N, RANK, b_v, b_k)
    U, Vb = q.new_zeros(N, P, D), q.new_zeros(N, P, D)
    G = _sketch(N, b_v * b_k, min(RANK + 4, a_v * a_k, b_v * b_k))
    acc, S = q.new_zeros(N, 1, 1), None
    ys = []

    def mT(x):
        return x.transpose(1, 2).contiguous()
    for t in range(0, T, P):
        c = min(P, T - t)
        qc, kc, hc, uc = (x[:, t:t + c] for x in (q, k, h, u))
        al, g = alpha[:, t:t + c, None], lg[:, t:t + c].cumsum(1)[..., None]
        low = torch.ones(c, c, dtype=torch.bool, device=q.device).tril()
        strict = torch.ones(c, c, dtype=torch.bool, device=q.device).tril(-1)
        old = torch.ones(c, P, dtype=torch.bool, device=q.device).triu()        # slot p still holds its old write up to token p
        Dm = (g - mT(g)).masked_fill(~low, -math.inf).exp()
        kT, VbT = mT(kc), mT(Vb)

        def past(x):
            r = torch.bmm(g.exp() * torch.bmm(x, VbT) * old, U)
            return r if S is None else r + (2 * (acc + g)).exp() * torch.bmm(x, mT(S))
        L = torch.bmm(hc, kT) * Dm * strict
        Un = torch.linalg.solve_triangular(torch.eye(c, dtype=q.dtype, device=q.device) + al * L,
                                           al * (uc - past(hc)), upper=False, unitriangular=True)
        ys.append(past(qc) + torch.bmm(torch.bmm(qc, kT) * Dm, Un))
        gl = g[:, -1:]
        U = torch.cat([Un, U[:, c:]], 1)
        Vb = torch.cat([kc * (gl - g).exp(), Vb[:, c:] * gl.exp()], 1)
        acc = acc + gl
        if (t + c) % every == 0:
            with torch.no_grad():
                f = acc.detach().exp()[..., None]
                A, Bf = _compact(A * f, Bf * f, mT(U.detach()), mT(Vb.detach()), G)
                S = _kron_matrix(A, Bf)
            acc = torch.zeros_like(acc)
    y = torch.cat(ys, 1).reshape(B, H, M, T, D).permute(0, 3, 1, 2, 4)
    f = acc.exp()[..., None]
    return y, (A * f, Bf * f, mT(U), mT(Vb))


def _lane_rope(x, M):
    """The layer's rotary embedding of lane-shared x [B,T,H,K] -> [B,T,H,M,K]:
    the second half of a pair reads the rotated first half; angles as the
    layer's float32 tables have them."""
    B, T, H, K = x.shape
    outs = []
    for m in range(M):
        frac, scale = (0.5, 0.25, 0.5, 0.5)[m], (1.0, 0.3, 0.5, 0.2)[m]
        d, width = int(K * frac // 2), int(K * 0.25) // 2
        if scale == 1.0 and d > width:
            outs.append(x)
            continue
        den = max(1, width - 1) if scale != 1.0 else max(1, d - 1)
        inv = 1.0 / (10000.0 ** (torch.arange(d, dtype=torch.float32, device=x.device) / den))
        ang = (torch.arange(T, dtype=torch.float32, device=x.device) * scale)[:, None] * inv
        cos, sin = ang.cos().to(x.dtype)[None, :, None], ang.sin().to(x.dtype)[None, :, None]
        x1 = x[..., :d] * cos - x[..., d:2 * d] * sin
        outs.append(torch.cat([x1, x1 * sin + x[..., d:2 * d] * cos, x[..., 2 * d:]], -1))
    return torch.stack(outs, 3)


def _layer64(x, P, every):
    M, D = x["b_proj"].shape[3], x["q"].shape[-1]
    b = torch.sigmoid(x["b_proj"] + 0.1 * x["proj_a"][..., None, None])
    w = torch.sigmoid(x["w_proj"] + 0.1 * x["proj_b"][..., None, None])
    dec = torch.exp(-F.softplus(x["decay_proj"]).clamp(max=5.0) * x["rates"]).mean(-1).clamp(max=0.999)
    v = x["v"].unsqueeze(3).expand_as(w)
    y, _ = _kron_window_scan(_lane_rope(x["q"], M), _lane_rope(x["k"], M), v, b, w, dec, P, every)
    routed = (torch.softmax(x["router"], -1).unsqueeze(-1) * y).sum(3)
    return F.normalize(routed, dim=-1, eps=1e-6) * math.sqrt(D) * x["norm"]


def _in_segments(step, S, T, xs, seg=64):
    """y [B,T,...] of S, y_t = step(S, x_t...), the tokens' states kept every
    ``seg`` tokens only when a gradient is wanted."""
    def part(S, *xc):
        ys = []
        for t in range(xc[0].shape[1]):
            S, y = step(S, *(x[:, t] for x in xc))
            ys.append(y)
        return S, torch.stack(ys, 1)
    out = []
    for t in range(0, T, seg):
        xc = [x[:, t:t + seg] for x in xs]
        if torch.is_grad_enabled():
            S, y = torch.utils.checkpoint.checkpoint(part, S, *xc, use_reentrant=False)
        else:
            S, y = part(S, *xc)
        out.append(y)
    return torch.cat(out, 1)


def _kmd2_64(q, k, v, g, be, bw, mix):
    B, T, H, r, D = q.shape
    qm = q[:, :, :, 0] if r == 1 else (q * mix[None, None, :, :, None]).sum(3)

    def step(S, qt, kt, vt, gt, bet, bwt):
        S = gt[..., None] * S
        m = (S * kt[..., None]).sum(-2)
        S = S + kt[..., None] * (bwt[..., None] * vt - bet[..., None] * m)[..., None, :]
        return S, (S * qt[..., None]).sum(-2)
    return _in_segments(step, q.new_zeros(B, H, D, D), T, (qm, k, v, g, be, bw))


def _small_inverse(Mx):
    """Inverse of symmetric positive [.., r, r] by Gauss-Jordan, r <= 4."""
    r = Mx.shape[-1]
    X = torch.cat([Mx, torch.eye(r, dtype=Mx.dtype, device=Mx.device).expand_as(Mx)], -1)
    for i in range(r):
        row = X[..., i:i + 1, :] / X[..., i:i + 1, i:i + 1]
        keep = torch.zeros(r, 1, dtype=Mx.dtype, device=Mx.device)
        keep[i] = 1.0
        X = (X - X[..., :, i:i + 1] * row) * (1 - keep) + row * keep
    return X[..., r:]


def _rls_64(q, K, V, Bg, Wg, a, mix, eps=0.5):
    B, T, H, ro, dk = q.shape
    r, dv = V.shape[3:]
    eye = torch.eye(r, dtype=q.dtype, device=q.device)
    qm = q[:, :, :, 0] if ro == 1 else (q * mix[None, None, :, :, None]).sum(3)

    def step(S, qt, Kt, Vt, Bt, Wt, at):
        S = S * at[..., None, :]
        Ke = Bt * Kt
        Tf = _small_inverse(eps * eye + Ke @ Ke.transpose(-1, -2).contiguous())
        S = S - (S @ Ke.transpose(-1, -2).contiguous()) @ (Tf @ Ke) + (Wt * Vt).transpose(-1, -2).contiguous() @ Kt
        return S, (S * qt[..., None, :]).sum(-1)
    return _in_segments(step, q.new_zeros(B, H, dv, dk), T, (qm, K, V, Bg, Wg, a))


def exact(case, seed):
    kind = case["kind"]
    raw = _tensors(case, seed)
    x = {n: t.double() if t.is_floating_point() else t for n, t in raw.items()}
    names = _grad_names(case)
    for n in names:
        x[n].requires_grad_(True)
    with torch.set_grad_enabled(bool(names)):
        if kind == "scan_train":
            y, _ = _dense_scan(x["q"], x["k"], x["v"], x["beta"], x["log_g"])
            return (y, *torch.autograd.grad(y, [x[n] for n in names], x["dy"]))
        if kind == "scan_prefill":
            return _dense_scan(x["q"], x["k"], x["v"], x["beta"], x["log_g"])
        if kind == "decode":
            gam = x["log_g"].exp()
            y = torch.empty(*gam.shape, case["D"], dtype=torch.float64, device=DEV)
            S = x["state"]
            for i in range(case["B"]):      # a sequence at a time: the states are gigabytes
                s = S[i].mul_(gam[i, ..., None, None])
                k, q, v = (x[n][i][:, None] for n in ("k", "q", "v"))
                r = x["a_w"][i, ..., None] * v - x["a_e"][i, ..., None] * (s * k[..., None]).sum(-2)
                s += k[..., None] * r[..., None, :]
                y[i] = (s * q[..., None]).sum(-2)
            pool = torch.empty_like(S)
            B = case["B"]
            base = list(range(B))
            slots = [base[(7 * i + 3) % B] for i in range(B)] if math.gcd(7, B) == 1 else base
            pool[torch.tensor(slots, device=DEV)] = S
            return y, pool
        if kind == "decode_gdn3":
            return _decode_gdn3_64(case, x)
        if kind == "layer_train":
            out = _layer64(x, case["P"], case["every"])
            return (out, *torch.autograd.grad(out, [x[n] for n in names], x["dout"]))
        if kind == "gdn3_prefill":
            B, T, H, D = x["q"].shape
            wide = (B, T, H, case["M"], D)
            y, s = _kron_window_scan(*(x[n].unsqueeze(3).expand(wide) for n in ("q", "k", "v")),
                                     *(x[n].unsqueeze(-1).expand(wide) for n in ("b", "w")), x["decay"], case["P"],
                                     case["every"])
            return (y, *s)
        if kind in ("kmd2_train", "kmd2_eval"):
            y = _kmd2_64(*(x[n] for n in ("q", "k", "v", "g", "beta_e", "beta_w", "out_mix")))
            return (y, *torch.autograd.grad(y, [x[n] for n in names], x["dy"])) if names else y
        y = _rls_64(*(x[n] for n in ("q", "K", "V", "Bg", "Wg", "a", "out_mix")))
        return (y, *torch.autograd.grad(y, [x[n] for n in names], x["dy"]))


def _decode_gdn3_64(case, x):
    B, H, M, D, P = (case[n] for n in ("B", "H", "M", "D", "P"))
    N = B * H * M
    A, Bf, U, Vb = (x[n].reshape(N, *x[n].shape[3:]) for n in ("A", "Bf", "U", "Vb"))
    q, k, b, w = (x[n].reshape(N, D) for n in ("q", "k", "b", "w"))
    v = x["v"].unsqueeze(2).expand(B, H, M, D).reshape(N, D)
    gam = x["decay"].clamp(0.0, 1.0).reshape(N, 1, 1)
    A, Bf, Vb = A * gam[..., None], Bf * gam[..., None], Vb * gam
    a_k, b_k = A.shape[-1], Bf.shape[-1]

    def read(z):
        X = z.reshape(N, 1, a_k, b_k)
        kron = torch.matmul(torch.matmul(A, X), Bf.transpose(-1, -2).contiguous()).sum(1).reshape(N, D)
        return kron + (U * (Vb * z[..., None]).sum(1, keepdim=True)).sum(-1)
    h = b * k
    al = _alpha((k * h).sum(-1, keepdim=True))
    un = al * (w * v - read(h))
    y = read(q) + (k * q).sum(-1, keepdim=True) * un
    pos = x["pos"].long().repeat_interleave(H * M)
    at = (pos % P).view(N, 1, 1).expand(N, D, 1)
    U, Vb = U.scatter(2, at, un[..., None]), Vb.scatter(2, at, k[..., None])
    ev = ((pos + 1) % case["every"] == 0).nonzero()[:, 0]
    if ev.numel():
        G = _sketch(N, Bf.shape[-1] * Bf.shape[-2], min(RANK + 4, A.shape[-1] * A.shape[-2], Bf.shape[-1] * Bf.shape[-2]))
        A[ev], Bf[ev] = _compact(A[ev], Bf[ev], U[ev], Vb[ev], G[ev])
    return (y.view(B, H, M, D), *(t.view(B, H, M, *t.shape[1:]) for t in (A, Bf, U, Vb)))
