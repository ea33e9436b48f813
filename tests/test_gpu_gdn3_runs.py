"""GDN3 forward over intervals of many sub-chunks, cut into runs: the window
carried from run to run, the state's keys and writes seen across ragged call
edges, against the CPU oracle (rel-L2 1e-4 in float32, 1e-2 in bf16, the
net writes twice that, the keys 1e-5)."""
import math

import pytest
import torch
import torch.nn.functional as F

from gdnx_amd import gdn3
from oracle import gdn3 as og

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rel_l2(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


# (D, P, K_c, t0, T): the smallest interval the runs take (3 sub-chunks), one
# batch, a run more than a batch, ragged starts inside a slot block and ends
# that leave the old writes in a block, intervals of one, two and many runs
CASES = [(128, 16, 48, 0, 96), (128, 16, 64, 5, 190), (128, 16, 1 << 20, 0, 1100), (64, 16, 512, 23, 1061),
         (128, 32, 512, 17, 700), (64, 32, 128, 0, 333), (128, 64, 1 << 20, 61, 900), (64, 64, 256, 70, 770),
         (128, 16, 256, 255, 258), (64, 64, 64 * 5, 3, 45)]


@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("D,P,Kc,t0,T", CASES)
def test_runs_match_oracle(gpu_lib, D, P, Kc, t0, T, io):
    print(f"case: gdn3 runs D={D} P={P} Kc={Kc} t0={t0} T={T} {io}", flush=True)
    B, H, M, R = 1, 1, 2, 4
    N = B * H * M
    f = (16, 16, 8, 8) if D == 128 else (8, 8, 8, 8)
    g = torch.Generator().manual_seed(D + P + T)
    q, k = (F.normalize(torch.randn(B, T, H, D, generator=g), dim=-1).to(io) for _ in range(2))
    v = torch.randn(B, T, H, D, generator=g).to(io)
    gate = (B, T, H, M, D) if (P + T) % 2 else (B, T, H, M)
    b, w = (torch.sigmoid(torch.randn(*gate, generator=g)) for _ in range(2))
    dec = torch.exp(-torch.rand(B, T, H, M, generator=g) * torch.tensor([0.1, 0.002])).clamp(max=1.0)
    st0 = None
    if t0:
        st0 = (torch.randn(N, R, f[0], f[1], generator=g) * 0.2, torch.randn(N, R, f[2], f[3], generator=g) * 0.1,
               torch.randn(N, D, P, generator=g) * 0.4,
               F.normalize(torch.randn(N, P, D, generator=g), dim=-1).transpose(1, 2).contiguous())
    wide = (B, T, H, M, D)
    ex = [x.double().unsqueeze(3).expand(wide) for x in (q, k, v)]
    gx = [x.double() if x.dim() == 5 else x.double().unsqueeze(-1).expand(wide) for x in (b, w)]
    yr, sr, _ = og.gdn3_recurrence(*ex, *gx, dec.double(), R=R, P=P, factors=f, compact_every=Kc,
                                   sign_mode="canonical", return_state=True, state0=st0, t0=t0)
    y, s, _ = gdn3.gdn3_recurrent_state(*(x.to(DEV) for x in (q, k, v, b, w, dec)), R=R, P=P, factors=f,
                                        compact_every=Kc, return_state=True, t0=t0,
                                        state0=None if st0 is None else tuple(x.to(DEV) for x in st0))
    torch.cuda.synchronize()
    tol = 1e-4 if io == torch.float32 else 1e-2
    assert rel_l2(y, yr) <= tol
    assert rel_l2(s[2], sr[2]) <= 2 * tol
    assert rel_l2(s[3], sr[3]) <= 1e-5     # keys decay in float32 from the inputs


# (D, P, K_c, t0, T, chains as H x M, per-channel gates, q / k / v per lane).  At
# d = 128 up to 128 workgroups (chains x runs) are split by value columns, so 132
# and more chains, or 66 with two runs, take the whole-row form.
WIDE = [(128, 16, 512, 0, 700, (1, 2), True, True), (128, 32, 1 << 20, 9, 800, (2, 1), True, False),
        (128, 64, 512, 0, 600, (1, 2), True, True), (128, 16, 48, 3, 100, (33, 4), True, True),
        (128, 16, 512, 0, 300, (33, 2), True, False), (128, 16, 512, 7, 300, (33, 2), False, True),
        (128, 32, 64, 0, 70, (44, 3), False, False), (128, 64, 1 << 20, 0, 280, (33, 2), True, True),
        (64, 16, 512, 11, 400, (33, 2), True, True), (64, 64, 128, 0, 150, (33, 4), False, True)]


def _wide_inputs(D, T, H, M, ch, lanes, io):
    g = torch.Generator().manual_seed(D + T + H)
    B = 1
    row = (B, T, H, M, D) if lanes else (B, T, H, D)
    q, k = (F.normalize(torch.randn(*row, generator=g), dim=-1).to(io) for _ in range(2))
    v = torch.randn(*row, generator=g).to(io)
    b, w = (torch.sigmoid(torch.randn(*((B, T, H, M, D) if ch else (B, T, H, M)), generator=g)) for _ in range(2))
    dec = torch.exp(-torch.rand(B, T, H, M, generator=g) * 0.05)
    return [q, k, v, b, w, dec], g


def _wide_oracle(xs, M, D, **kw):
    q, k, v, b, w, dec = xs
    wide = (*dec.shape, D)
    ex = [x if x.dim() == 5 else x.unsqueeze(3).expand(wide) for x in (q, k, v)]
    gx = [x if x.dim() == 5 else x.unsqueeze(-1).expand(wide) for x in (b, w)]
    return og.gdn3_recurrence(*ex, *gx, dec, R=4, sign_mode="canonical", **kw)


@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("D,P,Kc,t0,T,HM,ch,lanes", WIDE)
def test_runs_gate_and_lane_layouts(gpu_lib, D, P, Kc, t0, T, HM, ch, lanes, io):
    print(f"case: gdn3 runs D={D} P={P} Kc={Kc} t0={t0} T={T} HM={HM} ch={ch} lanes={lanes} {io}", flush=True)
    (H, M), R = HM, 4
    N, f = H * M, (16, 16, 8, 8) if D == 128 else (8, 8, 8, 8)
    xs, g = _wide_inputs(D, T, H, M, ch, lanes, io)
    st0 = None
    if t0:
        st0 = (torch.randn(N, R, f[0], f[1], generator=g) * 0.2, torch.randn(N, R, f[2], f[3], generator=g) * 0.1,
               torch.randn(N, D, P, generator=g) * 0.4,
               F.normalize(torch.randn(N, P, D, generator=g), dim=-1).transpose(1, 2).contiguous())
    kw = dict(P=P, factors=f, compact_every=Kc, return_state=True, t0=t0)
    yr, sr, _ = _wide_oracle([x.double() for x in xs], M, D, state0=st0, **kw)
    y, s, _ = gdn3.gdn3_recurrent_state(*(x.to(DEV) for x in xs), R=R,
                                        state0=None if st0 is None else tuple(x.to(DEV) for x in st0), **kw)
    torch.cuda.synchronize()
    tol = 1e-4 if io == torch.float32 else 1e-2
    assert rel_l2(y, yr) <= tol
    assert rel_l2(s[2], sr[2]) <= 2 * tol
    assert rel_l2(s[3], sr[3]) <= 1e-5


@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("D,P,Kc,T,HM,ch,lanes", [
    (128, 16, 512, 600, (1, 2), True, True), (128, 64, 1024, 700, (1, 2), False, False),
    (64, 32, 1024, 600, (1, 2), True, False), (128, 16, 512, 260, (33, 2), True, False)])
def test_gradients_over_runs(gpu_lib, D, P, Kc, T, HM, ch, lanes, io):
    """Training through intervals of several runs: the net writes and decays
    that every run stashes (tolerances as in the backward's own tests)."""
    print(f"case: gdn3 gradients over runs D={D} P={P} Kc={Kc} T={T} HM={HM} ch={ch} lanes={lanes} {io}", flush=True)
    H, M = HM
    f = (16, 16, 8, 8) if D == 128 else (8, 8, 8, 8)
    xs, g = _wide_inputs(D, T, H, M, ch, lanes, io)
    dy = torch.randn(1, T, H, M, D, generator=g).to(io)
    kw = dict(P=P, factors=f, compact_every=Kc)
    ref = [x.double().requires_grad_(True) for x in xs]
    yr = _wide_oracle(ref, M, D, **kw)
    want = torch.autograd.grad(yr, ref, dy.double())
    leaves = [x.to(DEV).requires_grad_(True) for x in xs]
    y = gdn3.gdn3_recurrent_state(*leaves, R=4, **kw)
    got = torch.autograd.grad(y, leaves, dy.to(DEV))
    torch.cuda.synchronize()
    tol = 1e-4 if io == torch.float32 else 1e-2
    assert rel_l2(y, yr) <= tol
    for name, a, r in zip(("dq", "dk", "dv", "db", "dw", "ddecay"), got, want):
        assert rel_l2(a, r) <= tol, name


@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("P,scale", [(16, 1.0), (16, 2.0), (64, 1.0), (64, 2.0)])
def test_runs_alike_keys(gpu_lib, P, scale, io):
    """Keys that are nearly one direction (a repeated token), decay near 1: the
    powers of L that make up T = (I + L)^-1 cancel.  With l the largest entry
    of L the factors' entries reach (1 + l)^15 where T's stay below 1, so
    products in float32 leave up to 2^-24 (1 + l)^15 in the net writes, and
    16-bit parts of them 2^-17 (1 + l)^15.  b = 1 keeps h = k exact in bf16."""
    print(f"case: gdn3 runs alike keys P={P} scale={scale} {io}", flush=True)
    B, T, H, M, D = 1, 133, 1, 2, 128
    g = torch.Generator().manual_seed(31 + P)
    base = F.normalize(torch.randn(B, 1, H, D, generator=g), dim=-1)
    k = (scale * F.normalize(base + 1e-3 * torch.randn(B, T, H, D, generator=g), dim=-1)).to(io)
    q = F.normalize(base + 0.5 * torch.randn(B, T, H, D, generator=g), dim=-1).to(io)
    v = (torch.randn(B, 1, H, D, generator=g) + 0.1 * torch.randn(B, T, H, D, generator=g)).to(io)
    one = torch.ones(B, T, H, M)
    dec = one * torch.tensor([1.0, 0.999])
    wide = (B, T, H, M, D)
    ex = [x.double().unsqueeze(3).expand(wide) for x in (q, k, v)]
    gx = one.double().unsqueeze(-1).expand(wide)
    cfg = dict(R=4, P=P, factors=(16, 16, 8, 8), compact_every=1 << 20, return_state=True)
    yr, sr, _ = og.gdn3_recurrence(*ex, gx, gx, dec.double(), sign_mode="canonical", **cfg)
    y, s, _ = gdn3.gdn3_recurrent_state(*(x.to(DEV) for x in (q, k, v, one, one, dec)), **cfg)
    torch.cuda.synchronize()
    kk = k.double().square().sum(-1).max().item()
    bound = 2.0 ** -24 * (1 + (1 - math.exp(-kk))) ** 15      # l = alpha(k.k) k.k
    assert rel_l2(s[2], sr[2]) <= bound
    assert rel_l2(y, yr) <= bound + (2.0 ** -9 if io == torch.bfloat16 else 0.0)   # y's own rounding
