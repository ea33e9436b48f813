"""GDN3 windows whose keys are nearly one direction (a repeated token) with
decays near 1, against the float64 CPU oracle: the powers of L that make up
T = (I + L)^-1 = (I - L)(I + L^2)(I + L^4)(I + L^8) are large there and cancel.

With l the largest entry of L the factors' entries reach (1 + l)^15 where T's
stay below 1, so that products in float32 leave up to 2^-24 (1 + l)^15 in the
net writes, and twice that in the gradients, which take T twice.  b = 1 keeps
h = b o k exact in bf16; what bf16 IO rounds besides (y, dy, the gradients) is
2^-9 a value."""
import math

import pytest
import torch
import torch.nn.functional as F

from gdnx_amd import gdn3
from oracle import gdn3 as og

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
IOS = pytest.mark.parametrize("io", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])


def rel_l2(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


def _alike(T, D, scale, io):
    g = torch.Generator().manual_seed(31 + T)
    B, H, M = 1, 1, 2
    base = F.normalize(torch.randn(B, 1, H, D, generator=g), dim=-1)
    k = (scale * F.normalize(base + 1e-3 * torch.randn(B, T, H, D, generator=g), dim=-1)).to(io)
    q = F.normalize(base + 0.5 * torch.randn(B, T, H, D, generator=g), dim=-1).to(io)
    v = (torch.randn(B, 1, H, D, generator=g) + 0.1 * torch.randn(B, T, H, D, generator=g)).to(io)
    one = torch.ones(B, T, H, M)
    kk = k.double().square().sum(-1).max().item()
    bound = 2.0 ** -24 * (2 - math.exp(-kk)) ** 15      # l = alpha(k.k) k.k = 1 - e^{-k.k}
    dy = torch.randn(B, T, H, M, D, generator=g).to(io)
    return [q, k, v, one, one.clone(), one * torch.tensor([1.0, 0.999])], dy, bound


def _oracle(xs, cfg):
    q, k, v, b, w, dec = xs
    wide = (*b.shape, q.shape[-1])
    return og.gdn3_recurrence(*(x.unsqueeze(3).expand(wide) for x in (q, k, v)),
                              *(x.unsqueeze(-1).expand(wide) for x in (b, w)), dec, sign_mode="canonical", **cfg)


def _cfg(D, P, Kc):
    return dict(R=4, P=P, factors=(16, 16, 8, 8) if D == 128 else (8, 8, 8, 8), compact_every=Kc)


@IOS
@pytest.mark.parametrize("D,scale", [(128, 1.0), (128, 2.0), (64, 1.0), (64, 2.0)])
def test_one_window_forward(gpu_lib, D, scale, io):
    """The layer's default regime (a compaction every 16 tokens), one window."""
    print(f"case: gdn3 alike keys, one window D={D} scale={scale} {io}", flush=True)
    xs, _, bound = _alike(16, D, scale, io)
    yr, sr, _ = _oracle([x.double() for x in xs], dict(_cfg(D, 16, 16), return_state=True))
    y, s, _ = gdn3.gdn3_recurrent_state(*(x.to(DEV) for x in xs), return_state=True, **_cfg(D, 16, 16))
    torch.cuda.synchronize()
    assert rel_l2(s[2], sr[2]) <= bound
    assert rel_l2(y, yr) <= bound + (2.0 ** -9 if io == torch.bfloat16 else 0.0)


@IOS
@pytest.mark.parametrize("D,P,Kc,T", [(128, 16, 16, 16), (64, 16, 16, 16), (128, 16, 64, 45), (64, 32, 64, 45)])
def test_gradients(gpu_lib, D, P, Kc, T, io):
    print(f"case: gdn3 alike keys, gradients D={D} P={P} Kc={Kc} T={T} {io}", flush=True)
    xs, dy, bound = _alike(T, D, 1.0, io)
    ref = [x.double().requires_grad_(True) for x in xs]
    want = torch.autograd.grad(_oracle(ref, _cfg(D, P, Kc)), ref, dy.double())
    leaves = [x.to(DEV).requires_grad_(True) for x in xs]
    got = torch.autograd.grad(gdn3.gdn3_recurrent_state(*leaves, **_cfg(D, P, Kc)), leaves, dy.to(DEV))
    torch.cuda.synchronize()
    errs = {n: rel_l2(a, r) for n, a, r in zip(("dq", "dk", "dv", "db", "dw", "ddecay"), got, want)}
    print("  " + " ".join(f"{n} {e:.1e}" for n, e in errs.items()), flush=True)
    for n, e in errs.items():
        assert e <= 2 * bound + (1e-2 if io == torch.bfloat16 else 0.0), n
