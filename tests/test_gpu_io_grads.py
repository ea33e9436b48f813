"""Gradients written in the IO dtype: bitwise the float32 ones cast to it."""
import pytest
import torch
import torch.nn.functional as F

from gdnx_amd import gdn3, layer, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("io", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("D,P,T,gate", [(128, 16, 53, "channel"), (64, 16, 16, "lane"), (128, 32, 70, "lane"),
                                        (64, 64, 130, "channel")])
def test_recurrence_backward_io_gradients(gpu_lib, D, P, T, gate, io):
    print(f"case: gdn3 bwd io grads D={D} P={P} T={T} {gate} {io}", flush=True)
    B, H, M = 2, 2, 3
    g = torch.Generator().manual_seed(T)
    f = (16, 16, 8, 8) if D == 128 else (8, 8, 8, 8)
    q, k, v = (F.normalize(torch.randn(B, T, H, M, D, generator=g), dim=-1).to(io).to(DEV) for _ in range(3))
    gs = (B, T, H, M, D) if gate == "channel" else (B, T, H, M)
    b, w = (torch.rand(*gs, generator=g).to(DEV) for _ in range(2))
    dec = (0.9 + 0.1 * torch.rand(B, T, H, M, generator=g)).to(DEV)
    dy = torch.randn(B, T, H, M, D, generator=g).to(io).to(DEV)
    G = gdn3.default_sketch(B * H * M, f[2] * f[3], 8, DEV)
    kw = dict(M=M, P=P, factors=f)
    _, _, _, st = ops.gdn3_chunk_fwd(q, k, v, b, w, dec, G, save_states=True, **kw)
    ref = ops.gdn3_chunk_bwd(q, k, v, b, w, dec, dy, st, **kw)
    got = ops.gdn3_chunk_bwd(q, k, v, b, w, dec, dy, st, io_grads=True, **kw)
    torch.cuda.synchronize()
    for r, o in zip(ref[:3], got[:3]):
        assert o.dtype == io and torch.equal(o, r.to(io))
    for r, o in zip(ref[3:], got[3:]):
        assert torch.equal(o, r)


@pytest.mark.parametrize("io", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("M,K,V", [(4, 128, 128), (1, 64, 32), (3, 96, 160), (4, 256, 256)])
def test_prologue_backward_io_gradients(gpu_lib, M, K, V, io):
    print(f"case: prologue bwd io grads M={M} K={K} V={V} {io}", flush=True)
    B, T, H = 2, 19, 3
    g = torch.Generator().manual_seed(M * K + V)

    def r(*s):
        return torch.randn(*s, generator=g).to(io).to(DEV)
    ins = (r(B, T, H, M, K), r(B, T, H), r(B, T, H, M, V), r(B, T, H), r(B, T, H, M, 4) * 3)
    rates = torch.tensor([0.05, 0.02, 0.005, 0.001], device=DEV)
    cos, sin = layer.lane_rope_tables(M, T, K, DEV)
    gr = [r(B, T, H, M, K), r(B, T, H, M, K), r(B, T, H, M, K).float(), r(B, T, H, M, V).float(),
          r(B, T, H, M).float()]
    ref = ops.gdn3_prologue_bwd(*ins, rates, cos, sin, *gr)
    got = ops.gdn3_prologue_bwd(*ins, rates, cos, sin, *gr, io_grads=True)
    torch.cuda.synchronize()
    for a, o in zip(ref, got):
        assert o.dtype == io and torch.equal(o, a.to(io))
