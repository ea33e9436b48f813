"""Per-channel-decay scans with a chain's state split over keys and value tiles:
outputs, final state, write norms and gradients at the edges of the chunk, of the
operands in flight (2, 3 and 4 chunks) and of the 1 / 2 / 4 value tiles a
workgroup takes, against the float64 oracle (rel-L2 1e-4: float32 throughout)."""
import pytest
import torch

from gdnx_amd import ops
from test_gpu_delta_chan import DEV, _inputs, _oracle, rel_l2

pytestmark = pytest.mark.gpu

# B H D T: chunks of 16 tokens around 1, 2, 4 and 8; chains at which the tiles of
# a workgroup change on 256 CUs (d = 128: 33 and 128, d = 64: 65 and 256)
CASES = [(1, 1, 128, 1), (1, 2, 128, 16), (2, 1, 64, 17), (1, 2, 64, 64), (1, 1, 128, 65), (1, 2, 128, 130),
         (2, 16, 128, 33), (3, 11, 128, 63), (3, 11, 128, 97), (8, 16, 128, 31), (8, 16, 128, 50), (5, 13, 64, 65),
         (16, 16, 64, 49), (16, 16, 64, 1), (16, 16, 64, 90)]


@pytest.mark.parametrize("B,H,D,T", CASES)
def test_chan_split_matches_oracle(gpu_lib, B, H, D, T):
    print(f"case: chan split B={B} H={H} D={D} T={T}", flush=True)
    x = _inputs(B, T, H, D, seed=B + T, with_state=True)
    gen = torch.Generator().manual_seed(T)
    dy = torch.randn(B, T, H, D, generator=gen)
    ds = torch.randn(B, H, D, D, generator=gen)
    ref = [t.double().requires_grad_(True) for t in x]
    yr, sr = _oracle(*ref)
    gr = torch.autograd.grad((yr * dy.double()).sum() + (sr * ds.double()).sum(), ref)
    q, k, v, be, bw, lg, st = (t.detach() for t in ref)
    r_ref = torch.empty(B, T, H, dtype=torch.float64)
    for t in range(T):
        st = lg[:, t].exp().unsqueeze(-1) * st
        r = bw[:, t, :, None] * v[:, t] - be[:, t, :, None] * (st * k[:, t].unsqueeze(-1)).sum(-2)
        st = st + k[:, t].unsqueeze(-1) * r.unsqueeze(-2)
        r_ref[:, t] = r.norm(dim=-1)
    dev = [t.to(DEV) for t in x]
    y0, s0, _ = ops.delta_chan_fwd(*dev)
    for save in (False, True):
        r_norm = torch.empty(B, T, H, device=DEV)
        y, s, stash = ops.delta_chan_fwd(*dev, save_states=save, r_norm=r_norm)
        assert torch.equal(y0, y) and torch.equal(s0, s)
        assert rel_l2(r_norm, r_ref) <= 1e-4
    y, s, stash = ops.delta_chan_fwd(*dev, save_states=True)
    grads = ops.delta_chan_bwd(*dev[:6], dy.to(DEV), stash, ds.to(DEV), want_dstate0=True)
    torch.cuda.synchronize()
    assert torch.equal(y0, y) and torch.equal(s0, s)
    assert rel_l2(y, yr) <= 1e-4
    assert rel_l2(s, sr) <= 1e-4
    for name, g, r in zip(("q", "k", "v", "beta_e", "beta_w", "log_g", "s0"), grads, gr):
        assert rel_l2(g, r) <= 1e-4, name
