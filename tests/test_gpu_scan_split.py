"""Scans whose value columns are split over two workgroups while chains are few,
and the gradient kernel's segments of 64, 128 and 256 tokens: outputs, final
state and gradients at the edges of each rule, against the oracle (rel-L2 1e-2
for bf16 IO, 1e-4 for float32)."""
import pytest
import torch

from gdnx_amd import gdn3
from oracle import delta, inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rel_l2(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


# chains B H M: 128 / 129 at d = 128 (4 | 8 waves a workgroup); segments per (b, h): 16 x 8 of 256 tokens
# would leave CUs idle (-> 128), 2 (-> 64), 64 x 5 would not
CASES = [(1, 16, 4, 70, 128, "bf16"), (1, 65, 1, 70, 128, "bf16"), (2, 16, 4, 33, 128, "bf16"),
         (3, 43, 1, 33, 128, "bf16"), (2, 16, 4, 70, 64, "bf16"), (3, 43, 1, 33, 64, "bf16"),
         (1, 16, 4, 2049, 64, "bf16"), (1, 2, 3, 129, 64, "bf16"), (4, 16, 1, 1100, 64, "bf16"),
         (1, 2, 1, 49, 64, "f32"), (1, 32, 2, 17, 128, "f32"), (1, 43, 3, 17, 128, "f32"), (1, 43, 3, 33, 64, "f32")]


@pytest.mark.parametrize("B,H,M,T,D,io", CASES)
def test_split_scans_match_oracle(gpu_lib, B, H, M, T, D, io):
    print(f"case: split scan B={B} H={H} M={M} T={T} D={D} {io}", flush=True)
    dt = torch.bfloat16 if io == "bf16" else torch.float32
    x = inputs.dense_inputs(B, T, H, D, M=M, seed=5 + T, decay="softplus", with_grad_out=True)
    names = ("q", "k", "v", "beta", "g")
    ins = [(x[n].to(dt) if n in "qkv" else x[n]).to(DEV).requires_grad_(True) for n in names]
    y, s = gdn3.gdn3_scan(*ins, return_state=True)
    grads = torch.autograd.grad(y, ins, x["dO"].to(dt).to(DEV))
    with torch.no_grad():
        y_inf = gdn3.gdn3_scan(*ins)
    torch.cuda.synchronize()
    ref = [(x[n].to(dt) if n in "qkv" else x[n]).double().requires_grad_(True) for n in names]
    a = delta.gdn3_dense_coeffs(ref[1], ref[3])
    yr, sr = delta.lane_delta(ref[0], ref[1], ref[2], a, a, ref[4], chunk=32)
    gr = torch.autograd.grad(yr, ref, x["dO"].to(dt).double())
    tol = 1e-2 if io == "bf16" else 1e-4
    assert rel_l2(y, yr) <= tol
    assert rel_l2(y_inf, yr) <= tol
    assert rel_l2(s, sr) <= tol
    for n, g, r in zip(names, grads, gr):
        assert rel_l2(g, r) <= tol, n
