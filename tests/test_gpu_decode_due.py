"""Which rows of a GDN3 decode batch compact, and on which workgroup."""
import pytest
import torch

from gdnx_amd import gdn3

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_decode_due_rows_spread_over_workgroups(gpu_lib):
    """The compactions of a decode batch with more rows than a workgroup has
    threads, at positions that repeat with a period, through slots in no order
    with empty rows among them: every row equals the same row stepped alone,
    bitwise, and the factors of exactly the due rows were compacted."""
    print("case: decode due rows, 600 rows", flush=True)
    NS, H, M, D, P, Kc = 600, 3, 2, 64, 16, 32
    g = torch.Generator().manual_seed(77)
    n_slots = NS + 5
    slots = torch.randperm(n_slots, generator=g)[:NS].to(torch.int32)
    slots[torch.tensor([0, 255, 256, 599])] = -1
    pos = (torch.arange(NS) * 5 % 64).to(torch.int32)
    pos[torch.tensor([30, 300])] = -1
    R, f = 4, (8, 8, 8, 8)
    state = [torch.randn(n_slots, H, M, *s, generator=g) * 0.2
             for s in ((R, 8, 8), (R, 8, 8), (D, P), (D, P))]
    q, k, v = (torch.nn.functional.normalize(torch.randn(NS, H, D, generator=g), dim=-1).bfloat16().to(DEV)
               for _ in range(3))
    b, w = (torch.rand(NS, H, M, generator=g).to(DEV) for _ in range(2))
    dec = (0.9 + 0.1 * torch.rand(NS, H, M, generator=g)).to(DEV)
    sl, ps = slots.to(DEV), pos.to(DEV)
    batch = [t.to(DEV) for t in state]
    alone = [t.to(DEV) for t in state]
    y = gdn3.gdn3_decode_step(q, k, v, b, w, dec, batch, ps, R=R, P=P, factors=f, compact_every=Kc, slots=sl)
    ys = [gdn3.gdn3_decode_step(q[i:i + 1], k[i:i + 1], v[i:i + 1], b[i:i + 1], w[i:i + 1], dec[i:i + 1], alone,
                                ps[i:i + 1], R=R, P=P, factors=f, compact_every=Kc, slots=sl[i:i + 1])
          for i in range(NS)]
    torch.cuda.synchronize()
    assert torch.equal(y, torch.cat(ys))
    for a, e in zip(batch, alone):
        assert torch.equal(a, e)
    due = (slots >= 0) & (pos >= 0) & ((pos + 1) % Kc == 0)
    rows = [int(s) for s in slots[due]]
    assert rows
    plain = [t.to(DEV) for t in state]     # the same step on an interval no row closes
    gdn3.gdn3_decode_step(q, k, v, b, w, dec, plain, ps, R=R, P=P, factors=f, compact_every=1 << 20, slots=sl)
    changed = (batch[0] != plain[0]).flatten(1).any(1).nonzero()[:, 0].tolist()
    assert sorted(rows) == changed
