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


@pytest.mark.parametrize("NS", [4095, 4097, 8500])
def test_decode_due_rows_beyond_one_batch(gpu_lib, NS):
    """More rows than are listed at once (4096), with and without slots: the
    same as the rows stepped a hundred and one at a time, bitwise."""
    print(f"case: decode due rows, {NS} rows", flush=True)
    H, M, D, P, Kc, R, f = 1, 1, 64, 16, 16, 4, (8, 8, 8, 8)
    g = torch.Generator().manual_seed(NS)
    pos = torch.randint(0, 64, (NS,), generator=g).to(torch.int32)
    state = [torch.randn(NS, H, M, *s, generator=g) * 0.2 for s in ((R, 8, 8), (R, 8, 8), (D, P), (D, P))]
    q, k, v = (torch.nn.functional.normalize(torch.randn(NS, H, D, generator=g), dim=-1).bfloat16().to(DEV)
               for _ in range(3))
    b, w = (torch.rand(NS, H, M, generator=g).to(DEV) for _ in range(2))
    dec = (0.9 + 0.1 * torch.rand(NS, H, M, generator=g)).to(DEV)
    ps = pos.to(DEV)
    for slots in (None, torch.randperm(NS, generator=g).to(torch.int32).to(DEV)):
        batch, parts = [t.to(DEV) for t in state], [t.to(DEV) for t in state]
        kw = dict(R=R, P=P, factors=f, compact_every=Kc)
        y = gdn3.gdn3_decode_step(q, k, v, b, w, dec, batch, ps, slots=slots, **kw)
        ys = []
        for i in range(0, NS, 101):
            c = slice(i, i + 101)
            st = parts if slots is not None else [t[c] for t in parts]
            ys.append(gdn3.gdn3_decode_step(q[c], k[c], v[c], b[c], w[c], dec[c], st, ps[c],
                                            slots=None if slots is None else slots[c], sketch=_sketch(c, slots, NS),
                                            **kw))
        torch.cuda.synchronize()
        assert torch.equal(y, torch.cat(ys))
        for a, e in zip(batch, parts):
            assert torch.equal(a, e)


def _sketch(c, slots, NS):
    """The sketch rows of the states that a call sees."""
    G = gdn3.default_sketch(NS, 64, 8, torch.device(DEV))
    return G if slots is not None else G[c]
