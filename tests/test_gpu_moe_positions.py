"""MoE permute: positions of experts in index rows (noted in LDS up to 256 entries,
searched for beyond), and the gradients of its two outputs one by one (GPU)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("topk,E", [(1, 511), (8, 32), (9, 32), (16, 64), (17, 511), (255, 511), (256, 300), (257, 511)])
def test_first_position_in_the_row(topk, E, dtype):
    """probs aligned with an index map follow the first position of an expert in its
    token's row: rows with repeated entries, entries outside [0, E), and 64-bit entries
    that are valid once truncated to 32 bits."""
    from primus_turbo.pytorch.ops import moe_permute

    T, H = 130, 64
    g = torch.Generator().manual_seed(topk * 1000 + E)
    idx = torch.randint(-2, E + 3, (T, topk), generator=g)
    idx[1::3] = idx[1::3, torch.randint(0, topk, (topk,), generator=g)]  # more repeats
    none = ~((idx >= 0) & (idx < E)).any(1)
    idx[none, -1] = torch.arange(T)[none] % E
    idx[-2], idx[-1] = -1, E  # tokens without a local expert come last
    entries = idx.clone()
    if dtype == torch.int64:
        entries[2::5] += 1 << 32
    tokens = torch.randn((T, H), generator=g).bfloat16()
    probs = torch.rand((T, topk), generator=g)
    rows, rim, per_expert, overflow, n, _, row_probs = moe_permute(
        tokens.cuda(), entries.to(dtype).cuda(), num_local_experts=E, num_topk=topk, probs=probs.cuda())

    first = [{} for _ in range(T)]
    for t in range(T):
        for k, e in enumerate(idx[t].tolist()):
            if 0 <= e < E:
                first[t].setdefault(e, k)
    order = [(t, first[t][e]) for e in range(E) for t in range(T) if e in first[t]]
    tt, kk = (torch.tensor(v, dtype=torch.long) for v in zip(*order))
    assert torch.equal(per_expert.cpu(), torch.tensor([sum(e in f for f in first) for e in range(E)]))
    assert not overflow.item() and int(n) == sum(bool(f) for f in first)
    assert torch.equal(rows.cpu(), tokens[tt]) and torch.equal(row_probs.cpu(), probs[tt, kk])
    rim = rim.cpu()
    for t in range(T):
        experts = sorted(first[t])
        assert rim[t, 2 * E].item() == len(experts)
        assert rim[t, E:E + len(experts)].tolist() == [first[t][e] for e in experts]


@pytest.mark.parametrize("layout", ["topk", "routing_map"])
@pytest.mark.parametrize("pad", [0, 16])
def test_gradients_of_one_output_alone(layout, pad):
    """A loss on the rows alone or on the rows' probs alone gives the gradients that
    explicit zeros for the other output give; probs that need no gradient take none."""
    from primus_turbo.pytorch.ops import moe_permute

    T, E, k, H = 75, 8, 3, 128
    g = torch.Generator().manual_seed(pad)
    idx = torch.rand((T, E), generator=g).argsort(1)[:, :k].cuda()
    probs = torch.rand((T, k if layout == "topk" else E), generator=g).cuda()
    tokens = torch.randn((T, H), generator=g).bfloat16().cuda()

    def call(p):
        t, p = tokens.clone().requires_grad_(), p.clone().requires_grad_(p.requires_grad)
        out = moe_permute(t, idx, num_local_experts=E, num_topk=k, probs=p, probs_layout=layout, pad_multiple=pad)
        return t, p, out[0], out[6]

    t, p, rows, row_probs = call(probs.clone().requires_grad_())
    g_rows = torch.randn(rows.shape, generator=g).bfloat16().cuda()
    g_probs = torch.randn(row_probs.shape, generator=g).cuda()
    for which, gr, gp in (("rows", g_rows, torch.zeros_like(g_probs)), ("probs", torch.zeros_like(g_rows), g_probs)):
        t, p, rows, row_probs = call(probs.clone().requires_grad_())
        want = torch.autograd.grad((rows, row_probs), (t, p), (gr, gp))
        t, p, rows, row_probs = call(probs.clone().requires_grad_())
        got = torch.autograd.grad(rows if which == "rows" else row_probs, (t, p), gr if which == "rows" else gp)
        assert all(x.dtype == y.dtype and torch.equal(x, y) for x, y in zip(got, want)), which
        assert any(x.any() for x in got)
    t, p, rows, row_probs = call(probs)
    assert not p.requires_grad
    (alone,) = torch.autograd.grad(rows, t, g_rows)
    t, p, rows, row_probs = call(probs.clone().requires_grad_())
    assert torch.equal(alone, torch.autograd.grad(rows, t, g_rows)[0])
