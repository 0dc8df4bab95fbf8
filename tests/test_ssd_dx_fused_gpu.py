"""dx of the SSD backward pass (ssd_dx_fused.hip, and ssd_dx_short.hip for lists of one and two heads) at the edges of its tiles: each chunk length, state count and headdim, lists
of one and of several heads, a last chunk of 1, 17 and Q - 1 positions, packed sequences, D per head, per (head, p) and none.
Reference: the quadratic form in float64 on the same bf16 operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _worst_tile(got, want):
    """The largest error of 16 positions of one head (or group), as a share of their norm.  (Whole tiles: the one or few terms
    of a single position can cancel, and leave a result that is small beside the rounding of each.)"""
    tiles = lambda t: t[:, :t.shape[1] // 16 * 16].double().unflatten(1, (-1, 16)).pow(2).sum((2, 4))
    return float((tiles(got.double() - want) / tiles(want)).max().sqrt())


# A rounding to bf16 is at most 2^-9 of the value, so a sum of 16 x 32 values and more that took three of them (operands of
# the products, chunk states, the result) is off by less than that many of its norm.  One position left out of 128
# comparable ones is 2^-3.5 of a row, 2^-5.5 of a tile
TILE = 3 * 2.0 ** -9


def _reference(dt, A, B, C, D, g, seq):
    """dx and the sum of its absolute terms."""
    b, L, H, P = g.shape
    live = torch.ones(L, L, device=g.device).tril().bool()[None].expand(b, L, L)
    if seq is not None:
        live = live & (seq[:, :, None] == seq[:, None, :])
    dx, size = torch.zeros(b, L, H, P, dtype=torch.float64, device=g.device), torch.zeros(b, L, H, P, dtype=torch.float64, device=g.device)
    for h in range(H):
        k = h // (H // B.shape[2])
        a = torch.cumsum(dt[:, :, h].double() * A[h].double(), 1)
        w = torch.where(live, torch.exp((a[:, :, None] - a[:, None, :]).clamp(max=0)) * dt[:, None, :, h].double(), 0.0)
        Ck, Bt, gh = C[:, :, k].double(), B[:, :, k].double().transpose(-1, -2).contiguous(), g[:, :, h].double()
        dx[:, :, h] = torch.matmul((torch.matmul(Ck, Bt) * w).transpose(-1, -2).contiguous(), gh)
        size[:, :, h] = torch.matmul((torch.matmul(Ck.abs(), Bt.abs()) * w).transpose(-1, -2).contiguous(), gh.abs())
    if D is not None:
        d = D.double() if D.dim() == 2 else D.double()[:, None]
        dx += d * g.double()
        size += (d * g.double()).abs()
    return dx, size


@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (1, 513, 8, 2, 64, 128, 64), (2, 127, 3, 1, 32, 64, 64), (1, 81, 2, 2, 64, 64, 64), (4, 1024, 24, 1, 32, 128, 64),
    (2, 641, 5, 1, 64, 128, 128), (4, 1024, 40, 1, 64, 64, 128), (1, 145, 4, 4, 32, 128, 128), (2, 383, 6, 2, 32, 64, 128),
    (4, 1024, 80, 1, 64, 128, 256), (1, 1025, 6, 2, 64, 128, 256), (2, 511, 3, 1, 64, 64, 256), (1, 785, 5, 5, 32, 128, 256),
    (4, 256, 4, 1, 32, 64, 256),
    # lists of 5 to 12 heads, one for each pair of headdim and states
    (4, 1009, 72, 1, 64, 128, 64), (3, 1009, 72, 1, 32, 128, 64), (8, 1009, 96, 1, 64, 64, 64), (8, 977, 96, 1, 32, 64, 64),
    (4, 1009, 72, 1, 64, 128, 128), (4, 1009, 72, 1, 32, 128, 128), (8, 1009, 96, 1, 64, 64, 128), (8, 977, 96, 1, 32, 64, 128),
    (4, 1009, 80, 1, 64, 128, 256), (4, 1009, 80, 1, 32, 128, 256), (4, 785, 96, 1, 64, 64, 256), (4, 1023, 96, 1, 32, 64, 256),
])
@pytest.mark.parametrize("packed,D_form", [(False, "head"), (True, "none"), (True, "channel")])
def test_dx(b, L, H, G, P, N, Q, packed, D_form):
    from mamba_amd.ops.triton import ssd_combined as sc
    gen = torch.Generator(device="cuda").manual_seed(L + Q + H)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    x, g, B, C = randn(b, L, H, P).requires_grad_(), randn(b, L, H, P), randn(b, L, G, N), randn(b, L, G, N)
    dt = 0.1 * torch.rand(b, L, H, device="cuda", generator=gen)
    A = -(0.1 + 5 * torch.rand(H, device="cuda", generator=gen))
    D = None if D_form == "none" else torch.randn(*((H,) if D_form == "head" else (H, P)), device="cuda", generator=gen).requires_grad_()
    seq = None
    if packed:
        ends = torch.tensor([0, L // 7, L // 7 + 1, L // 2 + 5], device="cuda")
        seq = (torch.arange(L, device="cuda")[:, None] >= ends).sum(-1).int()[None].expand(b, L).contiguous()
    sc.mamba_chunk_scan_combined(x, dt, A, B, C, Q, D=D, seq_idx=seq).backward(g)
    want, size = _reference(dt, A, B, C, None if D is None else D.detach(), g, seq)
    # the weighted products or the chunk states' gradients, and the result, are rounded to bf16: at most 2^-8 of each, twice
    err = (x.grad.double() - want).abs()
    assert bool((err <= 2 * 2.0 ** -8 * size + 1e-30).all()), float((err / (size + 1e-30)).max())
    assert _worst_tile(x.grad, want) < TILE
    if D is not None:  # of x and g as they are: fp32 sums of b L (and P) terms
        terms = x.detach().double() * g.double()
        dims = (0, 1) if D.dim() == 2 else (0, 1, 3)
        bound = 2.0 ** -24 * (16 + 4 * (b * L * P) ** 0.5) * terms.abs().sum(dims)
        assert bool(((D.grad.double() - terms.sum(dims)).abs() <= bound).all())


@pytest.mark.parametrize("L,H,P,N,Q", [(130, 2, 64, 128, 64), (100, 3, 32, 64, 128), (130, 1, 64, 128, 256)])
def test_rows_that_32_bit_offsets_do_not_reach(L, H, P, N, Q):
    """x and the gradient of the output as rows 2^22 values apart: the same dx as from dense rows."""
    from mamba_amd.ops.triton import ssd_combined as sc
    gen = torch.Generator(device="cuda").manual_seed(L + Q + H)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    x, g, B, C = randn(1, L, H, P), randn(1, L, H, P), randn(1, L, 1, N), randn(1, L, 1, N)
    dt, A = 0.1 * torch.rand(1, L, H, device="cuda", generator=gen), -(0.1 + 5 * torch.rand(H, device="cuda", generator=gen))
    rows = torch.empty(L << 22, device="cuda", dtype=torch.bfloat16)
    apart = lambda t, first: rows[first:].as_strided(t.shape, (L << 22, 1 << 22, P, 1)).copy_(t)
    got = []
    for xs, gs in ((x, g), (apart(x, 0), apart(g, 1 << 20))):
        leaf = xs.detach().requires_grad_()
        assert leaf.stride() == xs.stride()
        sc.mamba_chunk_scan_combined(leaf, dt, A, B, C, Q).backward(gs)
        got.append(leaf.grad)
    want, _ = _reference(dt, A, B, C, None, g, None)
    assert _worst_tile(got[1], want) < TILE and torch.equal(got[0], got[1])
