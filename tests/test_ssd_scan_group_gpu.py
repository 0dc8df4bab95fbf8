"""The forward chunk scan that keeps C B^T of the group (ssd_scan_group.hip): chunks of 64 and 128, state counts and headdims,
lists of one and of several heads, a last chunk of 1, 17 and Q - 1 positions, packed sequences, with and without gate, pre-gate
copy and D.  (64 states, or chunks of 64 with 128 states, with a gate are left to the one-tile form of ssd_scan_fused.hip: the
same check of that one.)  Reference: the stage's formula in float64 on the same bf16 operands."""
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


# (every problem has more workgroups than a card of 256 CUs; those whose lists are too short for this form, see
# ssd_scan_group_serves, are the same check of the one-tile form)
@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (2, 1025, 16, 8, 64, 128, 64), (4, 1024, 40, 10, 32, 128, 64), (1, 3025, 18, 6, 64, 64, 64), (3, 511, 64, 64, 32, 64, 64),
    (4, 2048, 24, 8, 64, 128, 128), (2, 1169, 48, 16, 64, 64, 128), (2, 2047, 40, 20, 32, 128, 128), (9, 129, 32, 32, 32, 64, 128),
    # lists of 8, 2, 8, 8 heads (chunk 64), of 4, 8, 4 (chunk 128)
    (4, 2047, 64, 8, 64, 128, 64), (4, 1025, 64, 8, 32, 128, 64), (4, 1937, 64, 8, 64, 64, 64), (4, 1985, 64, 8, 32, 64, 64),
    (4, 1169, 96, 8, 64, 64, 128), (4, 2047, 64, 8, 32, 128, 128), (4, 1937, 96, 6, 32, 64, 128),
])
@pytest.mark.parametrize("gate,pre,D_form,packed", [(False, False, "head", False), (False, False, "none", True), (True, True, "channel", True), (True, False, "head", False)])
def test_scan(b, L, H, G, P, N, Q, gate, pre, D_form, packed):
    from mamba_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(L + Q + H)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    nc = -(-L // Q)
    x, z, B, C, states = randn(b, L, H, P), randn(b, L, H, P), randn(b, L, G, N), randn(b, L, G, N), randn(b, nc, H, P, N)
    out, out_x = torch.full((b, L, H, P), 7.0, device="cuda").bfloat16(), torch.full((b, L, H, P), 7.0, device="cuda").bfloat16()
    dt = 0.1 * torch.rand(b, H, nc * Q, device="cuda", generator=gen)
    dt[:, :, L:] = 0
    dt = dt.reshape(b, H, nc, Q)
    dA = torch.cumsum(dt * -(0.1 + 5 * torch.rand(H, device="cuda", generator=gen))[None, :, None, None], -1).contiguous()
    D = None if D_form == "none" else torch.randn(*((H,) if D_form == "head" else (H, P)), device="cuda", generator=gen)
    seq = None
    if packed:
        ends = torch.tensor([0, L // 7, L // 7 + 1, L // 2 + 5], device="cuda")
        seq = ((torch.arange(L, device="cuda")[:, None] >= ends).sum(-1).int() - 1)[None].expand(b, L).contiguous()
    p = _lib.SsdParams()
    for k, v in dict(batch=b, seqlen=L, nheads=H, headdim=P, dstate=N, ngroups=G, chunk_size=Q, nchunks=nc, dtype=1).items():
        setattr(p, k, v)
    other = torch.zeros(1 << 12, device="cuda")  # fields that this stage does not read
    for k in ("dt", "A", "final_states"):
        setattr(p, k, other.data_ptr())
    for k, t in (("x", x), ("B", B), ("C", C), ("out", out)) + ((("z", z),) if gate else ()):
        setattr(p, k, t.data_ptr())
        for d, s in zip(("bs", "ls", "gs" if k in "BC" else "hs"), t.stride()):
            setattr(p, f"{k}_{d}", s)
    p.dt_out, p.dA_cumsum, p.states_lp = dt.data_ptr(), dA.data_ptr(), states.data_ptr()
    p.out_x = out_x.data_ptr() if gate and pre else None
    p.D, p.D_has_hdim = (D.data_ptr() if D is not None else None), int(D_form == "channel")
    p.seq_idx = seq.data_ptr() if packed else None
    assert lib.ssd_chunk_scan_fwd_fused_supported(p)
    _lib.check(lib.ssd_chunk_scan_fwd_fused(p, _lib.current_stream(x.device)), "ssd_chunk_scan_fwd_fused")
    torch.cuda.synchronize()
    pad = lambda t: torch.nn.functional.pad(t.double(), (0, 0, 0, 0, 0, nc * Q - L)).reshape(b, nc, Q, *t.shape[2:])
    ids = torch.full((b, nc * Q), -9, device="cuda")
    ids[:, :L] = 0 if seq is None else seq
    entered = torch.cat([torch.zeros(b, 1, device="cuda"), ids.reshape(b, nc, Q)[:, :-1, -1]], 1)[:, :, None]
    ids = ids.reshape(b, nc, Q)
    live = (ids[..., :, None] == ids[..., None, :]) & torch.ones(Q, Q, device="cuda").tril().bool()
    xs, Bs, Cs = pad(x), pad(B), pad(C)
    y, size = torch.zeros(b, nc, Q, H, P, dtype=torch.float64, device="cuda"), torch.zeros(b, nc, Q, H, P, dtype=torch.float64, device="cuda")
    for h in range(H):
        k = h // (H // G)
        a, w = dA[:, h].double(), dt[:, h].double()
        decay = torch.where(live, torch.exp((a[..., :, None] - a[..., None, :]).clamp(max=0)) * w[..., None, :], 0.0)
        carry = torch.where(ids == entered, torch.exp(a), 0.0)[..., None]
        Ck, Bt, Ht = Cs[:, :, :, k].contiguous(), Bs[:, :, :, k].transpose(-1, -2).contiguous(), states[:, :, h].double().transpose(-1, -2).contiguous()
        y[:, :, :, h] = torch.matmul(torch.matmul(Ck, Bt) * decay, xs[:, :, :, h].contiguous()) + carry * torch.matmul(Ck, Ht)
        size[:, :, :, h] = torch.matmul(torch.matmul(Ck.abs(), Bt.abs()) * decay, xs[:, :, :, h].abs().contiguous()) + carry * torch.matmul(Ck.abs(), Ht.abs())
    y, size = y.reshape(b, nc * Q, H, P)[:, :L], size.reshape(b, nc * Q, H, P)[:, :L]
    if D is not None:
        d = (D.double() if D.dim() == 2 else D.double()[:, None]) * x.double()
        y, size = y + d, size + d.abs()
    # the weighted products and the result are rounded to bf16, at most 2^-8 of each
    close = lambda got, want, scale: bool(((got.double() - want).abs() <= 2 * 2.0 ** -8 * scale + 1e-30).all())
    g = torch.nn.functional.silu(z.double())
    assert close(out, y * g, size * g.abs()) if gate else close(out, y, size)
    assert close(out_x, y, size) if gate and pre else bool((out_x == 7).all())
    assert _worst_tile(out, y * g if gate else y) < TILE
    assert not (gate and pre) or _worst_tile(out_x, y) < TILE
