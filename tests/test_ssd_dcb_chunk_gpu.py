"""The dCB stage of the SSD backward pass at the sizes where its two kernels and the edges of the one that holds a chunk's
whole triangle lie (ssd_dcb_chunk.hip): each chunk length, one and several head lists, a last chunk of 1 to Q positions,
packed sequences, both headdims.  Reference: the stage's formula in float64 on the same bf16 operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(x, g, B, C, dt, dA, Q, seq):
    """dCB (b, c, G, Q, Q), the ddA_cumsum share (b, H, c, Q), and the sums of the absolute terms of both."""
    b, L, H, P = x.shape
    G, nc = B.shape[2], dA.shape[2]
    pad = lambda t: torch.nn.functional.pad(t.double(), (0, 0, 0, 0, 0, nc * Q - L)).reshape(b, nc, Q, *t.shape[2:])
    ids = torch.full((b, nc * Q), -1, device=x.device)
    ids[:, :L] = 0 if seq is None else seq
    ids = ids.reshape(b, nc, Q)
    live = (ids[..., :, None] == ids[..., None, :]) & (ids[..., :, None] >= 0) & torch.ones(Q, Q, device=x.device).tril().bool()
    xs, gs, Bs, Cs = pad(x), pad(g), pad(B), pad(C)
    dCB = torch.zeros(b, nc, G, Q, Q, dtype=torch.float64, device=x.device)
    size = torch.zeros_like(dCB)
    dda, dda_size = torch.zeros(b, H, nc, Q, dtype=torch.float64, device=x.device), torch.zeros(b, H, nc, Q, dtype=torch.float64, device=x.device)
    for h in range(H):
        k = h // (H // G)
        a, w = dA[:, h].double(), dt[:, h].double()
        decay = torch.where(live, torch.exp((a[..., :, None] - a[..., None, :]).clamp(max=0)) * w[..., None, :], 0.0)
        prod = torch.matmul(gs[:, :, :, h], xs[:, :, :, h].transpose(-1, -2).contiguous())
        absl = torch.matmul(gs[:, :, :, h].abs(), xs[:, :, :, h].abs().transpose(-1, -2).contiguous())
        CB = torch.matmul(Cs[:, :, :, k], Bs[:, :, :, k].transpose(-1, -2).contiguous())
        CBabs = torch.matmul(Cs[:, :, :, k].abs(), Bs[:, :, :, k].abs().transpose(-1, -2).contiguous())
        dCB[:, :, k] += prod * decay
        size[:, :, k] += absl * decay
        terms, terms_abs = prod * decay * CB, absl * decay * CBabs
        dda[:, h] = terms.sum(-1) - terms.sum(-2)
        dda_size[:, h] = terms_abs.sum(-1) + terms_abs.sum(-2)
    return dCB, size, dda, dda_size


# (batch, seqlen, heads, groups, headdim, states, chunk): a list of 8 heads stored whole; several lists on short and long
# chunks; groups of 3 and of 1 head; a last chunk of 1, 17 and Q - 1 positions; many heads in few lists
@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (2, 1024, 16, 2, 64, 128, 64), (1, 961, 16, 1, 64, 128, 64), (2, 81, 20, 1, 32, 64, 64),
    (2, 1024, 24, 1, 64, 128, 128), (1, 1169, 16, 1, 64, 64, 128), (3, 2047, 12, 4, 64, 128, 128),
    (4, 2048, 80, 1, 64, 128, 256), (2, 24 * 256 + 1, 12, 4, 64, 128, 256), (1, 8192 - 239, 64, 1, 32, 128, 256),
])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("form_cb", [True, False])
def test_dcb_stage(b, L, H, G, P, N, Q, packed, form_cb):
    from mamba_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(L + Q + H)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    nc = -(-L // Q)
    x, g, B, C = randn(b, L, H, P), randn(b, L, H, P), randn(b, L, G, N), randn(b, L, G, N)
    dt = 0.1 * torch.rand(b, H, nc * Q, device="cuda", generator=gen)
    dt[:, :, L:] = 0
    dt = dt.reshape(b, H, nc, Q)
    dA = torch.cumsum(dt * -(0.1 + 5 * torch.rand(H, device="cuda", generator=gen))[None, :, None, None], -1).contiguous()
    seq = None
    if packed:
        ends = torch.tensor([0, L // 7, L // 7 + 1, L // 2 + 5], device="cuda")
        seq = (torch.arange(L, device="cuda")[:, None] >= ends).sum(-1).int()[None].expand(b, L).contiguous()
    start = torch.randn(b, H, nc, Q, device="cuda", generator=gen)   # what the stages before have left
    dda = start.clone()
    dCB = torch.zeros(b, nc, G, Q, Q, device="cuda")
    other = torch.zeros(1 << 12, device="cuda")                      # fields that this stage does not read
    p = _lib.SsdParams()
    for k, v in dict(batch=b, seqlen=L, nheads=H, headdim=P, dstate=N, ngroups=G, chunk_size=Q, nchunks=nc, dtype=1).items():
        setattr(p, k, v)
    for k in ("dt", "A", "ddt_out", "dB32", "dC32", "dx", "ddt", "dA", "states_lp", "dstates_lp", "out", "final_states"):
        setattr(p, k, other.data_ptr())
    for k, t in (("x", x), ("dout", g), ("B", B), ("C", C)):
        setattr(p, k, t.data_ptr())
        for d, s in zip(("bs", "ls", "gs" if k in "BC" else "hs"), t.stride()):
            setattr(p, f"{k}_{d}", s)
    p.dt_out, p.dA_cumsum, p.ddA_cumsum, p.dCB = dt.data_ptr(), dA.data_ptr(), dda.data_ptr(), dCB.data_ptr()
    p.seq_idx = seq.data_ptr() if packed else None
    stream = _lib.current_stream(x.device)
    if not form_cb:
        CB = torch.empty_like(dCB)
        p.CB = CB.data_ptr()
        _lib.check(lib.ssd_bmm_chunk_fwd(p, stream), "ssd_bmm_chunk_fwd")
    elif not lib.ssd_bwd_overwrites(p) & 4 and P == 64:
        pytest.skip("the library asks for CB here")
    _lib.check(lib.ssd_bwd_dcb(p, stream), "ssd_bwd_dcb")
    torch.cuda.synchronize()
    want, size, dda_want, dda_size = _reference(x, g, B, C, dt, dA, Q, seq)
    # fp32 sums of up to P (products), H / G (heads) and 2 Q (rows and columns) terms, exponents and a decay of a few units
    # each: 2^-24 times the terms' number is the bound of the worst order, its square root what rounding errors add up to
    eps = 2.0 ** -24
    low = torch.zeros(Q // 64, Q // 64, device="cuda").fill_(1).tril().bool().repeat_interleave(64, 0).repeat_interleave(64, 1)
    err = (dCB.double() - want).abs()
    assert bool((err <= eps * (16 + (P + H // G) ** 0.5 * 4) * size + 1e-30)[..., low].all()), float((err / (size + 1e-30))[..., low].max())
    derr = (dda.double() - start.double() - dda_want).abs()
    bound = eps * ((16 + (P + N + 2 * Q) ** 0.5 * 4) * dda_size + 4 * start.abs().double())
    assert bool((derr <= bound).all()), float((derr - bound).max())
