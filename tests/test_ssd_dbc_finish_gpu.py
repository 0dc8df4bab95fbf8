"""dB and dC of the SSD backward pass from the state-path launch (ssd_dbc_fused.hip), where it forms them whole (state path and
in-chunk products) and where it adds to sums that a later launch finishes: each chunk length, state count and headdim, groups
of one and of several heads, a last chunk of 1, 17 and Q - 1 positions, packed sequences.  Reference: the quadratic form in
float64 on the same bf16 operands."""
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


def _reference(x, dt, A, B, C, g, seq):
    """dB, dC and the sums of the absolute terms of both."""
    b, L, H, P = x.shape
    G = B.shape[2]
    live = torch.ones(L, L, device=x.device).tril().bool()[None].expand(b, L, L)
    if seq is not None:
        live = live & (seq[:, :, None] == seq[:, None, :])
    out = [torch.zeros(b, G, L, B.shape[3], dtype=torch.float64, device=x.device) for _ in range(4)]
    Bd, Cd = B.double().transpose(1, 2).contiguous(), C.double().transpose(1, 2).contiguous()
    for h in range(H):
        k = h // (H // G)
        a = torch.cumsum(dt[:, :, h].double() * A[h].double(), 1)
        w = torch.where(live, torch.exp((a[:, :, None] - a[:, None, :]).clamp(max=0)) * dt[:, None, :, h].double(), 0.0)
        gx = [(t(g[:, :, h].double()), t(x[:, :, h].double()).transpose(-1, -2).contiguous()) for t in (lambda v: v, torch.abs)]
        for i, (gh, xh) in enumerate(gx):
            m = torch.matmul(gh, xh) * w
            Bk, Ck = (Bd[:, k], Cd[:, k]) if i == 0 else (Bd[:, k].abs(), Cd[:, k].abs())
            out[2 * i][:, k] += torch.matmul(m.transpose(-1, -2).contiguous(), Ck)
            out[2 * i + 1][:, k] += torch.matmul(m, Bk)
    return [t.transpose(1, 2) for t in out]


# A term takes the rounding to bf16 (at most 2^-8 of it) of dCB or of a chunk state or its gradient, the result another one
FACTOR = 2 * 2.0 ** -8


def _check(B, C, want):
    for name, got, w, size in (("dB", B.grad, want[0], want[2]), ("dC", C.grad, want[1], want[3])):
        err = (got.double() - w).abs()
        assert bool((err <= FACTOR * size + 1e-30).all()), f"{name}: {float((err / (size + 1e-30)).max()):.3e}"
        assert _worst_tile(got, w) < TILE, name


def _inputs(b, L, H, G, P, N, packed):
    gen = torch.Generator(device="cuda").manual_seed(L + N + H)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    x, g = randn(b, L, H, P), randn(b, L, H, P)
    B, C = randn(b, L, G, N).requires_grad_(), randn(b, L, G, N).requires_grad_()
    dt = 0.1 * torch.rand(b, L, H, device="cuda", generator=gen)
    A = -(0.1 + 5 * torch.rand(H, device="cuda", generator=gen))
    seq = None
    if packed:
        ends = torch.tensor([0, L // 7, L // 7 + 1, L // 2 + 5], device="cuda")
        seq = (torch.arange(L, device="cuda")[:, None] >= ends).sum(-1).int()[None].expand(b, L).contiguous()
    return x.requires_grad_(), g, B, C, dt, A, seq


@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (1, 4033, 16, 8, 64, 128, 64), (2, 2047, 24, 8, 64, 64, 64), (2, 1041, 32, 32, 32, 128, 64), (4, 1024, 16, 8, 32, 64, 64),
    (2, 2049, 16, 16, 64, 128, 128), (2, 2048, 32, 16, 64, 64, 128), (2, 1937, 16, 8, 32, 128, 128), (4, 1151, 16, 16, 32, 64, 128),
    (2, 2304, 16, 16, 64, 128, 256), (2, 1809, 32, 16, 64, 64, 256), (2, 1793, 32, 32, 32, 128, 256), (4, 1279, 32, 16, 32, 64, 256),
])
@pytest.mark.parametrize("packed", [False, True])
def test_finished_dB_dC(monkeypatch, b, L, H, G, P, N, Q, packed):
    from mamba_amd import _lib
    from mamba_amd.ops.triton import ssd_combined as sc
    lib = _lib.load()
    seen, real = [], lib.ssd_bwd_overwrites
    monkeypatch.setattr(_lib, "torch_ext", lambda: None)
    monkeypatch.setattr(lib, "ssd_bwd_overwrites", lambda p: seen.append(real(p)) or seen[-1])
    x, g, B, C, dt, A, seq = _inputs(b, L, H, G, P, N, packed)
    sc.mamba_chunk_scan_combined(x, dt, A, B, C, Q, seq_idx=seq).backward(g)
    # (the Python host side, whose question to the library can be seen; the launch that follows is the C++ host side's as well)
    assert seen and seen[0] & 3 == 3, f"one workgroup does not hold a group here: {seen}"
    _check(B, C, _reference(x.detach(), dt, A, B.detach(), C.detach(), g, seq))


def _reference_dt_dA(x, dt, A, B, C, g, seq):
    """The gradients with respect to dt and A of the same form."""
    b, L, H, P = x.shape
    live = torch.ones(L, L, device=x.device).tril().bool()[None].expand(b, L, L)
    if seq is not None:
        live = live & (seq[:, :, None] == seq[:, None, :])
    ddt, dA = torch.zeros(b, L, H, dtype=torch.float64, device=x.device), torch.zeros(H, dtype=torch.float64, device=x.device)
    for h in range(H):
        k, t = h // (H // B.shape[2]), dt[:, :, h].double()
        a = torch.cumsum(t * A[h].double(), 1)
        w = torch.where(live, torch.exp((a[:, :, None] - a[:, None, :]).clamp(max=0)), 0.0)
        w *= torch.matmul(C[:, :, k].double(), B[:, :, k].double().transpose(-1, -2).contiguous())
        w *= torch.matmul(g[:, :, h].double(), x[:, :, h].double().transpose(-1, -2).contiguous())
        cols = w.sum(1)
        da = (w * t[:, None, :]).sum(2) - cols * t
        run = da.flip(1).cumsum(1).flip(1)
        ddt[:, :, h], dA[h] = cols + run * A[h].double(), (run * t).sum()
    return ddt, dA


# groups of 8 and of 17 to 40 heads: a workgroup's list is longer than the ring of ddA_cumsum rows, and the sums of dCB stay in
# one workgroup; a last chunk of any length
@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (4, 1009, 64, 8, 64, 64, 64), (16, 1009, 40, 2, 64, 128, 64), (4, 1009, 64, 8, 32, 128, 128), (16, 1009, 34, 2, 32, 64, 128),
    (32, 1009, 80, 2, 64, 128, 128), (8, 897, 64, 8, 64, 128, 256), (16, 2032, 80, 2, 64, 128, 256),
])
@pytest.mark.parametrize("packed", [False, True])
def test_finished_dB_dC_of_large_groups(monkeypatch, b, L, H, G, P, N, Q, packed):
    from mamba_amd import _lib
    from mamba_amd.ops.triton import ssd_combined as sc
    lib = _lib.load()
    sums = torch.full((2, b * L * G * N), 7.0, device="cuda")  # in the place of the sums that the other order writes
    real = lib.ssd_combined_bwd

    def combined(p, stream):
        p.dB32, p.dC32 = sums[0].data_ptr(), sums[1].data_ptr()
        return real(p, stream)

    monkeypatch.setattr(_lib, "torch_ext", lambda: None)
    monkeypatch.setattr(lib, "ssd_combined_bwd", combined)
    x, g, B, C, dt, A, seq = _inputs(b, L, H, G, P, N, packed)
    dt.requires_grad_(), A.requires_grad_()
    sc.mamba_chunk_scan_combined(x, dt, A, B, C, Q, seq_idx=seq).backward(g)
    assert bool((sums == 7).all()), "dB and dC were not finished in the state-path launch"
    args = [t.detach() for t in (x, dt, A, B, C)]
    _check(B, C, _reference(*args, g, seq))
    for name, got, want in zip(("ddt", "dA"), (dt.grad, A.grad), _reference_dt_dA(*args, g, seq)):
        assert float((got.double() - want).norm() / want.norm()) < TILE, name


# lists of 1, 5, 12, 16, 17 and 40 heads of larger groups, short and long last chunks
@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (1, 321, 20, 1, 64, 128, 64), (2, 500, 48, 2, 32, 128, 64), (1, 145, 32, 1, 64, 128, 128), (2, 1151, 34, 1, 64, 64, 128),
    (4, 1024, 80, 1, 64, 128, 256), (2, 897, 48, 2, 32, 128, 256), (1, 1009, 17, 1, 32, 64, 256),
])
@pytest.mark.parametrize("deterministic", [False, True])
def test_added_dB_dC(monkeypatch, b, L, H, G, P, N, Q, deterministic):
    from mamba_amd.ops.triton import ssd_combined as sc
    if deterministic:
        monkeypatch.setenv("MAMBA_DETERMINISTIC", "1")
    x, g, B, C, dt, A, seq = _inputs(b, L, H, G, P, N, True)
    sc.mamba_chunk_scan_combined(x, dt, A, B, C, Q, seq_idx=seq).backward(g)
    _check(B, C, _reference(x.detach(), dt, A, B.detach(), C.detach(), g, seq))
