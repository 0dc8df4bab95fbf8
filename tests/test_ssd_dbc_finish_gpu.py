"""dB and dC of the SSD backward pass from the state-path launch (ssd_dbc_fused.hip), where it forms them whole (state path and
in-chunk products) and where it adds to sums that a later launch finishes: each chunk length, state count and headdim, groups
of one and of several heads, a last chunk of 1, 17 and Q - 1 positions, packed sequences.  Reference: the quadratic form in
float64 on the same bf16 operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


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
    assert seen and seen[0] & 3 == 3, f"one workgroup does not hold a group here: {seen}"
    _check(B, C, _reference(x.detach(), dt, A, B.detach(), C.detach(), g, seq))


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
