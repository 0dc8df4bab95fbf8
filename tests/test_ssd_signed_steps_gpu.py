"""Steps of either sign (no softplus, dt_limit open below) through the chunked scan.  The kernels take the decay between two
positions apart at a position between them; with a step below zero in between, one of the two exponents is above zero while
their sum is not.  Reference: the quadratic form in float64 on the same operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(x, dt, A, B, C):
    L, H, G = x.shape[1], x.shape[2], B.shape[2]
    a = torch.cumsum(dt * A, 1).transpose(1, 2)
    w = torch.where(torch.ones(L, L, device=x.device).tril().bool(), a[..., :, None] - a[..., None, :], float("-inf")).exp()
    S = torch.matmul(C.transpose(1, 2), B.permute(0, 2, 3, 1).contiguous()).repeat_interleave(H // G, 1)
    return torch.matmul(S * w, (x * dt[..., None]).transpose(1, 2)).transpose(1, 2)


def _inputs(b, L, H, G, P, N):
    """A step below zero in front of every 16 positions, which no tile of 16 x 16 has inside; decay over any 16 of them."""
    gen = torch.Generator(device="cuda").manual_seed(L + H)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    x, g, B, C = randn(b, L, H, P), randn(b, L, H, P), randn(b, L, G, N), randn(b, L, G, N)
    dt = 0.01 + 0.05 * torch.rand(b, L, H, device="cuda", generator=gen)
    dt[:, 16::16] = -0.05
    return x, dt, -(0.5 + torch.rand(H, device="cuda", generator=gen)), B, C, g


# Operands of the products and the result are rounded to bf16 (at most 2^-9 of each, of either sign): two such roundings
BOUND = 2.0 ** -8
OPEN = (-float("inf"), float("inf"))


# more workgroups than a card of 256 CUs, one tile per wave and the group's C B^T kept, and few workgroups; two tiles per wave
@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (4, 2047, 64, 8, 64, 128, 64), (2, 2047, 80, 16, 64, 64, 64), (4, 2001, 64, 8, 32, 128, 128), (4, 2048, 24, 8, 64, 128, 128),
    (1, 1000, 8, 1, 64, 128, 128), (2, 1024, 40, 1, 64, 128, 256),
])
def test_forward(b, L, H, G, P, N, Q):
    from mamba_amd.ops.triton.ssd_combined import _mamba_chunk_scan_combined_fwd
    x, dt, A, B, C, _ = _inputs(b, L, H, G, P, N)
    y = _mamba_chunk_scan_combined_fwd(x, dt, A, B, C, Q, dt_limit=OPEN)[0].double()  # (keeps the chunk that is named)
    want = _reference(*[t.detach().double() for t in (x, dt, A, B, C)])
    assert float((y - want).norm() / want.norm()) <= BOUND


# dB and dC, whose in-chunk share is dCB: sizes at which one workgroup holds a chunk's whole triangle (ssd_dcb_chunk.hip; the
# tile pairs of ssd_bwd.hip cut both exponents at 0)
@pytest.mark.parametrize("b,L,H,G,P,N,Q", [
    (2, 2048, 40, 8, 64, 128, 128), (1, 2033, 16, 8, 64, 128, 64), (16, 1000, 40, 2, 32, 64, 64), (8, 1024, 64, 8, 64, 128, 256),
    (8, 1000, 64, 8, 32, 64, 128),
])
def test_dB_dC(b, L, H, G, P, N, Q):
    from mamba_amd.ops.triton.ssd_combined import mamba_chunk_scan_combined
    x, dt, A, B, C, g = _inputs(b, L, H, G, P, N)
    B.requires_grad_(), C.requires_grad_()
    got = torch.autograd.grad(mamba_chunk_scan_combined(x, dt, A, B, C, Q, dt_limit=OPEN), [B, C], g)
    Bd, Cd = B.detach().double().requires_grad_(), C.detach().double().requires_grad_()
    want = torch.autograd.grad(_reference(x.double(), dt.double(), A.double(), Bd, Cd), [Bd, Cd], g.double())
    for name, u, v in zip(("dB", "dC"), got, want):
        err = float((u.double() - v).norm() / v.norm())
        assert err <= BOUND, f"{name}: {err:.5f}"
