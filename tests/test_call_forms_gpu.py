"""The operators' calls beside their plain use: a projection's bias that does not fit, a projection of no rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return tuple(torch.randn(2, 64, 96, device="cuda", generator=g) for _ in range(2))


def _block_args(x, z):
    g = torch.Generator(device="cuda").manual_seed(0)
    rn = lambda *s: 0.2 * torch.randn(*s, device="cuda", generator=g)
    H, P, N = 2, 32, 16
    zxbcdt = torch.cat([z.transpose(1, 2), x.transpose(1, 2), rn(2, 96, 2 * N + H)], 2)
    return (zxbcdt, rn(H * P + 2 * N, 4), rn(H * P + 2 * N), rn(H), -torch.ones(H, device="cuda"), rn(H), 64), dict(
        rmsnorm_weight=rn(H * P), outproj_weight=rn(48, H * P), headdim=P)


@pytest.mark.parametrize("shape", [(47,), (1, 47), (0,)])
def test_block_bias_that_does_not_fit_is_refused(shape):
    x, z = _operands()
    args, kw = _block_args(x, z)
    from mamba_amd.ops.triton.ssd_combined import mamba_split_conv1d_scan_combined
    with pytest.raises(RuntimeError):
        mamba_split_conv1d_scan_combined(*args, outproj_bias=torch.zeros(shape, device="cuda"), **kw)


@pytest.mark.parametrize("shape", [(1,), (1, 48)])
def test_block_bias_is_broadcast(shape):
    from mamba_amd.ops.triton.ssd_combined import mamba_split_conv1d_scan_combined
    x, z = _operands()
    args, kw = _block_args(x, z)
    plain = mamba_split_conv1d_scan_combined(*args, **kw)
    out = mamba_split_conv1d_scan_combined(*args, outproj_bias=torch.full(shape, 0.5, device="cuda"), **kw)
    assert float((out - plain - 0.5).abs().max()) <= 1e-5 * float(plain.abs().max())


def test_block_projection_without_rows():
    from mamba_amd.ops.triton.ssd_combined import mamba_split_conv1d_scan_combined
    x, z = _operands()
    args, kw = _block_args(x, z)
    kw["outproj_weight"] = kw["outproj_weight"][:0]
    assert mamba_split_conv1d_scan_combined(*args, **kw).shape == (2, 96, 0)
    args = [t.bfloat16() for t in args[:3]] + list(args[3:])
    kw["outproj_weight"] = kw["outproj_weight"].bfloat16()
    assert mamba_split_conv1d_scan_combined(*args, **kw).shape == (2, 96, 0)
