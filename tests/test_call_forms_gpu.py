"""The operators' calls beside their plain use: forward-mode gradients, functorch's transforms, a jit trace, an in-place
write to the output, operands with the positions apart, a projection's bias that does not fit, a projection of no rows."""
import functools

import pytest
import torch
import torch.autograd.forward_ad as fwAD

pytestmark = pytest.mark.gpu


def _operands(seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return tuple(torch.randn(2, 64, 96, device="cuda", generator=g) for _ in range(2))


@functools.lru_cache(maxsize=None)
def _fixed(which, *shape):
    """Parameters of a call: the same tensor for every call of a test (a draw inside a traced call would be traced)."""
    return 0.2 * torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(which))


def _scan(x, z):
    """x, z: (2, 64, 96) on the GPU, as every call here takes them."""
    from mamba_amd.ops.selective_scan_interface import selective_scan_fn
    bc = _fixed(0, 2, 2, 1, 16, 96)
    return selective_scan_fn(x, torch.full_like(x, 0.1), -torch.ones(64, 16, device="cuda"), bc[0], bc[1], z=z)


def _ssd(x, z):
    from mamba_amd.ops.triton.ssd_combined import mamba_chunk_scan_combined
    bc = _fixed(0, 2, 2, 64, 1, 64)
    heads = lambda t: t.reshape(2, 64, 3, 32)
    return mamba_chunk_scan_combined(heads(x), torch.full((2, 64, 3), 0.1, device="cuda"), -torch.ones(3, device="cuda"), bc[0], bc[1], 64,
                                     z=heads(z))


def _inner(x, z):
    from mamba_amd.ops.selective_scan_interface import mamba_inner_fn
    return mamba_inner_fn(torch.cat([x, z], 1), _fixed(0, 64, 1, 4), _fixed(1, 64), _fixed(2, 4 + 32, 64), _fixed(3, 64, 4), _fixed(4, 32, 64), None,
                          -torch.ones(64, 16, device="cuda"), D=_fixed(5, 64), delta_bias=_fixed(6, 64))


def _block_args(x, z):
    H, P, N = 2, 32, 16
    zxbcdt = torch.cat([z.transpose(1, 2), x.transpose(1, 2), _fixed(0, 2, 96, 2 * N + H)], 2)
    return (zxbcdt, _fixed(1, H * P + 2 * N, 4), _fixed(2, H * P + 2 * N), _fixed(3, H), -torch.ones(H, device="cuda"), _fixed(4, H), 64), dict(
        rmsnorm_weight=_fixed(5, H * P), outproj_weight=_fixed(6, 48, H * P), headdim=P)


def _block(x, z):
    from mamba_amd.ops.triton.ssd_combined import mamba_split_conv1d_scan_combined
    args, kw = _block_args(x, z)
    return mamba_split_conv1d_scan_combined(*args, **kw)


def _conv(x, z):
    from mamba_amd.ops.causal_conv1d import causal_conv1d_fn
    return causal_conv1d_fn(x, torch.ones(64, 4, device="cuda"), activation="silu")


def _norm(x, z):
    from mamba_amd.ops.triton.layer_norm import rms_norm_fn
    return rms_norm_fn(x, torch.ones(96, device="cuda"), None, residual=z)


def _gated(x, z):
    from mamba_amd.ops.triton.layernorm_gated import rmsnorm_fn
    return rmsnorm_fn(x, torch.ones(96, device="cuda"), None, z=z)


CALLS = {f.__name__[1:]: f for f in (_scan, _ssd, _inner, _block, _conv, _norm, _gated)}
each_call = pytest.mark.parametrize("call", list(CALLS.values()), ids=list(CALLS))


@each_call
@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_is_refused(call, grad):
    """No operator has a forward-mode formula: a tangent is refused, never dropped."""
    x, z = _operands()
    with torch.set_grad_enabled(grad), fwAD.dual_level():
        dual = fwAD.make_dual(x, torch.ones_like(x))
        with pytest.raises(NotImplementedError):
            call(dual, z)


@each_call
def test_functorch_transforms_are_refused(call):
    x, z = _operands()
    with pytest.raises(RuntimeError):
        torch.func.jvp(lambda t: call(t, z), (x,), (torch.ones_like(x),))
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: call(x, z) + t)(torch.zeros(2, 1, device="cuda"))


@each_call
def test_traced_call_replays(call):
    """A jit trace holds the call itself, not the values it gave while it was traced."""
    x, z = _operands()
    with torch.no_grad():
        call(x, z)
        traced = torch.jit.trace(call, (x, z), check_trace=False)
        for seed in (1, 2, 3):
            x, z = _operands(seed)
            got, want = traced(x, z), call(x, z)  # (the block's projection: sums of 64 products in another order)
            assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())


@pytest.mark.parametrize("bias", [False, True])
def test_block_output_takes_in_place_writes(bias):
    from mamba_amd.ops.triton.ssd_combined import mamba_split_conv1d_scan_combined
    x, z = _operands()
    args, kw = _block_args(x, z)
    if bias:
        kw["outproj_bias"] = torch.zeros(48, device="cuda")
    args[0].requires_grad_()
    out = mamba_split_conv1d_scan_combined(*args, **kw)
    want, = torch.autograd.grad(out, args[0], torch.ones_like(out))
    out = mamba_split_conv1d_scan_combined(*args, **kw)
    out += 1.0
    got, = torch.autograd.grad(out, args[0], torch.ones_like(out))
    assert float((got - want).abs().max()) <= 1e-4 * float(want.abs().max())  # sums in another order (float atomics)


def test_strided_scan_operands_are_copied_once():
    """u, delta, z and B, C with the positions apart: one dense copy each in the forward pass (nothing of them remains
    but what the backward pass reads)."""
    from mamba_amd.ops.selective_scan_interface import selective_scan_fn
    g = torch.Generator(device="cuda").manual_seed(0)
    dim, L, n = 512, 1024, 16
    apart = lambda *s: torch.randn(*s[:-2], s[-1], s[-2], device="cuda", generator=g).transpose(-1, -2)
    u, delta, z, B, C = apart(2, dim, L), apart(2, dim, L), apart(2, dim, L), apart(2, 1, n, L), apart(2, 1, n, L)
    A = -torch.ones(dim, n, device="cuda")

    def allocations(*ops):
        leaves = [t.detach().requires_grad_() for t in ops]
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        out = selective_scan_fn(leaves[0], leaves[1], A, leaves[2], leaves[3], z=leaves[4], delta_softplus=True)
        return torch.cuda.memory_stats()["allocation.all.allocated"] - before, out, leaves

    dense = [t.contiguous() for t in (u, delta, B, C, z)]
    n_dense, want, want_leaves = allocations(*dense)
    n_apart, got, leaves = allocations(u, delta, B, C, z)
    assert n_apart - n_dense == 5
    assert torch.equal(got, want)
    dout = torch.randn(want.shape, device="cuda", generator=g)
    for a, b in zip(torch.autograd.grad(got, leaves, dout), torch.autograd.grad(want, want_leaves, dout)):
        assert torch.equal(a, b)


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
