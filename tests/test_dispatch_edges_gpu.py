"""The branches that the host rules choose by size, dtype and alignment, at the sizes where they can go wrong (edges of
tiles and segments, remainders, the smallest and largest of a range), against the oracles; the cases and tolerances of
the operators' own test files."""
import pytest
import torch

import test_causal_conv1d_gpu as conv
import test_layer_norm_gpu as norm
import test_layernorm_gated_gpu as gated
import test_mamba1_gpu as mamba1
import test_ssd_gpu as ssd

pytestmark = pytest.mark.gpu


# A sequence in segments: two tiles, the last of one position; rows of odd length; segments of unequal length; more than
# 16 states; constant B or C
@pytest.mark.parametrize("itype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,dim,dstate,seqlen,groups,var", [(1, 40, 16, 129, 1, True), (1, 64, 16, 777, 0, True), (2, 32, 24, 1000, 2, True),
                                                                (1, 16, 16, 1933, 1, True), (1, 32, 16, 515, 1, False)])
def test_scan_segments(batch, dim, dstate, seqlen, groups, var, itype):
    from mamba_amd import _lib
    p = _lib.MambaScanParams()
    p.batch, p.dim, p.seqlen, p.dstate, p.ngroups, p.dtype = batch, dim, seqlen, dstate, max(groups, 1), _lib.DTYPE_CODE[itype]
    assert all(_lib.load().mamba1_scan_segments(p, back) > 1 for back in (0, 1))
    mamba1._run_case(batch, dim, dstate, seqlen, itype, groups, var_B=var, var_C=var)


# The same with steps up to which nothing of the segment before is left (exp(-16 * 20) is zero), in every channel or in
# one position out of 16 among steps of 1e-3; the last segment is a tile of 1 and of 3 positions.  Tolerance: |A| step is
# at most 20 wherever a product still counts (exp(-20) = 2e-9), which an fp32 exponent holds to 20 * 2^-23, and a sum over
# a tile and 16 states adds about as much again: 5e-6 of each channel's norm.  dA and ddelta have a term
# adjoint * decay * state, formed as adjoint * (state - input): one rounding of adjoint * input, the larger the smaller the
# decay, is allowed beside that.
@pytest.mark.parametrize("seqlen", [129, 515, 771])
@pytest.mark.parametrize("step,rare", [(6.0, False), (20.0, False), (20.0, True)])
def test_scan_segments_large_steps(seqlen, step, rare):
    from mamba_amd.ops.selective_scan_interface import selective_scan_fn
    from oracle.mamba1 import selective_scan_oracle
    g = torch.Generator().manual_seed(seqlen)
    dim, n = 32, 16
    rn = lambda *s: torch.randn(*s, generator=g)
    delta = step * (0.8 + 0.2 * torch.rand(1, dim, seqlen, generator=g))
    if rare:
        delta = torch.where(torch.rand(1, dim, seqlen, generator=g) < 1 / 16, delta, 1e-3 * torch.rand(1, dim, seqlen, generator=g))
    delta[:, ::4] *= 1e-3  # channels in which the state does reach across the segments
    leaves = [rn(1, dim, seqlen), delta, -torch.arange(1, n + 1).float().repeat(dim, 1), rn(1, 1, n, seqlen), rn(1, 1, n, seqlen), rn(dim),
              rn(1, dim, seqlen)]
    dout = rn(1, dim, seqlen)
    ref = [t.double().requires_grad_() for t in leaves]
    want = selective_scan_oracle(*ref, compute_dtype=torch.float64)
    want = (want, *torch.autograd.grad(want, ref, dout.double()))
    got = [t.cuda().requires_grad_() for t in leaves]
    out = selective_scan_fn(*got)
    got = (out, *torch.autograd.grad(out, got, dout.cuda()))
    u, step, A, B, C, _, z = [t.detach()[0] if t.dim() > 2 else t.detach() for t in ref]  # (dim, L), A (dim, n), B and C (1, n, L)
    dy = dout[0].double() * torch.nn.functional.silu(z)
    term = (step * u * dy)[:, None] * B * C  # adjoint * input, (dim, n, L)
    rounding = dict(dA=(term * step[:, None]).norm(dim=2).norm(dim=1), ddelta=(term * A[..., None]).abs().sum(1).norm(dim=1))
    for name, a, b in zip(("out", "du", "ddelta", "dA", "dB", "dC", "dD", "dz"), got, want):
        a, b = a.detach().double().cpu(), b.detach()
        assert bool(torch.isfinite(a).all()), name
        if b.dim() > 1:
            a, b = a.flatten(0, -2), b.flatten(0, -2)  # per channel or state
        err, bound = (a - b).norm(dim=-1), 5e-6 * b.norm(dim=-1) + 2.0 ** -23 * rounding.get(name, 0.0)
        assert bool((err <= bound).all()), (name, float((err / bound).max()))


def test_scan_segments_nan_stays_in_its_segment():
    """A NaN in C reaches the gradients of its own position and the ones before it, not those between it and the last
    segment, whose first piece is read from 8 positions before the end of the row."""
    from mamba_amd.ops.selective_scan_interface import selective_scan_fn
    g = torch.Generator().manual_seed(0)
    dim, n, L, at = 32, 16, 771, 765
    rn = lambda *s: torch.randn(*s, generator=g).cuda()
    u, z, dout = rn(1, dim, L).requires_grad_(), rn(1, dim, L), rn(1, dim, L)
    A, B, C = -torch.arange(1, n + 1).float().repeat(dim, 1).cuda(), rn(1, 1, n, L), rn(1, 1, n, L)
    C[..., at] = float("nan")
    out = selective_scan_fn(u, torch.full_like(u, 0.01), A, B, C, z=z)
    du, = torch.autograd.grad(out, u, dout)
    nan = torch.isnan(du)[0].any(0)
    assert bool(nan[:at + 1].all()) and not bool(nan[at + 1:].any())


# channels next to each other, runs of 8 positions: below one run, its edges, one past; rows along the positions of a
# length that is no multiple of 8
@pytest.mark.parametrize("channel_last", [True, False])
@pytest.mark.parametrize("seqlen,seq_lens", [(2, None), (8, None), (9, None), (33, [5, 28]), (261, [100, 161])])
@pytest.mark.parametrize("width", [3, 4])
def test_conv_short_runs(seqlen, seq_lens, width, channel_last):
    conv._case(2, 264, seqlen, width, torch.bfloat16, channel_last, seq_lens=seq_lens)


# groups on the wide kernels that are no multiple of 512; parameters in bf16
@pytest.mark.parametrize("dim,group_size", [(2064, 1032), (3080, 3080), (8184, 8184)])
@pytest.mark.parametrize("wtype", [torch.float32, torch.bfloat16])
def test_gated_norm_wide_groups(dim, group_size, wtype):
    gated._case(37, dim, group_size, torch.bfloat16, norm_before_gate=False, has_bias=True, wtype=wtype)


# one, two, three and more rows per workgroup of the wide kernels (256 workgroups backward, 512 or 768 forward)
@pytest.mark.parametrize("rows", [256, 257, 600, 1100, 1800])
def test_gated_norm_wide_rows(rows):
    gated._case(rows, 5120, 5120, torch.bfloat16, norm_before_gate=False, has_bias=True)


@pytest.mark.parametrize("rows,dim", [(1, 8), (130, 2570), (700, 1032)])
def test_residual_norm_low_precision_parameters(rows, dim):
    from mamba_amd.ops.triton.layer_norm import layer_norm_fn
    g = torch.Generator().manual_seed(1)
    x, res, dy = (torch.randn(rows, dim, generator=g).cuda().bfloat16() for _ in range(3))
    w, b = (torch.randn(dim, generator=g).cuda().bfloat16() for _ in range(2))
    outs = []
    for wt in (torch.float32, torch.bfloat16):  # the same values either way
        leaves = [t.clone().requires_grad_() for t in (x, w.to(wt), b.to(wt), res)]
        out = layer_norm_fn(leaves[0], leaves[1], leaves[2], residual=leaves[3], eps=1e-5)
        outs.append((out, *torch.autograd.grad(out, leaves, dy)))
    for name, a, c in zip(("out", "dx", "dweight", "dbias", "dresidual"), *outs):
        norm._close(name, c, a, 1e-2 if name in ("dweight", "dbias") else 0, 1e-3)
    assert outs[1][2].dtype == torch.bfloat16


# chunk states and gradients on the wide kernels with a last chunk of any length; few heads (short head lists, several
# k steps in flight, the steps' sums in the chunk_state kernel); every chunk length, and all three operand types of the
# scan; 64 states on the tiled ones
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("seqlen,chunk,dstate,ngroups", [(1, 64, 128, 1), (65, 64, 128, 2), (129, 128, 128, 1), (257, 256, 128, 1), (415, 256, 64, 2),
                                                         (500, 128, 64, 1), (799, 256, 128, 4)])
@pytest.mark.parametrize("host", ["extension", "python"])  # python: the chunk length as it is given
def test_ssd_ragged(monkeypatch, seqlen, chunk, dstate, ngroups, dtype, host):
    from mamba_amd import _lib
    if host == "python":
        monkeypatch.setattr(_lib, "torch_ext", lambda: None)
    # (with the initial states dx and dB reach 60, where one bf16 step is 0.25: three times the absolute tolerance)
    ssd._bwd_case(2, seqlen, 4, 64, dstate, ngroups, chunk, dtype, has_init=True, grad_scale=3.0 if dtype == torch.bfloat16 else 1.0)


@pytest.mark.parametrize("seq_lens", [[3, 126, 70], [400, 13]])
def test_ssd_ragged_packed(seq_lens):
    ssd._bwd_case(1, sum(seq_lens), 24, 64, 128, 1, 256, torch.bfloat16, seq_lens=seq_lens)


# The chunk the kernels take for a call that names one: both sides of every line of the rule, for calls with and without
# gradients.  The forward pass at that chunk gives the same bits through the stage-level function, which keeps what it is
# given; every other chunk rounds elsewhere (the bound: bf16 inputs of the scan, 2^-8 of the largest output).
@pytest.mark.parametrize("heads,seqlen,groups,dstate,named,backward,chunk", [
    (8, 64, 1, 64, 256, False, 64), (8, 128, 1, 64, 256, True, 128),                  # one chunk
    (19, 1280, 1, 128, 64, False, 64), (24, 1024, 1, 128, 64, False, 128),            # 95, 96 workgroups of 256
    (53, 768, 1, 128, 256, False, 128), (40, 1024, 1, 128, 128, False, 256),          # 159, 160
    (112, 383, 1, 128, 128, False, 128), (127, 513, 1, 64, 256, False, 128), (128, 513, 1, 64, 256, False, 256),
    (64, 2815, 1, 64, 256, False, 256), (64, 2815, 1, 64, 64, False, 128), (64, 3072, 1, 64, 64, False, 256),
    (51, 1280, 1, 128, 64, True, 64), (32, 2048, 1, 128, 64, True, 128), (32, 3071, 8, 128, 256, True, 256),
    (24, 4096, 8, 64, 256, True, 128), (64, 3072, 1, 64, 256, True, 256), (64, 3072, 1, 128, 128, True, 256),
    (72, 4039, 8, 128, 256, True, 128), (64, 3072, 8, 128, 128, True, 128), (64, 8192, 8, 128, 128, True, 256)])
def test_ssd_chunk_rule(heads, seqlen, groups, dstate, named, backward, chunk):
    from mamba_amd.ops.triton.ssd_combined import _mamba_chunk_scan_combined_fwd, mamba_chunk_scan_combined
    g = torch.Generator(device="cuda").manual_seed(0)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()
    args = [rn(1, seqlen, heads, 64), rn(1, seqlen, heads), -torch.ones(heads, device="cuda"), rn(1, seqlen, groups, dstate),
            rn(1, seqlen, groups, dstate)]
    kw = dict(dt_bias=torch.full((heads,), -4.0, device="cuda"), dt_softplus=True)
    args[0].requires_grad_(backward)
    out, final = mamba_chunk_scan_combined(*args, named, return_final_states=True, **kw)
    with torch.no_grad():
        want, at_chunk = (_mamba_chunk_scan_combined_fwd(*args, q, **kw) for q in (named, chunk))
    assert torch.equal(out, at_chunk[0]) and torch.equal(final, at_chunk[5])
    assert float((out - want[0]).detach().abs().max()) <= 2.0 ** -8 * float(want[0].abs().max())
