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
