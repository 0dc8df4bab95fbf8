"""The grouped bf16 products (mamba_gemm in include/mamba_hip.h) against fp32 products of torch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# M, N, K: one element; edges of the 64 x 64 tile and of the 32-wide step; rows of every alignment; a ragged tail of k in
# the last of several splits; fewer rows than a piece of 8
SHAPES = [(1, 1, 1), (64, 64, 32), (65, 63, 33), (3, 200, 64), (80, 268, 100), (129, 5, 31), (96, 72, 2072), (48, 130, 4100)]


@pytest.mark.parametrize("a_kmajor", [True, False])
@pytest.mark.parametrize("b_kmajor", [True, False])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_grouped_products(a_kmajor, b_kmajor, out):
    from mamba_amd import _lib
    lib = _lib.load()
    g = torch.Generator().manual_seed(3)

    def operand(rows, k, kmajor):
        t = torch.randn(*((rows, k) if kmajor else (k, rows)), generator=g).to(device="cuda", dtype=torch.bfloat16)
        return t if kmajor else t.t()

    for first in range(0, len(SHAPES), 4):
        group, keep = (_lib.MambaGemm * 4)(), []
        for j, (M, N, K) in enumerate(SHAPES[first:first + 4]):
            A, B, bias = operand(M, K, a_kmajor), operand(N, K, b_kmajor), operand(1, N, True)[0].contiguous()
            with_bias, accumulate = j % 2 == 0, j >= 2
            D = torch.full((M, N + 3), 0.5, device="cuda", dtype=out)
            want = A.float() @ B.float().t() + (bias.float() if with_bias else 0) + (0.5 if accumulate else 0)
            ks = [(K, 1) if a_kmajor else (1, M), (K, 1) if b_kmajor else (1, N)]
            group[j] = _lib.MambaGemm(A.data_ptr(), B.data_ptr(), bias.data_ptr() if with_bias else None, D.data_ptr(), ks[0][0], ks[0][1],
                                      ks[1][0], ks[1][1], N + 3, M, N, K, _lib.DTYPE_CODE[out], int(accumulate), 0)
            keep.append((A, B, bias, D, want))
        floats = lib.mamba_gemm_plan(group, 4)
        assert floats >= 0 and (first == 0 or group[2].nsplit > 1)
        ws = torch.full((max(floats, 1),), float("nan"), device="cuda")
        _lib.check(lib.mamba_gemm(group, 4, ws.data_ptr(), _lib.current_stream(ws.device)), "mamba_gemm")
        for A, B, bias, D, want in keep:
            N = want.shape[1]
            rtol = 1e-2 if out == torch.bfloat16 else 1e-4
            torch.testing.assert_close(D[:, :N].float(), want, rtol=rtol, atol=1e-3 * want.abs().max().item() + 1e-4)
            assert bool((D[:, N:] == 0.5).all())
