"""The grouped bf16 products whose operands lie on 16 bytes (gemm_ring_kernel and gemm_wide_kernel in gemm.hip): edges of the tiles,
of the stages and of a split's k, every layout of both operands, beside values that must not be read into a result.
Reference: fp64 products."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# M, N multiples of 8 where the operand lies along its rows, K where one lies along k
SHAPES = [(8, 8, 8), (64, 64, 64), (72, 136, 72), (200, 56, 128), (64, 192, 200), (136, 64, 2072), (80, 72, 4104), (1000, 768, 1536)]
ODD_K = [(64, 128, 33), (72, 64, 97), (128, 136, 1001), (64, 64, 1)]        # both along their rows: any K
ODD_ROWS = [(65, 127, 64), (1, 3, 72), (100, 66, 2048), (129, 63, 4120)]     # both along k: any M and N


@pytest.mark.parametrize("a_k,b_k,shapes", [(a, b, SHAPES) for a in (True, False) for b in (True, False)] + [(False, False, ODD_K), (True, True, ODD_ROWS)])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_products(a_k, b_k, shapes, out):
    check(a_k, b_k, shapes, out, 3)


# Larger tiles: 128 x 128 without splits (a K shorter than the ring, ragged ones, a row of one element more than the tiles), with
# them, and 256 x 256; in one call with a product of 64 x 64
WIDE = [(2176, 2048, 16), (2056, 2184, 72), (72, 136, 72), (136, 200, 160008)]
WIDE_256 = [(1800, 1544, 3080), (1544, 1800, 3112), (64, 64, 64), (2048, 2048, 2056)]
WIDE_HELPED = [(2816, 3080, 9016), (64, 64, 64), (2568, 2824, 9016)]     # 143 and 132 tiles: the idle CUs take the ends of the sums
# 256 x 256 uncut, K shorter than a wave's ring and not, ragged: bias alone, neither, bias and what lay there, that alone (check)
WIDE_WHOLE = [(5128, 8200, 200), (5120, 16392, 104), (5128, 8200, 232), (8200, 16392, 64)]
WIDE_ODD_K = [(2184, 2056, 33), (136, 200, 160001), (64, 64, 33), (1800, 1544, 3081)]
WIDE_ODD_ROWS = [(2049, 2183, 72), (65, 129, 500008), (1, 3, 72), (1801, 1543, 3080)]
# how a product by itself goes: its sum whole, cut into parts, or whole with the idle CUs' help
FORMS = {tuple(WIDE): ["whole", "whole", None, "cut"], tuple(WIDE_256): ["cut", "cut", None, "cut"], tuple(WIDE_HELPED): ["helped", None, "helped"],
         tuple(WIDE_WHOLE): ["whole"] * 4}


@pytest.mark.parametrize("a_k,b_k,shapes", [(a, b, s) for a in (True, False) for b in (True, False) for s in (WIDE, WIDE_256, WIDE_HELPED, WIDE_WHOLE)] +
                         [(False, False, WIDE_ODD_K), (False, False, [(2816, 3080, 9009), (2568, 2824, 9009)]), (True, True, WIDE_ODD_ROWS)])
@pytest.mark.parametrize("out,pad", [(torch.bfloat16, 8), (torch.bfloat16, 3), (torch.float32, 3)])
def test_larger_tiles(a_k, b_k, shapes, out, pad):
    check(a_k, b_k, shapes, out, pad, FORMS.get(tuple(shapes)))


# what a plan would give helpers, or cut, runs whole without a plan and without a workspace
@pytest.mark.parametrize("shapes", [[WIDE_HELPED[0], WIDE[3], WIDE_256[0]], [(768, 1536, 2000), (64, 64, 64)]])
def test_whole_sums_need_no_workspace(shapes):
    check(False, False, shapes, torch.bfloat16, 8, planned=False)


def form(lib, product):
    group = (type(product) * 1)(product)
    floats, parts = lib.mamba_gemm_plan(group, 1), group[0].nsplit
    assert floats >= 0 and (floats == 0) == (parts == 1)
    return "cut" if parts > 1 else "helped" if parts < 0 else "whole"


def check(a_k, b_k, shapes, out, pad, forms=None, planned=True):
    from mamba_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(5)

    def operand(rows, k, along_k):  # 8 values of NaN behind every line and a line of them behind the last
        lines, n = (rows, k) if along_k else (k, rows)
        t = torch.full((lines + 1, (n + 7) // 8 * 8 + 8), float("nan"), device="cuda", dtype=torch.bfloat16)
        t[:lines, :n] = torch.randn(lines, n, device="cuda", generator=gen).bfloat16()
        t = t[:lines, :n]
        return t if along_k else t.t()

    for first in range(0, len(shapes), 4):
        count, keep = len(shapes[first:first + 4]), []
        group = (_lib.MambaGemm * 4)()
        for j, (M, N, K) in enumerate(shapes[first:first + 4]):
            A, B, bias = operand(M, K, a_k), operand(N, K, b_k), torch.randn(N, device="cuda", generator=gen).bfloat16()
            D = torch.full((M, N + pad), 0.5, device="cuda", dtype=out)
            with_bias, accumulate = j % 2 == 0, j >= 2
            D[:, :N] = torch.randn(M, N, device="cuda", generator=gen)
            want = A.double() @ B.double().t() + (bias.double() if with_bias else 0) + (D[:, :N].double() if accumulate else 0)
            size = A.double().abs() @ B.double().abs().t() + 1 + D[:, :N].double().abs()
            group[j] = _lib.MambaGemm(A.data_ptr(), B.data_ptr(), bias.data_ptr() if with_bias else None, D.data_ptr(), *A.stride(), *B.stride(),
                                      N + pad, M, N, K, _lib.DTYPE_CODE[out], int(accumulate), 0)
            keep.append((A, B, bias, D, want, size, K))
        for j, want_form in enumerate(forms or []):
            assert want_form in (None, form(lib, group[j])), shapes[j]
        floats = lib.mamba_gemm_plan(group, count)
        assert floats >= 0
        ws = torch.full((max(floats, 1),), float("nan"), device="cuda")
        if not planned:
            for product in group:
                product.nsplit = 1
        _lib.check(lib.mamba_gemm(group, count, ws.data_ptr() if planned else None, _lib.current_stream(ws.device)), "mamba_gemm")
        for A, B, bias, D, want, size, K in keep:
            N = want.shape[1]
            # fp32 sums of K terms, and one rounding to the result's type
            bound = 2.0 ** -24 * (16 + 4 * K ** 0.5) * size + (2.0 ** -8 if out == torch.bfloat16 else 0) * want.abs()
            assert bool(((D[:, :N].double() - want).abs() <= bound).all())
            assert bool((D[:, N:] == 0.5).all())
