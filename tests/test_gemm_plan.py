"""How the grouped bf16 products are planned (256 compute units, without a GPU too): the parts of the sum over k, and where a BLAS
library is the faster one."""
import pytest


def product(M, N, K, a_k=False, b_k=False):
    from mamba_amd import _lib
    a, b = (K, 1) if a_k else (1, M), (K, 1) if b_k else (1, N)
    return _lib.MambaGemm(4096, 4096, None, 4096, *a, *b, N, M, N, K, 1, 0, 0)   # (no memory is touched)


SHARED = -1


# 256 x 256 tiles that leave compute units idle, weight gradients of a mixer: the number of parts that was measured faster than the
# ones in brackets, -1 where idle units take the sums' ends; times in us
@pytest.mark.parametrize("M,N,K,want", [
    (1280, 2560, 16384, 5),        # 118 (-1: 146)
    (1408, 2816, 12288, 3),        # 128 (-1: 142)
    (1408, 2816, 16384, 3),        # 165 (-1: 178)
    (1536, 3072, 12288, 3),        # 133 (-1: 156)
    (1536, 3072, 16384, 3),        # 170 (-1: 201)
    (1536, 3072, 32768, 3),        # 322 (-1: 363)
    (1664, 3328, 12288, SHARED),   # 161 (2: 177)
    (1664, 3328, 16384, SHARED),   # 227 (2: 231)
    (1792, 3584, 12288, 2),        # 180 (-1: 197)
    (1792, 3584, 16384, 2),        # 232 (-1: 253)
    (1920, 3840, 32768, 2),        # 486 (-1: 535)
    (2048, 4096, 16384, 2),        # 264 (-1: 273)
    (2304, 4608, 16384, SHARED),   # 331 (1: 408)
    (2304, 4608, 32768, SHARED),   # 638 (1: 823)
    (2560, 5120, 16384, SHARED),   # 396 (1: 420)
    (2560, 5120, 32768, SHARED),   # 765 (1: 836)
])
@pytest.mark.parametrize("b_k", [False, True])
def test_parts_of_larger_tiles(M, N, K, want, b_k):
    from mamba_amd import _lib
    group = (_lib.MambaGemm * 1)(product(M, N, K, False, b_k))
    floats = _lib.load().mamba_gemm_plan(group, 1)
    tiles = -(-M // 256) * -(-N // 256)
    assert group[0].nsplit == want
    assert floats == 65536 * (tiles * want if want > 0 else tiles + 255)   # (a place per tile; the helpers' pieces lie at tile + helper)


# (which operands lie along k, sizes, whether the own kernels suit): both sides of each line
@pytest.mark.parametrize("a_k,b_k,M,N,K,want", [
    (True, True, 2000, 2000, 1000, 1), (True, True, 2000, 2000, 1008, 0),          # 8 GFLOP
    (False, True, 944, 2048, 4104, 1), (False, True, 944, 2048, 4096, 0),        # to 16 GFLOP: k over twice the larger side
    (False, True, 1024, 2048, 6144, 1), (False, True, 1024, 2048, 6136, 0),        # beyond: three times
    (False, False, 1024, 2048, 6144, 1), (False, False, 1024, 2048, 6136, 0),
    (False, False, 4080, 4088, 12264, 0), (False, False, 3840, 4088, 12264, 1),    # ... and fewer tiles of 256 x 256 than compute units
    (True, True, 1024, 1024, 4096, 0), (True, True, 2048, 2048, 6200, 0),          # both along k
    (True, True, 1024, 4096, 19992, 0), (True, True, 1024, 4096, 20000, 1),        # ... k from 20000 on
    (True, True, 128, 2048, 16384, 1), (True, True, 256, 2048, 12280, 0), (True, True, 256, 2048, 12288, 1),   # ... 48 times the shorter side
    (True, True, 160, 5120, 15360, 1), (True, True, 192, 5120, 15360, 1),          # (gradients of a 5120-channel mixer's projections)
    (True, False, 5120, 8192, 160, 1), (False, False, 5120, 8192, 192, 1), (True, False, 5120, 4096, 256, 1), (True, False, 5120, 4096, 264, 0),   # short k
    (True, False, 4864, 16384, 152, 1), (True, False, 5120, 16384, 160, 0), (False, False, 3072, 28672, 128, 0),   # ... up to 80 million results
    (False, False, 2047, 2048, 6144, 0),                                           # rows that lie on no 16 bytes
])
def test_where_the_own_kernels_suit(a_k, b_k, M, N, K, want):
    from mamba_amd import _lib
    assert _lib.load().mamba_gemm_suits(product(M, N, K, a_k, b_k)) == want
