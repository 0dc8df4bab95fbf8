"""The number of segments a forward Mamba-1 scan is cut into, by the library's rule (256 compute units, without a GPU too)."""
import pytest


# Scans that only scan_fwd_kernel takes: (batch, channels, positions, groups, states, input-independent B / C) and the number
# that was measured faster than the one in brackets, times in us
@pytest.mark.parametrize("b,d,L,G,N,const,want", [
    (2, 4160, 1261, 4, 4, 3, 1),      # 53 (5: 70)
    (3, 3776, 5821, 2, 8, 0, 1),      # 390 (2: 454)
    (2, 1552, 4029, 1, 64, 0, 5),     # 420 (32: 501)
    (6, 656, 2371, 4, 64, 3, 10),     # 291 (19: 334)
    (2, 2736, 684, 2, 64, 0, 1),      # 137 (6: 152)
    (4, 2336, 319, 1, 16, 3, 1),      # 39 (3: 41)
])
def test_scans_of_the_other_kernel(b, d, L, G, N, const, want):
    from mamba_amd import _lib
    p = _lib.MambaScanParams()
    for k, v in dict(batch=b, dim=d, seqlen=L, ngroups=G, dstate=N, bc_const=const, dtype=1).items():
        setattr(p, k, v)
    assert _lib.load().mamba1_scan_segments(p, 0) == want


# Scans that scan_fwd_serial_kernel takes, one sequence or a few of few channels, 16 states: the number that was measured the faster
# one; times in us
@pytest.mark.parametrize("b,d,L,want", [
    (1, 144, 192, 1),      # 12.2 (2: 13.5)
    (1, 768, 129, 1),      # 13.3 (2: 14.9)
    (1, 768, 192, 1),      # 12.2 (2: 13.8)
    (1, 768, 256, 1),      # 12.2 (2: 13.7)
    (1, 1024, 160, 1),     # 12.3 (2: 13.9)
    (1, 1536, 192, 1),     # 12.4 (2: 14.0)
    (1, 1536, 250, 1),     # 13.8 (2: 15.2)
    (1, 1536, 256, 1),     # 12.3 (2: 13.7)
    (1, 2048, 256, 1),     # 12.3 (2: 13.8)
    (2, 768, 129, 1),      # 13.3 (2: 15.0)
    (2, 1024, 256, 1),     # 12.3 (2: 13.9)
    (4, 768, 192, 1),      # 12.5 (2: 15.1)
    (8, 768, 256, 1),      # 15.5 (2: 18.8)
    (2, 1536, 257, 1),     # 18.2 (3: 21.3)
    (2, 2720, 274, 1),     # 22.2 (3: 23.5)
    (1, 768, 384, 3),      # 13.9 (1: 17.0)
    (1, 1536, 384, 3),     # 14.9 (1: 17.2)
    (2, 1024, 320, 3),     # 15.2 (1: 17.2)
    (1, 1536, 512, 4),     # 16.9 (1: 21.9)
    (1, 1536, 777, 7),     # 23.2 (1: 35.2)
])
def test_few_channels(b, d, L, want):
    from mamba_amd import _lib
    p = _lib.MambaScanParams()
    for k, v in dict(batch=b, dim=d, seqlen=L, ngroups=1, dstate=16, dtype=1).items():
        setattr(p, k, v)
    assert _lib.load().mamba1_scan_segments(p, 0) == want
