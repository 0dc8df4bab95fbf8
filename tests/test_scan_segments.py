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
