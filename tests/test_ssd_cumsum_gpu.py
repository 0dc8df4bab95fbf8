"""The cumsum stages of the SSD scan, forward (dt, dA_cumsum) and backward (ddt, dA, ddt_bias), where four heads of a position
are one access and where they are not: 16- and 32-bit steps, heads side by side or apart, a multiple of four of them or not,
rows off the 8 bytes, chunks of one to four waves, several chunks per workgroup and a ragged last one.  Reference: float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("layout", ["dense", "rows", "odd_rows", "apart"])
# few pairs of a chunk and four heads (a workgroup each), and 150 and more (several chunks in one)
@pytest.mark.parametrize("b,L,H,Q", [(2, 1000, 8, 64), (1, 2049, 12, 256), (1, 511, 6, 128), (2, 577, 4, 192), (1, 130, 3, 256), (3, 100, 20, 48),
                                     (2, 5000, 22, 64), (1, 9001, 20, 256), (1, 4999, 18, 128), (2, 3001, 17, 192), (4, 2011, 12, 48)])
def test_cumsum(b, L, H, Q, layout, dtype):
    from mamba_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(L + Q + H)
    rand = lambda *s: torch.rand(*s, device="cuda", generator=gen)
    width, step = {"dense": (H, 1), "rows": (H + 8, 1), "odd_rows": (H + 3, 1), "apart": (2 * H, 2)}[layout]
    first = 4 if layout == "rows" else 0
    dt = (rand(b, L, width) * 4 - 3).to(dtype)[:, :, first:first + H * step:step]
    ddt = torch.full((b, L, width), -7.0, device="cuda").to(dtype)[:, :, first:first + H * step:step]
    nc = -(-L // Q)
    A, bias = -(0.1 + rand(H)), rand(H) - 0.5
    dt_out, dA = torch.empty(b, H, nc, Q, device="cuda"), torch.empty(b, H, nc, Q, device="cuda")
    ddA, ddt_out = rand(b, H, nc, Q) - 0.5, rand(b, H, nc, Q) - 0.5
    g_A, g_bias = torch.zeros(H, device="cuda"), torch.zeros(H, device="cuda")
    other = torch.zeros(1 << 12, device="cuda")
    p = _lib.SsdParams()
    for k, v in dict(batch=b, seqlen=L, nheads=H, headdim=64, dstate=64, ngroups=1, chunk_size=Q, nchunks=nc, dtype=1,
                     dt_dtype={torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype], dt_softplus=1).items():
        setattr(p, k, v)
    for k in ("x", "B", "C", "dout", "dCB", "dB32", "dC32", "dx", "states_lp", "dstates_lp", "out", "final_states", "CB"):
        setattr(p, k, other.data_ptr())
    p.dt_min, p.dt_max = 0.05, 2.0
    p.dt, p.A, p.dt_bias, p.dt_out, p.dA_cumsum = dt.data_ptr(), A.data_ptr(), bias.data_ptr(), dt_out.data_ptr(), dA.data_ptr()
    p.ddt, p.ddA_cumsum, p.ddt_out, p.dA, p.ddt_bias = ddt.data_ptr(), ddA.data_ptr(), ddt_out.data_ptr(), g_A.data_ptr(), g_bias.data_ptr()
    for name, t in (("dt", dt), ("ddt", ddt)):
        for d, s in zip(("bs", "ls", "hs"), t.stride()):
            setattr(p, f"{name}_{d}", s)
    stream = _lib.current_stream(dt.device)
    _lib.check(lib.ssd_chunk_cumsum_fwd(p, stream), "ssd_chunk_cumsum_fwd")
    _lib.check(lib.ssd_chunk_cumsum_bwd(p, stream), "ssd_chunk_cumsum_bwd")
    torch.cuda.synchronize()
    x = dt.double() + bias.double()
    v = torch.nn.functional.softplus(x)
    w = torch.zeros(b, nc * Q, H, dtype=torch.float64, device="cuda")
    w[:, :L] = v.clamp(0.05, 2.0)
    w = w.reshape(b, nc, Q, H).permute(0, 3, 1, 2)
    eps = 2.0 ** -24  # sums of Q terms, and a few roundings of the softplus and its derivative
    assert torch.allclose(dt_out.double(), w, rtol=16 * eps, atol=16 * eps)
    want = torch.cumsum(w * A.double()[None, :, None, None], -1)
    assert bool(((dA.double() - want).abs() <= (16 + Q ** 0.5) * eps * want.abs() + 16 * eps).all())
    run = torch.flip(torch.cumsum(torch.flip(ddA.double(), [-1]), -1), [-1])
    size = torch.flip(torch.cumsum(torch.flip(ddA.double().abs(), [-1]), -1), [-1])
    to_pos = lambda t: t.permute(0, 2, 3, 1).reshape(b, nc * Q, H)[:, :L]
    inside = ((v >= 0.05) & (v <= 2.0)) * torch.sigmoid(x)
    edge = ((v - 0.05).abs() < 1e-6) | ((v - 2.0).abs() < 1e-6)  # either side of the clamp is right there
    want = to_pos(run * A.double()[None, :, None, None] + ddt_out.double()) * inside
    size_ddt = to_pos(size * A.double().abs()[None, :, None, None] + ddt_out.double().abs())
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]  # of a value just above a power of two
    bound = (16 + Q ** 0.5) * eps * size_ddt + half_ulp * 1.01 * want.abs() + (2.0 ** -25 if dtype == torch.float16 else 0)
    assert bool((((ddt.double() - want).abs() <= bound) | edge).all())
    n = b * nc * Q
    dA_terms = to_pos(run * w)
    assert bool(((g_A.double() - dA_terms.sum((0, 1))).abs() <= (32 + n ** 0.5) * eps * to_pos(size * w).sum((0, 1))).all())
    assert bool(((g_bias.double() - want.sum((0, 1))).abs() <= (((32 + n ** 0.5) * eps + edge) * size_ddt).sum((0, 1))).all())
