"""The forward scan with the lanes along the states (mamba1_scan_serial.hip) at its edges: lengths around its steps of 64
positions and the checkpoints every 128, rows off 16 bytes, a last workgroup that is not full, groups, segments, absent
operands.  The sizes are those the forward rule gives it (more than one workgroup of 32 channels per compute unit, or a
sequence in segments).  Reference: the recurrence in float64, position by position."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rms of a rounding to the type is 2^-9 / sqrt(3) of the value at most (bf16), 2^-12 / sqrt(3) (fp16); fp32: some 20
# roundings of 2^-24 and exponents of up to 2^5 whose rounding the exponential hands on
REL = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 2.0 ** -19}


def _reference(t, softplus):
    u, dl, A, B, C = (t[k].double() for k in ("u", "delta", "A", "B", "C"))
    b, d, L = u.shape
    G = B.shape[1]
    if t.get("delta_bias") is not None:
        dl = dl + t["delta_bias"].double()[None, :, None]
    if softplus:
        dl = torch.nn.functional.softplus(dl)
    h = torch.zeros(b, d, A.shape[1], dtype=torch.float64, device=u.device)
    out = torch.empty_like(u)
    for i in range(L):
        Bi, Ci = (x[..., i].repeat_interleave(d // G, 1) for x in (B, C))
        h = torch.exp(dl[:, :, i, None] * A) * h + (dl[:, :, i] * u[:, :, i])[..., None] * Bi
        out[:, :, i] = (h * Ci).sum(-1)
    if t.get("D") is not None:
        out = out + t["D"].double()[None, :, None] * u
    if t.get("z") is not None:
        out = out * torch.nn.functional.silu(t["z"].double())
    return out, h


def _check(t, softplus=True):
    from mamba_amd.ops.selective_scan_interface import selective_scan_fn
    with torch.no_grad():
        out, last = selective_scan_fn(t["u"], t["delta"], t["A"], t["B"], t["C"], t.get("D"), z=t.get("z"),
                                      delta_bias=t.get("delta_bias"), delta_softplus=softplus, return_last_state=True)
    want, h = _reference(t, softplus)
    assert torch.isfinite(out).all() and torch.isfinite(last).all()
    # the worst position and channel as well as the whole: an edge that is wrong is a small share of the values
    scale = want.abs().amax(dim=(1, 2), keepdim=True)
    assert float((out.double() - want).norm() / want.norm()) < REL[t["u"].dtype]
    assert float(((out.double() - want).abs() / scale).max()) < 2 * REL[t["u"].dtype]
    assert float((last.double() - h).norm() / h.norm()) < REL[torch.float32]


def _inputs(b, d, L, G, dtype, seed, off=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=g)
    row = lambda *s: randn(*s, L + off).to(dtype)[..., off:]   # off: rows that do not start on 16 bytes
    return dict(u=row(b, d), delta=row(b, d), z=row(b, d), B=row(b, G, 16), C=row(b, G, 16),
                A=-torch.rand(d, 16, device="cuda", generator=g) * 16 - 0.1, D=randn(d), delta_bias=randn(d) - 3)


@pytest.mark.parametrize("L", [8, 9, 63, 64, 65, 72, 127, 128, 129, 192, 200, 321])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_lengths(L, dtype):
    _check(_inputs(9, 1024, L, 1, dtype, L))


@pytest.mark.parametrize("b,d,G,off", [(9, 1008, 1, 0), (6, 1860, 2, 1), (10, 1040, 1, 3), (300, 16, 1, 0), (17, 1024, 4, 5)])
def test_channels_and_rows(b, d, G, off):
    _check(_inputs(b, d, 136, G, torch.bfloat16, b + off, off))


@pytest.mark.parametrize("drop", [("z",), ("D",), ("delta_bias",), ("z", "D", "delta_bias")])
@pytest.mark.parametrize("softplus", [True, False])
def test_absent_operands(drop, softplus):
    t = _inputs(9, 1024, 150, 1, torch.bfloat16, 5)
    if not softplus:
        t["delta"], t["delta_bias"] = t["delta"].abs() * 0.1, t["delta_bias"].abs() * 0.01   # (steps are not negative)
    _check({k: v for k, v in t.items() if k not in drop}, softplus)


@pytest.mark.parametrize("b,d,L", [(2, 944, 533), (2, 2224, 1409), (1, 1520, 2100)])
def test_segments(b, d, L):
    _check(_inputs(b, d, L, 1, torch.bfloat16, d))


def test_end_of_one_sequence_stays_in_it():
    """NaN in the last position reaches no other one; infinities in a channel reach no other channel."""
    from mamba_amd.ops.selective_scan_interface import selective_scan_fn
    t = _inputs(9, 1024, 130, 1, torch.bfloat16, 3)
    t["u"][:, 5, 129] = float("nan")
    t["u"][:, 7, 64] = float("inf")
    with torch.no_grad():
        out = selective_scan_fn(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], z=t["z"], delta_bias=t["delta_bias"],
                                delta_softplus=True)
    finite = torch.isfinite(out)
    assert not finite[:, 5, 129].any() and finite[:, 5, :129].all() and finite[:, 7, :64].all()
    finite[:, 5] = finite[:, 7] = True
    assert finite.all()


def test_the_measurement_hook_reaches_the_other_kernel():
    """MAMBA_AMD_FWD_MIN_LDS is for scan_fwd_kernel, and selects it: its fp32 sums are taken in another order than this one's."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    code = ("import sys; sys.path[:0] = [%r, %r]\n"
            "import hashlib, torch, test_mamba1_serial_gpu as t\n"
            "from mamba_amd.ops.selective_scan_interface import selective_scan_fn\n"
            "i = t._inputs(7, 3184, 192, 1, torch.float32, 5)\n"
            "t._check(i)\n"
            "y = selective_scan_fn(i['u'], i['delta'], i['A'], i['B'], i['C'], i['D'], z=i['z'], delta_bias=i['delta_bias'], delta_softplus=True)\n"
            "print(hashlib.sha256(y.cpu().numpy().tobytes()).hexdigest())\n") % (here, os.path.dirname(here))
    bits = set()
    for lds in ("", "1"):
        env = dict(os.environ)
        env.pop("MAMBA_AMD_FWD_MIN_LDS", None)
        if lds:
            env["MAMBA_AMD_FWD_MIN_LDS"] = lds
        bits.add(subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, check=True, timeout=100).stdout)
    assert len(bits) == 2


# one state per lane: few channels, whole and cut into segments, more of them than are read at a time, groups, ragged rows
@pytest.mark.parametrize("b,d,L,G,off", [(1, 1526, 8, 1, 0), (1, 1526, 65, 1, 0), (2, 770, 129, 1, 1), (1, 520, 777, 4, 3),
                                         (1, 96, 4100, 1, 0), (8, 1008, 256, 1, 0), (3, 1000, 127, 2, 2), (1, 1536, 256, 1, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_few_channels(b, d, L, G, off, dtype):
    _check(_inputs(b, d, L, G, dtype, d + L, off))


def test_few_channels_stay_apart():
    """NaN in the last position reaches no other one; infinities in a channel reach no other channel."""
    from mamba_amd.ops.selective_scan_interface import selective_scan_fn
    t = _inputs(1, 1024, 130, 1, torch.bfloat16, 3)
    t["u"][:, 5, 129] = float("nan")
    t["u"][:, 7, 64] = float("inf")
    with torch.no_grad():
        out = selective_scan_fn(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], z=t["z"], delta_bias=t["delta_bias"],
                                delta_softplus=True)
    bad = ~torch.isfinite(out)
    assert bad[:, 5, 129].all() and bad[:, 7, 64:].all()
    bad[:, 5, 129] = False
    bad[:, 7, 64:] = False
    assert not bad.any()
