"""The work that is timed when the framework's speed is looked at: what a program that trains or serves Mamba layers has
it do, through its public entry points.

Every case is a dict of plain values.  `op` names the path:

  scan   selective_scan_fn                           Mamba-1 scan, forward (prefill) or forward + backward (training)
  ssd    mamba_chunk_scan_combined                   Mamba-2 chunked scan, the same, also on packed rows
  inner  mamba_inner_fn                              Mamba-1 mixer after its input projection, forward + backward
  block  mamba_split_conv1d_scan_combined            Mamba-2 mixer after its input projection, forward + backward
  norm   rms_norm_fn with an fp32 residual stream    the add + norm in front of every mixer, forward + backward
  step1  causal_conv1d_update, selective_state_update                          one token of a Mamba-1 mixer
  step2  rms_norm_fn, causal_conv1d_update, selective_state_update, rmsnorm_fn one token of a Mamba-2 block
  state  selective_state_update                      the state update alone, as a bandwidth test

`listed()` has one or two cases of each, `draw()` gives more of the same ranges.
"""
import math

import torch

from mamba_amd.ops.causal_conv1d import causal_conv1d_update
from mamba_amd.ops.selective_scan_interface import mamba_inner_fn, selective_scan_fn
from mamba_amd.ops.triton.layer_norm import rms_norm_fn
from mamba_amd.ops.triton.layernorm_gated import rmsnorm_fn
from mamba_amd.ops.triton.selective_state_update import selective_state_update
from mamba_amd.ops.triton.ssd_combined import mamba_chunk_scan_combined, mamba_split_conv1d_scan_combined

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
WIDTH = 4       # convolution taps
HEADDIM = 64


def listed():
    return [
        # one token for one user: launches and host time are all there is
        dict(name="step2_b1", op="step2", batch=1, heads=80, dstate=128, groups=1, dtype="bf16", state="bf16", pooled=False),
        # one token for a few users of a small Mamba-1 model, states in a pool of rows (continuous batching)
        dict(name="step1_b7_pooled", op="step1", batch=7, dim=1536, dstate=16, dtype="bf16", state="fp32", pooled=True),
        # one token for a full serving batch (benchmark configuration 3)
        dict(name="state_b256", op="state", batch=256, heads=80, dstate=128, groups=1, dtype="bf16", state="fp32", pooled=False),
        # prefill of one prompt, whatever its length is, and the state that decoding starts from
        dict(name="scan_prefill_b1_l777", op="scan", batch=1, dim=1536, seqlen=777, dstate=16, dtype="bf16", grad=False),
        dict(name="ssd_prefill_b1_l1531", op="ssd", batch=1, seqlen=1531, heads=80, groups=1, dstate=128, chunk=256,
             dtype="bf16", gate=True, grad=False, sequences=0),
        # training in fp32 (benchmark configuration 0's shape)
        dict(name="scan_train_fp32", op="scan", batch=2, dim=1536, seqlen=2048, dstate=16, dtype="fp32", grad=True),
        # training at full size (benchmark configuration 1: the headline)
        dict(name="scan_train_large", op="scan", batch=8, dim=5120, seqlen=4096, dstate=16, dtype="bf16", grad=True),
        # benchmark configurations 2 and 4: training at full size, and one long row of packed sequences
        dict(name="ssd_train_large", op="ssd", batch=4, seqlen=4096, heads=80, groups=1, dstate=128, chunk=256,
             dtype="bf16", gate=True, grad=True, sequences=0),
        dict(name="ssd_train_packed", op="ssd", batch=1, seqlen=32768, heads=64, groups=8, dstate=128, chunk=256,
             dtype="bf16", gate=True, grad=True, sequences=16),
        # whole mixers in training: a small Mamba-2 block with fp32 weights under autocast on ragged sequences, and the
        # benchmark's Mamba-1 mixer
        dict(name="block_train_small", op="block", batch=2, seqlen=1000, heads=24, groups=1, dstate=128, chunk=256, amp=True),
        dict(name="inner_train_large", op="inner", batch=8, seqlen=4096, dim=5120, dstate=16, amp=False),
        # the add + norm of a training step: 16384 positions of d_model 2560
        dict(name="norm_train", op="norm", rows=16384, dim=2560, dtype="bf16"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _length(rng, low, high, aligned):
    """A sequence length over the logarithm of its range: any (prompts), or a multiple of 64 (cut training text)."""
    n = _log(rng, low, high)
    return max(64, n // 64 * 64) if aligned else n


def draw(rng):
    op = rng.choice(["scan", "scan", "ssd", "ssd", "ssd", "inner", "block", "norm", "step1", "step2", "state"])
    dtype = rng.choice(["bf16"] * 5 + ["fp16", "fp32"])
    if op == "scan":
        grad = rng.random() < 0.6
        batch, dim = _log(rng, 1, 8), _log(rng, 48, 320) * 16
        most = (8 * 5120 * 4096) // (2 if dtype == "fp32" else 1) // (batch * dim)
        seqlen = min(_length(rng, 16, 8192, grad and rng.random() < 0.6), most)
        return dict(op=op, batch=batch, dim=dim, seqlen=seqlen, dstate=16, dtype=dtype, grad=grad)
    if op == "ssd":
        grad = rng.random() < 0.6
        sequences = _log(rng, 2, 16) if rng.random() < 0.3 else 0
        groups = rng.choice([1, 1, 8])
        batch, heads = 1 if sequences else _log(rng, 1, 4), _log(rng, 2, 10) * 8
        most = (32768 * 64) // {"bf16": 1, "fp16": 4, "fp32": 4}[dtype] // (batch * heads)
        seqlen = min(_length(rng, 512 if sequences else 64, 32768 if sequences else 8192, grad and rng.random() < 0.6), most)
        return dict(op=op, batch=batch, seqlen=seqlen, heads=heads, groups=groups, dstate=rng.choice([64, 128, 128]),
                    chunk=rng.choice([64, 128, 256, 256, 256]), dtype=dtype, gate=rng.random() < 0.5, grad=grad,
                    sequences=sequences)
    if op == "inner":
        dim, batch = _log(rng, 12, 80) * 64, _log(rng, 1, 8)
        return dict(op=op, batch=batch, seqlen=_length(rng, 64, 4096, rng.random() < 0.6), dim=dim, dstate=16,
                    amp=rng.random() < 0.5)
    if op == "block":
        batch = _log(rng, 1, 4)
        return dict(op=op, batch=batch, seqlen=_length(rng, 64, 4096, rng.random() < 0.6), heads=_log(rng, 2, 10) * 8,
                    groups=rng.choice([1, 1, 8]), dstate=128, chunk=256, amp=rng.random() < 0.5)
    if op == "norm":
        return dict(op=op, rows=_log(rng, 64, 32768), dim=_log(rng, 96, 640) * 8, dtype=dtype)
    batch, state, pooled = _log(rng, 1, 256), rng.choice(["fp32", dtype]), rng.random() < 0.3
    if op == "step1":
        return dict(op=op, batch=batch, dim=_log(rng, 48, 320) * 16, dstate=16, dtype=dtype, state=state, pooled=pooled)
    return dict(op=op, batch=batch, heads=_log(rng, 2, 10) * 8, dstate=128, groups=rng.choice([1, 1, 8]), dtype=dtype,
                state=state, pooled=pooled)


# ------------------------------------------------------------------------------------------------ inputs
def _maker(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    randn = lambda *s: torch.randn(*s, device="cuda", generator=g)
    rand = lambda *s: torch.rand(*s, device="cuda", generator=g)
    return g, randn, rand


def _dt_bias(rand, n):
    """softplus^-1 of step sizes spread over the logarithm of [1e-3, 1e-1], as the layers initialise it."""
    dt = torch.exp(rand(n) * math.log(100.0) + math.log(1e-3))
    return dt + torch.log(-torch.expm1(-dt))


def _leaf(*tensors):
    for t in tensors:
        t.requires_grad_()


def _prepare_scan(c, seed):
    _, randn, rand = _maker(seed)
    b, d, L, n, dtype = c["batch"], c["dim"], c["seqlen"], c["dstate"], DTYPES[c["dtype"]]
    s = dict(u=randn(b, d, L).to(dtype), delta=randn(b, d, L).to(dtype), z=randn(b, d, L).to(dtype),
             B=randn(b, 1, n, L).to(dtype), C=randn(b, 1, n, L).to(dtype),
             A=-torch.arange(1, n + 1, device="cuda", dtype=torch.float32).repeat(d, 1).contiguous(),
             D=torch.ones(d, device="cuda"), delta_bias=_dt_bias(rand, d))
    if c["grad"]:
        _leaf(*s.values())
        s["dout"] = randn(b, d, L).to(dtype)
    return s


def _run_scan(c, s):
    args = [s[k] for k in ("u", "delta", "A", "B", "C", "D", "z", "delta_bias")]
    if not c["grad"]:
        with torch.no_grad():
            return selective_scan_fn(*args, delta_softplus=True, return_last_state=True)
    out = selective_scan_fn(*args, delta_softplus=True)
    return (out, *torch.autograd.grad(out, args, s["dout"]))


def _seq_idx(lengths):
    ids = torch.repeat_interleave(torch.arange(len(lengths), dtype=torch.int32), torch.tensor(lengths))
    return ids[None].to("cuda")


def _prepare_ssd(c, seed):
    _, randn, rand = _maker(seed)
    b, L, h, g, n, dtype = c["batch"], c["seqlen"], c["heads"], c["groups"], c["dstate"], DTYPES[c["dtype"]]
    s = dict(x=randn(b, L, h, HEADDIM).to(dtype), dt=randn(b, L, h).to(dtype), A=-(1 + 15 * rand(h)),
             B=randn(b, L, g, n).to(dtype), C=randn(b, L, g, n).to(dtype), D=rand(h), dt_bias=_dt_bias(rand, h))
    if c["gate"]:
        s["z"] = randn(b, L, h, HEADDIM).to(dtype)
    if c["sequences"]:
        s["initial_states"] = 0.1 * randn(b, h, HEADDIM, n)
    if c["grad"]:
        _leaf(*s.values())
        s["dout"] = randn(b, L, h, HEADDIM).to(dtype)
    if c["sequences"]:
        part = torch.rand(c["sequences"], generator=torch.Generator().manual_seed(seed)) + 0.2
        ends = (part.cumsum(0) / part.sum() * L).long().tolist()
        ends[-1] = L
        s["seq_idx"] = _seq_idx([e - a for a, e in zip([0] + ends, ends)])
    return s


def _run_ssd(c, s):
    call = lambda: mamba_chunk_scan_combined(
        s["x"], s["dt"], s["A"], s["B"], s["C"], c["chunk"], D=s["D"], z=s.get("z"), dt_bias=s["dt_bias"],
        initial_states=s.get("initial_states"), seq_idx=s.get("seq_idx"), dt_softplus=True,
        return_final_states=not c["grad"] or bool(c["sequences"]))
    if not c["grad"]:
        with torch.no_grad():
            return call()
    r = call()
    outs = r if isinstance(r, tuple) else (r,)
    leaves = [s[k] for k in ("x", "dt", "A", "B", "C", "D", "dt_bias", "z", "initial_states") if k in s]
    return (*outs, *torch.autograd.grad(outs[0], leaves, s["dout"]))


def _prepare_inner(c, seed):
    _, randn, rand = _maker(seed)
    b, L, d, n = c["batch"], c["seqlen"], c["dim"], c["dstate"]
    rank, model, weights = math.ceil(d // 2 / 16), d // 2, torch.float32 if c["amp"] else torch.bfloat16
    s = dict(xz=randn(b, 2 * d, L).bfloat16(), conv_w=(0.3 * randn(d, 1, WIDTH)).to(weights), conv_b=(0.1 * randn(d)).to(weights),
             x_proj=(randn(rank + 2 * n, d) / math.sqrt(d)).to(weights), dt_proj=(randn(d, rank) / math.sqrt(rank)).to(weights),
             out_proj=(randn(model, d) / math.sqrt(d)).to(weights),
             A=-torch.arange(1, n + 1, device="cuda", dtype=torch.float32).repeat(d, 1).contiguous(),
             D=torch.ones(d, device="cuda"), delta_bias=_dt_bias(rand, d))
    _leaf(*s.values())
    s["dout"] = randn(b, L, model).bfloat16()
    return s


def _run_inner(c, s):
    leaves = [s[k] for k in ("xz", "conv_w", "conv_b", "x_proj", "dt_proj", "out_proj", "A", "D", "delta_bias")]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=c["amp"]):
        out = mamba_inner_fn(*leaves[:6], None, s["A"], None, None, s["D"], delta_bias=s["delta_bias"], delta_softplus=True)
    return (out, *torch.autograd.grad(out, leaves, s["dout"]))


def _prepare_block(c, seed):
    _, randn, rand = _maker(seed)
    b, L, h, g, n = c["batch"], c["seqlen"], c["heads"], c["groups"], c["dstate"]
    d, weights = h * HEADDIM, torch.float32 if c["amp"] else torch.bfloat16
    conv = d + 2 * g * n
    s = dict(zxbcdt=(0.5 * randn(b, L, d + conv + h)).bfloat16(), conv_w=(0.3 * randn(conv, WIDTH)).to(weights),
             conv_b=(0.1 * randn(conv)).to(weights), dt_bias=_dt_bias(rand, h), A=-(1 + 15 * rand(h)), D=rand(h),
             norm_w=1 + 0.1 * randn(d), out_w=(randn(d // 2, d) / math.sqrt(d)).to(weights))
    _leaf(*s.values())
    s["dout"] = randn(b, L, d // 2).bfloat16()
    return s


def _run_block(c, s):
    leaves = [s[k] for k in ("zxbcdt", "conv_w", "conv_b", "dt_bias", "A", "D", "norm_w", "out_w")]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=c["amp"]):
        out = mamba_split_conv1d_scan_combined(*leaves[:6], c["chunk"], rmsnorm_weight=s["norm_w"], outproj_weight=s["out_w"],
                                               headdim=HEADDIM, ngroups=c["groups"], norm_before_gate=False)
    return (out, *torch.autograd.grad(out, leaves, s["dout"]))


def _prepare_norm(c, seed):
    _, randn, _ = _maker(seed)
    rows, d, dtype = c["rows"], c["dim"], DTYPES[c["dtype"]]
    s = dict(x=randn(rows, d).to(dtype), weight=(1 + 0.1 * randn(d)).to(dtype), residual=randn(rows, d))
    _leaf(*s.values())
    s["dy"], s["dresidual"] = randn(rows, d).to(dtype), randn(rows, d)
    return s


def _run_norm(c, s):
    outs = rms_norm_fn(s["x"], s["weight"], None, residual=s["residual"], eps=1e-5, prenorm=True, residual_in_fp32=True)
    return (*outs, *torch.autograd.grad(outs, [s["x"], s["weight"], s["residual"]], [s["dy"], s["dresidual"]]))


def _rows_in_pool(c, g):
    """With a pool, twice as many state rows as the batch, and the row of every entry."""
    rows = 2 * c["batch"] if c["pooled"] else c["batch"]
    return rows, torch.randperm(rows, generator=g, device="cuda")[:c["batch"]].int() if c["pooled"] else None


def _prepare_step1(c, seed):
    g, randn, rand = _maker(seed)
    b, d, n, dtype = c["batch"], c["dim"], c["dstate"], DTYPES[c["dtype"]]
    rows, index = _rows_in_pool(c, g)
    return dict(x=randn(b, d).to(dtype), z=randn(b, d).to(dtype), dt=randn(b, d).to(dtype), B=randn(b, n).to(dtype),
                C=randn(b, n).to(dtype), conv_state=randn(rows, d, WIDTH).to(dtype), index=index,
                ssm_state=(0.1 * randn(rows, d, n)).to(DTYPES[c["state"]]), conv_w=(0.4 * randn(d, WIDTH)).to(dtype),
                conv_b=(0.1 * randn(d)).to(dtype), D=torch.ones(d, device="cuda"), dt_bias=_dt_bias(rand, d),
                A=-torch.arange(1, n + 1, device="cuda", dtype=torch.float32).repeat(d, 1).contiguous())


def _run_step1(c, s):
    with torch.no_grad():
        x = causal_conv1d_update(s["x"], s["conv_state"], s["conv_w"], s["conv_b"], "silu", conv_state_indices=s["index"])
        y = selective_state_update(s["ssm_state"], x, s["dt"], s["A"], s["B"], s["C"], s["D"], z=s["z"], dt_bias=s["dt_bias"],
                                   dt_softplus=True, state_batch_indices=s["index"])
    return y, s["conv_state"], s["ssm_state"]


def _prepare_step2(c, seed):
    g, randn, rand = _maker(seed)
    b, h, n, groups, dtype = c["batch"], c["heads"], c["dstate"], c["groups"], DTYPES[c["dtype"]]
    rows, index = _rows_in_pool(c, g)
    d = h * HEADDIM
    conv = d + 2 * groups * n
    per_head = dict(A=-(1 + 15 * rand(h)), D=rand(h), dt_bias=_dt_bias(rand, h))
    return dict(hidden=randn(b, d // 2).to(dtype), residual=randn(b, d // 2), block_norm_w=(1 + 0.1 * randn(d // 2)).to(dtype),
                zxbcdt=randn(b, d + conv + h).to(dtype), index=index,
                conv_state=randn(rows, WIDTH, conv).to(dtype).transpose(1, 2),   # channel-contiguous, as the layer allocates it
                ssm_state=(0.1 * randn(rows, h, HEADDIM, n)).to(DTYPES[c["state"]]), conv_w=(0.4 * randn(conv, WIDTH)).to(dtype),
                conv_b=(0.1 * randn(conv)).to(dtype), norm_w=(1 + 0.1 * randn(d)).to(dtype),
                A=per_head["A"][:, None, None].expand(h, HEADDIM, n), D=per_head["D"][:, None].expand(h, HEADDIM),
                dt_bias=per_head["dt_bias"][:, None].expand(h, HEADDIM))


def _run_step2(c, s):
    b, h, n, groups = c["batch"], c["heads"], c["dstate"], c["groups"]
    d = h * HEADDIM
    with torch.no_grad():
        # the projections between these calls are the program's own matrix products
        normed, residual = rms_norm_fn(s["hidden"], s["block_norm_w"], None, residual=s["residual"], eps=1e-5, prenorm=True,
                                       residual_in_fp32=True)
        z, xBC, dt = torch.split(s["zxbcdt"], [d, d + 2 * groups * n, h], dim=-1)
        xBC = causal_conv1d_update(xBC, s["conv_state"], s["conv_w"], s["conv_b"], "silu", conv_state_indices=s["index"])
        x, B, C = torch.split(xBC, [d, groups * n, groups * n], dim=-1)
        y = selective_state_update(s["ssm_state"], x.view(b, h, HEADDIM), dt[:, :, None].expand(b, h, HEADDIM), s["A"],
                                   B.view(b, groups, n), C.view(b, groups, n), s["D"], z=None, dt_bias=s["dt_bias"],
                                   dt_softplus=True, state_batch_indices=s["index"])
        y = rmsnorm_fn(y.view(b, d), s["norm_w"], None, z=z, eps=1e-5, group_size=d // groups, norm_before_gate=False)
    return normed, residual, y, s["conv_state"], s["ssm_state"]


def _prepare_state(c, seed):
    g, randn, rand = _maker(seed)
    b, h, n, groups, dtype = c["batch"], c["heads"], c["dstate"], c["groups"], DTYPES[c["dtype"]]
    rows, index = _rows_in_pool(c, g)
    return dict(state=(0.1 * randn(rows, h, HEADDIM, n)).to(DTYPES[c["state"]]), x=randn(b, h, HEADDIM).to(dtype),
                z=randn(b, h, HEADDIM).to(dtype), dt=randn(b, h).to(dtype)[:, :, None].expand(b, h, HEADDIM),
                A=(-(1 + 15 * rand(h)))[:, None, None].expand(h, HEADDIM, n), B=randn(b, groups, n).to(dtype),
                C=randn(b, groups, n).to(dtype), D=rand(h)[:, None].expand(h, HEADDIM), index=index,
                dt_bias=_dt_bias(rand, h)[:, None].expand(h, HEADDIM))


def _run_state(c, s):
    with torch.no_grad():
        y = selective_state_update(s["state"], s["x"], s["dt"], s["A"], s["B"], s["C"], s["D"], z=s["z"], dt_bias=s["dt_bias"],
                                   dt_softplus=True, state_batch_indices=s["index"])
    return y, s["state"]


OPS = {"scan": (_prepare_scan, _run_scan), "ssd": (_prepare_ssd, _run_ssd), "inner": (_prepare_inner, _run_inner),
       "block": (_prepare_block, _run_block), "norm": (_prepare_norm, _run_norm), "step1": (_prepare_step1, _run_step1),
       "step2": (_prepare_step2, _run_step2), "state": (_prepare_state, _run_state)}


def prepare(case, seed):
    return case, OPS[case["op"]][0](case, seed)


def run(state):
    case, tensors = state
    return OPS[case["op"]][1](case, tensors)


# ------------------------------------------------------------------------------------------------ what the work is
_SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}


def _scan_flops(elements, grad):
    """Per (position, channel, state): the exponent, exp, input term, recurrence and output forward; backward the same
    recurrence again, its adjoint, and the terms of the gradients of the step, A, B and C."""
    return elements * (7 + (19 if grad else 0))


def _ssd_flops(b, L, h, g, n, chunk, grad):
    """The chunked form's products with the causal halves counted once; each product has two gradients."""
    q = min(chunk, L)
    return b * L * (h * (q * HEADDIM + 4 * n * HEADDIM) + g * q * n) * (3 if grad else 1)


def work(case):
    c = case
    op, e = c["op"], _SIZE[c.get("dtype", "bf16")]
    if op == "scan":
        b, d, L, n = c["batch"], c["dim"], c["seqlen"], c["dstate"]
        x, bc, per_channel = b * d * L, b * n * L, d * (n + 2)
        if c["grad"]:   # u, delta, z, dout, out, du, ddelta, dz; B, C, dB, dC; parameters and their gradients
            return {"bytes": e * (8 * x + 4 * bc) + 8 * per_channel, "flops": _scan_flops(x * n, True)}
        return {"bytes": e * (4 * x + 2 * bc) + 4 * (per_channel + b * d * n), "flops": _scan_flops(x * n, False)}
    if op == "ssd":
        b, L, h, g, n = c["batch"], c["seqlen"], c["heads"], c["groups"], c["dstate"]
        x, bc, steps, states = b * L * h * HEADDIM, b * L * g * n, b * L * h, b * h * HEADDIM * n
        flops = _ssd_flops(b, L, h, g, n, c["chunk"], c["grad"])
        tensors = 2 + int(c["gate"])
        if c["grad"]:
            more = 3 * states * 4 if c["sequences"] else 0   # initial and final states, gradient of the initial ones
            return {"bytes": e * ((2 * tensors) * x + 4 * bc + 2 * steps) + more + 24 * h, "flops": flops}
        return {"bytes": e * (tensors * x + 2 * bc + steps) + 4 * states * (2 if c["sequences"] else 1) + 12 * h, "flops": flops}
    if op == "inner":
        b, L, d, n = c["batch"], c["seqlen"], c["dim"], c["dstate"]
        rank, model, w = math.ceil(d // 2 / 16), d // 2, 4 if c["amp"] else 2
        weights = d * (WIDTH + 1) + (rank + 2 * n) * d + d * rank + model * d
        products = 2 * b * L * ((rank + 2 * n) * d + d * rank + model * d)
        return {"bytes": 2 * b * L * (2 * 2 * d + 2 * model) + 2 * w * weights + 8 * d * (n + 2),
                "flops": 3 * products + _scan_flops(b * L * d * n, True)}
    if op == "block":
        b, L, h, g, n = c["batch"], c["seqlen"], c["heads"], c["groups"], c["dstate"]
        d, w = h * HEADDIM, 4 if c["amp"] else 2
        conv = d + 2 * g * n
        weights = conv * (WIDTH + 1) + d // 2 * d
        return {"bytes": 2 * b * L * (2 * (d + conv + h) + 2 * (d // 2)) + 2 * w * weights + 8 * (3 * h + d),
                "flops": 3 * 2 * b * L * d * (d // 2) + _ssd_flops(b, L, h, g, n, c["chunk"], True)}
    if op == "norm":
        x = c["rows"] * c["dim"]   # x, dy, y, dx; residual, dresidual, their sum and its gradient
        return {"bytes": x * (4 * e + 4 * 4) + 2 * e * c["dim"], "flops": 15 * x}
    b, n, es = c["batch"], c["dstate"], _SIZE[c["state"]]
    if op == "step1":
        d = c["dim"]
        return {"bytes": b * d * (2 * n * es + 2 * WIDTH * e + 4 * e) + 2 * b * n * e + d * (e * (WIDTH + 1) + 4 * (n + 2)),
                "flops": b * d * (7 * n + 2 * WIDTH + 10)}
    h, g = c["heads"], c["groups"]
    d, ssm = h * HEADDIM, b * h * HEADDIM * n
    if op == "state":
        return {"bytes": 2 * ssm * es + e * b * (3 * d + 2 * g * n + h) + 12 * h, "flops": 7 * ssm}
    conv = d + 2 * g * n
    return {"bytes": 2 * ssm * es + e * b * (2 * WIDTH * conv + d + conv + h + d + 2 * (d // 2)) + 8 * b * (d // 2)
            + e * (conv * (WIDTH + 1) + d + d // 2) + 12 * h,
            "flops": 7 * ssm + 2 * WIDTH * b * conv + 20 * b * d}


def tolerance(case):
    """Set by the least precise type that results pass through."""
    types = {case.get("dtype", "bf16"), case.get("state", "fp32")}
    if "bf16" in types:
        return {"rel": 1e-2}
    return {"rel": 2e-3} if "fp16" in types else {"rel": 3e-5}
