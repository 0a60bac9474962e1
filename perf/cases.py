"""What a user of this framework has it do, as cases to be timed: training, prefill and decode through the public
entry points, with and without the precision state, bare and inside the layers' glue.

Shapes are those of the repository's benchmark configurations (c0 .. c4) and of the layer configurations that its tests
and notes name (16 heads of 48 x 48, 48 x 96, 96 x 192), and generic ones of the same kind in `draw`.  A case is one
pass of one `path`:

* ``train``     chunk_palimpsa forward + backward: outputs and every gradient
* ``prefill``   chunk_palimpsa forward without autograd, final state handed to the decode that follows
* ``prompt``    fused_recurrent_palimpsa over a short prompt, final state returned
* ``decode``    fused_recurrent_palimpsa, one token per sequence, state in and state out (a generation loop)
* ``step``      DecodeStep.step(), the bound decode of a server: state updated in place
* ``layer``     Palimpsa layer between projections and output projection: glue, operator, glue; forward + backward
* ``mamba``     the same for the MetaMamba2 layer
* ``gla``       chunk_simple_gla forward + backward (layers with the precision state off)
* ``gla_decode``  fused_recurrent_simple_gla, one token per sequence, state in and state out
"""
import math

import numpy as np
import torch

from palimpsa_amd.ops.layer_glue import (metamamba2_inputs, metamamba2_output_norm, palimpsa_inputs,
                                         palimpsa_output_norm)
from palimpsa_amd.ops.palimpsa import DecodeStep, chunk_palimpsa, fused_recurrent_palimpsa
from palimpsa_amd.ops.simple_gla import chunk_simple_gla, fused_recurrent_simple_gla

TRAINING = ("train", "layer", "mamba", "gla")

# no drawn case does more than the largest listed one (the packed training batch and the long prefill are equals)
MOST_FLOPS = 1.69e11


def case(name, path, B, T, H, dk, dv, Hq=None, dtype="bf16", gates="fp32", init=False, var=False, docs=0):
    """``Hq`` heads of q, k; ``docs`` > 0: one packed row of documents of that length in the mean; ``init``: an initial
    state is passed in; ``var``: the uncertainty output is asked for (and used by the loss)."""
    c = dict(path=path, B=B, T=T, H=H, Hq=Hq or H, dk=dk, dv=dv, dtype=dtype, gates=gates, init=init, var=var, docs=docs)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one conversation, token by token, on the 170M configuration: the call is all latency
        case("decode_one", "decode", 1, 1, 16, 48, 48, init=True),
        # a serving batch with bound tensors (c3): memory bandwidth
        case("step_b256", "step", 256, 1, 16, 128, 128, init=True),
        # a short fp32 evaluation through the token-serial entry point (c0)
        case("prompt_fp32", "prompt", 2, 256, 4, 32, 32, dtype="fp32"),
        # the next turn of a conversation: an odd number of tokens on top of a kept state
        case("prefill_turn", "prefill", 1, 777, 16, 48, 48, init=True),
        # a long document (c4)
        case("prefill_long", "prefill", 1, 65536, 16, 128, 128, init=True),
        # training batch of the headline metric (c1)
        case("train_c1", "train", 8, 2048, 12, 64, 64, gates="bf16"),
        # packed ragged training batch (c2)
        case("train_packed", "train", 1, 32768, 16, 96, 96, docs=1024),
        # fp32 training with every option on, the topology of the reference's own check
        case("train_fp32", "train", 2, 512, 4, 32, 32, dtype="fp32", init=True, var=True),
        # a layer of the 170M Palimpsa configuration in training
        case("layer_170m", "layer", 8, 2048, 16, 48, 48),
        # a layer of the 170M MetaMamba2 configuration, B and C shared by pairs of heads, on a ragged length
        case("mamba_170m", "mamba", 4, 1531, 16, 48, 96, Hq=8),
        # the 760M configuration without the precision state in training
        case("gla_760m", "gla", 8, 2048, 16, 96, 192),
        # and its decode on a small serving batch
        case("gla_decode", "gla_decode", 32, 1, 16, 96, 192, init=True),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    square = [(32, 32), (48, 48), (64, 64), (80, 80), (96, 96)]
    while True:
        path = rng.choice(["train", "train", "prefill", "prefill", "prompt", "decode", "step", "layer", "mamba", "gla",
                           "gla_decode"])
        H = rng.choice([2, 3, 4, 6, 8, 12, 16, 24])
        dtype = "fp32" if path in ("train", "prefill", "prompt", "decode") and rng.random() < 0.25 else "bf16"
        wide = [(128, 128), (128, 64), (96, 192)] if dtype == "bf16" else [(128, 64)]
        dk, dv = rng.choice(square + [(48, 96), (65, 31)] + wide)
        gates = "bf16" if path in ("train", "prefill", "prompt") and rng.random() < 0.25 else "fp32"
        Hq, init, var, docs, T = H, False, False, 0, 1
        if path in TRAINING or path == "prefill":
            T = _between(rng, 65, 8192 if path == "gla" else 32768)
            B = _between(rng, 1, 16)
            if path in ("train", "prefill"):
                init, var = rng.random() < 0.4, rng.random() < 0.2
            if path in ("train", "gla", "prefill") and rng.random() < 0.3 and T > 512:
                B, docs = 1, _between(rng, 64, 2048)
        elif path == "prompt":
            B, T, init = _between(rng, 1, 16), _between(rng, 2, 512), rng.random() < 0.5
        else:
            B, init = _between(rng, 1, 256), True
        if path in ("layer", "mamba", "step", "gla", "gla_decode"):
            dk, dv = rng.choice([(48, 48), (48, 96), (64, 64), (96, 96), (96, 192), (128, 128)])
        if path in ("train", "layer", "mamba", "gla") and H % 2 == 0 and rng.random() < 0.25:
            Hq = H // 2
        if path == "mamba" and H * dv > 4096:
            continue
        c = case(None, path, B, T, H, dk, dv, Hq, dtype, gates, init, var, docs)
        w = work(c)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= 4e9:
            return c


def _documents(T, mean):
    """cu_seqlens of a packed row: lognormal document lengths (sigma 1) clipped to [16, 4 mean]."""
    rng, cu = np.random.RandomState(T + mean), [0]
    while cu[-1] < T:
        n = int(np.clip(rng.lognormal(math.log(mean) - 0.5, 1.0), 16, 4 * mean))
        cu.append(min(T, cu[-1] + n))
    return cu


def _rows_dtype(c):
    return torch.float32 if c["dtype"] == "fp32" else torch.bfloat16


class _Random:
    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32):
        return torch.randn(*shape, generator=self.gen, device=self.dev).to(dtype)

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=self.gen, device=self.dev)


def prepare(c, seed):
    r = _Random(seed)
    B, T, H, Hq, dk, dv, path = (c[n] for n in ("B", "T", "H", "Hq", "dk", "dv", "path"))
    dt = _rows_dtype(c)
    s = {"path": path, "var": c["var"], "cu": None, "mu": None, "I": None}
    N = B
    if c["docs"]:
        cu = _documents(T, c["docs"])
        N = len(cu) - 1
        s["cu"] = torch.tensor(cu, dtype=torch.int32, device=r.dev)
    if path == "layer":
        leaves = dict(q_raw=r.normal(B, T, Hq, dk, dtype=dt), k_raw=r.normal(B, T, Hq, dk, dtype=dt),
                      x=r.normal(B, T, H, dv, dtype=dt), dt_raw=(r.normal(B, T, H) - 1.0).to(dt), dt_bias=r.normal(H),
                      bs_raw=r.normal(B, T, H, dtype=dt), b_raw=r.normal(B, T, H, dv, dtype=dt),
                      b_scale=r.uniform(0.5, 1.5, H))
        more = dict(gate=r.normal(B, T, H, dv, dtype=dt), weight=r.uniform(0.5, 1.5, dv), D=r.uniform(0.5, 1.5, H),
                    A=r.uniform(0.1, 2.0, H))
    elif path == "mamba":
        leaves = dict(C=0.5 * r.normal(B, T, Hq, dk, dtype=dt), Bm=0.5 * r.normal(B, T, Hq, dk, dtype=dt),
                      x=r.normal(B, T, H, dv, dtype=dt), dt_raw=(r.normal(B, T, H) - 1.0).to(dt), dt_bias=r.normal(H),
                      b_raw=r.normal(B, T, H, dv, dtype=dt), b_scale=r.uniform(0.5, 1.5, H))
        more = dict(gate=r.normal(B, T, H * dv, dtype=dt), weight=r.uniform(0.5, 1.5, H * dv), D=r.uniform(0.5, 1.5, H),
                    A_log=r.uniform(-1.0, 1.5, H))
    else:
        # unit q and k rows, positive b, gates in (0, 1) and one decay rate per head, as the layers hand them over
        unit = lambda: torch.nn.functional.normalize(r.normal(B, T, Hq, dk), dim=-1).to(dt)  # noqa: E731
        leaves = dict(q=unit(), k=unit(), v=r.normal(B, T, H, dv, dtype=dt))
        gt = torch.sigmoid(r.normal(B, T, H)).to(torch.bfloat16 if c["gates"] == "bf16" else torch.float32)
        rate = r.uniform(0.05, 2.0, H)
        if path in ("gla", "gla_decode"):
            leaves["g"] = -gt * rate
            if c["init"]:
                s["S"] = 0.1 * r.normal(N, H, dk, dv)
        else:
            leaves.update(b=torch.sigmoid(r.normal(B, T, H, dv)).to(dt), gt=gt, g=rate, Ip=r.uniform(0.5, 1.5, H))
            if c["init"]:
                s["mu"] = 0.1 * r.normal(N, H, dv, dk)
                s["I"] = leaves["Ip"].view(1, H, 1, 1) + torch.nn.functional.softplus(r.normal(N, H, dv, dk))
        more = {}
    s["leaves"], s["more"] = leaves, more
    if path in TRAINING:
        for x in list(leaves.values()) + list(more.values()):
            x.requires_grad_(True)
        # the gradient of a regression: partly along the values that the outputs are made of
        along = leaves["x" if path in ("layer", "mamba") else "v"].detach().float()
        s["do"] = [(0.7 * along + 0.7 * r.normal(B, T, H, dv)).to(dt)]
        if c["var"]:
            s["do"].append(r.uniform(0.0, 0.2, B, T, H, dv).to(dt))
        if path in ("layer", "mamba"):
            s["Ip"] = torch.ones(H, device=r.dev)
        for n in ("mu", "I"):
            if s[n] is not None:
                s[n].requires_grad_(True)
    if path == "step":
        s["step"] = DecodeStep(B, H, dk, dv, r.dev, dt, tokens=T)
        s["step"].bind(*[leaves[n] for n in ("q", "k", "v", "b", "gt", "g", "Ip")], s["mu"], s["I"])
    return s


def run(s):
    path, x, m = s["path"], s["leaves"], s["more"]
    if path == "step":
        return s["step"].step(), s["mu"], s["I"]
    if path == "decode" or path == "prompt":
        with torch.no_grad():
            return fused_recurrent_palimpsa(**x, initial_mu_state=s["mu"], initial_I_state=s["I"], output_final_state=True)
    if path == "prefill":
        with torch.no_grad():
            return chunk_palimpsa(**x, initial_mu_state=s["mu"], initial_I_state=s["I"], chunk_size=64,
                                  output_final_state=True, output_uncertainty=s["var"], cu_seqlens=s["cu"])
    if path == "gla_decode":
        with torch.no_grad():
            return fused_recurrent_simple_gla(**x, initial_state=s["S"], output_final_state=True)
    wanted = list(x.values()) + list(m.values())
    if path == "train":
        out = chunk_palimpsa(**x, initial_mu_state=s["mu"], initial_I_state=s["I"], chunk_size=64,
                             output_uncertainty=s["var"], cu_seqlens=s["cu"])
        out = list(out) if s["var"] else [out]
        wanted += [s[n] for n in ("mu", "I") if s[n] is not None]
    elif path == "gla":
        out = [chunk_simple_gla(**x, cu_seqlens=s["cu"])[0]]
    elif path == "layer":
        q, k, v, b, gt = palimpsa_inputs(**x)
        o = chunk_palimpsa(q, k, v, b, gt, m["A"], s["Ip"], chunk_size=64)
        out = [palimpsa_output_norm(o, x["x"], m["D"], m["gate"], m["weight"], 1e-6)]
    else:
        v, b, dt = metamamba2_inputs(x["x"], x["dt_raw"], x["dt_bias"], x["b_raw"], x["b_scale"])
        o = chunk_palimpsa(x["C"], x["Bm"], v, b, dt, m["A_log"].exp(), s["Ip"], scale=1.0, chunk_size=64)
        out = [metamamba2_output_norm(o, x["x"], m["D"], m["gate"], m["weight"], 1e-5)]
    grads = torch.autograd.grad(out, wanted, s["do"])
    return [o.detach() for o in out] + list(grads)


def work(c):
    """Each tensor of the call read or written once.  Operations: those of the recurrence itself, per token, head and
    state entry.  With the precision state, forward: decay and update of both states (6), the division, product with q
    and sum (4): 10; forward and backward 35.  Without it 5 and 15."""
    B, T, H, Hq, dk, dv, path = (c[n] for n in ("B", "T", "H", "Hq", "dk", "dv", "path"))
    e = 4 if c["dtype"] == "fp32" else 2
    train, gla = path in TRAINING, path in ("gla", "gla_decode")
    tokens = B * T
    N = len(_documents(T, c["docs"])) - 1 if c["docs"] else B
    value_rows = 1 if gla else 2                                   # v, and b
    qk, v = tokens * Hq * dk * e, tokens * H * dv * e
    gate = tokens * H * (2 if c["gates"] == "bf16" else 4)
    out = v * (2 if c["var"] else 1)
    state = N * H * dk * dv * 4 * (1 if gla else 2)
    total = 2 * qk + value_rows * v + gate + out
    if train:                                                      # gradient of the outputs in, of the inputs out
        total += out + 2 * qk + value_rows * v + gate
        total += 2 * state if c["init"] else 0
        if path in ("layer", "mamba"):                             # gate rows and their gradient
            total += 2 * v
    else:
        total += state * (2 if c["init"] else 1)
    per_entry = {(False, False): 10, (False, True): 35, (True, False): 5, (True, True): 15}[gla, train]
    return {"bytes": total, "flops": per_entry * tokens * H * dk * dv}


def tolerance(c):
    """bf16 rows: products and results rounded to 8 bits, sums in fp32.  fp32 rows: the token-serial kernels compute in
    fp32, the chunked ones promise 1e-4 of the fp32 recurrence."""
    if c["dtype"] == "fp32":
        return {"rel": 1e-4 if c["path"] in ("train", "prefill") else 1e-5}
    if c["path"] == "gla":       # the gate's gradient is a suffix sum over the sequence of differences of rounded products
        return {"rel": 3e-2}
    if c["path"] in TRAINING:    # single entries of the gates' gradients are sums over a row that cancel
        return {"rel": 1.5e-2, "max": 0.9}
    return {"rel": 1e-2}
