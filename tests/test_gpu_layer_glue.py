"""pal_prologue_* / pal_epilogue_* (the layer's element-wise work either side of the operator) against the
CPU restatement of the reference lines (oracle/layer_glue_oracle.py), forward and backward.

Bars: fp32 rows max relative error <= 1e-4 (measured against the largest reference entry); bf16 rows <= 2e-2
absolute on the outputs (all O(1)) and <= 5e-2 on gradients normalised by the largest reference entry.
"""
import pytest
import torch

from oracle import layer_glue_oracle as lo
from tests import helpers as hp

pytestmark = pytest.mark.gpu


def _inputs(lead, Hqk, H, dk, dv, seed, dtype):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)
    a = dict(q_raw=r(*lead, Hqk, dk), k_raw=r(*lead, Hqk, dk), x=r(*lead, H, dv), dt_raw=r(*lead, H) - 2.0,
             dt_bias=r(H), bs_raw=r(*lead, H), b_raw=r(*lead, H, dv), b_scale=r(H) + 1.0)
    for n in ("q_raw", "k_raw", "x", "dt_raw", "bs_raw", "b_raw"):
        a[n] = a[n].to(dtype)
    return a


NAMES = ("q_raw", "k_raw", "x", "dt_raw", "dt_bias", "bs_raw", "b_raw", "b_scale")
SHAPES = [
    ((2, 70), 4, 4, 64, 64, torch.bfloat16),
    ((1, 33), 2, 6, 48, 48, torch.bfloat16),     # repeated q/k heads, 6 lanes of an 8-lane group
    ((3, 17), 3, 3, 96, 192, torch.bfloat16),
    ((5,), 1, 2, 8, 256, torch.bfloat16),
    ((2, 40), 2, 4, 32, 64, torch.float32),
]


@pytest.mark.parametrize("lead,Hqk,H,dk,dv,dtype", SHAPES)
@pytest.mark.parametrize("with_b", [True, False])
def test_prologue_forward_backward(gpu_device, lead, Hqk, H, dk, dv, dtype, with_b):
    from palimpsa_amd.ops.layer_glue import palimpsa_inputs
    a = _inputs(lead, Hqk, H, dk, dv, 0, dtype)
    if not with_b:
        a["b_raw"] = a["b_scale"] = None
    dev = gpu_device
    leaves = {n: (None if a[n] is None else a[n].to(dev).clone().requires_grad_(True)) for n in NAMES}
    outs = palimpsa_inputs(**leaves)
    ref_leaves = {n: (None if a[n] is None else a[n].double().clone().requires_grad_(True)) for n in NAMES}
    refs = lo.prologue(**ref_leaves, model_dtype=dtype)
    out_tol, grad_tol = (hp.BF16_OUT_ABS_TOL, hp.BF16_GRAD_NORM_TOL) if dtype == torch.bfloat16 else (1e-4, 1e-4)
    gen = torch.Generator().manual_seed(1)
    loss = 0.0
    loss_ref = 0.0
    for name, y, r in zip(("q", "k", "v", "b", "gt"), outs, refs):
        if r is None:
            assert y is None
            continue
        assert y.shape == r.shape, name
        assert y.dtype == (torch.float32 if name == "gt" else dtype)
        assert hp.max_abs(y.float(), r) <= out_tol * max(1.0, r.abs().max().item()), name
        wgt = torch.randn(r.shape, generator=gen).to(y.dtype)
        loss = loss + (y.float() * wgt.to(dev).float()).sum()
        loss_ref = loss_ref + (r * wgt.double()).sum()
    loss.backward()
    loss_ref.backward()
    for n in NAMES:
        if a[n] is None:
            continue
        g, r = leaves[n].grad, ref_leaves[n].grad
        assert g.shape == r.shape and g.dtype == leaves[n].dtype, n
        err = hp.max_rel(g, r)
        assert err <= grad_tol, (n, err)


def test_prologue_zero_rows_and_reproducibility(gpu_device):
    from palimpsa_amd.ops.layer_glue import palimpsa_inputs
    a = _inputs((4, 300), 2, 4, 64, 64, 2, torch.bfloat16)
    a["q_raw"][0, 5] = 0     # a zero row: the norm is clamped, the output row is zero, gradients stay finite
    dev = gpu_device

    def run():
        leaves = {n: a[n].to(dev).clone().requires_grad_(True) for n in NAMES}
        outs = palimpsa_inputs(**leaves)
        sum((y.float() ** 2).sum() for y in outs).backward()
        return outs, [leaves[n].grad for n in NAMES]

    o1, g1 = run()
    o2, g2 = run()
    assert (o1[0][0, 5] == 0).all()
    for x in list(o1) + g1:
        assert torch.isfinite(x.float()).all()
    for x, y in zip(list(o1) + g1, list(o2) + g2):
        assert torch.equal(x, y)       # per-head sums are taken in a fixed order


@pytest.mark.parametrize("lead,H,dv,dtype", [
    ((2, 70), 4, 64, torch.bfloat16),
    ((1, 33), 6, 48, torch.bfloat16),
    ((3, 17), 3, 192, torch.bfloat16),
    ((5,), 2, 256, torch.bfloat16),
    ((2, 40), 4, 64, torch.float32),
])
@pytest.mark.parametrize("residual,gated", [(True, True), (False, True), (True, False), (False, False)])
def test_epilogue_forward_backward(gpu_device, lead, H, dv, dtype, residual, gated):
    from palimpsa_amd.ops.layer_glue import palimpsa_output_norm
    gen = torch.Generator().manual_seed(3)
    o = torch.randn(*lead, H, dv, generator=gen).to(dtype)
    x = torch.randn(*lead, H, dv, generator=gen).to(dtype) if residual else None
    D = torch.randn(H, generator=gen) if residual else None
    gate = torch.randn(*lead, H, dv, generator=gen).to(dtype) if gated else None
    w = 1.0 + 0.2 * torch.randn(dv, generator=gen)
    dy = torch.randn(*lead, H, dv, generator=gen).to(dtype)
    eps = 1e-6
    dev = gpu_device
    ts = [o, x, D, gate, w]
    leaves = [None if t is None else t.to(dev).clone().requires_grad_(True) for t in ts]
    y = palimpsa_output_norm(leaves[0], leaves[1], leaves[2], leaves[3], leaves[4], eps)
    y.backward(dy.to(dev))
    refs = [None if t is None else t.double().clone().requires_grad_(True) for t in ts]
    y_ref = lo.epilogue(refs[0], refs[1], refs[2], refs[3], refs[4], eps)
    y_ref.backward(dy.double())
    out_tol, grad_tol = (hp.BF16_OUT_ABS_TOL, hp.BF16_GRAD_NORM_TOL) if dtype == torch.bfloat16 else (1e-4, 1e-4)
    assert y.dtype == dtype and y.shape == y_ref.shape
    assert hp.max_abs(y.float(), y_ref) <= out_tol * max(1.0, y_ref.abs().max().item())
    for name, t, r in zip(("o", "x", "D", "gate", "weight"), leaves, refs):
        if t is None:
            continue
        assert t.grad.shape == r.grad.shape and t.grad.dtype == t.dtype, name
        err = hp.max_rel(t.grad, r.grad)
        assert err <= grad_tol, (name, err)


def test_layer_slice_end_to_end(gpu_device):
    """Projections' outputs -> prologue -> chunk_palimpsa -> epilogue, with autograd through all three, against the
    same chain built from the oracles (the operator one in float64)."""
    from oracle import palimpsa_oracle as po
    from palimpsa_amd.ops.layer_glue import palimpsa_inputs, palimpsa_output_norm
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    B, T, H, d = 1, 96, 2, 32
    a = _inputs((B, T), H, H, d, d, 4, torch.bfloat16)
    gen = torch.Generator().manual_seed(5)
    gate = torch.randn(B, T, H, d, generator=gen).bfloat16()
    w = 1.0 + 0.1 * torch.randn(d, generator=gen)
    Dp = torch.randn(H, generator=gen)
    A = torch.rand(H, generator=gen) * 4 + 0.5
    Ip = torch.ones(H)
    dy = torch.randn(B, T, H, d, generator=gen).bfloat16()
    dev = gpu_device
    leaves = {n: a[n].to(dev).clone().requires_grad_(True) for n in NAMES}
    q, k, v, b, gt = palimpsa_inputs(**leaves)
    o = chunk_palimpsa(q, k, v, b, gt, A.to(dev), Ip.to(dev), chunk_size=64)
    y = palimpsa_output_norm(o, leaves["x"], Dp.to(dev), gate.to(dev), w.to(dev), 1e-6)
    y.backward(dy.to(dev))

    refl = {n: a[n].double().clone().requires_grad_(True) for n in NAMES}
    q_r, k_r, v_r, b_r, gt_r = lo.prologue(**refl, model_dtype=torch.bfloat16)
    o_r, _, _, _ = po.palimpsa_recurrence(q_r, k_r, v_r, b_r, gt_r, A.double(), Ip.double(), scale=d ** -0.5,
                                          compute_dtype=torch.float64)
    y_r = lo.epilogue(o_r, refl["x"], Dp, gate, w, 1e-6)
    y_r.backward(dy.double())
    assert hp.max_abs(y.float(), y_r) <= 2 * hp.BF16_OUT_ABS_TOL * max(1.0, y_r.abs().max().item())
    for n in NAMES:
        err = hp.max_rel(leaves[n].grad, refl[n].grad)
        assert err <= 2 * hp.BF16_GRAD_NORM_TOL, (n, err)


def test_random_shape_sweep(gpu_device):
    """Seeded random shapes of both glue kernels (head dims any multiple of 8 up to 256, odd token counts, repeated
    q/k heads), forward and backward against the oracle."""
    import random
    from palimpsa_amd.ops.layer_glue import palimpsa_inputs, palimpsa_output_norm
    rng = random.Random(4321)
    dev = gpu_device
    for case in range(12):
        Hqk = rng.choice([1, 2, 3])
        H = Hqk * rng.choice([1, 2, 4])
        dk, dv = 8 * rng.randint(1, 32), 8 * rng.randint(1, 32)
        lead = (rng.randint(1, 3), rng.randint(1, 90))
        dtype = rng.choice([torch.bfloat16, torch.bfloat16, torch.float32])
        a = _inputs(lead, Hqk, H, dk, dv, 3000 + case, dtype)
        leaves = {n: a[n].to(dev).clone().requires_grad_(True) for n in NAMES}
        outs = palimpsa_inputs(**leaves)
        refl = {n: a[n].double().clone().requires_grad_(True) for n in NAMES}
        refs = lo.prologue(**refl, model_dtype=dtype)
        gen = torch.Generator().manual_seed(4000 + case)
        loss = loss_ref = 0.0
        out_tol, grad_tol = (hp.BF16_OUT_ABS_TOL, hp.BF16_GRAD_NORM_TOL) if dtype == torch.bfloat16 else (1e-4, 1e-4)
        tag = (case, lead, Hqk, H, dk, dv, dtype)
        for y, r in zip(outs, refs):
            assert hp.max_abs(y.float(), r) <= out_tol * max(1.0, r.abs().max().item()), tag
            wgt = torch.randn(r.shape, generator=gen).to(y.dtype)
            loss = loss + (y.float() * wgt.to(dev).float()).sum()
            loss_ref = loss_ref + (r * wgt.double()).sum()
        loss.backward()
        loss_ref.backward()
        for n in NAMES:
            assert hp.max_rel(leaves[n].grad, refl[n].grad) <= grad_tol, (n,) + tag
        # epilogue on the same shape
        o = torch.randn(*lead, H, dv, generator=gen).to(dtype)
        gate = torch.randn(*lead, H, dv, generator=gen).to(dtype)
        Dp, w = torch.randn(H, generator=gen), 1.0 + 0.2 * torch.randn(dv, generator=gen)
        dy = torch.randn(*lead, H, dv, generator=gen).to(dtype)
        ts = [o, a["x"], Dp, gate, w]
        lv = [t.to(dev).clone().requires_grad_(True) for t in ts]
        palimpsa_output_norm(*lv, 1e-5).backward(dy.to(dev))
        rv = [t.double().clone().requires_grad_(True) for t in ts]
        lo.epilogue(*rv, 1e-5).backward(dy.double())
        for name, t, r in zip(("o", "x", "D", "gate", "weight"), lv, rv):
            assert hp.max_rel(t.grad, r.grad) <= grad_tol, (name,) + tag


def test_full_size_headline_shape(gpu_device):
    """Both glue kernels at the headline shape (B=8, T=2048, H=12, d=64, bf16), forward and backward against the
    oracle; the per-head and per-column sums of the backward run over 16384 tokens per head."""
    from palimpsa_amd.ops.layer_glue import palimpsa_inputs, palimpsa_output_norm
    lead, H, d = (8, 2048), 12, 64
    a = _inputs(lead, H, H, d, d, 7, torch.bfloat16)
    dev = gpu_device
    leaves = {n: a[n].to(dev).clone().requires_grad_(True) for n in NAMES}
    outs = palimpsa_inputs(**leaves)
    refl = {n: a[n].double().clone().requires_grad_(True) for n in NAMES}
    refs = lo.prologue(**refl, model_dtype=torch.bfloat16)
    gen = torch.Generator().manual_seed(8)
    loss = loss_ref = 0.0
    for y, r in zip(outs, refs):
        assert hp.max_abs(y.float(), r) <= hp.BF16_OUT_ABS_TOL * max(1.0, r.abs().max().item())
        wgt = torch.randn(r.shape, generator=gen).to(y.dtype)
        loss = loss + (y.float() * wgt.to(dev).float()).sum()
        loss_ref = loss_ref + (r * wgt.double()).sum()
    loss.backward()
    loss_ref.backward()
    for n in NAMES:
        assert hp.max_rel(leaves[n].grad, refl[n].grad) <= hp.BF16_GRAD_NORM_TOL, n
    o = torch.randn(*lead, H, d, generator=gen).bfloat16()
    gate = torch.randn(*lead, H, d, generator=gen).bfloat16()
    Dp, w = torch.randn(H, generator=gen), 1.0 + 0.2 * torch.randn(d, generator=gen)
    dy = torch.randn(*lead, H, d, generator=gen).bfloat16()
    ts = [o, a["x"], Dp, gate, w]
    lv = [t.to(dev).clone().requires_grad_(True) for t in ts]
    y = palimpsa_output_norm(*lv, 1e-6)
    y.backward(dy.to(dev))
    rv = [t.double().clone().requires_grad_(True) for t in ts]
    y_ref = lo.epilogue(*rv, 1e-6)
    y_ref.backward(dy.double())
    assert hp.max_abs(y.float(), y_ref.detach()) <= hp.BF16_OUT_ABS_TOL * max(1.0, y_ref.abs().max().item())
    for name, t, r in zip(("o", "x", "D", "gate", "weight"), lv, rv):
        assert hp.max_rel(t.grad, r.grad) <= hp.BF16_GRAD_NORM_TOL, name


# ------------------------------------------------------------------ the MetaMamba2 layer's form of the same kernels
MAMBA_SHAPES = [
    ((2, 70), 12, 64, torch.bfloat16),      # 768 entries per token: two passes of the wave, the second half full
    ((1, 33), 6, 48, torch.bfloat16),       # 288 entries: one partial pass
    ((3, 17), 16, 192, torch.bfloat16),     # 3072 entries
    ((5,), 2, 256, torch.bfloat16),
    ((2, 40), 4, 64, torch.float32),
    ((2, 300), 16, 96, torch.bfloat16),     # more tokens than one workgroup takes
    ((2, 21), 16, 128, torch.bfloat16),     # 2048 entries: the longest token the backward keeps in registers
]


@pytest.mark.parametrize("lead,H,dv,dtype", MAMBA_SHAPES)
@pytest.mark.parametrize("with_b,limit", [(True, (0.0, float("inf"))), (True, (0.05, 0.4)), (False, (0.05, 0.4))])
def test_mamba_prologue_forward_backward(gpu_device, lead, H, dv, dtype, with_b, limit):
    from palimpsa_amd.ops.layer_glue import metamamba2_inputs
    a = _inputs(lead, 1, H, 8, dv, 10, dtype)
    names = ("x", "dt_raw", "dt_bias", "b_raw", "b_scale")
    if not with_b:
        a["b_raw"] = a["b_scale"] = None
    dev = gpu_device
    leaves = {n: (None if a[n] is None else a[n].to(dev).clone().requires_grad_(True)) for n in names}
    outs = metamamba2_inputs(**leaves, dt_limit=limit)
    ref_leaves = {n: (None if a[n] is None else a[n].double().clone().requires_grad_(True)) for n in names}
    refs = lo.mamba_prologue(**ref_leaves, dt_limit=limit)
    out_tol, grad_tol = (hp.BF16_OUT_ABS_TOL, hp.BF16_GRAD_NORM_TOL) if dtype == torch.bfloat16 else (1e-4, 1e-4)
    gen = torch.Generator().manual_seed(11)
    loss, loss_ref = 0.0, 0.0
    for name, y, r in zip(("v", "b", "dt"), outs, refs):
        if r is None:
            assert y is None
            continue
        assert y.shape == r.shape and y.dtype == (torch.float32 if name == "dt" else dtype), name
        assert hp.max_abs(y.float(), r) <= out_tol * max(1.0, r.abs().max().item()), name
        wgt = torch.randn(r.shape, generator=gen).to(y.dtype)
        loss = loss + (y.float() * wgt.to(dev).float()).sum()
        loss_ref = loss_ref + (r * wgt.double()).sum()
    # the clamp is live in the bounded cases: some time steps on either side
    if limit[1] < 1.0:
        assert (refs[2] == limit[0]).any() and (refs[2] == limit[1]).any() and ((refs[2] > limit[0]) & (refs[2] < limit[1])).any()
    loss.backward()
    loss_ref.backward()
    for n in names:
        if a[n] is None:
            continue
        g, r = leaves[n].grad, ref_leaves[n].grad
        assert g.shape == r.shape and g.dtype == leaves[n].dtype, n
        err = hp.max_rel(g, r)
        assert err <= grad_tol, (n, err)


@pytest.mark.parametrize("lead,H,dv,dtype", MAMBA_SHAPES)
@pytest.mark.parametrize("residual,gated", [(True, True), (False, True), (True, False), (False, False)])
def test_mamba_epilogue_forward_backward(gpu_device, lead, H, dv, dtype, residual, gated):
    from palimpsa_amd.ops.layer_glue import metamamba2_output_norm
    gen = torch.Generator().manual_seed(12)
    o = torch.randn(*lead, H, dv, generator=gen).to(dtype)
    x = torch.randn(*lead, H, dv, generator=gen).to(dtype) if residual else None
    D = torch.randn(H, generator=gen) if residual else None
    gate = torch.randn(*lead, H * dv, generator=gen).to(dtype) if gated else None      # the layer's gate is [.., H dv]
    w = 1.0 + 0.2 * torch.randn(H * dv, generator=gen)
    dy = torch.randn(*lead, H, dv, generator=gen).to(dtype)
    dev = gpu_device
    names = ("o", "x", "D", "gate", "w")
    vals = dict(o=o, x=x, D=D, gate=gate, w=w)
    leaves = {n: (None if vals[n] is None else vals[n].to(dev).clone().requires_grad_(True)) for n in names}
    y = metamamba2_output_norm(leaves["o"], leaves["x"], leaves["D"], leaves["gate"], leaves["w"], 1e-5)
    ref_leaves = {n: (None if vals[n] is None else vals[n].double().clone().requires_grad_(True)) for n in names}
    y_ref = lo.mamba_epilogue(ref_leaves["o"], ref_leaves["x"], ref_leaves["D"], ref_leaves["gate"], ref_leaves["w"], 1e-5)
    out_tol, grad_tol = (hp.BF16_OUT_ABS_TOL, hp.BF16_GRAD_NORM_TOL) if dtype == torch.bfloat16 else (1e-4, 1e-4)
    assert y.shape == o.shape and y.dtype == dtype
    assert hp.max_abs(y.float(), y_ref.detach()) <= out_tol * max(1.0, y_ref.abs().max().item())
    y.backward(dy.to(dev))
    y_ref.backward(dy.double())
    for n in names:
        if vals[n] is None:
            continue
        g, r = leaves[n].grad, ref_leaves[n].grad
        assert g.shape == r.shape and g.dtype == leaves[n].dtype, n
        err = hp.max_rel(g, r)
        assert err <= grad_tol, (n, err)


def test_mamba_glue_is_reproducible_and_rejects_wide_tokens(gpu_device):
    from palimpsa_amd.ops.layer_glue import metamamba2_inputs, metamamba2_output_norm
    dev = gpu_device
    a = _inputs((3, 500), 1, 12, 8, 64, 13, torch.bfloat16)

    def run():
        lv = {n: a[n].to(dev).clone().requires_grad_(True) for n in ("x", "dt_raw", "dt_bias", "b_raw", "b_scale")}
        D = torch.ones(12, device=dev, requires_grad=True)
        w = torch.ones(768, device=dev, requires_grad=True)
        v, b, dt = metamamba2_inputs(**lv, dt_limit=(0.0, 0.5))
        y = metamamba2_output_norm(v * b, lv["x"], D, v, w)
        (y.float() ** 2).sum().backward()
        return [y.detach(), dt.detach()] + [t.grad for t in lv.values()] + [D.grad, w.grad]

    for p, q in zip(run(), run()):
        assert torch.isfinite(p.float()).all() and torch.equal(p, q)      # sums over tokens are taken in a fixed order
    with pytest.raises(ValueError):
        metamamba2_output_norm(torch.zeros(2, 32, 256, device=dev), None, None, None, torch.ones(32 * 256, device=dev))


def test_mamba_layer_slice_end_to_end(gpu_device):
    """MetaMamba2.forward between its convolution and out_proj (layers/meta_mamba2.py:276-363): inputs from the
    projections, the operator with scale = 1 and B, C rows of two groups shared by eight heads, residual + gated norm
    over the token; forward and all gradients against the oracles chained the same way."""
    from oracle import palimpsa_oracle as po
    from palimpsa_amd.ops.layer_glue import metamamba2_inputs, metamamba2_output_norm
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    dev = gpu_device
    B, T, H, G, dk, dv = 2, 130, 8, 2, 64, 32
    gen = torch.Generator().manual_seed(14)
    r = lambda *s: torch.randn(*s, generator=gen)
    vals = dict(C=(0.5 * r(B, T, G, dk)).bfloat16(), Bm=(0.5 * r(B, T, G, dk)).bfloat16(), x=r(B, T, H, dv).bfloat16(),
                dt_raw=(r(B, T, H) - 1.0).bfloat16(), dt_bias=0.3 * r(H), b_raw=r(B, T, H, dv).bfloat16(), b_scale=r(H) + 1.0,
                A_log=torch.log(torch.arange(1, H + 1).float()), Ip_log=0.2 * r(H), D=1.0 + 0.1 * r(H),
                gate=r(B, T, H * dv).bfloat16(), w=1.0 + 0.1 * r(H * dv))
    dy = r(B, T, H, dv).bfloat16()

    lv = {n: t.to(dev).clone().requires_grad_(True) for n, t in vals.items()}
    v, b, dt = metamamba2_inputs(lv["x"], lv["dt_raw"], lv["dt_bias"], lv["b_raw"], lv["b_scale"], dt_limit=(0.0, 2.0))
    o = chunk_palimpsa(lv["C"], lv["Bm"], v, b, dt, lv["A_log"].exp(), lv["Ip_log"].exp(), scale=1.0, chunk_size=16)
    y = metamamba2_output_norm(o, lv["x"], lv["D"], lv["gate"], lv["w"], 1e-5)
    y.backward(dy.to(dev))

    rl = {n: t.double().clone().requires_grad_(True) for n, t in vals.items()}
    v_r, b_r, dt_r = lo.mamba_prologue(rl["x"], rl["dt_raw"], rl["dt_bias"], rl["b_raw"], rl["b_scale"], dt_limit=(0.0, 2.0))
    rep = H // G
    o_r = po.palimpsa_recurrence(rl["C"].repeat_interleave(rep, dim=2), rl["Bm"].repeat_interleave(rep, dim=2), v_r, b_r,
                                 dt_r, rl["A_log"].exp(), rl["Ip_log"].exp(), scale=1.0, compute_dtype=torch.float64)[0]
    y_r = lo.mamba_epilogue(o_r, rl["x"], rl["D"], rl["gate"], rl["w"], 1e-5)
    y_r.backward(dy.double())
    assert hp.max_abs(y.float(), y_r.detach()) <= hp.BF16_OUT_ABS_TOL * max(1.0, y_r.abs().max().item())
    for n in vals:
        err = hp.max_rel(lv[n].grad, rl[n].grad)
        assert err <= hp.BF16_GRAD_NORM_TOL, (n, err)


# ------------------------------------------------------------------ how rows are dealt out
@pytest.mark.parametrize("lead,Hqk,H,dk,dv", [
    ((1,), 16, 16, 48, 48),       # one token: most row slots are empty
    ((9,), 16, 16, 48, 48),       # a workgroup's tokens and one more
    ((300,), 24, 24, 48, 96),     # groups of eight heads, rows of two widths
    ((3, 41), 4, 16, 64, 64),     # q, k of four heads each: the third and fourth gradient are fetched late
    ((77,), 5, 40, 16, 16),       # an odd number of q, k heads beside groups of eight
    ((130,), 64, 64, 8, 16),      # more heads than row slots
    ((40,), 256, 256, 8, 8),      # a head to every thread: more sums per head than threads
    ((9,), 4, 512, 16, 8),        # two groups of them
])
def test_rows_over_heads_and_tokens(gpu_device, lead, Hqk, H, dk, dv):
    test_prologue_forward_backward(gpu_device, lead, Hqk, H, dk, dv, torch.bfloat16, True)
    test_epilogue_forward_backward(gpu_device, lead, H, dv, torch.bfloat16, True, True)


@pytest.mark.parametrize("tokens", [1, 4097, 5121, 13315])       # four tokens a wave: ragged ends of one and of three
def test_mamba_epilogue_tokens_per_wave(gpu_device, tokens):
    test_mamba_epilogue_forward_backward(gpu_device, (tokens,), 2, 16, torch.float32, True, True)
    test_mamba_epilogue_forward_backward(gpu_device, (tokens,), 4, 152, torch.bfloat16, True, True)
