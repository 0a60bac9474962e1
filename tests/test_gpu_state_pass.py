"""The two ways the chunked entry points build the states at the start of every tile — per-tile contributions
by all tiles in parallel followed by a scan, or one pass per (sequence, head) with the running state in
registers — must agree: same algorithm, same bf16 operands, fp32 sums taken in a different order.  Each form is
also checked against the oracle (Palimpsa) or the float64 closed form (scalar-gated path) on its own, so that
neither is only ever compared with the other.
"""
import math

import pytest
import torch

from tests import helpers as hp

pytestmark = pytest.mark.gpu


@pytest.fixture
def state_pass_mode():
    from palimpsa_amd import _lib
    yield _lib.set_state_pass_mode
    _lib.set_state_pass_mode(0)


def _pal_inputs(B, T, H, dk, dv, seed, dev):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)
    inp = dict(
        q=torch.nn.functional.normalize(r(B, T, H, dk), dim=-1), k=torch.nn.functional.normalize(r(B, T, H, dk), dim=-1),
        v=r(B, T, H, dv), b=torch.rand(B, T, H, dv, generator=gen) + 0.1,
        gt=torch.nn.functional.softplus(r(B, T, H)) * 0.2, g=torch.linspace(0.3, 3.0, H), Ip=torch.linspace(0.5, 2.0, H))
    return hp.to_device(hp.rounded(inp, torch.bfloat16), dev)


def _run_palimpsa(inp, mu0, I0, cu, grads):
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    names = ("q", "k", "v", "b", "gt", "g", "Ip")
    leaves = {n: inp[n].detach().clone().requires_grad_(grads) for n in names}
    st = [s.detach().clone().requires_grad_(grads) for s in (mu0, I0)] if mu0 is not None else [None, None]
    o, fmu, fI = chunk_palimpsa(*[leaves[n] for n in names], initial_mu_state=st[0], initial_I_state=st[1],
                                output_final_state=True, cu_seqlens=cu)
    out = [o, fmu, fI]
    if grads:
        gen = torch.Generator().manual_seed(5)
        do = torch.randn(o.shape, generator=gen).to(o)
        (o.float() * do.float()).sum().backward()
        out += [leaves[n].grad for n in names] + ([s.grad for s in st] if mu0 is not None else [])
    return out


@pytest.mark.parametrize("case", ["batched", "varlen_ragged", "wide_heads", "init_state_grads", "key_slices"])
def test_palimpsa_forms_agree(gpu_device, state_pass_mode, case):
    dev = gpu_device
    cu = mu0 = I0 = None
    grads = False
    if case == "batched":
        inp = _pal_inputs(3, 300, 4, 64, 64, 1, dev)
    elif case == "varlen_ragged":       # full and partial tiles, a one-token document
        inp = _pal_inputs(1, 64 + 1 + 130 + 257, 2, 32, 48, 2, dev)
        cu = torch.tensor([0, 64, 65, 195, 452], dtype=torch.int32, device=dev)
    elif case == "wide_heads":            # few (sequence, head) pairs: the one-pass form also slices the key columns
        inp = _pal_inputs(2, 129, 2, 256, 144, 3, dev)
    elif case == "key_slices":            # the same with an initial state, at the shape class of a long single prefill
        inp = _pal_inputs(1, 300, 12, 128, 128, 6, dev)
        gen = torch.Generator().manual_seed(10)
        mu0 = (torch.randn(1, 12, 128, 128, generator=gen) * 0.3).to(dev)
        I0 = (torch.rand(1, 12, 128, 128, generator=gen) + inp["Ip"].cpu()[None, :, None, None]).to(dev)
    else:
        inp = _pal_inputs(2, 200, 3, 48, 96, 4, dev)
        gen = torch.Generator().manual_seed(9)
        mu0 = (torch.randn(2, 3, 96, 48, generator=gen) * 0.3).to(dev)
        I0 = (torch.rand(2, 3, 96, 48, generator=gen) + inp["Ip"].cpu()[None, :, None, None]).to(dev)
        grads = True
    state_pass_mode(1)
    a = _run_palimpsa(inp, mu0, I0, cu, grads)
    state_pass_mode(2)
    b = _run_palimpsa(inp, mu0, I0, cu, grads)
    assert hp.max_abs(a[0].float(), b[0].float()) <= 1e-2            # outputs: bf16, a last-bit flip at most
    assert hp.max_rel(a[1], b[1]) <= 1e-4 and hp.max_rel(a[2], b[2]) <= 1e-4   # fp32 final states: order of sums only
    for x, y in zip(a[3:], b[3:]):
        assert hp.max_rel(x.float(), y.float()) <= 2e-2
    # the one-pass form against the oracle
    o_ref, _, fmu_ref, fI_ref = hp.oracle_forward({k: v.cpu() for k, v in inp.items()}, mu0=None if mu0 is None else mu0.cpu(),
                                                  I0=None if I0 is None else I0.cpu(), cu=None if cu is None else cu.cpu().tolist())
    assert hp.max_abs(b[0].float(), o_ref) <= hp.BF16_OUT_ABS_TOL
    assert hp.max_rel(b[1], fmu_ref) <= 2e-2 and hp.max_rel(b[2], fI_ref) <= 2e-2


@pytest.mark.parametrize("dk,dv", [(16, 64), (48, 48), (80, 64), (96, 32), (128, 48), (176, 32), (192, 16), (256, 16)])
def test_wide_value_slices_agree(gpu_device, state_pass_mode, dk, dv):
    """Enough heads that a workgroup takes several blocks of value rows, over the widths of the staged key rows; two tiles
    and a ragged third. Tolerances as above: the forms differ in the order of fp32 sums."""
    inp = _pal_inputs(2, 129 + dk % 7, 96, dk, dv, dk + dv, gpu_device)
    state_pass_mode(1)
    a = _run_palimpsa(inp, None, None, None, False)
    state_pass_mode(2)
    b = _run_palimpsa(inp, None, None, None, False)
    assert hp.max_abs(a[0].float(), b[0].float()) <= 1e-2
    assert hp.max_rel(a[1], b[1]) <= 1e-4 and hp.max_rel(a[2], b[2]) <= 1e-4


@pytest.mark.parametrize("dk,dv", [(64, 64), (48, 20), (80, 48)])       # even and odd numbers of columns per lane
@pytest.mark.parametrize("case", ["usual", "no_decay", "strong", "mixed", "growth", "huge", "nan"])
def test_scaled_and_plain_tiles(gpu_device, state_pass_mode, dk, dv, case):
    """Outputs of the tiles over what decides between their two forms, and over what makes the scaled one start again,
    against the oracle in float64: bf16 rows, so the results' rounding is the tolerance."""
    inp = _pal_inputs(2, 150, 3, dk, dv, dk, "cpu")
    gen = torch.Generator().manual_seed(dv)
    mu0 = torch.randn(2, 3, dv, dk, generator=gen) * 0.3
    I0 = torch.rand(2, 3, dv, dk, generator=gen) + inp["Ip"][None, :, None, None]
    if case == "no_decay":
        inp["g"] = torch.zeros(3)
    elif case == "strong":            # 2^-60 and less over eight tokens, a gate that leaves nothing among them
        inp["g"] = torch.tensor([40.0, 80.0, 2000.0])
    elif case == "mixed":             # one step of one tile decays too much
        inp["gt"][:, 70] = 30.0
    elif case == "growth":
        inp["gt"][:, 20:30] *= -0.2
    elif case == "huge":              # the product of two precisions overflows, the quotients do not
        I0 *= 1e24
    elif case == "nan":
        inp["v"][0, 40, 1, 3] = float("nan")
    state_pass_mode(2)
    o = _run_palimpsa(hp.to_device(inp, gpu_device), mu0.to(gpu_device), I0.to(gpu_device), None, False)[0].float().cpu()
    o_ref = hp.oracle_forward(inp, mu0=mu0, I0=I0, dtype=torch.float64)[0].float()
    assert torch.equal(torch.isnan(o), torch.isnan(o_ref))
    assert hp.max_abs(o.nan_to_num(), o_ref.nan_to_num()) <= hp.BF16_OUT_ABS_TOL


@pytest.mark.parametrize("dk,dv", [(32, 32), (48, 48), (64, 64), (80, 96), (128, 64), (192, 48)])
def test_decay_applied_after_8_to_64_tokens(gpu_device, state_pass_mode, dk, dv):
    """The scaled form applies the decay to the state after 64, 32, 16 or 8 tokens, the longest whose decay stays above 2^-30:
    heads on either side of each line and far from them, full and ragged tiles, against the oracle in float64.  bf16 rows:
    half a unit of the result (2^-9) and as much for the rows' products."""
    bits = torch.tensor([0.0, 0.3, 0.468, 0.47, 0.93, 0.945, 1.87, 1.88, 3.0, 6.0])   # of decay a token; 30 / 64 = 0.46875
    H = bits.numel()
    inp = _pal_inputs(1, 64 * 3 + 41, H, dk, dv, dk + dv, "cpu")
    inp["g"] = bits * math.log(2.0)
    inp["gt"] = torch.ones_like(inp["gt"])
    inp["gt"][:, 64:128] = torch.rand(1, 64, H, generator=torch.Generator().manual_seed(3)) * 2.0   # one tile of uneven decays
    gen = torch.Generator().manual_seed(dv)
    mu0 = torch.randn(1, H, dv, dk, generator=gen) * 0.3
    I0 = torch.rand(1, H, dv, dk, generator=gen) + inp["Ip"][None, :, None, None]
    state_pass_mode(2)
    o = _run_palimpsa(hp.to_device(inp, gpu_device), mu0.to(gpu_device), I0.to(gpu_device), None, False)[0].float().cpu()
    o_ref = hp.oracle_forward(inp, mu0=mu0, I0=I0, dtype=torch.float64)[0].float()
    for h in range(H):
        assert hp.max_rel(o[:, :, h], o_ref[:, :, h]) <= 2.0 ** -8, h


@pytest.mark.parametrize("tiles,dtype,case", [(257, torch.bfloat16, "usual"), (129, torch.bfloat16, "usual"),
                                              (257, torch.bfloat16, "strong"), (257, torch.bfloat16, "huge"),
                                              (257, torch.bfloat16, "uncertainty"), (257, torch.float32, "usual")])
def test_walks_over_several_tiles(gpu_device, monkeypatch, tiles, dtype, case):
    """The windows of a long sequence keep the state of every fourth (second) tile only and walk on from it; windows that
    keep all of them give the same final states, and the outputs up to what the states between are rounded to."""
    from palimpsa_amd import _lib
    from palimpsa_amd.ops.palimpsa import chunk as chunk_mod, chunk_palimpsa
    H, d = 24, 64
    T = 64 * (2 * tiles - 1) - 20     # the last window ends in a ragged tile; a walk of one or two tiles ends the first
    monkeypatch.setattr(chunk_mod, "_WINDOW_STATE_BYTES", tiles * 2 * 4 * H * d * d)
    inp = _pal_inputs(1, T, H, d, d, 31, gpu_device)
    inp = {n: x.to(dtype) if n in "qkvb" else x for n, x in inp.items()}
    if case == "strong":
        inp["g"] = torch.linspace(0.5, 90.0, H, device=gpu_device)
    gen = torch.Generator().manual_seed(32)
    mu0 = (torch.randn(1, H, d, d, generator=gen) * 0.2).to(gpu_device)
    I0 = (torch.rand(1, H, d, d, generator=gen) + 0.5).to(gpu_device) * (1e24 if case == "huge" else 1.0)
    kw = dict(initial_mu_state=mu0, initial_I_state=I0, output_final_state=True, output_uncertainty=case == "uncertainty")
    with torch.no_grad():
        o, mu, I = chunk_palimpsa(**inp, **kw)
        monkeypatch.setattr(_lib, "PAL_FLAG_SPARSE_STATES", 0)
        o_all, mu_all, I_all = chunk_palimpsa(**inp, **kw)
    assert torch.equal(mu, mu_all) and torch.equal(I, I_all)
    o, o_all = ((z if isinstance(z, tuple) else (z,)) for z in (o, o_all))
    for x, y in zip(o, o_all):
        if dtype == torch.float32:
            assert hp.max_rel(x, y) <= hp.FP32_REL_TOL
        else:
            assert hp.max_abs(x.float(), y.float()) <= hp.BF16_OUT_ABS_TOL


@pytest.mark.parametrize("H,dk,dv,tiles", [(16, 128, 128, 128), (16, 96, 192, 130), (24, 128, 64, 129), (16, 128, 112, 160)])
@pytest.mark.parametrize("case", ["usual", "strong", "uncertainty", "no_init"])
def test_state_pass_in_segments(gpu_device, monkeypatch, H, dk, dv, tiles, case):
    """Windows that keep every fourth tile's state cut the walk that makes them into segments, whose states count from the
    start of their segment (bf16 rows, few heads): final states and outputs against windows that keep all states.  A second
    window of fewer tiles, the last of them ragged.  The states differ by the order of fp32 sums over 10^4 tokens."""
    from palimpsa_amd import _lib
    from palimpsa_amd.ops.palimpsa import chunk as chunk_mod, chunk_palimpsa
    T = 64 * (2 * tiles - 27) - 20
    monkeypatch.setattr(chunk_mod, "_WINDOW_STATE_BYTES", tiles * 2 * 4 * H * dk * dv)
    inp = _pal_inputs(1, T, H, dk, dv, 77, gpu_device)
    inp = {n: x.to(torch.bfloat16) if n in "qkvb" else x for n, x in inp.items()}
    # slow decays: states of earlier segments reach far into the later ones; or none that survives a tile
    inp["g"] = torch.linspace(0.5, 90.0, H, device=gpu_device) if case == "strong" else torch.logspace(-5, 0, H, device=gpu_device)
    gen = torch.Generator().manual_seed(5)
    kw = dict(output_final_state=True, output_uncertainty=case == "uncertainty")
    if case != "no_init":
        kw["initial_mu_state"] = (torch.randn(1, H, dv, dk, generator=gen) * 0.2).to(gpu_device)
        kw["initial_I_state"] = (torch.rand(1, H, dv, dk, generator=gen) + 0.5).to(gpu_device)
    with torch.no_grad():
        o, mu, I = chunk_palimpsa(**inp, **kw)
        monkeypatch.setattr(_lib, "PAL_FLAG_SPARSE_STATES", 0)
        o_all, mu_all, I_all = chunk_palimpsa(**inp, **kw)
    for h in range(H):
        assert hp.max_rel(mu[:, h], mu_all[:, h]) <= 1e-5 and hp.max_rel(I[:, h], I_all[:, h]) <= 1e-5, h
    o, o_all = ((z if isinstance(z, tuple) else (z,)) for z in (o, o_all))
    for x, y in zip(o, o_all):
        assert hp.max_abs(x.float(), y.float()) <= hp.BF16_OUT_ABS_TOL


@pytest.mark.parametrize("H,dk,dv", [(16, 128, 128), (16, 128, 112)])
def test_segments_whose_decay_leaves_the_range_of_fp32(gpu_device, monkeypatch, H, dk, dv):
    """Gates above 1, or states far above 1, over more tokens than fp32 has powers of two: what the tile by tile walk over the
    same window keeps finite stays finite in segments, to the rounding of fp32 sums.  Heads: nothing before a growth of 2^368;
    a state of 2^-100 that grows by 2^184; one of 2^100 that decays by 2^-184; and ordinary ones."""
    from palimpsa_amd import _lib
    from palimpsa_amd.ops.palimpsa import chunk as chunk_mod, chunk_palimpsa
    tiles, grown = 128, 80
    T = 64 * tiles + 64 * 8
    monkeypatch.setattr(chunk_mod, "_WINDOW_STATE_BYTES", tiles * 2 * 4 * H * dk * dv)
    inp = _pal_inputs(1, T, H, dk, dv, 78, gpu_device)
    inp = {n: x.to(torch.bfloat16) if n in "qkvb" else x for n, x in inp.items()}
    inp["g"] = torch.full((H,), 0.6931472, device=gpu_device)        # f = 2^-gt
    inp["gt"] = 0.02 * torch.rand(1, T, H, generator=torch.Generator().manual_seed(3)).to(gpu_device)
    quiet = slice(0, 64 * grown)
    inp["gt"][:, quiet, :12] = 0
    inp["gt"][:, :64 * grown, 0:4] = inp["gt"][:, :32 * grown, 4:8] = -0.071875     # 2^147 over a segment of 32 tiles
    inp["gt"][:, :32 * grown, 8:12] = 0.071875
    for n in ("v", "b"):
        inp[n][:, quiet, :12] = 0
    gen = torch.Generator().manual_seed(5)
    mu0, I0 = torch.randn(1, H, dv, dk, generator=gen) * 0.2, inp["Ip"].cpu().view(1, H, 1, 1).expand(1, H, dv, dk).clone()
    mu0[:, 0:4], mu0[:, 4:8], mu0[:, 8:12] = 0, mu0[:, 4:8] * 2.0 ** -100, mu0[:, 8:12] * 2.0 ** 100
    kw = dict(output_final_state=True, initial_mu_state=mu0.to(gpu_device), initial_I_state=I0.to(gpu_device))
    with torch.no_grad():
        o, mu, I = chunk_palimpsa(**inp, **kw)
        monkeypatch.setattr(_lib, "PAL_FLAG_SPARSE_STATES", 0)
        o_all, mu_all, I_all = chunk_palimpsa(**inp, **kw)
    for x in (o_all, mu_all, I_all, o, mu, I):
        assert bool(torch.isfinite(x).all())
    for h in range(H):
        assert hp.max_rel(mu[:, h], mu_all[:, h]) <= 1e-5 and hp.max_rel(I[:, h], I_all[:, h]) <= 1e-5, h
        for w in (slice(0, 64 * grown), slice(64 * grown, None)):
            x, y = o[:, w, h].float(), o_all[:, w, h].float()
            if float(y.abs().max()) < hp.BF16_OUT_ABS_TOL or float(y.abs().max()) > 100:   # one bf16 rounding on either side
                assert hp.max_rel(x, y) <= 2.0 ** -7, (h, w)
            else:
                assert hp.max_abs(x, y) <= hp.BF16_OUT_ABS_TOL, (h, w)


@pytest.mark.parametrize("T", [64, 64 * 9 + 5, 64 * 21])
def test_scan_of_few_and_of_many_heads(gpu_device, state_pass_mode, T):
    """The scan over the tiles takes one or four state entries per thread, by the number of heads: the same sums in the same
    order, so the final states are the same bits."""
    inp = _pal_inputs(4, T, 20, 64, 64, T, gpu_device)
    few = {n: x[:1, :, :3].contiguous() if x.dim() > 1 else x[:3] for n, x in inp.items()}
    state_pass_mode(1)
    a = _run_palimpsa(inp, None, None, None, False)
    b = _run_palimpsa(few, None, None, None, False)
    assert torch.equal(a[1][:1, :3], b[1]) and torch.equal(a[2][:1, :3], b[2])
    assert hp.max_abs(a[0][:1, :, :3].float(), b[0].float()) <= 1e-2


def _gla_inputs(B, T, H, dk, dv, seed):
    gen = torch.Generator().manual_seed(seed)
    q = torch.nn.functional.normalize(torch.randn(B, T, H, dk, generator=gen), dim=-1).bfloat16()
    k = torch.nn.functional.normalize(torch.randn(B, T, H, dk, generator=gen), dim=-1).bfloat16()
    v = torch.randn(B, T, H, dv, generator=gen).bfloat16()
    g = -torch.nn.functional.softplus(torch.randn(B, T, H, generator=gen)) * torch.linspace(0.05, 2.0, H)
    S0 = torch.randn(B, H, dk, dv, generator=gen) * 0.2
    do = torch.randn(B, T, H, dv, generator=gen).bfloat16()
    return q, k, v, g, S0, do


def _run_gla(x, dev, cu=None):
    from palimpsa_amd.ops.simple_gla import chunk_simple_gla
    q, k, v, g, S0, do = x
    leaves = [t.to(dev).clone().requires_grad_(True) for t in (q, k, v, g, S0)]
    o, S = chunk_simple_gla(q=leaves[0], k=leaves[1], v=leaves[2], g=leaves[3], initial_state=leaves[4],
                            output_final_state=True, cu_seqlens=cu)
    (o.float() * do.to(dev).float()).sum().backward()
    return [o, S] + [t.grad for t in leaves]


@pytest.mark.parametrize("shape", [(2, 200, 3, 64, 64), (1, 777, 2, 96, 192), (2, 65, 2, 256, 32), (3, 64, 1, 16, 16)])
def test_simple_gla_forms_agree_forward_and_backward(gpu_device, state_pass_mode, shape):
    x = _gla_inputs(*shape, seed=21)
    state_pass_mode(1)
    a = _run_gla(x, gpu_device)
    state_pass_mode(2)
    b = _run_gla(x, gpu_device)
    assert hp.max_abs(a[0].float(), b[0].float()) <= 1e-2
    assert hp.max_rel(a[1], b[1]) <= 1e-4                     # fp32 final state
    names = ("dq", "dk", "dv", "dg", "dS0")
    for n, p, r in zip(names, a[2:], b[2:]):
        assert hp.max_rel(p.float(), r.float()) <= 2e-2, n


def test_simple_gla_one_pass_form_against_closed_form(gpu_device, state_pass_mode):
    from tests.test_gpu_simple_gla import _closed_form
    B, T, H, dk, dv = 2, 260, 3, 64, 32
    q, k, v, g, S0, do = _gla_inputs(B, T, H, dk, dv, seed=22)
    state_pass_mode(2)
    got = _run_gla((q, k, v, g, S0, do), gpu_device)
    leaves = [t.double().clone().requires_grad_(True) for t in (q, k, v, g, S0)]
    o_ref, S_ref = _closed_form(*leaves[:4], dk ** -0.5, leaves[4])
    (o_ref * do.double()).sum().backward()
    assert hp.max_abs(got[0].float(), o_ref) <= hp.BF16_OUT_ABS_TOL
    assert hp.max_rel(got[1], S_ref) <= 1e-2
    for n, p, r in zip(("dq", "dk", "dv", "dg", "dS0"), got[2:], leaves):
        assert hp.max_rel(p.float(), r.grad) <= hp.BF16_GRAD_NORM_TOL, n


def test_varlen_simple_gla_forms_agree(gpu_device, state_pass_mode):
    from palimpsa_amd.ops.simple_gla import chunk_simple_gla
    dev = gpu_device
    lens = [1, 64, 0, 100, 300]
    T = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=dev)
    q, k, v, g, _, do = _gla_inputs(1, T, 2, 48, 96, seed=23)
    outs = []
    for mode in (1, 2):
        state_pass_mode(mode)
        leaves = [t.to(dev).clone().requires_grad_(True) for t in (q, k, v, g)]
        o, S = chunk_simple_gla(q=leaves[0], k=leaves[1], v=leaves[2], g=leaves[3], output_final_state=True, cu_seqlens=cu)
        (o.float() * do.to(dev).float()).sum().backward()
        outs.append([o, S] + [t.grad for t in leaves])
    a, b = outs
    assert a[1].shape[0] == len(lens)
    assert hp.max_abs(a[0].float(), b[0].float()) <= 1e-2
    assert hp.max_rel(a[1], b[1]) <= 1e-4
    for p, r in zip(a[2:], b[2:]):
        assert hp.max_rel(p.float(), r.float()) <= 2e-2
