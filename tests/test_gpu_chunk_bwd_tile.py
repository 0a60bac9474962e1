"""The chunked backward's tile kernel at the edges of its launches: one and several groups of key columns and slices of
value rows (64, 48, 32, 16 of each), tiles that end inside a step, at a step, in the first or the second half; with and
without the uncertainty output and an initial state; fp32 rows at the fp32 bar, bf16 rows at the bf16 one."""
import pytest
import torch

from oracle import palimpsa_oracle as po
from tests import helpers as hp

pytestmark = pytest.mark.gpu

NAMES = ("q", "k", "v", "b", "gt", "g", "Ip")


@pytest.mark.parametrize("dk,dv", [(16, 64), (16, 48), (32, 16), (32, 80), (48, 96), (64, 112), (80, 32), (96, 48), (128, 64)])
@pytest.mark.parametrize("rows", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_tile_kernel_launches(gpu_device, dk, dv, rows):
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    H = 2
    for T, var, init in ((3, False, False), (33, True, False), (64, False, True), (103, True, True)):
        inp = hp.rounded(po.make_inputs(1, T, H, dk, dv, seed=dk + dv + T), rows)
        inp["g"] = torch.tensor([0.3, 5.0])
        gen = torch.Generator().manual_seed(T)
        mu0 = I0 = None
        if init:
            mu0 = 0.1 * torch.randn(1, H, dv, dk, generator=gen)
            I0 = inp["Ip"].view(1, H, 1, 1) + torch.rand(1, H, dv, dk, generator=gen)
        o_ref, _, _, _ = hp.oracle_forward(inp, mu0=mu0, I0=I0, dtype=torch.float64)
        # squared-error loss: dO correlated with the state, dg and dIp well conditioned
        do = (o_ref - 0.3 * torch.randn(1, T, H, dv, generator=gen)).float()
        dov = 0.3 * torch.randn(1, T, H, dv, generator=gen) if var else None
        ref = hp.oracle_grads(inp, do, dov, mu0=mu0, I0=I0)
        leaves = {n: inp[n].to(gpu_device).clone().requires_grad_(True) for n in NAMES}
        if init:
            leaves["mu0"], leaves["I0"] = (x.to(gpu_device).requires_grad_(True) for x in (mu0, I0))
        out = chunk_palimpsa(*[leaves[n] for n in NAMES], initial_mu_state=leaves.get("mu0"), initial_I_state=leaves.get("I0"),
                             output_uncertainty=var)
        loss = ((out[0] if var else out).float() * do.to(gpu_device)).sum()
        if var:
            loss = loss + (out[1].float() * dov.to(gpu_device)).sum()
        got = torch.autograd.grad(loss, list(leaves.values()))
        for n, x in zip(leaves, got):
            err = hp.max_rel(x, ref[n])
            assert err <= (hp.CHUNK_FP32_GRAD_TOL if rows == torch.float32 else hp.BF16_GRAD_NORM_TOL), (T, var, init, n, err)


@pytest.mark.parametrize("dk,dv", [(16, 16), (32, 32), (48, 48), (64, 64), (80, 80), (96, 128)])
@pytest.mark.parametrize("rows", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_gate_gradient_of_strongly_decaying_tokens(gpu_device, dk, dv, rows):
    """dgt_t is f_t times a number of the order of the other gradients (what flows back against the state before the
    token), however small f_t is: that number is held to the bar of the other gradients, entry by entry.  Where there is
    no state before a token its gradient is exactly zero."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    H, T = 2, 150
    inp = hp.rounded(po.make_inputs(1, T, H, dk, dv, seed=dk + dv), rows)
    inp["g"] = torch.tensor([1.0, 2.0])
    inp["gt"][:, ::5] = 9.0                     # f = e^-9, e^-18
    for var in (False, True):
        gen = torch.Generator().manual_seed(T)
        o_ref, _, _, _ = hp.oracle_forward(inp, dtype=torch.float64)
        do = (o_ref - 0.3 * torch.randn(1, T, H, dv, generator=gen)).float()
        dov = 0.3 * torch.randn(1, T, H, dv, generator=gen) if var else None
        ref = hp.oracle_grads(inp, do, dov)["gt"]
        leaves = [inp[n].to(gpu_device).requires_grad_(True) for n in NAMES]
        out = chunk_palimpsa(*leaves, output_uncertainty=var)
        loss = ((out[0] if var else out).float() * do.to(gpu_device)).sum()
        if var:
            loss = loss + (out[1].float() * dov.to(gpu_device)).sum()
        dgt = torch.autograd.grad(loss, leaves[4])[0].double().cpu()
        assert bool((dgt[:, 0] == 0).all())
        f = torch.exp(-inp["gt"].double() * inp["g"].double())
        err = hp.max_rel(dgt / f, ref / f)
        assert err <= (hp.CHUNK_FP32_GRAD_TOL if rows == torch.float32 else hp.BF16_GRAD_NORM_TOL), (var, err)


@pytest.mark.parametrize("dk,dv", [(16, 64), (32, 80), (48, 96), (64, 112), (80, 80), (96, 96), (96, 192), (112, 16), (128, 64), (160, 48),
                                   (176, 32), (192, 80)])
@pytest.mark.parametrize("rows", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_small_passes_agree_with_large_ones(gpu_device, dk, dv, rows):
    """Few tiles: the rectangles of a wide head side by side, their parts summed by a kernel of its own.  Many tiles: one
    after the other.  The same rows as a small pass and as the first rows of a large one: the same gradients, up to the
    rounding of the results and the order of their sums (48 rows of another batch entry per tile stay apart)."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    if rows == torch.float32 and max(dk, dv) > 128:
        pytest.skip("fp32 rows take head dims up to 128")
    H, few, many = 4, 1, 24          # 24 tiles of 4 heads a pass of few rows, 576 of many
    T = 64 * 6 - 11                  # the last tile is ragged
    inp = hp.to_device(hp.rounded(po.make_inputs(many, T, H, dk, dv, seed=dk + dv), rows), gpu_device)
    gen = torch.Generator(device=gpu_device).manual_seed(3)
    do, dov = (torch.randn(many, T, H, dv, generator=gen, device=gpu_device) for _ in range(2))
    mu0 = 0.1 * torch.randn(many, H, dv, dk, generator=gen, device=gpu_device)
    I0 = inp["Ip"].view(1, H, 1, 1) + torch.rand(many, H, dv, dk, generator=gen, device=gpu_device)
    for var, init in ((False, False), (True, True)):
        got = []
        for B in (few, many):
            leaves = [(inp[n][:B] if inp[n].dim() > 1 else inp[n]).clone().requires_grad_(True) for n in NAMES]
            state = [x[:B].clone().requires_grad_(True) for x in (mu0, I0)] if init else [None, None]
            out = chunk_palimpsa(*leaves, *state, output_uncertainty=var)
            out = list(out) if var else [out]
            got.append(torch.autograd.grad(out, leaves[:5] + [x for x in state if x is not None],
                                           [g[:B].to(rows) for g in (do, dov)][:len(out)]))
        for n, x, y in zip(NAMES[:5] + ("mu0", "I0"), *got):
            # 2 x 2 roundings of operands, and for bf16 results one of 2^-9 on each side
            bar = 4 * 2.0 ** -17 if rows == torch.float32 else (4 if n == "gt" else 6) * 2.0 ** -9
            assert hp.max_rel(x, y[:few]) <= bar, (var, init, n, hp.max_rel(x, y[:few]))


@pytest.mark.parametrize("dk,dv", [(16, 16), (32, 64), (48, 48), (64, 64), (96, 80)])
@pytest.mark.parametrize("rows", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_scaled_and_plain_tiles(gpu_device, dk, dv, rows):
    """A tile of bf16 rows without the uncertainty is worked with the decay of a step taken out of the state, or in plain form
    where a step decays below 2^-48, the decay since its start exceeds 1, or v, b, k, the state or Ip are large; fp32 rows and the
    uncertainty always in plain form.  Heads on either side of each line (every one with tiles of both kinds), as a small pass, in
    slices of 16 rows and mostly eight tokens a step, and repeated in the batch until the pieces run whole, one after the other;
    gradients head by head against the float64 recurrence."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    H, T, many = 6, 64 * 4 + 21, 18                  # 5 tiles of 6 heads, or 540 of them
    base = po.make_inputs(1, T, H, dk, dv, seed=dk + dv)
    base["g"] = torch.full((H,), 0.6931472)          # f = 2^-gt
    gt = 0.3 * torch.rand(1, T, H, generator=torch.Generator().manual_seed(1))
    gt[:, 70:, 1] = 11.9                             # four tokens: 2^-47.6, eight 2^-95
    gt[:, 70:90, 2] = 5.99                           # eight: 2^-47.92
    gt[:, 70:90, 3] = 6.01                           # eight: 2^-48.08
    gt[:, 100::64, 4] = 80.0                         # single tokens
    gt[:, 100:120, 5] = -0.05                        # f > 1
    base["gt"] = gt
    gen = torch.Generator().manual_seed(T)
    mu0 = 0.1 * torch.randn(1, H, dv, dk, generator=gen)
    I0 = base["Ip"].view(1, H, 1, 1) + torch.rand(1, H, dv, dk, generator=gen)
    noise = torch.randn(1, T, H, dv, generator=gen)
    unc = 0.3 * torch.rand(1, T, H, dv, generator=gen)
    # rows and states beyond their lines, and just inside
    cases = [("none", 1.0)] + [(n, 2.0 ** 24) for n in "vbk"] + [("state", 2.0 ** 70), ("Ip", 2.0 ** 70)]
    cases += [("v", 2.0 ** 17), ("b", 2.0 ** 3), ("k", 2.0 ** 3), ("Ip", 2.0 ** 13)]
    for what, size in cases:
        raw, m0, i0 = dict(base), mu0, I0
        if what in "vbk":
            raw[what] = base[what].clone()
            raw[what][:, 130:140] *= size
        if what == "state":
            m0, i0 = mu0.clone(), I0.clone()
            i0[:, ::2] *= size
        if what == "Ip":
            raw["Ip"] = base["Ip"] * torch.tensor([size, 1, size, 1, size, 1])
            i0 = raw["Ip"].view(1, H, 1, 1) * (I0 / base["Ip"].view(1, H, 1, 1))
        inp = hp.rounded(raw, rows)
        o_ref, _, _, _ = hp.oracle_forward(inp, mu0=m0, I0=i0, dtype=torch.float64)
        do = (o_ref - 0.3 * noise * o_ref.abs().mean(dim=(0, 1, 3), keepdim=True)).float()   # as large as the head's outputs
        do = do.to(rows).float()
        for var in (False, True) if what in ("none", "b") else (False,):
            dov = unc.to(rows).float() if var else None
            ref = hp.oracle_grads(inp, do, dov, mu0=m0, I0=i0)
            for copies in (1, many):
                rep = lambda x: x.to(gpu_device).repeat(copies, *[1] * (x.dim() - 1)) if x.dim() > 1 else x.to(gpu_device)
                leaves = {n: rep(inp[n]).clone().requires_grad_(True) for n in NAMES}
                leaves["mu0"], leaves["I0"] = (rep(x).clone().requires_grad_(True) for x in (m0, i0))
                out = chunk_palimpsa(*[leaves[n] for n in NAMES], initial_mu_state=leaves["mu0"], initial_I_state=leaves["I0"],
                                     output_uncertainty=var)
                grads = [rep(x).to(rows) for x in ((do, dov) if var else (do,))]
                got = torch.autograd.grad(list(out) if var else [out], list(leaves.values()), grads)
                for n, x in zip(leaves, got):
                    assert bool(torch.isfinite(x).all()), (what, size, var, copies, n)
                    if what in ("state", "Ip") and size > 1 and n in ("gt", "g", "I0", "Ip"):
                        continue   # <dM, M> + <dJ, J> with M = mu I: two terms whose difference is smaller by the size of I
                    x = x[-1:] if x.dim() > 1 else x / copies
                    dim = {"g": 0, "Ip": 0, "mu0": 1, "I0": 1}.get(n, 2)
                    for h in range(H):
                        err = hp.max_rel(x.select(dim, h), ref[n].select(dim, h))
                        bar = hp.CHUNK_FP32_GRAD_TOL if rows == torch.float32 else hp.BF16_GRAD_NORM_TOL
                        assert err <= bar, (what, size, var, copies, n, h, err)


@pytest.mark.parametrize("dk,dv", [(16, 16), (32, 64), (48, 48), (64, 64), (96, 80)])
@pytest.mark.parametrize("case", ["fp32", "fp32-var", "bf16", "bf16-var"])
@pytest.mark.parametrize("end", ["large", "small"])
def test_gradients_at_the_ends_of_the_range(gpu_device, dk, dv, case, end):
    """Strong decays inside a step (f = 2^-54.5), where what is divided by a decay is largest and what is multiplied by one
    least: gradients of the outputs of 2^90 stay finite, and with a precision of 2^60 gradients of 2^-32 keep their bits.  Head
    by head against the float64 recurrence; as a small pass, and repeated in the batch until its pieces run one after the other."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    rows, var = torch.float32 if case.startswith("fp32") else torch.bfloat16, case.endswith("var")
    H, T, many = 4, 64 * 3 + 21, 33                   # 4 tiles of 4 heads, or 528 of them
    inp = hp.rounded(po.make_inputs(1, T, H, dk, dv, seed=dk + dv), rows)
    inp["g"] = torch.full((H,), 0.6931472)            # f = 2^-gt
    inp["gt"] = 0.3 * torch.rand(1, T, H, generator=torch.Generator().manual_seed(1))
    inp["gt"][:, 97::8] = 54.5
    gen = torch.Generator().manual_seed(T)
    mu0 = 0.1 * torch.randn(1, H, dv, dk, generator=gen)
    if end == "small":
        inp["Ip"] = inp["Ip"] * 2.0 ** 60
    I0 = inp["Ip"].view(1, H, 1, 1) * (1 + torch.rand(1, H, dv, dk, generator=gen))
    size = 2.0 ** 90 if end == "large" else 2.0 ** -32
    do = (size * torch.randn(1, T, H, dv, generator=gen)).to(rows).float()
    dov = (size * torch.rand(1, T, H, dv, generator=gen)).to(rows).float() if var else None
    ref = hp.oracle_grads(inp, do, dov, mu0=mu0, I0=I0)
    for n_copies in (1, many):
        per_row = {n: x.to(gpu_device).repeat(n_copies, *[1] * (x.dim() - 1)) for n, x in inp.items() if x.dim() > 1}
        leaves = {n: per_row.get(n, inp[n].to(gpu_device)).clone().requires_grad_(True) for n in NAMES}
        states = [x.to(gpu_device).repeat(n_copies, 1, 1, 1) for x in (mu0, I0)]
        out = chunk_palimpsa(*[leaves[n] for n in NAMES], *states, output_uncertainty=var)
        grads = [x.to(rows).to(gpu_device).repeat(n_copies, 1, 1, 1) for x in ((do, dov) if var else (do,))]
        got = torch.autograd.grad(list(out) if var else [out], [leaves[n] for n in "qkvb"], grads)
        for n, x in zip("qkvb", got):
            assert bool(torch.isfinite(x).all()), (n_copies, n)
            for h in range(H):
                err = hp.max_rel(x[-1:, :, h], ref[n][:, :, h])
                assert err <= (hp.CHUNK_FP32_GRAD_TOL if rows == torch.float32 else hp.BF16_GRAD_NORM_TOL), (n_copies, n, h, err)
                if n == "b" and end == "small":
                    continue   # (in the strong steps do r mu k^2 itself is below fp32's range)
                err = hp.max_rel(x[-1:, 97:104, h], ref[n][:, 97:104, h])   # tokens of the strong steps by themselves
                assert err <= (hp.CHUNK_FP32_GRAD_TOL if rows == torch.float32 else hp.BF16_GRAD_NORM_TOL), (n_copies, n, h, err)


@pytest.mark.parametrize("few", [1, 5, 8, 10])
@pytest.mark.parametrize("dk,dv", [(16, 48), (32, 64), (48, 48), (64, 48), (64, 64)])
@pytest.mark.parametrize("rows", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_small_passes_of_heads_of_one_piece(gpu_device, dk, dv, rows, few):
    """A head that is one piece is cut into slices of 16 or 32 value rows where a pass has few tiles: the same rows as such a
    pass (24, 120, 192, 240 tiles of heads: either slice, on both sides of the lines) and as the first of 576, which are whole.
    Bars as above."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    H, many, T = 4, 24, 64 * 6 - 11
    inp = hp.to_device(hp.rounded(po.make_inputs(many, T, H, dk, dv, seed=dk * dv), rows), gpu_device)
    gen = torch.Generator(device=gpu_device).manual_seed(few)
    do, dov = (torch.randn(many, T, H, dv, generator=gen, device=gpu_device) for _ in range(2))
    for var in (False, True):
        got = []
        for B in (few, many):
            leaves = [(inp[n][:B] if inp[n].dim() > 1 else inp[n]).clone().requires_grad_(True) for n in NAMES]
            out = chunk_palimpsa(*leaves, output_uncertainty=var)
            out = list(out) if var else [out]
            got.append(torch.autograd.grad(out, leaves[:5], [g[:B].to(rows) for g in (do, dov)][:len(out)]))
        for n, x, y in zip(NAMES, *got):
            bar = 4 * 2.0 ** -17 if rows == torch.float32 else (4 if n == "gt" else 6) * 2.0 ** -9
            assert hp.max_rel(x, y[:few]) <= bar, (var, n, hp.max_rel(x, y[:few]))
