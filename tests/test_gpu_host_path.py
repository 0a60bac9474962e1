"""The native host path of the eager calls against the Python route, which a call with a strided row tensor takes: the same
kernels on the same values, so results, states and gradients are equal bit for bit."""
import pytest
import torch

from oracle import palimpsa_oracle as po
from tests import helpers as hp

pytestmark = pytest.mark.gpu

NAMES = ("q", "k", "v", "b", "gt", "g", "Ip")


def _strided(x):
    return torch.cat([x, x], -1)[..., : x.shape[-1]]


def _taken(host, monkeypatch, name):
    """A list that grows by one entry per call of the extension's function: whether it served the call."""
    real, taken = getattr(host, name), []

    def call(*args):
        r = real(*args)
        taken.append(r is not None)
        return r

    monkeypatch.setattr(host, name, call)
    return taken


@pytest.mark.parametrize("rows", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("T,init,var,cu,bf16_gates", [(1, True, False, None, False), (70, False, True, None, True),
                                                      (150, True, True, [0, 17, 17, 150], False)])
def test_native_and_python_routes_agree(gpu_device, monkeypatch, rows, T, init, var, cu, bf16_gates):
    from palimpsa_amd import _lib as L
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa, fused_recurrent_palimpsa
    from palimpsa_amd.ops.simple_gla import fused_recurrent_simple_gla
    B, H, dk, dv = 1 if cu else 2, 4, 32, 48
    inp = hp.rounded(po.make_inputs(B, T, H, dk, dv, seed=T), rows)
    x = {n: inp[n].to(gpu_device) for n in NAMES}
    x["q"], x["k"] = x["q"][:, :, :2].contiguous(), x["k"][:, :, :2].contiguous()   # two heads share a q/k row
    if bf16_gates:
        x["gt"] = x["gt"].bfloat16()
    N = len(cu) - 1 if cu else B
    cu_t = None if cu is None else torch.tensor(cu, dtype=torch.int32, device=gpu_device)
    s = dict(initial_mu_state=torch.randn(N, H, dv, dk, device=gpu_device),
             initial_I_state=2 + torch.rand(N, H, dv, dk, device=gpu_device)) if init else {}
    host = L.host()

    def run(f, native, grad):
        y = {n: (t.clone().requires_grad_(grad)) for n, t in list(x.items()) + list(s.items())}
        args = [y[n] for n in NAMES]
        assert args[0].is_contiguous()
        if not native:
            args[0] = _strided(args[0])
            assert not args[0].is_contiguous()
        with torch.set_grad_enabled(grad):
            out = f(*args, **{n: y[n] for n in s}, output_final_state=True, output_uncertainty=var, cu_seqlens=cu_t)
        o = list(out[0]) if var else [out[0]]
        res = o + list(out[1:])
        if grad:
            res += torch.autograd.grad([z.float().square().sum() for z in o], list(y.values()))
        return res

    for f, grad in ((chunk_palimpsa, False), (chunk_palimpsa, True), (fused_recurrent_palimpsa, False)):
        if f is chunk_palimpsa or cu is None:   # (a packed token-serial call is not a plain one)
            taken = _taken(host, monkeypatch, "chunk_fwd" if f is chunk_palimpsa else "recurrent_fwd")
            run(f, True, grad)
            run(f, False, grad)
            assert taken == [True, False], (f.__name__, grad)
        for a, b in zip(run(f, True, grad), run(f, False, grad)):
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), (f.__name__, grad)
    if cu is None:
        g = -x["gt"].float()
        S = torch.randn(N, H, dk, dv, device=gpu_device) if init else None
        taken = _taken(host, monkeypatch, "gla_recurrent_fwd")
        a = fused_recurrent_simple_gla(x["q"], x["k"], x["v"], g, initial_state=S, output_final_state=True)
        b = fused_recurrent_simple_gla(_strided(x["q"]), x["k"], x["v"], g, initial_state=S, output_final_state=True)
        assert taken == [True, False]
        assert all(torch.equal(y, z) for y, z in zip(a, b))


def _plain_call(dev, T=3, H=2, dk=16, dv=16, grad=()):
    inp = po.make_inputs(1, T, H, dk, dv, seed=5)
    x = [inp[n].to(dev) for n in NAMES]
    for i in grad:
        x[i].requires_grad_(True)
    return x


@pytest.mark.parametrize("which", range(9), ids=list(NAMES) + ["mu0", "I0"])
@pytest.mark.parametrize("grad_mode", [False, True])
def test_forward_mode_stays_refused(gpu_device, which, grad_mode):
    """No operator has a forward-mode formula: a dual number is refused, with gradients on or off, and never comes back
    without its tangent."""
    import torch.autograd.forward_ad as fw
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa, fused_recurrent_palimpsa
    x = _plain_call(gpu_device)
    s = [torch.zeros(1, 2, 16, 16, device=gpu_device), torch.ones(1, 2, 16, 16, device=gpu_device)]
    for f in (chunk_palimpsa, fused_recurrent_palimpsa):
        with fw.dual_level(), torch.set_grad_enabled(grad_mode):
            y = x + s
            y[which] = fw.make_dual(y[which], torch.ones_like(y[which]))
            with pytest.raises(NotImplementedError):
                f(*y[:7], initial_mu_state=y[7], initial_I_state=y[8])


@pytest.mark.filterwarnings("ignore")
def test_traced_call_runs_the_kernels_again(gpu_device):
    """torch.jit.trace records the call as an operation that the trace repeats on its inputs, not the allocation of its
    outputs alone."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa, fused_recurrent_palimpsa
    x = _plain_call(gpu_device)
    with torch.no_grad():
        for f in (chunk_palimpsa, fused_recurrent_palimpsa):
            traced = torch.jit.trace(lambda q: f(q, *x[1:]), (x[0],), check_trace=False)
            for q in (x[0], 2.0 * x[0], x[0].flip(1).contiguous()):
                junk = torch.full_like(x[2], 1e6)   # what an unfilled output would be likely to hold
                del junk
                assert torch.equal(traced(q), f(q, *x[1:])), f.__name__


def test_transforms_and_dispatch_modes_take_the_python_route(gpu_device):
    from torch.utils._python_dispatch import TorchDispatchMode

    from palimpsa_amd import _lib as L
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    x = _plain_call(gpu_device)
    native = (*x, None, None, 1.0, False, 0, None, None, 1 << 30)
    assert L.host().chunk_fwd(*native) is not None

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert L.host().chunk_fwd(*native) is None
        assert chunk_palimpsa(*x).shape == x[2].shape
    with pytest.raises(RuntimeError):   # the Function has no vmap rule
        torch.vmap(lambda q: chunk_palimpsa(q, *x[1:]))(torch.stack([x[0]] * 2))
    with pytest.raises(RuntimeError):   # nor one for functorch's gradients
        torch.func.grad(lambda q: chunk_palimpsa(q, *x[1:]).sum())(x[0])


def test_library_codes_raise_what_the_python_route_raises(gpu_device):
    """A code of the library, forward or backward (there on a thread of the autograd engine): the same exception from both
    routes.  The library's functions are replaced by ones that return the code and launch nothing."""
    import ctypes as C

    from palimpsa_amd import _lib as L
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    host, lib = L.host(), L.load()
    addresses = {n: C.cast(getattr(lib, n), C.c_void_p).value for n in L._HOST_FUNCTIONS}
    fwd_t = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_void_p, C.c_void_p)
    bwd_t = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p)
    try:
        for code in (L.PAL_E_WORKSPACE, L.PAL_E_ALIGN, L.PAL_E_DIM, 700):
            with pytest.raises(Exception) as want:
                L.check(code, "pal_chunk_bwd")
            x = _plain_call(gpu_device, grad=range(7))
            host.bind([*(dict(addresses, pal_chunk_bwd=C.cast(f := bwd_t(lambda *a: code), C.c_void_p).value)).values()], L.check)
            out = chunk_palimpsa(*x)
            assert "ChunkNode" in out.grad_fn.name()
            with pytest.raises(Exception) as got:
                out.sum().backward()
            assert type(got.value) is type(want.value) and str(got.value) == str(want.value)
            assert getattr(got.value, "code", None) == getattr(want.value, "code", None)
            host.bind([*(dict(addresses, pal_chunk_fwd=C.cast(f := fwd_t(lambda *a: code), C.c_void_p).value)).values()], L.check)  # noqa: F841
            with pytest.raises(type(want.value)):
                chunk_palimpsa(*x)
    finally:
        host.bind([*addresses.values()], L.check)
    chunk_palimpsa(*x).sum().backward()


def test_saved_tensor_hooks(gpu_device):
    """What a hook hands back is what the backward uses, and nothing that the kernels would misread."""
    from torch.autograd.graph import save_on_cpu, saved_tensors_hooks

    from palimpsa_amd.ops.palimpsa import chunk_palimpsa

    def grads(hooks):
        x = _plain_call(gpu_device, T=150, grad=range(7))
        with hooks:
            out = chunk_palimpsa(*x, initial_mu_state=s[0], initial_I_state=s[1])
        assert "ChunkNode" in out.grad_fn.name()
        return torch.autograd.grad(out.square().sum(), x)

    s = [torch.zeros(1, 2, 16, 16, device=gpu_device), torch.ones(1, 2, 16, 16, device=gpu_device)]
    seen = []
    want = grads(saved_tensors_hooks(lambda t: seen.append(t.shape) or t, lambda t: t))
    assert (3, 2, 16, 16) in seen      # the states at the starts of the tiles among them
    assert all(torch.equal(a, b) for a, b in zip(grads(save_on_cpu()), want))
    for change in (lambda t: t.double(), lambda t: t[:1], lambda t: t.cpu(), lambda t: t.transpose(-1, -2)):
        with pytest.raises(ValueError):
            grads(saved_tensors_hooks(lambda t: t, lambda t: change(t) if t.shape == (3, 2, 16, 16) else t))


def test_calls_on_a_stream_of_their_own(gpu_device):
    """Kernels, outputs and workspaces of a call belong to the stream that is current for it, those of the backward to the
    forward's."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa, fused_recurrent_palimpsa
    x = _plain_call(gpu_device, T=150, grad=range(7))
    want = chunk_palimpsa(*x)
    want_g = torch.autograd.grad(want.square().sum(), x)
    with torch.no_grad():
        want_r = fused_recurrent_palimpsa(*x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            big = torch.randn(4096, 4096, device=gpu_device)
            big = big @ big                                   # keeps the stream busy ahead of the call
            y = [(t.detach() + 0 * big[0, 0]).requires_grad_(True) for t in x]   # ready on this stream only
            out = chunk_palimpsa(*y)
            got_g = torch.autograd.grad(out.square().sum(), y)
            with torch.no_grad():
                got_r = fused_recurrent_palimpsa(*y)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(out, want) and torch.equal(got_r, want_r)
    assert all(torch.equal(a, b) for a, b in zip(got_g, want_g))


@pytest.mark.parametrize("reentrant", [False, True])
def test_activation_checkpointing(gpu_device, reentrant):
    """torch.utils.checkpoint runs the forward again inside the backward and stops it by an exception from a hook."""
    from torch.utils.checkpoint import checkpoint

    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    x = _plain_call(gpu_device, T=150, grad=range(7))

    def f(*a):
        return chunk_palimpsa(*a).square()

    want = torch.autograd.grad(f(*x).sum(), x)
    y = checkpoint(f, *x, use_reentrant=reentrant)
    if reentrant:
        y.sum().backward()
        got = [t.grad for t in x]
    else:
        got = torch.autograd.grad(y.sum(), x)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    with torch.inference_mode():
        from palimpsa_amd import _lib as L
        assert L.host().chunk_fwd(*[t.detach() for t in x], None, None, 1.0, False, 0, None, None, 1 << 30) is not None


@pytest.mark.filterwarnings("ignore")
def test_call_traced_without_gradients_differentiates(gpu_device):
    """A short pass traced without gradients keeps no tile states; run with gradients, its backward fills them."""
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa
    x = _plain_call(gpu_device)
    with torch.no_grad():
        traced = torch.jit.trace(lambda *a: chunk_palimpsa(*a), tuple(x), check_trace=False)
    grads = []
    for f in (traced, chunk_palimpsa):
        leaves = [t.detach().clone().requires_grad_(True) for t in x]
        junk = torch.full((1 << 16,), 1e6, device=gpu_device)   # what unfilled states would be likely to hold
        del junk
        grads.append(torch.autograd.grad(f(*leaves).float().square().sum(), leaves))
    for a, r in zip(*grads):
        assert (a.float() - r.float()).abs().max() <= 5e-2 * r.float().abs().max()
