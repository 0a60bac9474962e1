"""The chunked forward's output kernel at the edges of its layouts: column counts per lane (and padded columns), waves
per workgroup that divide the value rows unevenly, tile lengths around the staging step, one and two value rows per lane
(few and many tiles), uncertainty output; fp32 rows against the token-serial kernel at the fp32 bar."""
import pytest
import torch

from oracle import palimpsa_oracle as po
from tests import helpers as hp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("many", [False, True], ids=["one row per lane", "two rows per lane"])
@pytest.mark.parametrize("dk,dv", [(16, 256), (32, 96), (48, 80), (64, 112), (80, 80), (96, 16), (112, 48), (128, 144), (144, 32),
                                   (176, 64), (208, 16), (256, 48)])
def test_output_kernel_layouts(gpu_device, dk, dv, many):
    from palimpsa_amd.ops.palimpsa import chunk_palimpsa, fused_recurrent_palimpsa
    B, H = (24, 12) if many else (1, 2)
    for T, var in ((1, False), (9, True), (71, True)) if not many else ((73, False),):
        inp = po.make_inputs(B, T, H, dk, dv, seed=dk + dv + T)
        inp["g"] = torch.linspace(0.1, 6.0, H)
        d = hp.to_device(inp, gpu_device)
        args = [d[n] for n in ("q", "k", "v", "b", "gt", "g", "Ip")]
        out = [f(*args, output_uncertainty=var) for f in (chunk_palimpsa, fused_recurrent_palimpsa)]
        for x, ref in zip(*(o if var else (o,) for o in out)):
            assert torch.isfinite(x).all() and hp.max_rel(x, ref) <= hp.FP32_REL_TOL, (T, var)
