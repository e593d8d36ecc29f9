"""GPU: H*v of torch tensors follows the work that made its input and comes
before the work that reads its result, on torch's default stream and on
another, for each form of the standalone H*v."""
import numpy as np
import pytest
import torch

from nadvibs_amd import torch_ops
from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem

pytestmark = pytest.mark.gpu

# the step tables, the shaped form, the run-time compiled FP32 kernel (by default), the fast-block form
FORMS = {"steps": ("NV_HV_KERNEL", "steps"), "shaped": ("NV_HV_KERNEL", "generic"), "default": None,
         "fast-block": ("NV_HV_FB", "1")}


@pytest.mark.parametrize("own", [False, True], ids=["default stream", "own stream"])
@pytest.mark.parametrize("form", list(FORMS))
def test_hv_is_ordered_with_torch(form, own, monkeypatch):
    """Bits of the same H*v after a synchronisation."""
    for v in ("NV_HV_KERNEL", "NV_HV_FB"):
        monkeypatch.delenv(v, raising=False)
    if FORMS[form]:
        monkeypatch.setenv(*FORMS[form])
    p = make_problem(4, [3, 5, 4, 4, 4, 4], 2, (400, 2500), 200.0, 60.0, 40.0, seed=6)
    gen = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randn(2048, 2048, generator=gen, device="cuda")
    xs = [torch.randn(p.n, generator=gen, device="cuda", dtype=torch.float64) for _ in range(3)]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream() if own else torch.cuda.default_stream()
    with Engine(p) as eng:
        for prec in ("f64", "f32"):
            want = []
            for x in xs:
                want.append(torch_ops.hv(eng, x, prec))
                torch.cuda.synchronize()
            want = [w + 1.0 for w in want]
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                x = torch.zeros_like(xs[0])
                got = []
                for xi in xs * 4:
                    b = a
                    for _ in range(6):  # the input is late
                        b = b @ a
                    x.copy_(xi + 0.0 * b[0, 0].nan_to_num(0.0, 0.0, 0.0).double())
                    y = torch_ops.hv(eng, x, prec)
                    got.append(y + 1.0)
            torch.cuda.synchronize()
            for k, g in enumerate(got):
                assert torch.equal(g, want[k % 3]), (prec, k)
    assert np.isfinite(float(got[0][0]))
