"""GPU: the drop-in operators give the same result, and are seen in the same way, whether or not the
call passes their autograd kernels: no gradient asked for, gradients, torch.func transforms, dispatch
modes, traces; attributes as arrays, lists and tensors."""
import numpy as np
import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from fanbeamctrecon_tensorflowop_amd import ops, workloads
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu

N, SIDE, VIEWS, COLS = 2, 24, 20, 40
CALLS = {"fp_fan_curve": (ops.fp_fan_curve, (N, SIDE, SIDE), (N, VIEWS, COLS)),
         "bp_fan_curve": (ops.bp_fan_curve, (N, VIEWS, COLS), (N, SIDE, SIDE)),
         "fbp_fan_curve": (ops.fbp_fan_curve, (N, VIEWS, COLS), (N, SIDE, SIDE)),
         "back_projection": (ops.BackProjection, (N, VIEWS, COLS), (N, SIDE, SIDE))}


@pytest.fixture(scope="module")
def scan():
    p, a = workloads.scan(nx=SIDE, rfov=12.0, sid=60.0, sdd=110.0, n_cols=COLS, dcol_rad=0.0125, n_views=VIEWS)
    p = np.array(p, dtype=np.float32)
    p[11] = N
    return p, np.asarray(a, dtype=np.float32)


def _fn(name, scan):
    f = CALLS[name][0]
    p, a = scan
    return lambda x: f(x, a, p, [N, SIDE, SIDE], [N, VIEWS, COLS])


@pytest.mark.parametrize("name", sorted(CALLS))
def test_routes(name, scan):
    f, shape = _fn(name, scan), CALLS[name][1]
    x = torch.rand(shape, device="cuda")
    y = f(x)
    assert not y.requires_grad and y.grad_fn is None
    xg = x.clone().requires_grad_(True)
    yg = f(xg)
    assert yg.requires_grad and torch.equal(yg.detach(), y)
    w = torch.rand_like(y)
    g, = torch.autograd.grad((yg * w).sum(), xg)
    with torch.no_grad():
        assert torch.equal(f(xg), y) and not f(xg).requires_grad
    with pytest.raises(RuntimeError):  # torch.func transforms are refused, not passed by
        torch.func.grad(lambda t: (f(t) * w).sum())(x)
    xh = x.clone().requires_grad_(True)
    (f(xh) * w).sum().backward()
    assert torch.equal(xh.grad, g)

    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Log():
        assert torch.equal(f(x), y)
    assert any(name in s for s in seen)
    traced = make_fx(f)(x)
    assert name in traced.code and torch.equal(traced(x), y)


def test_attributes(scan):
    p, a = scan
    x = torch.rand(CALLS["fp_fan_curve"][1], device="cuda")
    y = ops.fp_fan_curve(x, a, p, [N, SIDE, SIDE], [N, VIEWS, COLS])
    assert torch.equal(y, FanBeamPlan(p, a).fp(x))
    for aa, pp in ((a.tolist(), p.tolist()), (torch.from_numpy(a), torch.from_numpy(p)),
                   (a.astype(np.float64), p.astype(np.float64)), (tuple(a), tuple(p)), (a.reshape(1, -1), p)):
        assert torch.equal(ops.fp_fan_curve(x, aa, pp, (N, SIDE, SIDE), np.array([N, VIEWS, COLS])), y)
    with pytest.raises(ValueError):
        ops.fp_fan_curve(x.cpu(), a, p, [N, SIDE, SIDE], [N, VIEWS, COLS])
