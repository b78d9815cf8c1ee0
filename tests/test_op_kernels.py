"""The drop-in operators' kernels are closed to Dynamo: called from a frame that Dynamo leaves to Python, an
op runs as one opaque call, as it does with the kernel that custom_op makes."""
import os
from typing import List

import pytest
import torch
import torch._dynamo

from fanbeamctrecon_tensorflowop_amd import torch_ops, workloads

P, A = ([float(v) for v in t] for t in workloads.small_scan())


def _graphs(op, x, *args):
    """The result of a call and the calls of the compiled graphs, where the caller's frame runs in Python."""
    graphs = []

    def backend(gm, example_inputs):
        graphs.append([str(n.target) for n in gm.graph.nodes if n.op.startswith("call")])
        return gm.forward

    def skipped(x):
        with open(os.devnull):  # Dynamo leaves this frame to Python and goes on with its callees
            return op(x, *args) * 2.0

    torch._dynamo.reset()
    f = torch.compile(skipped, backend=backend)
    y = f(x)
    assert torch.equal(f(x), y)
    torch._dynamo.reset()
    return y, graphs


@pytest.fixture(scope="module")
def lib():
    lib = torch.library.Library("fbct_kernel_test", "FRAGMENT")
    yield lib
    lib._destroy()


def _body(x: torch.Tensor, angle: List[float], parameter: List[float]) -> torch.Tensor:
    assert not torch.compiler.is_compiling()
    return x * float(torch_ops._plan(angle, parameter).n_views)


def test_kernel_is_opaque(lib):
    schema = "(Tensor x, float[] angle, float[] parameter) -> Tensor"
    lib.define("direct" + schema)
    lib.impl("direct", torch_ops._device_kernel(_body), "CPU")
    torch.library.custom_op("fbct_kernel_test::custom", mutates_args=())(_body)
    for name in ("direct", "custom"):
        torch.library.register_fake("fbct_kernel_test::" + name)(lambda x, angle, parameter: torch.empty_like(x))
    ops = torch.ops.fbct_kernel_test
    x = torch.ones(3)
    want, wrapped = _graphs(ops.custom, x, A, P)
    got, direct = _graphs(ops.direct, x, A, P)
    assert torch.equal(got, want) and torch.equal(want, torch.full((3,), 720.0))
    assert direct == wrapped == []


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["fp_fan_curve", "fbp_fan_curve"])
def test_device_kernels_are_opaque(name):
    _, shape_in, shape_out = {"fp_fan_curve": (0, [1, 256, 256], [1, 360, 512]),
                              "fbp_fan_curve": (0, [1, 360, 512], [1, 256, 256])}[name]
    op = getattr(torch.ops.fbct, name)
    x = torch.rand(shape_in, device="cuda")
    vol, proj = [1, 256, 256], [1, 360, 512]
    y, graphs = _graphs(op, x, A, P, vol, proj)
    assert torch.equal(y, op(x, A, P, vol, proj) * 2.0)
    assert not graphs, graphs  # nothing of the kernel
