"""What ``int8_linear_forward`` and ``int8_linear_backward`` do before a kernel is given addresses.

The native library is replaced by one that notes the calls it gets, and the decodes by the eager
one, so that routing, refusals and the torch products of the library paths run on the CPU.
"""

from __future__ import annotations

import types

import pytest
import torch

from moss_offload import quant_kernels as qk

SIZES = {"small": (64, 128), "library": (16384, 1024)}  # out_features, in_features: below and above LIBRARY_WEIGHT


class _Library:
    """Notes the names of the calls; its workspace sizes are zero."""

    def __init__(self) -> None:
        self.names: list[str] = []

    def __getattr__(self, name):
        def call(*args):
            if "bytes" not in name:
                self.names.append(name)
            return 0

        return call


@pytest.fixture
def library(monkeypatch) -> _Library:
    lib = _Library()
    monkeypatch.setattr(qk, "_native", types.SimpleNamespace(load=lambda: lib, check=lambda name, rc: None))
    monkeypatch.setattr(qk, "_stream", lambda tensor: 0)

    def eager(weight, scale, out=None):
        return qk.decode(weight, scale, torch.bfloat16)

    monkeypatch.setattr(qk, "decode_hip", eager)
    monkeypatch.setattr(qk, "decode_transposed_hip", lambda weight, scale: eager(weight, scale).t().contiguous())
    return lib


def _operands(size: str, rows: int = 20):
    out_features, in_features = SIZES[size]
    g = torch.Generator().manual_seed(out_features + rows)
    weight = torch.randint(-127, 128, (out_features, in_features), dtype=torch.int8, generator=g)
    scale = 0.001 + 0.01 * torch.rand(out_features, generator=g)
    return (torch.randn(rows, in_features, generator=g).bfloat16(), torch.randn(rows, out_features, generator=g).bfloat16(),
            weight, scale)


@pytest.mark.parametrize("size", SIZES)
def test_calls_that_fit_reach_a_kernel_by_address(library, size) -> None:
    x, dy, w, s = _operands(size)
    qk.int8_linear_forward(x, w, s, torch.zeros(w.shape[0]))
    qk.int8_linear_forward(x, w, s[:, None], torch.zeros(1, w.shape[0]))
    qk.int8_linear_backward(dy, w, s, x.shape)
    assert library.names == ["mo_int8_strip_forward", "mo_int8_strip_forward", "mo_int8_strip_backward"]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("path", ["auto", "strip", "fused"])
@pytest.mark.parametrize("fault", ["float32", "wide", "bias", "scale", "scale dtype", "weight", "gradient"])
def test_operands_that_do_not_fit_raise_before_any_kernel(library, size, path, fault) -> None:
    x, dy, w, s = _operands(size)
    bias = None
    if fault == "float32":
        x = x.float()
    elif fault == "wide":
        x = torch.cat([x, x], 1)
    elif fault == "bias":
        bias = torch.zeros(16)
    elif fault == "scale":
        s = s[:16].clone()
    elif fault == "scale dtype":
        s = s.bfloat16()
    elif fault == "weight":
        w = w.t().contiguous().t()
    with pytest.raises(RuntimeError):
        if fault == "gradient":
            qk.int8_linear_backward(dy[:, 16:], w, s, x.shape, path=path)
        else:
            qk.int8_linear_forward(x, w, s, bias, path=path)
    assert library.names == []


@pytest.mark.parametrize("shape", [(), (1,), (20, 16384)])
def test_a_bias_that_broadcasts_is_added_by_torch(library, shape) -> None:
    x, _, w, s = _operands("library")
    bias = torch.randn(shape).bfloat16()
    got = qk.int8_linear_forward(x, w, s, bias)
    assert library.names == []
    want = torch.nn.functional.linear(x, qk.decode(w, s, torch.bfloat16), bias)
    assert torch.equal(got, want)


def test_the_reference_interface_refuses_activations_of_another_type(library) -> None:
    x, _, w, s = _operands("library")
    with pytest.raises(RuntimeError):
        qk.triton_int8_linear_forward(x.float(), w, s, None, torch.bfloat16, torch.bfloat16)
    assert library.names == []


@pytest.mark.parametrize("size", ["library", "long"])
@pytest.mark.parametrize("backward", [False, True])
def test_a_call_without_rows_asks_no_launch_plan(library, monkeypatch, size, backward) -> None:
    monkeypatch.setattr(qk, "_splits", lambda *args: pytest.fail("a plan of no tiles"))
    shape = (16384, 1024)
    if size == "long":  # the reduction at least four times the output width, in the call's direction
        shape = (16384, 1024) if backward else (1024, 16384)
    w, s = torch.zeros(shape, dtype=torch.int8), torch.ones(shape[0])
    if backward:
        got = qk.int8_linear_backward(torch.zeros(0, shape[0]).bfloat16(), w, s, torch.Size((0, shape[1])))
    else:
        got = qk.int8_linear_forward(torch.zeros(0, shape[1]).bfloat16(), w, s)
    assert got.shape == (0, shape[1] if backward else shape[0]) and library.names == []


def _call(backward, x, dy, w, s):
    if backward:
        return lambda t: qk.int8_linear_backward(t, w, s, t.shape[:-1] + (w.shape[1],)), dy
    return lambda t: qk.int8_linear_forward(t, w, s), x


@pytest.mark.parametrize("size,rows", [("library", 20), ("small", 20), ("small", 2100), ("small", 2700)])
@pytest.mark.parametrize("backward", [False, True])
def test_graphs_tangents_and_batches_go_through_the_product(library, size, backward, rows) -> None:
    """Reverse mode, forward mode and vmap give what the product of the decoded weight gives, at
    weights and rows of the strips' and of the library path."""

    x, dy, w, s = _operands(size, rows)
    call, t = _call(backward, x, dy, w, s)
    decoded = qk.decode(w, s, torch.bfloat16)
    linear = (lambda v: v @ decoded) if backward else (lambda v: v @ decoded.t())
    leaf, tangent = t.clone().requires_grad_(True), torch.ones_like(t)

    out = call(leaf)
    (got,) = torch.autograd.grad(out.float().sum(), leaf)
    other = t.clone().requires_grad_(True)
    (want,) = torch.autograd.grad(linear(other).float().sum(), other)
    assert torch.equal(got, want)
    with torch.autograd.forward_ad.dual_level():
        y = torch.autograd.forward_ad.unpack_dual(call(torch.autograd.forward_ad.make_dual(t, tangent))).tangent
    assert torch.equal(y, linear(tangent))
    assert torch.equal(torch.func.jvp(call, (t,), (tangent,))[1], linear(tangent))
    assert torch.equal(torch.func.grad(lambda v: call(v).float().sum())(t), want)
    assert torch.vmap(call)(torch.stack([t, tangent])).shape == (2, *linear(t).shape)
    assert library.names == []
    with torch.no_grad():  # nothing to carry on
        assert not call(leaf).requires_grad
    if rows == 20:
        assert len(library.names) == 1


def test_second_derivatives_go_through_the_frozen_linear(library, monkeypatch) -> None:
    from moss_offload import dit

    monkeypatch.setattr(qk, "unsupported_reason", lambda *args: None)
    x, _, w, s = _operands("library")
    module = dit.FrozenInt8Linear(w, s, torch.bfloat16, backend="hip")
    first = module(x)
    assert library.names == ["mo_int8_strip_forward"]
    t, seed = x.clone().requires_grad_(True), torch.ones_like(first).requires_grad_(True)
    (grad,) = torch.autograd.grad(module(t), t, seed, create_graph=True)
    (second,) = torch.autograd.grad(grad.float().sum(), seed)
    decoded = qk.decode(w, s, torch.bfloat16)
    assert torch.equal(second, torch.ones_like(x) @ decoded.t())


@pytest.mark.filterwarnings("ignore")  # torch.jit.trace is deprecated
def test_what_watches_the_operators_sees_the_product(library) -> None:
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    class Subclass(torch.Tensor):
        pass

    x, dy, w, s = _operands("library")
    for backward in (False, True):
        call, t = _call(backward, x, dy, w, s)
        with FlopCounterMode(display=False) as counter:
            call(t)
        assert counter.get_total_flops() == 2 * 20 * w.numel()
        assert "mm" in make_fx(call)(t).code
        assert ("aten::matmul" if backward else "aten::linear") in str(torch.jit.trace(call, t, check_trace=False).graph)
        assert type(call(t.as_subclass(Subclass))) is Subclass
    assert library.names == []


def test_autocast_to_another_type_keeps_its_result_type(library) -> None:
    x, dy, w, s = _operands("library")
    with torch.autocast("cpu", dtype=torch.float16):
        assert qk.int8_linear_forward(x, w, s).dtype == torch.float16
        assert qk.int8_linear_backward(dy, w, s, x.shape).dtype == torch.float16
    assert library.names == []
    with torch.autocast("cpu", dtype=torch.bfloat16):
        assert qk.int8_linear_forward(x, w, s).dtype == torch.bfloat16
    assert library.names == ["mo_int8_strip_forward"]


@pytest.mark.parametrize("rows,out_features,in_features,want", [
    (2559, 6160, 4096 + 16, "library"), (2560, 3088, 6160, "transposed"), (320, 6160, 3088, "library"),
    (2560, 2032, 12304, "library"), (2560, 2048, 12304, "transposed"), (2560, 6144, 3088, "transposed"),
    (2560, 6160, 3088, "library"), (2560, 3072, 8192, "library"), (2559, 3072, 3072, "strip"),
])
def test_input_gradients_on_the_transposed_weight(rows, out_features, in_features, want) -> None:
    """Only from the strips' rows on and for reductions it was measured at; reductions that are no
    multiple of 64 are not the strips' at any rows."""

    weight = torch.empty(out_features, in_features, dtype=torch.int8, device="meta")
    matrix = torch.empty(16, dtype=torch.bfloat16)
    assert qk._route("auto", rows, weight, out_features, in_features, True, matrix, None) == want


@pytest.mark.parametrize("rows,width,splits,want", [
    (5376, 3072, True, "strip"), (5377, 3072, True, "fused"), (5377, 3072, False, "strip"),
    (6143, 2560, True, "strip"), (2559, 8192, True, "strip"), (2560, 8192, True, "fused"),
    (6144, 3072, True, "fused"), (6144, 3072, False, "library"),
])
def test_long_input_gradients_leave_the_strips_to_a_split_plan(library, monkeypatch, rows, width, splits, want) -> None:
    monkeypatch.setattr(qk, "_splits", lambda *args: splits)
    weight = torch.empty(4 * width, width, dtype=torch.int8, device="meta")
    matrix = torch.empty(16, dtype=torch.bfloat16)
    assert qk._route("auto", rows, weight, 4 * width, width, True, matrix, None) == want


@pytest.mark.parametrize("cus", [32, 256])
def test_the_strips_tiles_are_counted_by_cu(monkeypatch, cus) -> None:
    """Forwards of 1600 rows (13 row tiles of 128) are strips from half a round of the CUs to hardly
    more than one, long input gradients whose plan splits up to two rounds."""

    monkeypatch.setattr(qk, "_splits", lambda *args: True)
    for columns in range(1, 30):  # of 256
        tiles = 13 * columns
        assert qk._strips(1600, 512, 256 * columns, False, False, cus) == (cus <= 2 * tiles and 32 * tiles <= 33 * cus)
    for columns in range(1, 30):
        assert qk._strips(2560, 1 << 20, 256 * columns, True, True, cus) == (20 * columns <= 2 * cus)


def test_a_named_buffer_ends_no_graph_silently(library) -> None:
    """With a buffer torch's product refuses operands that want a graph; the smaller weights' kernels
    write it, as a caller that names one asks for."""

    x, _, w, s = _operands("library")
    with pytest.raises(RuntimeError, match="out="):
        qk.int8_linear_forward(x.clone().requires_grad_(True), w, s, out=torch.empty(20, w.shape[0]).bfloat16())
    assert library.names == []
    x, _, w, s = _operands("small")
    qk.int8_linear_forward(x.clone().requires_grad_(True), w, s, out=torch.empty(20, w.shape[0]).bfloat16())
    assert library.names == ["mo_int8_linear_forward"]
