"""The strip kernels (mo_int8_strip_forward / backward): every tile shape, tails, splits.

Each case is held to the fp64 product of the decoded weight within the bound of fp32 accumulation
plus the final bf16 rounding, in both directions. The sizes put a ragged edge everywhere one can
be: last row tiles of one to four 32-row tiles, output columns that end inside a column tile, K
groups of unequal or no steps, odd step counts, a last split shorter than the others.
``tests/test_cpu_int8_strip.py`` pins which shape the plan gives each case.
"""

from __future__ import annotations

import pytest
import torch

from moss_offload import _native, quant_kernels

from gpu_util import requires_gpu
from test_cpu_int8_strip import CASES
from test_gpu_int8_gemm import DEV, _operands, _within_accumulation_bound

pytestmark = requires_gpu


@pytest.mark.parametrize("rows,cols,reduction", [c[:3] for c in CASES])
@pytest.mark.parametrize("direction", ["forward", "bias", "backward"])
def test_strip_matches_fp64_reference(rows, cols, reduction, direction) -> None:
    if direction == "backward":
        x, w, scale, b = _operands(rows, reduction, cols, seed=rows + cols)
        w, scale = _operands(1, cols, reduction, seed=rows + 3 * cols)[1:3]  # [out = reduction][in = cols]
        got = quant_kernels.int8_linear_backward(x, w, scale, torch.Size((rows, cols)), path="strip")
        again = quant_kernels.int8_linear_backward(x, w, scale, torch.Size((rows, cols)), path="strip")
        decoded = quant_kernels.decode(w, scale, torch.bfloat16).double()
    else:
        x, w, scale, b = _operands(rows, reduction, cols, seed=rows + cols, bias=direction == "bias")
        got = quant_kernels.int8_linear_forward(x, w, scale, b, path="strip")
        again = quant_kernels.int8_linear_forward(x, w, scale, b, path="strip")
        decoded = quant_kernels.decode(w, scale, torch.bfloat16).double().t()
    assert got.shape == (rows, cols)
    assert torch.equal(got.view(torch.int16), again.view(torch.int16))
    exact = x.double() @ decoded
    if b is not None:
        exact = exact + b.double()
    _within_accumulation_bound(got, exact, x.double().abs() @ decoded.abs(), reduction)


@pytest.mark.parametrize("rows,features", [(128, 64), (3136, 3136), (1040, 448)])
def test_strip_reproduces_the_decoded_weight_bitwise(rows, features) -> None:
    """One-hot operands: each output is one product plus zeros, whatever the split."""

    eye = torch.eye(features, dtype=torch.bfloat16, device=DEV)
    _, w, scale, _ = _operands(1, features, rows, seed=rows)
    decoded = quant_kernels.decode(w, scale, torch.bfloat16)
    y = quant_kernels.int8_linear_forward(eye, w, scale, path="strip")
    assert torch.equal(y.view(torch.int16), decoded.t().contiguous().view(torch.int16))
    _, w, scale, _ = _operands(1, rows, features, seed=rows + 1)
    dx = quant_kernels.int8_linear_backward(eye, w, scale, torch.Size((features, rows)), path="strip")
    assert torch.equal(dx.view(torch.int16), quant_kernels.decode(w, scale, torch.bfloat16).view(torch.int16))


def test_unsplit_strip_adds_in_the_order_of_the_other_tiles() -> None:
    # 2047 x 4096 from 704: one K group, no split; the fused path runs the small tile
    x, w, scale, _ = _operands(2047, 704, 4096, seed=3)
    assert torch.equal(quant_kernels.int8_linear_forward(x, w, scale, path="strip").view(torch.int16),
                       quant_kernels.int8_linear_forward(x, w, scale, path="fused").view(torch.int16))
    _, w, scale, _ = _operands(1, 4096, 704, seed=4)
    shape = torch.Size((2047, 4096))
    assert torch.equal(quant_kernels.int8_linear_backward(x, w, scale, shape, path="strip").view(torch.int16),
                       quant_kernels.int8_linear_backward(x, w, scale, shape, path="fused").view(torch.int16))


@pytest.mark.parametrize("out_f,in_f", [(16, 16), (48, 80), (144, 272), (4112, 16), (3072, 1040)])
def test_transposed_decode_matches_the_decode_bitwise(out_f, in_f) -> None:
    _, w, scale, _ = _operands(1, in_f, out_f, seed=out_f + in_f)
    scale[::7] = -scale[::7]
    scale[::11] = 1.0 + 2.0**-8  # halfway between two bf16 values
    got = quant_kernels.decode_transposed_hip(w, scale)
    want = quant_kernels.decode(w, scale, torch.bfloat16).t().contiguous()
    assert got.shape == (in_f, out_f) and torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_input_gradients_above_the_strips_take_the_transposed_weight() -> None:
    rows, in_f, out_f = 4608, 1104, 2048
    _, w, scale, _ = _operands(1, in_f, out_f, seed=8)
    dy = _operands(rows, out_f, 16, seed=9)[0]
    shape = torch.Size((rows, in_f))
    got = quant_kernels.int8_linear_backward(dy, w, scale, shape)
    named = quant_kernels.int8_linear_backward(dy, w, scale, shape, path="transposed")
    assert torch.equal(got.view(torch.int16), named.view(torch.int16))
    buf = torch.empty(rows * in_f, dtype=torch.bfloat16, device=DEV)
    out = quant_kernels.int8_linear_backward(dy, w, scale, shape, out=buf)
    assert out.data_ptr() == buf.data_ptr()
    decoded = quant_kernels.decode(w, scale, torch.bfloat16).double()
    for y in (got, out):
        _within_accumulation_bound(y, dy.double() @ decoded, dy.double().abs() @ decoded.abs(), out_f)
    with pytest.raises(ValueError, match="input gradient"):
        quant_kernels.int8_linear_forward(dy, w.t().contiguous(), scale[:in_f], path="transposed")


def test_strip_refuses_what_it_cannot_run() -> None:
    x, w, scale, _ = _operands(64, 80, 64, seed=5)  # a reduction of 80
    with pytest.raises(_native.EngineError, match="multiples of 64"):
        quant_kernels.int8_linear_forward(x, w, scale, path="strip")
    lib = _native.load()
    x, w, scale, _ = _operands(33, 3072, 1040, seed=6)
    y = torch.empty(33, 1040, dtype=torch.bfloat16, device=DEV)
    need = lib.mo_int8_strip_workspace_bytes(33, 1040, 3072)
    assert need >= 2 * 33 * 1040 * 4
    work = torch.empty(need, dtype=torch.uint8, device=DEV)
    stream = torch.cuda.current_stream(DEV).cuda_stream
    rc = lib.mo_int8_strip_forward(x.data_ptr(), w.data_ptr(), scale.data_ptr(), 0, y.data_ptr(), 33, 3072, 1040,
                                   work.data_ptr(), need - 256, stream)
    assert rc == _native.MO_E_INVALID and b"workspace" in lib.mo_last_error()
    # no workspace: the same product without a split
    _native.check("mo_int8_strip_forward", lib.mo_int8_strip_forward(
        x.data_ptr(), w.data_ptr(), scale.data_ptr(), 0, y.data_ptr(), 33, 3072, 1040, 0, 0, stream))
    decoded = quant_kernels.decode(w, scale, torch.bfloat16).double().t()
    _within_accumulation_bound(y, x.double() @ decoded, x.double().abs() @ decoded.abs(), 3072)


def test_operands_off_the_grid_run_as_on_the_library_path() -> None:
    rows, out_f, in_f = 33, 6144, 3072
    x, w, scale, b = _operands(rows, in_f, out_f, seed=12, bias=True)
    dy = _operands(rows, out_f, 16, seed=13)[0]
    for backward, a, width in ((False, x, out_f), (True, dy, in_f)):
        off = torch.empty(a.numel() + 1, dtype=torch.bfloat16, device=DEV)[1:].view(a.shape)
        off.copy_(a)
        out = torch.empty(rows * width + 1, dtype=torch.bfloat16, device=DEV)[1:]
        decoded = quant_kernels.decode(w, scale, torch.bfloat16).double()
        decoded = decoded if backward else decoded.t()
        for matrix, buffer in ((off, None), (a, out)):
            def call(path):
                if backward:
                    return quant_kernels.int8_linear_backward(matrix, w, scale, torch.Size((rows, width)), out=buffer,
                                                              path=path)
                return quant_kernels.int8_linear_forward(matrix, w, scale, b, out=buffer, path=path)

            named = call("library").clone()
            got = call("auto")
            assert torch.equal(got.view(torch.int16), named.view(torch.int16))
            exact = a.double() @ decoded + (0 if backward else b.double())
            _within_accumulation_bound(got, exact, a.double().abs() @ decoded.abs(), a.shape[1])


@pytest.mark.parametrize("out_f,in_f", [(3072, 12288), (24576, 3072), (1024, 4096), (6144, 3072)])
def test_calls_without_rows(out_f, in_f) -> None:
    """Long and short reductions of either direction: the sizes are planned, small weights are refused."""

    lib = _native.load()
    assert lib.mo_int8_forward_workspace_bytes(0, in_f, out_f) == 0
    assert lib.mo_int8_backward_workspace_bytes(0, in_f, out_f) == out_f * in_f  # the transposed weight
    _, w, scale, _ = _operands(1, in_f, out_f, seed=14)
    x = torch.empty(0, in_f, dtype=torch.bfloat16, device=DEV)
    dy = torch.empty(0, out_f, dtype=torch.bfloat16, device=DEV)
    if w.numel() < quant_kernels.LIBRARY_WEIGHT:
        with pytest.raises(_native.EngineError):
            quant_kernels.int8_linear_forward(x, w, scale)
        with pytest.raises(_native.EngineError):
            quant_kernels.int8_linear_backward(dy, w, scale, x.shape)
    else:
        assert quant_kernels.int8_linear_forward(x, w, scale).shape == (0, out_f)
        assert quant_kernels.int8_linear_backward(dy, w, scale, x.shape).shape == (0, in_f)


@pytest.mark.parametrize("rows,cols,reduction", [c[:3] for c in CASES])
@pytest.mark.parametrize("direction", ["forward", "backward"])
def test_infinities_and_nans_stay_where_they_belong(rows, cols, reduction, direction) -> None:
    """Positive operands, so that an infinite factor gives infinities and no NaN: the zeros that the
    kernels multiply past a tile's edges, a K group's end and the last step must not meet it."""

    g = torch.Generator().manual_seed(rows + cols)
    x = (0.5 + torch.rand(rows, reduction, generator=g)).bfloat16().to(DEV)
    shape = (cols, reduction) if direction == "forward" else (reduction, cols)
    w = torch.randint(1, 128, shape, dtype=torch.int8, generator=g).to(DEV)
    scale = (0.001 + 0.01 * torch.rand(shape[0], generator=g)).to(DEV)

    def call(x, scale):
        if direction == "forward":
            return quant_kernels.int8_linear_forward(x, w, scale, path="strip")
        return quant_kernels.int8_linear_backward(x, w, scale, torch.Size((rows, cols)), path="strip")

    clean = call(x, scale)
    assert clean.isfinite().all()
    inf_row, nan_row = rows - 1, rows // 2
    special = x.clone()
    special[nan_row, reduction - 1] = float("nan")
    special[inf_row, 0] = float("inf")  # the only row of a call of one: the infinity
    if inf_row == nan_row:
        special[inf_row, reduction - 1] = 1.0
    got = call(special, scale)
    assert (got[inf_row] == float("inf")).all()
    assert inf_row == nan_row or got[nan_row].isnan().all()
    other = torch.ones(rows, dtype=torch.bool, device=DEV)
    other[[inf_row, nan_row]] = False
    assert torch.equal(got[other].view(torch.int16), clean[other].view(torch.int16))

    infinite = scale.clone()
    infinite[-1] = float("inf")
    got = call(x, infinite)
    if direction == "forward":  # one column; the others as they were
        assert (got[:, -1] == float("inf")).all()
        assert torch.equal(got[:, :-1].contiguous().view(torch.int16), clean[:, :-1].contiguous().view(torch.int16))
    else:
        assert (got == float("inf")).all()
