"""Weight-only int8 linear on MFMA: drop-in for the Triton path of MOSS-Image's
``training/quant_kernels.py`` (:100-228, ``triton_int8_linear_forward/backward``).

The GEMMs are hand-written gfx950 kernels in ``csrc/mo_gemm.hip`` (bf16 MFMA; the int8
weight decoded to bf16 in registers on its way into the MFMA): the strip kernels for calls with
few rows (``mo_int8_strip_forward`` / ``backward``), large tiles above them
(``mo_int8_linear_forward`` / ``backward``). From ``LIBRARY_ROWS`` rows or ``LIBRARY_WEIGHT``
weight elements up, a call above the strips whose reduction is not long against its output width
instead decodes the weight in one HIP pass (``mo_int8_decode``) and runs the same library GEMM as
the eager path, bit for bit equal to it and faster by the decode.

Backend selection mirrors the reference's ``auto | eager | triton``
with ``hip`` in place of ``triton``: ``auto`` takes the HIP kernels whenever the call is
supported (bf16 activations and weight dtype on a HIP device, int8 weights, fp32 scales,
feature sizes multiples of 16, contiguous operands) and the eager path otherwise; an explicit
``hip`` request that is not supported raises. The eager path is the reference's own eager
backend (decode the weight, then ``F.linear``), not a substitute for a missing library.

The reference's module interface for this path is kept under its own names, so that
``training/quantization.py`` runs unchanged on top of this module: ``validate_quantized_backend``,
``resolve_quantized_backend`` (``"triton"`` names the fused-kernel backend, here the HIP
kernels), ``autocast_compute_dtype``, ``triton_is_available``, ``triton_int8_linear_forward``
and ``triton_int8_linear_backward`` (reference ``quant_kernels.py:30-99, 294-374``). The HIP
kernels take bf16 activations and a bf16 weight dtype; the reference's Triton kernels also take
fp16 and fp32, which ``auto`` sends to the eager path here.
"""

from __future__ import annotations

import functools

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from . import _native

BACKENDS = {"auto", "eager", "hip", "triton"}  # "triton": the reference's name for "hip"


def unsupported_reason(tokens: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor,
                       weight_dtype: torch.dtype) -> str | None:
    """Why the HIP kernels cannot run this call (None when they can)."""

    if tokens.device.type != "cuda":
        return "the input is not on a HIP device"
    if weight.device != tokens.device or scale.device != tokens.device:
        return "the quantized weight and scale are not on the input device"
    if tokens.dtype != torch.bfloat16 or weight_dtype != torch.bfloat16:
        return f"only bf16 activations and weights are supported (got {tokens.dtype}, {weight_dtype})"
    if weight.dtype != torch.int8 or scale.dtype != torch.float32:
        return "weights must be int8 and scales float32"
    if weight.ndim != 2 or tokens.shape[-1] != weight.shape[1]:
        return "input and weight dimensions do not match"
    out_features, in_features = weight.shape
    if in_features % 16 or out_features % 16:
        return "feature sizes must be multiples of 16"
    if not weight.is_contiguous() or not scale.is_contiguous():
        return "weight and scale must be contiguous"
    if tokens.numel() == 0:
        return "empty input"
    return None


def resolve_backend(backend: str, tokens: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor,
                    weight_dtype: torch.dtype) -> str:
    """``auto`` -> ``hip`` or ``eager``; an explicit ``hip`` must be supported."""

    if backend not in BACKENDS:
        raise ValueError("quantized backend must be auto, eager or hip.")
    if backend == "triton":
        backend = "hip"
    if backend == "eager":
        return backend
    reason = unsupported_reason(tokens, weight, scale, weight_dtype)
    if backend == "auto":
        return "eager" if reason is not None else "hip"
    if reason is not None:
        raise RuntimeError(f"HIP int8 backend is unavailable: {reason}.")
    return backend


def decode(weight: torch.Tensor, scale: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """The decoded weight, bf16(q * bf16(scale)) for bf16 (reference quant_kernels.py:126-131)."""

    return weight.to(dtype) * scale.to(dtype)[:, None]


# Calls with few rows run the strip kernels (mo_int8_strip_*, reductions of whole steps of 64). The
# other paths pay for a decode of the whole weight (8 to 40 us), or for a grid of large tiles that
# does not fill the GPU. Measured on the 256 CUs of an MI355X (the rows hold for those; a partition
# keeps the tiles a CU, unmeasured), us, strip / fused / library:
#   rows                       320           700           1000          1450          2100          2693          4608
#   forward
#    3072 from 3072         15/28/31      25/31/32      30/35/36      41/48/46      43/54/49      54/78/55     82/102/71
#    3072 from 12288       36/109/61      62/68/92     81/85/100   117/112/134   149/150/275   205/295/307   308/413/258
#    16384 from 3072        37/46/58      73/81/84      92/85/98   134/144/145   201/197/230   252/233/329   396/389/442
#    24576 from 3072        56/76/85   108/117/147   136/139/161   209/213/219   288/282/298   367/370/396   599/589/608
#   input gradient
#    3072 from 3072         15/38/31      26/37/37      31/42/50      43/56/49      42/62/53      60/94/73     82/115/81
#    3072 from 24576      58/284/205   108/148/267   148/174/275   220/257/344   287/349/421   404/701/651   611/931/833
#    12288 from 3072        35/53/54      64/93/72      77/96/90   119/141/153   155/173/160   196/224/197   302/339/313
# - input gradients below STRIP_ROWS_BACKWARD rows, and below STRIP_LONG_ROWS where the reduction is
#   at least LONG_REDUCTION times the output width, for which the library's kernel is erratic (3072
#   from 24576, strip / library: 3569 rows 490/769, 3884 rows 542/525, 4784 rows 643/877, 5350 rows
#   694/645, 5477 rows 814/1216), unless the fused plan splits such a reduction and the 128 x 256
#   tiles no longer fit the CUs two at a time (5350 rows are 504, 5589 are 528 and take 831 against
#   750 of the fused kernels, 6090 rows 874/824; 5589 from 16384 559/514; 45 random calls past 512
#   tiles: fused 7 % faster on average, 5 % slower at worst);
# - forwards below STRIP_ROWS rows, and up to STRIP_ROWS_NARROW while their 128 x 256 tiles fill half
#   a round of the CUs but hardly more than one (past it a second round starts: 3300 rows of 3072 from 8192 take
#   175, the library 143; under half a round the large tiles split the reduction as well and the
#   two are within 10 %: 2047 rows of 1040 from 3072, 28 / 31 / 31). Long reductions that the fused
#   plan splits stay there from STRIP_LONG_ROWS_FORWARD rows (1700 rows of 3072 from 12288: 129 / 126).
STRIP_ROWS = 1536
STRIP_LONG_ROWS_FORWARD = 1280
STRIP_TILES, STRIP_ROWS_NARROW = (1 / 2, 33 / 32), 2816  # tiles a CU
STRIP_ROWS_BACKWARD = 2560
STRIP_LONG_ROWS = 6144
STRIP_LONG_TILES = 2  # a CU
# Any other call with at least LIBRARY_ROWS rows, or a weight of at least LIBRARY_WEIGHT elements,
# decodes the weight once (mo_int8_decode) and runs the library GEMM on it, unless its reduction is
# at least LONG_REDUCTION times its output width and the fused kernels' launch plan splits that
# reduction (rows that do not fill a round of large tiles): there the fused kernels run, as for any
# call left. Measured, library time / fused time (forward, input gradient):
#   rows:                4096       8192       17792
#   qkvo 3072x3072       0.89 0.75  0.91 0.89  0.86 0.90
#   up_gate 24576x3072   0.88 0.70  0.85 0.86  0.83 1.04
#   down 3072x12288      0.74 0.88  0.90 0.89  1.04 0.91
# The rule takes the fused kernels for up_gate's input gradient (24576-long reduction) and down's
# forward (12288) at 17792 rows, where the library's GEMM runs its weakest and the split reduction
# fills the GPU. On square and wide shapes the library's MFMA loop runs 10-15 % faster than the
# fused kernels' (which also decode each weight tile again for every row tile).
LIBRARY_ROWS = 2048
LIBRARY_WEIGHT = 16 << 20
LONG_REDUCTION = 4
# Input gradients left to the library decode the weight transposed (mo_int8_decode_transposed), so
# that its GEMM reads both operands along the reduction. Library on the weight as stored / transposed,
# decode included, us:
#   rows                  3400      4608      5700      6400      8192      11000     14000     17792
#   3072 from 3072       73/66     85/74   113/115   118/122   146/133   198/178   229/201   307/258
#   12288 from 3072    235/206   312/271   422/363   399/350   501/430   704/654   841/749  1103/945
# Not for reductions outside TRANSPOSED_REDUCTION (6200 rows of 3072 from 1040: 65/77; 5550 rows of
# 5552 from 18384: 1372/1613), nor below STRIP_ROWS_BACKWARD rows, where the decode is most of the call
# and writes its rows in shorter pieces (1246 rows of 13168 from 3536: 161/224, 14 rows of 8896 from
# 12112: 113/152), nor for outputs a power of two wide, where the library's kernel for it is erratic
# (8192 from 3072: 2800 rows 135/197, 4000 rows 169/150, 5700 rows 280/326), nor for long reductions
# (3072 from 24576: 7800 rows 1483/1536, 8192 rows 1044/923, 8600 rows 1409/1487). Of 125 random calls
# inside the range 8 are over 4 % slower (24 % at worst), the mean is 5 % faster.
TRANSPOSED_REDUCTION = (2048, 6144)
PATHS = ("auto", "fused", "library", "strip", "transposed")


def decode_hip(weight: torch.Tensor, scale: torch.Tensor, *, out: torch.Tensor | None = None) -> torch.Tensor:
    """``decode(weight, scale, bfloat16)`` in one HIP pass (``mo_int8_decode``), bit for bit."""

    lib = _native.load()
    _check_weight(weight, scale)
    out_features, in_features = weight.shape
    out = _output(out, (out_features, in_features), weight.device, "decoded-weight")
    _native.check("mo_int8_decode", lib.mo_int8_decode(weight.data_ptr(), scale.data_ptr(), out.data_ptr(),
                                                       out_features, in_features, _stream(weight)))
    return out


def decode_transposed_hip(weight: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
    """``decode(weight, scale, bfloat16).t()``, contiguous, in one HIP pass, bit for bit."""

    lib = _native.load()
    _check_weight(weight, scale)
    out_features, in_features = weight.shape
    out = torch.empty((in_features, out_features), dtype=torch.bfloat16, device=weight.device)
    _native.check("mo_int8_decode_transposed", lib.mo_int8_decode_transposed(
        weight.data_ptr(), scale.data_ptr(), out.data_ptr(), out_features, in_features, _stream(weight)))
    return out


def _matrix(tensor: torch.Tensor) -> torch.Tensor:
    # the two calls that change nothing on a matrix take as long on the host as all checks together
    if tensor.ndim == 2 and tensor.is_contiguous():
        return tensor
    return tensor.reshape(-1, tensor.shape[-1]).contiguous()


def _check_weight(weight: torch.Tensor, scale: torch.Tensor) -> None:
    """Every path hands the weight and its scales to a kernel by address: what they must be for that."""

    if weight.ndim != 2 or weight.dtype != torch.int8 or not weight.is_contiguous():
        raise RuntimeError("HIP int8 weight must be a contiguous int8 matrix.")
    if scale.dtype != torch.float32 or scale.numel() != weight.shape[0] or not scale.is_contiguous() \
            or scale.get_device() != weight.get_device():
        raise RuntimeError("HIP int8 scale must be contiguous float32 on the weight's device, one a row of the weight.")


def _misfit(matrix: torch.Tensor, weight: torch.Tensor, features: int, bias: torch.Tensor | None = None,
            outputs: int = 0) -> str | None:
    """Why the kernels that take the activations by address cannot read them (None when they can):
    they rely on the sizes they are given."""

    if matrix.dtype != torch.bfloat16 or matrix.get_device() != weight.get_device() or matrix.shape[1] != features:
        return f"expected bfloat16 rows of {features} on the weight's device"
    if bias is not None and (bias.numel() != outputs or bias.shape[-1:] != (outputs,)
                             or bias.get_device() != weight.get_device()):
        return f"expected a bias of {outputs} on the weight's device"
    return None


def _by_address(*operands: torch.Tensor | None) -> bool:
    """Whether a kernel that is given the operands' addresses does all that torch's product does with
    them: there is no graph or tangent to carry on, and nothing that traces, batches or watches the
    operators of the call."""

    if torch._C._functorch.peek_interpreter_stack() is not None or torch._C._len_torch_dispatch_stack() \
            or torch._C._get_tracing_state() is not None:
        return False
    graph, dual = torch.is_grad_enabled(), forward_ad._current_level >= 0
    for t in operands:
        if t is None:
            continue
        if type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter or graph and t.requires_grad:
            return False
        if dual and forward_ad.unpack_dual(t).tangent is not None:
            return False
    return True


def _autocast_dtype(tensor: torch.Tensor) -> torch.dtype:
    kind = tensor.device.type
    return torch.get_autocast_dtype(kind) if torch.is_autocast_enabled(kind) else torch.bfloat16


def _route(path: str, rows: int, weight: torch.Tensor, reduction: int, width: int, backward: bool,
           matrix: torch.Tensor, out: torch.Tensor | None, bias: torch.Tensor | None = None, *,
           misfit: str | None = None) -> str:
    """The path a call takes: ``strip``, ``library``, ``transposed`` or ``fused``. ``matrix``: the
    activations; ``out``: the output buffer (None: a new one). ``misfit``: ``_misfit``'s reason; such
    a call is left to torch's matrix product, which refuses it or, for a bias that broadcasts or a
    matrix that autocast converts, takes it. So is a call that is more than its bytes (see
    ``_by_address``), unless it names a buffer, which no graph can go through."""

    if path not in PATHS:
        raise ValueError(f"path must be one of {PATHS}")
    if path == "transposed" and not backward:
        raise ValueError("the transposed path is the input gradient's")
    if misfit and path in ("strip", "fused"):
        raise RuntimeError(f"HIP int8 operands do not fit: {misfit}.")
    if path != "auto":
        return path
    plain = not misfit and _by_address(matrix, out, bias)
    if misfit or not plain and out is None:
        return "library"
    if torch._C._is_any_autocast_enabled() and _autocast_dtype(matrix) != torch.bfloat16:
        plain = False  # torch's product returns autocast's type, the strips bfloat16
    long_reduction = reduction >= LONG_REDUCTION * width
    # What the strip kernels' and the transposed decode's argument checks refuse and the library path
    # takes (activations or outputs off the 16-byte grid, no rows, larger weights) stays with it. No
    # rows of a smaller weight stay with the fused kernels, which refuse them.
    fits = weight.numel() < 1 << 31 and all(size % 16 == 0 and size <= 1 << 20 for size in weight.shape)
    if (plain and rows and fits and reduction % 64 == 0 and matrix.data_ptr() % 16 == 0
            and (out is None or out.data_ptr() % 16 == 0)
            and _strips(rows, reduction, width, backward, long_reduction, _cus(matrix.get_device()))):
        return "strip"
    if rows < LIBRARY_ROWS and weight.numel() < LIBRARY_WEIGHT:
        return "fused"
    if rows == 0:
        return "library"
    if long_reduction and _splits(rows, width, reduction, backward):
        return "fused"
    if (backward and fits and rows >= STRIP_ROWS_BACKWARD and not long_reduction and width & (width - 1)
            and TRANSPOSED_REDUCTION[0] <= reduction <= TRANSPOSED_REDUCTION[1]):
        return "transposed"
    return "library"


@functools.lru_cache(maxsize=None)
def _cus(index: int) -> int:
    """CUs of a device (256 of an MI355X, fewer of a partition of it; off a HIP device as many)."""

    return torch.cuda.get_device_properties(index).multi_processor_count if index >= 0 else 256


def _strips(rows: int, reduction: int, width: int, backward: bool, long_reduction: bool, cus: int) -> bool:
    """Whether a call runs the strip kernels on a device of ``cus`` CUs (see ``STRIP_ROWS``)."""

    tiles = -(-rows // 128) * -(-width // 256) / cus
    if backward:
        if rows < STRIP_ROWS_BACKWARD or not long_reduction:
            return rows < STRIP_ROWS_BACKWARD
        return rows < STRIP_LONG_ROWS and (tiles <= STRIP_LONG_TILES or not _splits(rows, width, reduction, True))
    if long_reduction and rows >= STRIP_LONG_ROWS_FORWARD and _splits(rows, width, reduction, False):
        return False
    return rows < STRIP_ROWS or (rows <= STRIP_ROWS_NARROW and STRIP_TILES[0] <= tiles <= STRIP_TILES[1])


def _splits(rows: int, width: int, reduction: int, backward: bool) -> bool:
    """Whether the fused kernels' launch plan splits the call's reduction."""

    lib = _native.load()
    if not backward:
        return lib.mo_int8_forward_workspace_bytes(rows, reduction, width) > 0
    return lib.mo_int8_backward_workspace_bytes(rows, width, reduction) > (width * reduction + 255) // 256 * 256


def _stream(tensor: torch.Tensor) -> int:
    return torch.cuda.current_stream(tensor.device).cuda_stream


def _output(out: torch.Tensor | None, shape: tuple[int, int], device: torch.device, what: str) -> torch.Tensor:
    if out is None:
        return torch.empty(shape, dtype=torch.bfloat16, device=device)
    if out.dtype != torch.bfloat16 or not out.is_contiguous() or out.numel() != shape[0] * shape[1] \
            or out.device != device:
        raise ValueError(f"HIP {what} buffer has the wrong dtype, size or device, or is not contiguous.")
    return out.view(shape)


def _workspace(nbytes: int, device: torch.device) -> torch.Tensor | None:
    # fp32 partial sums of split reductions, the transposed weight of the fused input gradient: freed
    # to the caching allocator after the call; stream order keeps it alive for the kernels
    return torch.empty(nbytes, dtype=torch.uint8, device=device) if nbytes else None


def int8_linear_forward(tokens: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor,
                        bias: torch.Tensor | None = None, *, out: torch.Tensor | None = None,
                        path: str = "auto") -> torch.Tensor:
    """``tokens @ decode(weight).T (+ bias)``; the call must be supported. ``path``: ``strip`` (the
    MFMA kernels for few rows; ``in_features`` a multiple of 64), ``fused`` (the MFMA kernels on
    large tiles), ``library`` (``decode_hip``, then the same ``addmm``/``mm`` as the reference's
    eager path, bit for bit), ``auto`` (by rows and shape, see ``STRIP_ROWS`` and
    ``LIBRARY_ROWS``). The result of ``strip`` and ``fused`` has no graph; ``auto`` takes the library
    path where one is wanted."""

    lib = _native.load()
    _check_weight(weight, scale)
    matrix = _matrix(tokens)
    rows = matrix.shape[0]
    out_features, in_features = weight.shape
    if bias is not None:
        bias = bias.to(torch.bfloat16).contiguous()
    misfit = _misfit(matrix, weight, in_features, bias, out_features)
    route = _route(path, rows, weight, in_features, out_features, False, matrix, out, bias, misfit=misfit)
    if route == "library":
        decoded = decode_hip(weight, scale)
        if out is None:
            # the eager path's own call (F.linear): with an output buffer, PyTorch-ROCm picks
            # a different GEMM solution on some shapes, up to 15 % slower at qkvo's
            result = F.linear(matrix, decoded, bias)
        else:
            out = _output(out, (rows, out_features), tokens.device, "output")
            result = torch.mm(matrix, decoded.t(), out=out) if bias is None else \
                torch.addmm(bias, matrix, decoded.t(), out=out)
        return result.reshape(*tokens.shape[:-1], out_features)
    out = _output(out, (rows, out_features), tokens.device, "output")
    if route == "strip":
        name, call = "mo_int8_strip_forward", lib.mo_int8_strip_forward
        nbytes = lib.mo_int8_strip_workspace_bytes(rows, out_features, in_features)
    else:
        name, call = "mo_int8_linear_forward", lib.mo_int8_linear_forward
        nbytes = lib.mo_int8_forward_workspace_bytes(rows, in_features, out_features)
    workspace = _workspace(nbytes, tokens.device)
    _native.check(name, call(matrix.data_ptr(), weight.data_ptr(), scale.data_ptr(),
                             0 if bias is None else bias.data_ptr(), out.data_ptr(), rows, in_features, out_features,
                             0 if workspace is None else workspace.data_ptr(), nbytes, _stream(tokens)))
    return out.reshape(*tokens.shape[:-1], out_features)


def int8_linear_backward(gradient: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor,
                         input_shape: torch.Size, *, out: torch.Tensor | None = None,
                         path: str = "auto") -> torch.Tensor:
    """``gradient @ decode(weight)``: the input gradient of the frozen int8 linear (``path`` as in
    ``int8_linear_forward``; ``strip`` needs ``out_features`` a multiple of 64; ``transposed``: the
    library GEMM on ``decode_transposed_hip``'s weight)."""

    lib = _native.load()
    _check_weight(weight, scale)
    matrix = _matrix(gradient.to(torch.bfloat16))
    rows = matrix.shape[0]
    out_features, in_features = weight.shape
    route = _route(path, rows, weight, out_features, in_features, True, matrix, out,
                   misfit=_misfit(matrix, weight, out_features))
    if route == "transposed":
        decoded = decode_transposed_hip(weight, scale)
        if out is None:
            return F.linear(matrix, decoded).reshape(input_shape)
        out = _output(out, (rows, in_features), gradient.device, "input-gradient")
        torch.mm(matrix, decoded.t(), out=out)
        return out.reshape(input_shape)
    if route == "library":
        if out is None:  # the eager path's call (see int8_linear_forward)
            return matrix.matmul(decode_hip(weight, scale)).reshape(input_shape)
        out = _output(out, (rows, in_features), gradient.device, "input-gradient")
        torch.mm(matrix, decode_hip(weight, scale), out=out)
        return out.reshape(input_shape)
    out = _output(out, (rows, in_features), gradient.device, "input-gradient")
    if route == "strip":
        name, call = "mo_int8_strip_backward", lib.mo_int8_strip_backward
        nbytes = lib.mo_int8_strip_workspace_bytes(rows, in_features, out_features)
    else:
        name, call = "mo_int8_linear_backward", lib.mo_int8_linear_backward
        nbytes = lib.mo_int8_backward_workspace_bytes(rows, in_features, out_features)
    workspace = _workspace(nbytes, gradient.device)
    _native.check(name, call(matrix.data_ptr(), weight.data_ptr(), scale.data_ptr(), out.data_ptr(), rows, in_features,
                             out_features, 0 if workspace is None else workspace.data_ptr(), nbytes,
                             _stream(gradient)))
    return out.reshape(input_shape)


def launch_plan(rows: int, cols: int, reduction: int, cus: int, kernel: str = "registers") -> list[dict]:
    """The fused kernels' launches for a call with a workspace (``mo_int8_launch_plan``): ``cols``
    output columns (out_features for the forward, in_features for the input gradient) from a
    ``reduction`` (in_features, or out_features) on a device of ``cus`` CUs. Each part is
    ``{"tile": "large" | "small" | "split", "row0", "rows", "splits", "split_steps"}``."""

    import ctypes

    lib = _native.load()
    code = {"registers": _native.MO_INT8_KERNEL_REGISTERS, "lds": _native.MO_INT8_KERNEL_LDS}[kernel]
    n = ctypes.c_uint32(0)
    raw = (ctypes.c_uint32 * 10)()
    _native.check("mo_int8_launch_plan", lib.mo_int8_launch_plan(rows, cols, reduction, cus, code, ctypes.byref(n), raw))
    names = ("large", "small", "split")
    return [{"tile": names[raw[5 * i]], "row0": raw[5 * i + 1], "rows": raw[5 * i + 2], "splits": raw[5 * i + 3],
             "split_steps": raw[5 * i + 4]} for i in range(n.value)]


def strip_plan(rows: int, cols: int, reduction: int, cus: int, may_split: bool = True) -> dict:
    """The strip kernels' plan (``mo_int8_strip_plan``): ``{"rows", "cols"}`` of the output tile,
    ``"k_groups"`` of a workgroup, ``"splits"`` and ``"split_steps"`` of the reduction."""

    import ctypes

    raw = (ctypes.c_uint32 * 5)()
    _native.check("mo_int8_strip_plan", _native.load().mo_int8_strip_plan(rows, cols, reduction, cus, int(may_split),
                                                                          raw))
    return dict(zip(("rows", "cols", "k_groups", "splits", "split_steps"), raw))


def set_kernel(kernel: str) -> None:
    """Which kernel takes the large tiles of the fused path, process-wide: ``registers`` (default:
    weights decoded in registers, activations through LDS) or ``lds`` (the weight tile decoded
    into LDS). Same results bit for bit; for measuring one against the other."""

    code = {"registers": _native.MO_INT8_KERNEL_REGISTERS, "lds": _native.MO_INT8_KERNEL_LDS}[kernel]
    _native.check("mo_int8_set_kernel", _native.load().mo_int8_set_kernel(code))


# ---- the reference module's interface (training/quant_kernels.py), same names and meaning ----

def validate_quantized_backend(backend: str) -> str:
    """``auto``, ``eager`` or ``triton`` (reference ``quant_kernels.py:30-33``)."""

    if backend not in {"auto", "eager", "triton"}:
        raise ValueError("quantized backend must be auto, eager or triton.")
    return backend


def triton_is_available() -> bool:
    """Whether the fused-kernel backend can run: the HIP library loads and a HIP device is
    present (reference ``quant_kernels.py:36-38``, with the HIP kernels in place of Triton)."""

    if not torch.cuda.is_available():
        return False
    try:
        _native.load()
    except (OSError, RuntimeError):
        return False
    return True


def resolve_quantized_backend(backend: str, tokens: torch.Tensor, weight: torch.Tensor,
                              scale: torch.Tensor) -> str:
    """``auto`` -> ``triton`` when the fused kernels support the call, else ``eager``; an explicit
    ``triton`` must be supported (reference ``quant_kernels.py:64-79``). The weight dtype is
    the input's, as the reference's callers convert the input to it before the kernel."""

    selected = validate_quantized_backend(backend)
    if selected == "eager":
        return selected
    reason = unsupported_reason(tokens, weight, scale, tokens.dtype)
    if reason is None and not triton_is_available():
        reason = "the HIP library or device is unavailable"
    if selected == "auto":
        return "eager" if reason is not None else "triton"
    if reason is not None:
        raise RuntimeError(f"Triton quantized backend is unavailable: {reason}.")
    return selected


def autocast_compute_dtype(tokens: torch.Tensor, module_dtype: torch.dtype) -> torch.dtype:
    """The dtype autocast gives a linear on ``tokens`` (reference ``quant_kernels.py:82-96``)."""

    if tokens.device.type != "cuda" or not torch.is_autocast_enabled("cuda"):
        return module_dtype
    return torch.get_autocast_dtype("cuda")


def triton_int8_linear_forward(tokens: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor,
                               bias: torch.Tensor | None, output_dtype: torch.dtype, weight_dtype: torch.dtype,
                               *, out: torch.Tensor | None = None) -> torch.Tensor:
    """Reference ``quant_kernels.py:294-334`` on the HIP kernel: bf16 output and weight dtype."""

    if output_dtype != torch.bfloat16 or weight_dtype != torch.bfloat16:
        raise TypeError(f"HIP int8 kernels compute in bf16 (got output {output_dtype}, weight {weight_dtype}).")
    if bias is not None and (bias.device != tokens.device or not bias.is_contiguous()):
        raise RuntimeError("Triton quantized bias must be contiguous and on the input device.")
    return int8_linear_forward(tokens, weight, scale, bias, out=out)


def triton_int8_linear_backward(gradient: torch.Tensor, weight: torch.Tensor, scale: torch.Tensor,
                                input_shape: torch.Size, input_dtype: torch.dtype, weight_dtype: torch.dtype,
                                *, out: torch.Tensor | None = None) -> torch.Tensor:
    """Reference ``quant_kernels.py:337-373`` on the HIP kernel: the input gradient only."""

    if input_dtype != torch.bfloat16 or weight_dtype != torch.bfloat16:
        raise TypeError(f"HIP int8 kernels compute in bf16 (got input {input_dtype}, weight {weight_dtype}).")
    return int8_linear_backward(gradient.contiguous(), weight, scale, input_shape, out=out)

