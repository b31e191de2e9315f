"""Tensor-argument checks shared by the operator entries.

Mirrors the checks the reference's TensorKernel applies before a launch
(src/runtime/torch.py:94-167): shape, dtype, device, contiguity and pairwise
disjointness of the external tensors. Launchers themselves never read tensor
values, as in the reference (docs/operators/sparse-mla.md:83-84).
"""

from __future__ import annotations

import ctypes as ct
import functools

import torch

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


_STORAGE_NAMES = {"bf16": "bf16", "f16": "f16", torch.bfloat16: "bf16", torch.float16: "f16"}


def storage_dtype(value) -> str:
    """Normalise a DTYPE constexpr ("bf16"/"f16", torch dtype or an object named so)."""
    if isinstance(value, (str, torch.dtype)) and value in _STORAGE_NAMES:
        return _STORAGE_NAMES[value]
    if isinstance(value, torch.dtype):
        for name, dt in DTYPES.items():
            if dt == value:
                return name
    name = str(getattr(value, "name", value)).lower().replace("torch.", "")
    aliases = {"bfloat16": "bf16", "float16": "f16", "half": "f16", "bf16": "bf16", "f16": "f16"}
    if name not in aliases:
        raise ValueError(f"unsupported storage dtype {value!r}; expected bf16 or f16")
    return aliases[name]


def require(condition: bool, message: str) -> None:
    if not condition:
        raise ValueError(message)


def check_tensor(name, tensor, shape, dtype, device=None):
    require(isinstance(tensor, torch.Tensor), f"{name} must be a torch.Tensor")
    require(tuple(tensor.shape) == tuple(shape), f"{name} shape {tuple(tensor.shape)} != {tuple(shape)}")
    require(tensor.dtype == dtype, f"{name} dtype {tensor.dtype} != {dtype}")
    require(tensor.is_cuda, f"{name} must live on a ROCm device")
    require(tensor.is_contiguous(), f"{name} must be contiguous")
    if device is not None:
        require(tensor.device == device, f"{name} is on {tensor.device}, expected {device}")


def _span(tensor):
    start = tensor.data_ptr()
    return start, start + tensor.numel() * tensor.element_size()


def check_disjoint(named):
    """Every written tensor must not overlap any other external tensor (read
    tensors may share memory with each other, as read-only caches do)."""
    spans = [(name, *_span(t), write) for name, t, write in named if t.numel()]
    for i, (a, a0, a1, aw) in enumerate(spans):
        if not aw:
            continue
        for j, (b, b0, b1, _) in enumerate(spans):
            if j != i and a0 < b1 and b0 < a1:
                first, second = (a, b) if i < j else (b, a)
                raise ValueError(f"external tensors {first} and {second} overlap")


class Operand:
    """Shape, dtype and bytes that a call of given sizes expects of one tensor."""

    __slots__ = ("name", "shape", "dtype", "nbytes")

    def __init__(self, name, shape, dtype):
        self.name = name
        self.shape = torch.Size(shape)
        self.dtype = dtype
        self.nbytes = self.shape.numel() * dtype.itemsize


def operand_pointers(operands, tensors, written):
    """(device index, data pointers) of a call's tensors after the checks of
    ``check_tensor`` and, for the operand at index ``written``, of
    ``check_disjoint``, each tensor looked at once (an eager call of a few
    microseconds on the GPU is otherwise bound by its checks); a failure is
    reported by those two."""
    device = tensors[0].get_device() if isinstance(tensors[0], torch.Tensor) and tensors[0].is_cuda else -1
    pointers = []
    for o, t in zip(operands, tensors):
        if (device < 0 or not isinstance(t, torch.Tensor) or t.dtype is not o.dtype or t.shape != o.shape
                or t.get_device() != device or not t.is_contiguous()):
            check_tensor(o.name, t, o.shape, o.dtype, tensors[0].device if pointers else None)
        pointers.append(t.data_ptr())
    start = pointers[written]
    end = start + operands[written].nbytes
    for i, p in enumerate(pointers):
        if p < end and start < p + operands[i].nbytes and i != written:
            check_disjoint([(o.name, t, i == written) for i, (o, t) in enumerate(zip(operands, tensors))])
    return device, pointers


_PLAIN = frozenset((bool, int, float, str, ct.CDLL))


def kept_by_value(build):
    """``build(*sizes)``, its last 64 results kept where every argument is a
    plain number or text (or the library), which nobody can change under the
    key; 1, 1.0 and True are different keys, since a float is refused where a
    count is due. Sizes that are not kept cost 3 us more (a decode loop whose
    cache grows by one each step: attention 10.9 -> 14.1 us of host time with its
    two launches, top-k 6.7 -> 9.5). Other number-likes (NumPy scalars and arrays, tensors), whose
    value may change or that have no hash, are built for each call."""
    kept = functools.lru_cache(maxsize=64, typed=True)(build)

    @functools.wraps(build)
    def plan(*sizes):
        return kept(*sizes) if _PLAIN.issuperset(map(type, sizes)) else build(*sizes)

    return plan


def raw_stream(device_index) -> int:
    """Handle of the current stream of a device."""
    return torch._C._cuda_getCurrentRawStream(device_index)


def stream_handle(device) -> int:
    return torch.cuda.current_stream(device).cuda_stream
