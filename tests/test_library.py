"""CPU checks of the product boundary: the C-ABI library builds for gfx950,
loads, and exports every entry point include/sandyrt_hip.h declares (no
compute calls -- there is no GPU here)."""
import ctypes
import os
import re

import pytest

from sandyrt_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "sandyrt_hip.h")).read()
    return sorted(set(re.findall(r"^\w[\w\s\*]*?\b(sandy_hip_\w+)\s*\(", text, re.M)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert "sandy_hip_paged_attention" in syms and "sandy_hip_norm" in syms
    assert len(syms) >= 15


def test_library_exports_every_declared_symbol():
    assert os.path.exists(_lib.LIB_PATH), "run sandyrt_amd.build.build() first"
    lib = ctypes.CDLL(_lib.LIB_PATH)
    missing = [s for s in declared_symbols() if not hasattr(lib, s)]
    assert not missing, f"not exported: {missing}"
    assert set(_lib.exported_symbols()) == set(declared_symbols())


def test_version_string():
    assert _lib.lib().sandy_hip_version().decode().startswith("sandyrt-hip")


def test_code_object_targets_gfx950():
    data = open(_lib.LIB_PATH, "rb").read()
    assert b"gfx950" in data


def test_paged_operand_checks_on_the_host():
    """sandy_hip_paged_to_dense / _stage reject descriptors the reference's
    pack_tensor_arg rejects (CudaKernelUtils.cuh:290-374) before any device
    work, so these run without a GPU."""
    import pytest

    def pt(**kw):
        s = _lib.SandyPagedTensor()
        s.pages, s.dtype, s.rank = 0x1000, _lib.F32, 3
        for i, d in enumerate([2, 3, 4]):
            s.dims[i] = d
        s.grow_dim, s.page_size, s.page_count = 1, 2, 2
        for k, v in kw.items():
            setattr(s, k, v)
        return ctypes.pointer(s)

    dst = _lib.SandyTensor()
    dst.rank, dst.dtype = 3, _lib.F32
    for i, (d, st) in enumerate([(2, 12), (3, 4), (4, 1)]):
        dst.dims[i], dst.strides[i] = d, st
    dst.data = 0x2000
    cases = [
        (pt(page_size=3), "page_size must be a power of two"),
        (pt(page_size=0), "page_size must be > 0"),
        (pt(grow_dim=3), "grow_dim out of range"),
        (pt(page_count=-1), "page_count must be >= 0"),
        (pt(pages=None), "page table is null"),
        (pt(dtype=_lib.U8), "unsupported dtype"),
    ]
    for p, msg in cases:
        with pytest.raises(_lib.SandyError, match=msg):
            _lib.call("sandy_hip_paged_to_dense", p, ctypes.byref(dst), stream=0)
    bad = _lib.SandyTensor.from_buffer_copy(dst)
    bad.dims[2] = 5
    with pytest.raises(_lib.SandyError, match="destination must be a contiguous tensor"):
        _lib.call("sandy_hip_paged_to_dense", pt(), ctypes.byref(bad), stream=0)
    with pytest.raises(_lib.SandyError, match="slot out of range"):
        _lib.call("sandy_hip_paged_stage", pt(), ctypes.c_int32(-1), ctypes.byref(dst), stream=0)


def test_packed_arguments():
    """Tensor and node arguments packed as bytes: the fields the C structs
    hold, for every rank and view, and nodes told apart by content (a node
    list changed in place, the sign of a zero constant)."""
    import torch

    from sandyrt_amd import _lib, ops

    base = torch.arange(2 * 3 * 4 * 5, dtype=torch.float32).view(2, 3, 4, 5)
    for t in (base, base[1:, :, 2:].permute(2, 0, 3, 1), base[1, 2, 3, 4], base.view(1, 1, 1, 1, 2, 3, 4, 5).bfloat16(),
              base[:0], torch.zeros(3, dtype=torch.int64)):
        d = _lib.desc(t).contents
        n = t.dim()
        assert (d.data or 0) == t.data_ptr() and d.storage_offset == 0
        assert d.dtype == _lib._TORCH_TO_CODE[t.dtype] and d.rank == n
        assert list(d.dims) == list(t.shape) + [0] * (8 - n) and list(d.strides) == list(t.stride()) + [0] * (8 - n)
    with pytest.raises(_lib.SandyError, match="rank 9"):
        _lib.desc(base.view(1, 1, 1, 1, 1, 2, 3, 4, 5))

    nodes = [ops.ScalarNode(0, ops.LOAD, 1), ops.ScalarNode(1, ops.CONST, constant=0.0),
             ops.ScalarNode(2, ops.MUL, operands=[0, 1])]
    first = [(n.id, n.op, n.dtype, n.input_index, n.constant, n.operand_count, list(n.operands)) for n in ops._nodes(nodes)]
    assert first == [(0, 0, 0, 1, 0.0, 0, [0, 0]), (1, 1, 0, 0, 0.0, 0, [0, 0]), (2, 4, 0, 0, 0.0, 2, [0, 1])]
    nodes[1].constant = -0.0
    assert str(ops._nodes(nodes)[1].constant) == "-0.0"
    nodes[1].constant = 3.5
    assert ops._nodes(nodes)[1].constant == 3.5


def test_node_constants_by_value():
    """A scalar node's constant is any object with a float value, taken at the
    call: booleans and zeros, numpy scalars, and a tensor changed in place
    between calls; an op past int32 wraps as a C field does (and is rejected)."""
    import numpy as np
    import torch

    from sandyrt_amd import ops

    def constant(v):
        return ops._nodes([ops.ScalarNode(0, ops.CONST, constant=v)])[0].constant

    for v, want in ((False, 0.0), (True, 1.0), (0, 0.0), (np.float32(0.0), 0.0), (np.float32(1.5), 1.5),
                    (np.array(2.5), 2.5), (torch.tensor(0.0), 0.0), (float("inf"), float("inf"))):
        assert constant(v) == want
    assert constant(float("nan")) != constant(float("nan"))
    t = torch.tensor(2.0)
    assert constant(t) == 2.0
    t.fill_(3.0)
    assert constant(t) == 3.0
    assert ops._nodes([ops.ScalarNode(0, 2 ** 31 + 5)])[0].op == 5 - 2 ** 31
    assert ops._nodes([ops.ScalarNode(0, -1)])[0].op == -1
