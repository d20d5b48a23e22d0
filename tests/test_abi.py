"""The C-ABI library loads, exports every symbol include/helix_hip.h declares, and rejects bad
arguments on the host with the reference's TensorError variants — no GPU needed."""
import ctypes
import re
from pathlib import Path

import numpy as np
import pytest
import torch

from helixml_amd import _ffi

ROOT = Path(__file__).resolve().parent.parent
HEADER = ROOT / "include" / "helix_hip.h"


def declared_functions():
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(hx_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_expected_entry_points():
    names = declared_functions()
    for must in ("hx_selective_scan_fwd", "hx_selective_state_update", "hx_s4_ref_fwd",
                 "hx_s4d_complex_fwd", "hx_linear_f32", "hx_matmul_f32", "hx_init", "hx_malloc",
                 "hx_free", "hx_last_error"):
        assert must in names


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(str(_ffi.LIB_PATH))
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, f"declared but not exported: {missing}"


def test_binding_covers_header():
    assert set(declared_functions()) == set(_ffi.SIGNATURES)


def test_version():
    assert _ffi.lib().hx_version() >= 0x000100


@pytest.mark.parametrize("dstate", [0, 65])
def test_scan_rejects_dstate(dstate):
    rc = _ffi.lib().hx_selective_scan_fwd(1, 4, 4, dstate, 0, 1, *([None] * 11), None)
    assert rc == _ffi.UnsupportedOperation.status
    assert "dstate" in _ffi.last_error()
    with pytest.raises(_ffi.UnsupportedOperation):
        _ffi.check(rc)


def test_scan_rejects_dtype_and_negative_sizes():
    L = _ffi.lib()
    assert L.hx_selective_scan_fwd(1, 4, 4, 16, 7, 1, *([None] * 11), None) == _ffi.DTypeMismatch.status
    assert L.hx_selective_scan_fwd(-1, 4, 4, 16, 0, 1, *([None] * 11), None) == _ffi.InvalidDimension.status


def test_scan_empty_batch_is_noop():
    # batch == 0: nothing to do, no device call, OK
    assert _ffi.lib().hx_selective_scan_fwd(0, 4, 4, 16, 0, 1, *([None] * 11), None) == 0


def test_scan_null_pointers_rejected():
    rc = _ffi.lib().hx_selective_scan_fwd(1, 4, 4, 16, 0, 1, *([None] * 11), None)
    assert rc == _ffi.InvalidInput.status


@pytest.mark.parametrize("dtype,size", [(_ffi.HX_F32, 4), (_ffi.HX_BF16, 2)])
@pytest.mark.parametrize("dim", [1, 3, 7, 15, 17, 33])
def test_scan_paired_kernel_bounds_every_operand(dtype, size, dim):
    """The automatic scan kernel addresses the rows of u (dim wide) and of B and C (16 wide) with 32-bit byte
    offsets: it takes a size (and asks for a workspace, which no other kernel does for these dims) only while the
    wider of the two, 96 steps of read-ahead included, stays below 2^31 bytes."""
    first = -(-2 ** 31 // (max(dim, 16) * size)) - 96  # the first length past the bound
    size_of = lambda L: _ffi.lib().hx_selective_scan_workspace_size(1, L, dim, 16, dtype)  # noqa: E731
    assert size_of(first - 1) > 0 and size_of(first) == 0 and size_of(2 ** 28 + 1) == 0


@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="launches nothing only where there is no device")
@pytest.mark.parametrize("M,N,K", [(1999, 768, 1536), (777, 1024, 2048), (4096, 2048, 512)])
def test_gemm_without_its_lds_falls_through(M, N, K):
    """Where a device does not grant a kernel its LDS, the automatic choice goes on to one that needs none; it
    refuses no size for it. Without a device every grant fails, and so does the launch that is reached at last (the
    operands are never touched)."""
    p = 4096
    rc = _ffi.lib().hx_gemm_bf16(M, N, K, p, K, p, K, None, 0, _ffi.HX_BF16, p, N, N, None, 0, N, None, 0, None)
    assert rc == _ffi.BackendError.status, _ffi.last_error()


@pytest.mark.parametrize("dim,L,cut", [
    (128 * 64, 479, False), (128 * 64, 480, True), (96 * 64 - 3, 359, False), (96 * 64 - 3, 360, True), (1, 319, False), (1, 320, True),
    (191 * 64, 717, True), (192 * 64, 1023, False), (192 * 64 - 1, 1024, True), (256 * 64 - 1, 4096, False), (256 * 64, 1024, True)])
def test_s4d_segments_where_a_second_pass_pays(dim, L, cut):
    """Sequences whose end states leave nothing out (below 1024 steps, or dims that are no multiple of 4) are cut, which
    takes a workspace, only where the second pass is repaid: with tiles of 64 channels, from 15/4 steps a tile, none from
    192 below 1024 steps and from 256 at any length."""
    assert (_ffi.lib().hx_s4d_workspace_size(1, L, dim, 16) > 0) == cut


def test_s4_ref_rejects():
    L = _ffi.lib()
    assert L.hx_s4_ref_fwd(4, 0, 4, 0.1, *([None] * 7), None, 0, None) == _ffi.UnsupportedOperation.status
    assert L.hx_s4_ref_fwd(4, 16, 4, 0.1, *([None] * 7), None, 0, None) == _ffi.InvalidInput.status
    assert L.hx_s4_ref_fwd(0, 16, 4, 0.1, *([None] * 7), None, 0, None) == 0


def test_s4_discretize_is_the_reference_libm_formula():
    """hx_s4_discretize (host) = expf(f32(a_real*dt)) * cosf(f32(a_imag*dt)) in f32, as
    S4Block::discretize (crates/nn/src/ssm.rs:113-120) computes it; the oracle's restatement of
    the same function is pinned by the S4 reference-mode tests."""
    rng = np.random.default_rng(5)
    ar = rng.standard_normal(16).astype(np.float32)
    ai = rng.standard_normal(16).astype(np.float32) * np.float32(3)
    a = np.empty(16, np.float32)
    assert _ffi.lib().hx_s4_discretize(16, 0.1, ar.ctypes.data, ai.ctypes.data, a.ctypes.data) == 0
    tr = (ar * np.float32(0.1)).astype(np.float32)
    ti = (ai * np.float32(0.1)).astype(np.float32)
    ref = (np.exp(tr.astype(np.float64)) * np.cos(ti.astype(np.float64)))
    assert np.abs(a - ref).max() <= 2e-7 * np.abs(ref).max()
    # A_real = 0 (the reference's default init, ssm.rs:42): a = cos(dt * A_imag) exactly as f32 cosf
    ar0 = np.zeros(16, np.float32)
    assert _ffi.lib().hx_s4_discretize(16, 0.1, ar0.ctypes.data, ai.ctypes.data, a.ctypes.data) == 0
    assert np.abs(a - np.cos(ti.astype(np.float64))).max() <= 1.2e-7
    assert _ffi.lib().hx_s4_discretize(65, 0.1, None, None, None) == _ffi.UnsupportedOperation.status
    assert _ffi.lib().hx_s4_discretize(4, 0.1, None, None, None) == _ffi.InvalidInput.status


def test_workspace_sizes():
    L = _ffi.lib()
    # config 4 scan (batch 1, L 65536, d 2048): segmented, 16 segments x 3 x 32768 floats (end
    # states, entry states, decays)
    assert L.hx_selective_scan_workspace_size(1, 65536, 2048, 16, 0) == 16 * 3 * 2048 * 16 * 4
    # config 2 (batch 8, L 2048, d 1536) fills the GPU unsegmented: no workspace
    assert L.hx_selective_scan_workspace_size(8, 2048, 1536, 16, 0) == 0
    assert L.hx_selective_scan_workspace_size(1, 8192, 64, 7, 0) == 0  # generic kernel
    assert L.hx_s4_ref_workspace_size(64, 16, 100) >= (16 * 64 + 100 * 16) * 4
    assert L.hx_s4_ref_parallel_workspace_size(2048, 16, 65536) >= (2048 + 65536) * 16 * 4
    assert L.hx_s4d_workspace_size(1, 65536, 2048, 16) > 0
    assert L.hx_s4d_workspace_size(1, 100, 64, 8) == 0


def test_scan_ws_rejects_short_workspace():
    buf = (ctypes.c_uint8 * 64)()
    rc = _ffi.lib().hx_selective_scan_fwd_ws(1, 4, 4, 16, 0, 1, *([None] * 11), None, 64, None)
    assert rc == _ffi.InvalidInput.status  # NULL workspace with a size
    del buf


def test_linear_rejects_bad_act():
    assert _ffi.lib().hx_linear_f32(2, 2, 2, None, None, None, 5, None, None) == _ffi.InvalidInput.status


def test_set_scan_variant_validation():
    assert _ffi.lib().hx_set_scan_variant(3) == _ffi.InvalidInput.status
    assert _ffi.lib().hx_set_scan_variant(0) == 0


def test_error_mapping_covers_tensor_error_variants():
    # status codes mirror tensor_core::TensorError (crates/tensor-core/src/error.rs:7-37)
    assert {c.__name__ for c in _ffi._BY_STATUS.values()} == {
        "ShapeMismatch", "InvalidDimension", "DeviceMismatch", "DTypeMismatch",
        "UnsupportedOperation", "AllocationFailed", "BackendError", "SerializationError",
        "InvalidInput", "InvalidCheckpoint"}
