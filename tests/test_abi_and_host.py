"""C-ABI surface and host-side (Python) logic, runnable without a GPU: no kernel is launched."""
import ctypes as C
import os
import re
import subprocess
import sys
import warnings

import numpy as np
import pytest
import torch

import mojo_amd
from mojo_amd import QuantizationConfig, QuantizationEncoding as QE, _lib, build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "qmm.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(qmm_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = C.CDLL(_lib.LIB_PATH)
    names = declared_symbols()
    assert len(names) >= 11
    for name in names:
        assert hasattr(lib, name), f"{name} declared in include/qmm.h but not exported"
    assert set(names) == set(_lib.SIGNATURES), "ctypes signatures out of step with the header"


def test_block_params_and_errors_from_c():
    lib = _lib.load()
    assert lib.qmm_version() >= 100
    e, b = C.c_int64(), C.c_int64()
    for code, want in ((0, (32, 18)), (1, (256, 144)), (2, (256, 210)), (8, (32, 34))):
        assert lib.qmm_block_params(code, C.byref(e), C.byref(b)) == 0
        assert (e.value, b.value) == want
    assert lib.qmm_block_params(3, C.byref(e), C.byref(b)) == -1  # GPTQ has no fixed block
    assert b"no block layout" in lib.qmm_last_error()
    assert lib.qmm_block_params(0, None, None) == -1


def test_argument_validation_happens_before_any_launch():
    """Every invalid-argument status is produced on the host; pointers here are never dereferenced."""
    lib = _lib.load()
    fake = C.c_void_p(0x1000)
    rhs = (C.c_void_p * 1)(0x2000)

    def matmul(enc, m, k, n, cfg=None, n_rhs=1, lhs=fake, dt=0, ws=None, ws_bytes=0, rhs_arr=rhs):
        return lib.qmm_matmul(enc, cfg, lhs, dt, m, k, rhs_arr, n_rhs, n, fake, ws, ws_bytes, 0, None)

    assert matmul(1, 1, 4100, 8) == -1 and b"multiple of the block size" in lib.qmm_last_error()
    # the reserved bf16-weights mode has no kernel: refused, never silently ignored
    assert lib.qmm_matmul(1, None, fake, 0, 1, 4096, rhs, 1, 8, fake, None, 0, _lib.QMM_FLAG_W_BF16, None) == -2
    assert b"W_BF16" in lib.qmm_last_error()
    assert matmul(1, 0, 4096, 8) == -1 and b"positive" in lib.qmm_last_error()
    assert matmul(1, 1, 4096, 8, lhs=None) == -1
    assert matmul(7, 1, 4096, 8) == -1 and b"unknown encoding" in lib.qmm_last_error()
    assert matmul(1, 1, 4096, 8, dt=2) == -1  # fp16 lhs is not part of the contract
    assert matmul(1, 1, 4096, 8, n_rhs=2) == -1
    assert matmul(1, 1, 4096, 8, lhs=C.c_void_p(0x1004)) == -1 and b"aligned" in lib.qmm_last_error()
    assert matmul(1, 1, 4096, 8, rhs_arr=(C.c_void_p * 1)(0x2008)) == -1  # Q4_K blocks need 16-byte alignment
    assert matmul(0, 2, 4096, 8) == -4 and b"workspace" in lib.qmm_last_error()  # Q4_0 needs its Q8_0 planes
    assert matmul(3, 1, 4096, 8) == -1 and b"GPTQ" in lib.qmm_last_error()
    bad = _lib.GptqConfig(8, 128, 0, 1)
    rhs3 = (C.c_void_p * 3)(0x2000, 0x3000, 0x4000)
    assert matmul(3, 1, 4096, 8, cfg=C.byref(bad), n_rhs=3, rhs_arr=rhs3) == -2
    assert matmul(3, 1, 4096, 8, cfg=C.byref(_lib.GptqConfig(4, 128, 1, 1)), n_rhs=3, rhs_arr=rhs3) == -1  # desc_act without g_idx
    assert b"g_idx" in lib.qmm_last_error()
    assert lib.qmm_quantize_gptq(C.byref(_lib.GptqConfig(4, 128, 1, 1)), fake, 8, 256, fake, fake, fake, fake, None) == -2  # desc_act
    assert lib.qmm_dequantize_gptq(C.byref(_lib.GptqConfig(4, 128, 1, 1)), fake, fake, fake, None, 8, 256, fake, 0, None) == -1
    assert lib.qmm_quantize_gptq(C.byref(_lib.GptqConfig(4, 128, 0, 0)), fake, 8, 256, fake, fake, fake, fake, None) == -2  # sym=False
    assert matmul(3, 1, 4096, 8, cfg=C.byref(_lib.GptqConfig(4, 100, 0, 1)), n_rhs=3, rhs_arr=rhs3) == -1
    assert lib.qmm_dequantize(1, fake, 4, 100, fake, 0, None) == -1
    assert lib.qmm_dequantize(8, fake, 4, 256, fake, 0, None) == -1
    assert lib.qmm_quantize(1, fake, 0, 256, fake, None) == -1
    assert lib.qmm_matmul_workspace_bytes(0, 0, 16, 4096, 4096) == 16 * 4096 + 2 * 16 * 128 * 4
    assert lib.qmm_matmul_workspace_bytes(1, 0, 2, 4096, 4096) == 0  # Q4_K decode reads the lhs as it is
    assert lib.qmm_matmul_workspace_bytes(1, 0, 8, 4096, 4096) == 0  # up to 8 rows the kernel narrows the lhs itself
    assert lib.qmm_matmul_workspace_bytes(1, 0, 12, 4096, 4096) >= 2 * 12 * 4096 * 2  # fp16 hi and residual planes
    assert lib.qmm_matmul_workspace_bytes(1, 1, 2048, 14336, 4096) >= 2048 * 4096 * 2
    # one-row decode of the K-quants needs none on any projection shape; a few rows on a long K hold the partial results of
    # the parts of K that lie side by side in the grid (Q4_K: four groups of 4096 columns; Q6_K: four rounds)
    for enc in (1, 2, 4):
        for n, k in ((4096, 4096), (14336, 4096), (4096, 14336), (128256, 4096)):
            assert lib.qmm_matmul_workspace_bytes(enc, 0, 1, n, k) == 0, (enc, n, k)
    assert lib.qmm_matmul_workspace_bytes(1, 0, 4, 4096, 14336) == 4 * 4 * 4096 * 4
    assert lib.qmm_matmul_workspace_bytes(2, 0, 4, 4096, 14336) == 4 * 4 * 4096 * 4
    # flags that change the workspace: a bf16 result that the kernel does not store itself goes through an fp32 copy; Q8_K
    # activations outside the integer kernel go through fp32 rows of d8 * code
    f = lib.qmm_matmul_workspace_bytes_flags
    assert f(1, 0, 1, 4096, 4096, _lib.QMM_FLAG_OUT_BF16) == 0                      # Q4_K decode stores bf16 itself
    assert f(2, 0, 1, 4096, 4096, _lib.QMM_FLAG_OUT_BF16) == 4096 * 4               # Q6_K decode: fp32 result in the workspace
    assert f(1, 0, 4, 4096, 4096, _lib.QMM_FLAG_ACT_Q8K) == 0                       # the integer kernel
    assert 4 * 4096 < f(2, 0, 4, 4096, 4096, _lib.QMM_FLAG_ACT_Q8K) < 4 * 4096 * 2  # Q6_K, few rows: Q8_K codes, scales and sums
    assert f(2, 0, 40, 4096, 4096, _lib.QMM_FLAG_ACT_Q8K) >= 40 * 4096 * 4          # Q6_K, many rows: round-tripped fp32 rows
    assert f(1, 0, 2048, 14336, 4096, 0) == lib.qmm_matmul_workspace_bytes(1, 0, 2048, 14336, 4096)
    # Q5_K / Q6_K prefill: lhs planes and weight planes (2 bytes per weight and plane; Q6_K has two)
    assert lib.qmm_matmul_workspace_bytes(2, 1, 2048, 14336, 4096) >= 2 * 14336 * 4096 * 2
    assert lib.qmm_matmul_workspace_bytes(4, 1, 2048, 14336, 4096) >= 14336 * 4096 * 2
    assert lib.qmm_matmul_workspace_bytes(0, 1, 2048, 14336, 4096) >= 14336 * 4096 * 2 + 2048 * 4096 * 2  # Q4_0: plane + lhs codes
    # bf16 output without the workspace it needs, Q8_K activations for an encoding that has none
    assert lib.qmm_matmul(2, None, fake, 0, 1, 4096, rhs, 1, 8, fake, None, 0, _lib.QMM_FLAG_OUT_BF16, None) == -4
    assert b"bf16" in lib.qmm_last_error()
    ws = C.c_void_p(0x100000)
    assert lib.qmm_matmul(0, None, fake, 0, 1, 4096, rhs, 1, 8, fake, ws, 1 << 30, _lib.QMM_FLAG_ACT_Q8K, None) == -2
    assert lib.qmm_matmul(1, None, fake, 0, 1, 4096, rhs, 1, 8, fake, None, 0, 8, None) == -1 and b"flag" in lib.qmm_last_error()
    # Q8_K activations and a bf16 result together: a workspace of exactly the quoted size passes the size check of the outer and
    # of the inner call (encodings 4, 2, 1 = Q5_K, Q6_K, Q4_K at 8 rows go through the fp32 round trip of the lhs); one byte less
    # is refused.  K = 100 makes a call that got past the size checks fail on the block size instead of reaching a launch.
    both = _lib.QMM_FLAG_ACT_Q8K | _lib.QMM_FLAG_OUT_BF16
    for enc in (4, 2, 1):
        for rows in (8, 40):  # the integer kernels (passes of four rows); the fp32 round trip of the lhs
            need = f(enc, 0, rows, 512, 4096, both)
            assert need >= rows * 512 * 4 + (rows * 4096 * 4 if rows > 16 else 0)
            assert lib.qmm_matmul(enc, None, fake, 0, rows, 4096, rhs, 1, 512, fake, ws, need - 1, both, None) == -4
            assert lib.qmm_matmul(enc, None, fake, 0, rows, 100, rhs, 1, 512, fake, ws, max(f(enc, 0, rows, 512, 100, both), 1 << 20), both, None) == -1
            assert b"block size" in lib.qmm_last_error()
    # the normalisation prologue
    g = C.c_void_p(0x3000)
    rn = lib.qmm_matmul_rmsnorm
    assert rn(0, None, fake, 0, None, 1e-5, 1, 4096, rhs, 1, 8, fake, None, 0, 0, None) == -1               # no gamma
    assert rn(0, None, fake, 0, g, -1.0, 1, 4096, rhs, 1, 8, fake, None, 0, 0, None) == -1 and b"eps" in lib.qmm_last_error()
    assert rn(0, None, fake, 2, g, 1e-5, 1, 4096, rhs, 1, 8, fake, None, 0, 0, None) == -1                  # fp16 x
    assert rn(1, None, fake, 0, g, 1e-5, 1, 4096, rhs, 1, 8, fake, None, 0, 0, None) == -4                  # Q4_K: needs room for the normalised rows
    assert lib.qmm_matmul_rmsnorm_workspace_bytes(1, 0, 1, 8, 4096, 0) == 4096 * 4
    assert lib.qmm_matmul_rmsnorm_workspace_bytes(1, 1, 3, 8, 4096, 0) == 3 * 4096 * 2


def test_workspace_figures_of_the_optional_weight_planes():
    """Host arithmetic only.  Large Q4_K / GPTQ prefill problems (more than 512 lhs rows, 160 or more tiles of 256 x 256)
    are quoted with room for fp16 weight planes, 2 bytes per weight; the same matrices with fewer rows, and small matrices,
    are quoted for the kernels that unpack as they go (lhs planes only).  Q5_K / Q6_K always need their planes beyond 64
    rows (Q6_K two of them; Q5_K from 33 rows where K is no multiple of 512).  Planes kept across calls: the buffer holds
    them with both forms of the Q4_K / Q5_K min operands, and a call's workspace then only the lhs."""
    lib = _lib.load()
    n, k = 14336, 4096
    bf16 = _lib.QMM_BF16
    for enc in (QE.Q4_K, QE.GPTQ):
        big = lib.qmm_matmul_workspace_bytes(enc.code, bf16, 2048, n, k)
        mid = lib.qmm_matmul_workspace_bytes(enc.code, bf16, 512, n, k)
        small_matrix = lib.qmm_matmul_workspace_bytes(enc.code, bf16, 2048, 2048, k)  # 8 x 8 tiles
        assert big >= 2 * n * k + 2048 * k * 2, enc
        assert mid < 32 << 20 and small_matrix < 64 << 20, enc
    assert lib.qmm_matmul_workspace_bytes(QE.Q5_K.code, bf16, 65, n, k) >= 2 * n * k
    assert lib.qmm_matmul_workspace_bytes(QE.Q5_K.code, bf16, 40, n, k) == 0
    assert lib.qmm_matmul_workspace_bytes(QE.Q5_K.code, bf16, 40, n, 4096 + 256) >= 2 * n * (4096 + 256)
    assert lib.qmm_matmul_workspace_bytes(QE.Q6_K.code, bf16, 70, n, k) >= 4 * n * k
    assert lib.qmm_matmul_workspace_bytes(QE.Q6_K.code, bf16, 64, n, k) == 0
    for enc, per_weight in ((QE.Q4_K, 2), (QE.Q5_K, 2), (QE.Q6_K, 4)):
        held = lib.qmm_repack_bytes(enc.code, None, n, k)
        assert per_weight * n * k * (1.125 if per_weight == 2 else 1) <= held < per_weight * n * k * 1.2, enc  # (one extension block per eight)
        ws = lib.qmm_matmul_repacked_workspace_bytes(enc.code, bf16, 2048, n, k)
        assert 2048 * k * 2 <= ws < 2048 * k * 2 * 1.2 + (1 << 20), enc
    cfg = _lib.GptqConfig(4, 128, 0, 1)
    assert 2 * n * k <= lib.qmm_repack_bytes(QE.GPTQ.code, C.byref(cfg), n, k) < 2.1 * n * k
    assert lib.qmm_repack_bytes(QE.GPTQ.code, C.byref(_lib.GptqConfig(4, 64, 0, 1)), n, k) == 0      # groups of 64: no plane GEMM
    assert lib.qmm_repack_bytes(QE.GPTQ.code, C.byref(_lib.GptqConfig(4, 128, 1, 1)), n, k) == 0     # act-order
    assert 2 * n * k <= lib.qmm_repack_bytes(QE.Q4_0.code, None, n, k) < 2.1 * n * k
    assert lib.qmm_repack_bytes(QE.Q8_0.code, None, n, k) == 0 and lib.qmm_repack_bytes(QE.Q4_K.code, None, n, 4096 + 32) == 0
    fake = C.c_void_p(0x1000)
    assert lib.qmm_repack(QE.Q8_0.code, None, (C.c_void_p * 1)(0x1000), 1, n, k, fake, 1 << 40, None) == -2
    assert lib.qmm_repack(QE.Q4_K.code, None, (C.c_void_p * 1)(0x1000), 1, n, k, fake, 16, None) == -4
    assert lib.qmm_matmul_repacked(QE.Q4_K.code, None, fake, bf16, 2048, k, None, 0, fake, 1 << 40, n, fake, None, 0, 1, None) == -2  # flags
    assert lib.qmm_matmul_repacked(QE.Q4_K.code, None, fake, bf16, 2048, k, None, 0, fake, 16, n, fake, None, 0, 0, None) == -1      # buffer too small
    assert lib.qmm_matmul_repacked(QE.Q4_K.code, None, fake, bf16, 2048, k, None, 0, C.c_void_p(0x1000), 1 << 40, n, fake, None, 0, 0, None) == -4  # no workspace


def test_quantization_encoding_metadata():
    assert QE.Q4_0.block_parameters == mojo_amd.BlockParameters(32, 18)
    assert QE.Q4_K.block_parameters.block_size == 144 and QE.Q6_K.block_parameters.block_size == 210
    assert QE.Q5_K.block_parameters == mojo_amd.BlockParameters(256, 176) and QE.Q5_K.is_gguf and QE.Q5_K.code == 4
    assert QE.Q4_K.is_gguf and QE.Q6_K.is_gguf and QE.Q4_0.is_gguf and not QE.GPTQ.is_gguf
    assert QE.Q4_K.name == "Q4_K" and QE.GPTQ.code == 3
    assert QE.Q4_K.packed_row_bytes(4096) == 2304 and QE.Q6_K.packed_row_bytes(4096) == 3360
    with pytest.raises(ValueError):
        QE.Q4_K.packed_row_bytes(4100)
    with pytest.raises(ValueError):
        QE.GPTQ.block_parameters
    cfg = QuantizationConfig()
    assert (cfg.quant_method, cfg.bits, cfg.group_size, cfg.desc_act, cfg.sym) == ("gptq", 4, 128, False, True)


def test_host_shim_rejects_bad_calls_without_touching_the_gpu():
    a = torch.zeros(1, 256)
    w = torch.zeros(4, 144, dtype=torch.uint8)
    with pytest.raises(ValueError, match="GPU"):
        mojo_amd.qmatmul(QE.Q4_K, None, a, w)  # no CPU fallback, by design
    with pytest.raises(TypeError):
        mojo_amd.qmatmul("Q4_K", None, a, w)
    with pytest.raises(TypeError):
        mojo_amd.qmatmul(QE.Q4_K, None, np.zeros((1, 256), np.float32), w)
    with pytest.raises(ValueError, match="GPU"):
        mojo_amd.dequantize(QE.Q4_K, w)
    with pytest.raises(ValueError, match="GPU"):
        mojo_amd.quantize(QE.Q4_0, a)


def test_missing_library_is_an_error_not_a_fallback(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", os.path.join(ROOT, "mojo_amd", "does_not_exist.so"))
    with pytest.raises(RuntimeError, match="not built"):
        _lib.load()


def test_product_never_imports_the_oracle():
    """The shipped package and the C sources must not reference the oracle directory."""
    for base, _, files in os.walk(os.path.join(ROOT, "mojo_amd")):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp")):
                text = open(os.path.join(base, f), errors="ignore").read()
                assert "import oracle" not in text and "qmm_oracle" not in text and "oracle/" not in text, f


def test_act_order_beyond_the_direct_gemm_stays_with_the_look_up_kernel():
    """The sorted columns are for the direct GEMM, which takes up to 2^32 weights; no room is asked for them where it does not serve the call (the GEMM
    that unpacks tiles, the next in line, has ten times the error of the look-up kernel)."""
    lib, cfg = _lib.load(), C.byref(_lib.GptqConfig(4, 128, 1, 1))
    for m in (9, 17, 200):
        least = lib.qmm_matmul_workspace_bytes(QE.GPTQ.code, _lib.QMM_BF16, m, 1 << 17, 1 << 15)
        assert lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, QE.GPTQ.code, cfg, _lib.QMM_BF16, m, (1 << 17) - 8, 1 << 15, 0) > (1 << 31)
        assert lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, QE.GPTQ.code, cfg, _lib.QMM_BF16, m, 1 << 17, 1 << 15, 0) <= least


def without_call_module(monkeypatch):
    """As on an installation where ``_call.so`` is missing: ``from . import _call`` raises ImportError."""
    monkeypatch.setattr(_lib, "_call", None)
    monkeypatch.delattr(mojo_amd, "_call", raising=False)
    monkeypatch.setitem(sys.modules, "mojo_amd._call", None)


def test_calls_are_served_without_the_call_module(monkeypatch):
    without_call_module(monkeypatch)
    lhs, w = torch.zeros(1, 256), torch.zeros((8, 144), dtype=torch.uint8)
    with pytest.warns(RuntimeWarning, match="_call.so"):
        with pytest.raises(ValueError, match="must live on the GPU"):  # the Python code behind the module looked at the call
            mojo_amd.qmatmul(QE.Q4_K, None, lhs, w)
    with warnings.catch_warnings():  # the warning comes once
        warnings.simplefilter("error")
        gamma = torch.ones(256)
        for call in (lambda: mojo_amd.qmatmul(QE.Q4_K, None, lhs, w), lambda: mojo_amd.qmatmul_grouped(QE.Q4_K, lhs, [w]),
                     lambda: mojo_amd.qmatmul_swiglu(QE.Q4_K, lhs, w, w), lambda: mojo_amd.qmatmul_rmsnorm(QE.Q4_K, None, lhs, gamma, 1e-5, w),
                     lambda: mojo_amd.dequantize(QE.Q4_K, w), lambda: mojo_amd.quantize(QE.Q4_K, lhs),
                     lambda: mojo_amd.quantize_gptq(torch.zeros(8, 256))):
            with pytest.raises(ValueError, match="must live on the GPU"):
                call()


def test_a_call_module_that_does_not_compile_is_no_build_error(monkeypatch, tmp_path):
    call = tmp_path / "_call.so"
    call.write_bytes(b"an older module")
    monkeypatch.setattr(build, "CALL", str(call))
    monkeypatch.setattr(build, "HIPCC", "/bin/false")
    with pytest.warns(RuntimeWarning, match="ctypes"):
        build._build_call(force=True, verbose=False)
    assert not call.exists()


def test_a_call_module_of_another_torch_is_rebuilt_and_not_loaded(monkeypatch, tmp_path):
    assert _lib.call_is_current(_lib.CALL_PATH) and _lib.call().compiled_for == _lib.call_stamp()
    old = _lib.call_stamp().encode()
    monkeypatch.setattr(torch, "__version__", torch.__version__ + "x")  # as after an update of torch
    assert old != _lib.call_stamp().encode() and not _lib.call_is_current(_lib.CALL_PATH)
    monkeypatch.setattr(_lib, "_call", None)
    with pytest.warns(RuntimeWarning, match="another torch"):
        assert _lib.call().matmul() is None
    call = tmp_path / "_call.so"  # newer than every source
    call.write_bytes(old)
    compiled = []
    monkeypatch.setattr(build, "CALL", str(call))
    monkeypatch.setattr(build.subprocess, "run", lambda cmd, **kw: compiled.append(cmd) or subprocess.CompletedProcess(cmd, 0, "", ""))
    build._build_call(force=False, verbose=False)
    assert len(compiled) == 1
    call.write_bytes(_lib.call_stamp().encode())
    build._build_call(force=False, verbose=False)
    assert len(compiled) == 1  # current: nothing to do


def wanted(enc, m, n, k, at, lhs=_lib.QMM_BF16, group=0):
    """gemm_direct.hip's answer to: does the direct GEMM, or a kernel behind it there, serve weights at that address?"""
    call = getattr(C.CDLL(_lib.LIB_PATH), "_ZN3qmm18gemm_direct_wantedEiillliPKv")
    call.argtypes, call.restype = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_void_p], C.c_bool
    return call(enc.code, lhs, m, n, k, group, at)


def test_q6_k_between_multiples_of_four_is_not_served_beyond_the_direct_range():
    """The staged GEMM, on which the range beyond rests, does not take such tensors; the direct and the shared one would be up to half as slow again there as the
    GEMM that unpacks the weights once."""
    for m, n, k in ((700, 14336, 4096), (1000, 11008, 4096), (1500, 4096, 4096)):
        assert wanted(QE.Q6_K, m, n, k, 0x10000) and wanted(QE.Q6_K, m, n, k, 0x10004)
        assert not wanted(QE.Q6_K, m, n, k, 0x10002)
    assert wanted(QE.Q6_K, 400, 4096, 4096, 0x10002)  # (within it they serve it)


def test_q6_k_that_ends_between_multiples_of_four_is_not_served_beyond_the_direct_range():
    """An odd number of blocks: the staged GEMM reads whole multiples of four and would read beyond the last one."""
    for m, n, k in ((700, 14337, 2304), (800, 14337, 2304), (1500, 4095, 3840)):
        assert not wanted(QE.Q6_K, m, n, k, 0x10000) and wanted(QE.Q6_K, m, n - 1, k, 0x10000)
        assert wanted(QE.Q6_K, m, n, k + 256, 0x10000)


def test_long_rows_go_to_the_staged_gemm():
    """K of 2^23 and more, below 2^27: by row tiles of 64, whose loads need no offsets from one 32 rows' operands to another's."""
    call = getattr(C.CDLL(_lib.LIB_PATH), "_ZN3qmm24gemm_direct_takes_stagedEiillli")
    call.argtypes, call.restype = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64, C.c_int], C.c_bool
    for enc, lhs, m, n, group in ((QE.GPTQ, _lib.QMM_BF16, 600, 8, 128), (QE.GPTQ, _lib.QMM_F32, 800, 64, 128), (QE.Q4_K, _lib.QMM_F32, 1000, 64, 0), (QE.Q5_K, _lib.QMM_BF16, 1600, 8, 0)):
        assert all(call(enc.code, lhs, m, n, k, group) for k in (2**23 - 256, 2**23, 2**23 + 256, 2**25))


def test_workgroups_beside_the_slabs_find_a_place():
    """Act-order: rows of the lhs and the zeroing of results share the launch that sorts the weights where no group of compute units, of four in each XCD that take workgroups in turn, gets more rounds of
    long ones than the weights alone would have: counted out here one by one."""
    room = getattr(C.CDLL(_lib.LIB_PATH), "_ZN3qmm14order_lhs_roomElllll")
    room.argtypes, room.restype = [C.c_int64] * 5, C.c_int

    def rounds(slabs, at_once, m, rows, zeroing):
        worst = 0
        for xcd in range(8):
            per, each, long = -(-slabs // 8), 8 // rows, [0] * 4
            for turn in range(-(-m // 64) * each):  # (gptq_order_kernel's rows of a workgroup)
                if (turn // each * 8 + xcd) * 8 + turn % each * rows < m:
                    long[turn % 4] += 1
            first = -(-m // 64) * each + zeroing // 8
            for i in range(max(0, min(per, slabs - xcd * per))):
                long[(first + i) % 4] += 1
            worst = max(worst, *long)
        return -(-worst // (at_once // 32))

    shared = apart = 0
    for slabs in (1, 8, 129, 232, 237, 245, 254, 256, 257, 480, 512, 700, 1016):
        for at_once, rows in ((256, 1), (256, 4), (512, 2), (256, 8)):
            alone = -(-(-(-slabs // 8)) // 4)
            alone = -(-alone // (at_once // 32))
            for m in (1, 8, 13, 29, 64, 66, 300, 1000):
                for zeros in (0, 1, 13 * 7560, 29 * 7400, 1 << 21):
                    got, most = room(slabs, at_once, m, rows, zeros), -(-min(1024, -(-zeros // 4096)) // 8) * 8
                    if got < 0:
                        apart += 1
                        assert all(rounds(slabs, at_once, m, rows, most + 8 * i) > alone for i in range(4))
                        continue
                    shared += 1
                    assert got % 8 == 0 and most <= got < most + 32
                    if at_once == 256 or alone == 1:  # (two a compute unit, several rounds: always)
                        assert rounds(slabs, at_once, m, rows, got) == alone
    assert shared > 300 and apart > 300


def test_operands_of_long_rows_do_not_overlap(tmp_path):
    """The places of a row tile's operands, as the preparation of the lhs works them out, against 64-bit arithmetic: with K = 2^25 (fp32) and 2^26 (bf16) they pass 32 bits."""
    if not os.path.exists(build.HIPCC):
        pytest.skip("needs hipcc")
    checks = "\n".join(f"static_assert(qmm::operand_offset({k // 16 - 1}, {row}, {g}, {per}) == {(k // 16 - 1) * 1024 * per + (row + 32 * g) * 16}LL);"
                       for per, k in ((1, 256), (2, 256), (1, 2**26 + 256), (2, 2**25 + 256), (1, 2**31 - 256), (2, 2**31 - 256)) for row, g in ((0, 0), (31, 1)))
    source = tmp_path / "places.hip"
    source.write_text('#include "gemm_direct.h"\n' + checks + "\n")
    proc = subprocess.run([build.HIPCC, "-std=c++17", "--offload-arch=gfx950", "--cuda-host-only", "-fsyntax-only", f"-I{build.CSRC}", str(source)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-3000:]


def test_no_tensors_means_none_is_looked_at():
    """n_rhs = 0 with an array all the same (here one that ends where memory does): an error, not a read of its first entry."""
    import mmap

    lib, libc, page = _lib.load(), C.CDLL(None, use_errno=True), mmap.PAGESIZE
    pages = mmap.mmap(-1, 2 * page)
    base = C.addressof(C.c_char.from_buffer(pages))
    libc.mprotect.argtypes = [C.c_void_p, C.c_size_t, C.c_int]
    assert libc.mprotect(base + page, page, 0) == 0
    end, m, n, k = C.cast(base + page, C.POINTER(C.c_void_p)), 64, 4096, 4096
    at, packed = 1 << 20, lib.qmm_repack_bytes(QE.Q5_K.code, None, n, k)
    need = lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_REPACKED, QE.Q5_K.code, None, _lib.QMM_BF16, m, n, k, 0)
    assert need > 0 and packed > 0
    assert lib.qmm_matmul_repacked(QE.Q5_K.code, None, at, _lib.QMM_BF16, m, k, end, 0, at, packed, n, at, at, need, 0, None) == -1
    assert lib.qmm_matmul(QE.Q5_K.code, None, at, _lib.QMM_BF16, m, k, end, 0, n, at, at, need, _lib.QMM_FLAG_OUT_BF16, None) == -1
    libc.mprotect(base + page, page, 3)


def test_every_switch_that_the_fallback_test_throws_exists():
    """The library ignores names that it does not know: a setting with one would test nothing."""
    from test_gpu_fallback_kernels import SETTINGS

    text = ""
    for name in os.listdir(build.CSRC):
        with open(os.path.join(build.CSRC, name)) as f:
            text += f.read()
    switches = {s for line in text.split("\n") if "kernel_disabled(" in line for s in re.findall(r'"(\w+)"', line)}
    variables = set(re.findall(r'(?:getenv|is_one)\("(\w+)"\)', text))
    assert {v for setting in SETTINGS for v in setting} <= variables
    assert {s for setting in SETTINGS for s in setting.get("QMM_DISABLE", "").split(",") if s} <= switches


def test_grouped_workspace_is_not_what_the_matrices_need_one_after_the_other():
    """Matrices that share a launch for few rows have their groups of K next to each other; whatever else is kept there, the lhs of the direct GEMM for one, is kept once."""
    lib = _lib.load()

    def figures(enc, m, k, ns):
        each = [lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, enc.code, None, _lib.QMM_F32, m, n, k, 0) for n in ns]
        return lib.qmm_matmul_grouped_workspace_bytes(enc.code, _lib.QMM_F32, m, k, len(ns), (C.c_int64 * len(ns))(*ns)), each

    for enc, m, k, ns in [(QE.Q5_K, 32, 4096, [4096] * 16), (QE.Q6_K, 40, 4096, [1024, 4096]), (QE.Q4_0, 300, 2048, [2048] * 3), (QE.Q4_K, 1, 4096, [4096, 1024])]:
        got, each = figures(enc, m, k, ns)
        assert got == max(each), (enc, m, k, ns)
    assert figures(QE.Q4_K, 4, 14336, [1024, 256, 512])[0] == 4 * 4 * 4 * 1792  # four groups, fp32 [4, 1792]
    assert figures(QE.Q4_K, 4, 14336, [1024] * 9)[0] == 4 * 4 * 4 * 4096  # four matrices a launch
    assert lib.qmm_matmul_grouped_workspace_bytes(QE.Q4_K.code, 0, 4, 4096, 0, None) == 0
