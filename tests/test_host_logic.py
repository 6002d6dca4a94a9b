"""Host-side logic without a GPU: the Python mirror of the reference's extension surface (gemm_amd) and
the built neoGEMM module reject what they must, and nothing falls back to a CPU computation."""
import pytest
import torch

import gemm_amd


def test_surface_names():
    # the reference's names (nemgemmV03.cu:396-399, v01.cu:314-317) plus C = gemm(A, B)
    for mod in (gemm_amd, __import__("neoGEMM")):
        assert callable(mod.gemm) and callable(mod.neoGemmV1) and callable(mod.neogemm)
    import neoGEMM
    assert neoGEMM.version() == gemm_amd.version()


def test_no_cpu_path():
    A = torch.zeros(8, 8, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="GPU"):
        gemm_amd.gemm(A, A)
    with pytest.raises(ValueError, match="GPU"):
        gemm_amd.neoGemmV1(A, A, A.clone())
    import neoGEMM
    with pytest.raises(RuntimeError, match="GPU"):
        neoGEMM.gemm(A, A)
    with pytest.raises(RuntimeError, match="GPU"):
        neoGEMM.neoGemmV1(A=A, B=A, C=A.clone())   # the reference's keyword names


def test_type_checks_come_first():
    with pytest.raises(TypeError):
        gemm_amd.gemm([1, 2], torch.zeros(2, 2))
    # dtype and rank are checked after the device in both wrappers; on CPU tensors the device error wins
    import neoGEMM
    with pytest.raises(RuntimeError):
        neoGEMM.gemm(torch.zeros(4, 4), torch.zeros(4, 4))


def test_missing_library_is_an_error(monkeypatch):
    from gemm_amd import _abi
    monkeypatch.setattr(_abi, "_lib", None)
    monkeypatch.setattr(_abi, "LIB_PATH", "/nonexistent/libneogemm.so")
    with pytest.raises(RuntimeError, match="no CPU or PyTorch fallback"):
        _abi.load()


def test_error_class_carries_status():
    e = gemm_amd.NeoGemmError(-3, "shape")
    assert e.status == -3 and "variant" in str(e)


def test_a_transposed_view_of_the_output_is_copied():
    """gemm_scaled(C.t(), X, C): A is read while C is written, so a view of C's memory must not be read in place."""
    C, X = torch.zeros(256, 256, dtype=torch.bfloat16), torch.zeros(256, 256, dtype=torch.bfloat16)
    A, _, lda, _, a_layout, _ = gemm_amd._describe(C.t(), X, out=C)
    assert a_layout == gemm_amd.A_MK and lda == 256 and A.data_ptr() != C.data_ptr()
    # part of it shared: rows 100 .. 355 of a buffer whose rows 0 .. 255 are C
    buf = torch.zeros(356, 256, dtype=torch.bfloat16)
    A, _, _, _, a_layout, _ = gemm_amd._describe(buf[100:].t(), X, out=buf[:256])
    assert a_layout == gemm_amd.A_MK and not gemm_amd._overlap(A, buf)
    # neighbours share nothing and are read in place
    both = torch.zeros(512, 256, dtype=torch.bfloat16)
    A, _, lda, _, a_layout, _ = gemm_amd._describe(both[:256].t(), X, out=both[256:])
    assert a_layout == gemm_amd.A_KM and A.data_ptr() == both.data_ptr()


def test_scratch_of_captured_and_of_large_calls_is_not_kept(monkeypatch):
    """A buffer whose address a graph replays must not be dropped when a later call outgrows it: captured calls take their own."""
    import contextlib
    import types

    capturing = [False]
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: types.SimpleNamespace(cuda_stream=7))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(gemm_amd, "_workspaces", {})
    monkeypatch.setattr(gemm_amd, "_MAX_KEPT", 4096, raising=False)
    cpu = torch.device("cpu")
    kept = gemm_amd._workspace(cpu, 1000)
    assert gemm_amd._workspace(cpu, 500) is kept
    capturing[0] = True
    a, b = gemm_amd._workspace(cpu, 500), gemm_amd._workspace(cpu, 2000)
    assert a is not kept and a.numel() >= 500 and b.numel() >= 2000
    capturing[0] = False
    assert gemm_amd._workspace(cpu, 500) is kept
    assert gemm_amd._workspace(cpu, 4097).numel() >= 4097 and gemm_amd._workspace(cpu, 500) is kept
