"""CPU-side checks of the C ABI: the library loads, exports every symbol include/f3d_hip.h declares,
and rejects bad arguments with the reference's messages before touching a GPU."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "flash3dtransformer_amd", "lib", "libf3d_hip.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()
    L = ctypes.CDLL(LIB)
    L.f3d_last_error.restype = ctypes.c_char_p
    return L


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "f3d_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(f3d_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_symbol_is_exported(lib):
    names = declared_symbols()
    assert len(names) >= 15
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, f"declared in include/f3d_hip.h but not exported: {missing}"


def test_module_state_roundtrip(lib):
    assert lib.f3d_set_sync_stream(1) == 1 and lib.f3d_get_sync_stream() == 1
    assert lib.f3d_set_sync_stream(0) == 0 and lib.f3d_get_sync_stream() == 0
    lib.f3d_get_seed.restype = ctypes.c_uint32
    assert lib.f3d_get_seed() == 3407
    lib.f3d_set_seed(ctypes.c_uint32(11))
    assert lib.f3d_get_seed() == 11
    lib.f3d_set_seed(ctypes.c_uint32(3407))
    assert lib.f3d_set_psh_rebalance(7) != 0 and b"rebalance" in lib.f3d_last_error()
    assert lib.f3d_set_psh_rebalance(1) == 0
    assert lib.f3d_get_quantiser() == 0
    assert lib.f3d_set_quantiser(1) == 0 and lib.f3d_get_quantiser() == 1
    assert lib.f3d_set_quantiser(2) != 0 and b"quantiser mode" in lib.f3d_last_error()
    assert lib.f3d_set_quantiser(0) == 0 and lib.f3d_get_quantiser() == 0


def _psh_call(lib, *, num_bucket=64, divisor=1024, pad_to=512, total_n=512, hash_type=1, num_vox=0xFFFF):
    u32, vp = ctypes.c_uint32, ctypes.c_void_p
    dummy = vp(16)  # never dereferenced: validation fails first
    return lib.f3d_batch_psh_scatter_pad_hash(dummy, dummy, dummy, dummy, dummy, u32(1), u32(total_n), u32(total_n),
                                              u32(num_bucket), u32(divisor), u32(512), u32(num_vox), dummy, dummy,
                                              dummy, dummy, dummy, u32(pad_to), ctypes.c_float(0.0), u32(hash_type),
                                              ctypes.c_int(0), vp(0))


def test_psh_argument_errors_match_reference(lib):
    # src/psh/batch_psh_bucket_dispatcher.cu:239-250
    assert _psh_call(lib, divisor=512) == 1 and b"bucket divisor too small" in lib.f3d_last_error()
    assert _psh_call(lib, pad_to=100) == 1 and b"smaller than the input length" in lib.f3d_last_error()
    assert _psh_call(lib, hash_type=5) == 1 and b"hash_type=5 is unsupported" in lib.f3d_last_error()
    assert _psh_call(lib, hash_type=0) == 1
    # src/common/kernel_dispatcher.cuh:73-82
    assert _psh_call(lib, num_bucket=48, divisor=2048) == 2 and b"No kernel found" in lib.f3d_last_error()


def test_no_alloc_psh_rejects_batches_beyond_its_scratch_array(lib):
    """the entry point that allocates nothing says so when a batch does not fit its fixed scratch array
    (argument validation: no GPU is touched)"""
    u32, vp = ctypes.c_uint32, ctypes.c_void_p
    dummy = vp(16)

    def call(batch, per_cloud, nb):
        div = -(-65535 // nb)
        return lib.f3d_batch_psh_scatter_pad_hash_noalloc(
            dummy, dummy, dummy, dummy, dummy, u32(batch), u32(batch * per_cloud), u32(per_cloud), u32(nb), u32(div),
            u32(512), u32(0xFFFF), dummy, dummy, dummy, dummy, dummy, u32(batch * per_cloud), ctypes.c_float(0.0),
            u32(1), ctypes.c_int(0), vp(0))
    assert call(256, 262144, 512) == 2
    msg = lib.f3d_last_error()
    assert b"scratch" in msg and b"f3d_batch_psh_scatter_pad_hash" in msg
    # the same argument errors as the allocating entry point come first
    assert lib.f3d_batch_psh_scatter_pad_hash_noalloc(
        dummy, dummy, dummy, dummy, dummy, u32(1), u32(512), u32(512), u32(64), u32(512), u32(512), u32(0xFFFF), dummy,
        dummy, dummy, dummy, dummy, u32(512), ctypes.c_float(0.0), u32(1), ctypes.c_int(0), vp(0)) == 1
    assert b"bucket divisor too small" in lib.f3d_last_error()


@pytest.mark.parametrize("m,n,k,act", [(0, 64, 64, 0), (16, 0, 640, 0), (16, 0, 64, 2)])
def test_linear_without_outputs_launches_nothing(lib, m, n, k, act):
    """no rows or no columns: done, whatever the kernel that the other sizes would choose, and before a device is selected"""
    p, none, u = ctypes.c_void_p(4096), ctypes.c_void_p(0), ctypes.c_uint32
    end = ctypes.c_int(0), none
    assert lib.f3d_linear_bf16(p, u(k), p, none, none, u(0), p, u(64), u(m), u(n), u(k), u(act), *end) == 0
    if k == 64:
        assert lib.f3d_ln_linear_bf16(p, u(k), p, none, ctypes.c_float(1e-5), p, none, none, u(0), p, u(64), u(m), u(n), u(k),
                                      u(act), *end) == 0


def test_staged_buffer_is_not_kept_by_a_call_that_prepares_nothing(lib):
    """a refused call, an empty one and none at all: f3d_staged_weights_kept says no, and ends the staging"""
    at = lambda a: ctypes.c_void_p(a)
    u, f = ctypes.c_uint32, ctypes.c_float

    def ln_linear(x, m):
        return lib.f3d_ln_linear_bf16(at(x), u(256), at(4096), None, f(1e-5), at(8192), None, None, u(0), at(16384), u(64), u(m), u(64),
                                      u(256), u(0), 0, None)
    assert lib.f3d_staged_weights_kept() == 0
    for call in (lambda: ln_linear(2, 8) != 0, lambda: ln_linear(32768, 0) == 0, lambda: True):
        assert lib.f3d_stage_weights(at(65536), ctypes.c_size_t(1 << 20), 0) == 0
        assert call()
        assert lib.f3d_staged_weights_kept() == 0


def test_library_builds_without_torch(monkeypatch, capsys, tmp_path):
    """the native driver is left out with a word, where torch is absent or on request; it is compiled anew for another torch"""
    import subprocess
    import sys

    import torch
    from flash3dtransformer_amd.csrc import build
    ran = []
    monkeypatch.setattr(subprocess, "run", lambda cmd, **kw: (ran.append(cmd[0]), subprocess.CompletedProcess(cmd, 0, "", ""))[1])
    monkeypatch.setattr(build, "_compile", lambda src, incremental: src)
    with monkeypatch.context() as m:
        m.setitem(sys.modules, "torch", None)
        build.build(verbose=False)
    assert ran == ["hipcc"] and "native driver is not built" in capsys.readouterr().err
    build.build(verbose=False, host=False)
    assert ran == ["hipcc"] * 2
    monkeypatch.setattr(build, "OBJ_DIR", str(tmp_path))
    monkeypatch.setattr(build, "HOST_LIB", os.path.join(build.OBJ_DIR, "_f3d_host.so"))
    open(build.HOST_LIB, "w").close()
    os.utime(build.HOST_LIB, (2e9, 2e9))
    ran.clear()
    for version in ("2.0", "2.0", "2.1"):
        monkeypatch.setattr(torch, "__version__", version)
        build._build_host(incremental=True)
    assert ran == ["g++", "g++"]
