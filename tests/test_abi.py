"""CPU checks of the boundary: the shared library loads without a GPU, exports every symbol that
include/rwkv_hip.h declares, and argument errors come back as error codes (never a crash or exit)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "rwkv_hip.h")).read()
    return sorted(set(re.findall(r"\b(rwkv_hip_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from rwkv_lightning_cuda_amd import hip
    lib = hip.load()
    names = declared_symbols()
    assert len(names) >= 55
    for n in names:
        assert hasattr(lib, n), n
    assert sorted(hip.EXPORTS) == names


def test_errors_are_codes_not_crashes():
    from rwkv_lightning_cuda_amd import hip
    lib = hip.load()
    assert hip.device_count() >= 0
    # shape checks run on the host before anything touches a device
    rc = lib.rwkv_hip_wkv7(None, 1, 1, 100, 1, 0, 0, None, None, None, None, None, None, None, None)
    assert rc == -1 and b"H*64" in lib.rwkv_hip_last_error()
    m = ctypes.c_void_p(0)
    assert lib.rwkv_hip_model_create(ctypes.byref(m), 1, 100, 1, 64, 64, 8, 8, 8, 8) == -1
    assert b"C must equal H*N" in lib.rwkv_hip_last_error()
    assert lib.rwkv_hip_model_create(ctypes.byref(m), 1, 64, 1, 64, 64, 8, 8, 8, 1024) == -1
    assert lib.rwkv_hip_model_create(ctypes.byref(m), 2, 64, 1, 64, 64, 8, 8, 8, 8) == 0
    assert lib.rwkv_hip_model_set_tensor(m, 5, 10, ctypes.c_void_p(16)) == -1      # layer out of range
    assert lib.rwkv_hip_model_set_matrix(m, 0, 0, 1, ctypes.c_void_p(16), None, None) == -1   # W8 without scale
    assert lib.rwkv_hip_model_set_matrix(m, 0, 0, 2, ctypes.c_void_p(16), ctypes.c_void_p(16), ctypes.c_void_p(16)) == -1  # W4, K=64
    n = ctypes.c_uint64(0)
    assert lib.rwkv_hip_model_weight_bytes(m, ctypes.byref(n)) == 0 and n.value > 0
    assert lib.rwkv_hip_model_destroy(m) == 0
    assert lib.rwkv_hip_sample(None, 1, 6, None, None, None, None, ctypes.c_double(0), ctypes.c_double(0),
                               ctypes.c_double(1), ctypes.c_double(1), 0, ctypes.c_double(1), ctypes.c_uint64(0),
                               ctypes.c_uint64(0)) == -1
    assert b"multiple of 4" in lib.rwkv_hip_last_error()


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from rwkv_lightning_cuda_amd import hip
    monkeypatch.setattr(hip, "_lib", None)
    monkeypatch.setattr(hip, "LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(hip.RwkvHipError, match="no CPU fallback"):
        hip.load()


def test_workspace_queries_that_repeat_cost_no_search():
    """A decode step asks about ten times which tile and K split its products take, with the answers of the step before; the
    search over all of them took 10 us a query (three formats), 30 to 140 us of host time in front of every step.  A repeated
    query costs the call's own 1.5 us; and threads that ask for more shapes than are kept get what one thread gets."""
    import threading
    import time
    from rwkv_lightning_cuda_amd import hip
    shapes = [(8, 4096, 4096), (8, 16384, 4096), (8, 4096, 16384), (8, 65536, 4096)]
    best = 1e9
    for _ in range(10):
        start = time.perf_counter()
        for _ in range(50):
            for shape in shapes:
                hip.linear_packed_workspace(*shape)
        best = min(best, (time.perf_counter() - start) / 200 * 1e6)
    print("%.2f us a query" % best)
    assert best <= 5.0
    many = [(M, N, K) for M in (3, 17, 64, 100, 512, 2048) for N in (64, 768, 2048, 16384) for K in (256, 768, 4096, 16384)]
    want = [hip.linear_packed_workspace(*shape) for shape in many]
    got = [[] for _ in range(4)]

    def ask(out):
        for _ in range(5):
            out.append([hip.linear_packed_workspace(*shape) for shape in many])

    threads = [threading.Thread(target=ask, args=(out,)) for out in got]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(row == want for out in got for row in out)


@pytest.mark.parametrize("fmt,M,N,K,tile", [("w8", 208, 12288, 4096, (128, 128, 1)), ("w8", 256, 16384, 4096, (128, 128, 1)),
                                            ("w8", 256, 65536, 4096, (256, 256, 1)), ("f16", 384, 12288, 4096, (128, 256, 1)),
                                            ("f16", 208, 4096, 16384, (128, 128, 4)), ("f16", 512, 65536, 4096, (128, 256, 1))])
def test_the_operator_of_some_hundred_rows_takes_the_tile_that_is_fastest(fmt, M, N, K, tile):
    """Up to 512 rows the operator went by the time of a 128 x 256 tile that is not there any more, and the estimate of the ones that are
    knew nothing of what few row tiles take out of HBM.  The fastest of every tile and split as measured; the next one takes 1.08 to
    1.3 times as long.  Without a workspace there is no split, and no other tile where there was none."""
    from rwkv_lightning_cuda_amd import hip
    problem = [({"f16": hip.FMT_F16, "w8": hip.FMT_W8}[fmt], N)]
    assert hip.linear_packed_plan(M, K, problem, hip.linear_packed_workspace(M, N, K))[0] == tile
    assert hip.linear_packed_plan(M, K, problem, 0)[0][2] == 1
    if tile[2] == 1:
        assert hip.linear_packed_plan(M, K, problem, 0)[0] == tile


def test_no_workspace_is_asked_for_that_no_launch_takes():
    """From 513 rows on every launch runs with the splits that fit: the query is what the largest choice of the three formats takes (1300 x
    4704 x 2560 asked for the two planes of a tile that was not looked at)."""
    from rwkv_lightning_cuda_amd import hip
    for M, N, K in ((1300, 4704, 2560), (1030, 3872, 512), (2049, 832, 8192), (1038, 1056, 10240), (600, 768, 3072)):
        need = hip.linear_packed_workspace(M, N, K)
        splits = [hip.linear_packed_plan(M, K, [(fmt, N)], 1 << 40)[0][2] for fmt in (hip.FMT_W8, hip.FMT_W4, hip.FMT_F16)]
        assert need == (max(splits) * M * N * 4 if max(splits) > 1 else 0)
