"""The C-ABI library loads and exports every symbol include/qimm.h declares
(no compute calls: this runs without a GPU), and its error paths are codes."""
import ctypes as C
import os
import re
import subprocess

import pytest

import qimm
from test_gpu_kernels import BF16_ROWS_CASES, bf16_rows_route

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "qimm.h")


def header_functions():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(qimm_[a-z0-9_]+)\s*\(", src)))


def test_header_declares_the_entry_points():
    names = header_functions()
    for must in ("qimm_ctx_create", "qimm_weight_upload", "qimm_dequant", "qimm_qmatmul",
                 "qimm_attention", "qimm_block_create", "qimm_block_forward", "qimm_kv_create"):
        assert must in names


def test_library_exports_every_declared_symbol():
    lib = qimm.load()
    missing = [n for n in header_functions() if not hasattr(lib, n)]
    assert not missing, missing
    out = subprocess.run(["nm", "-D", "--defined-only", qimm.LIB_PATH], capture_output=True, text=True).stdout
    exported = set(re.findall(r"\bT (qimm_[a-z0-9_]+)", out))
    assert set(header_functions()) <= exported


def test_python_binding_covers_the_header():
    assert sorted(n for n, _, _ in qimm.SIGNATURES) == header_functions()


def test_abi_version_and_status_strings():
    lib = qimm.load()
    assert lib.qimm_abi_version() == 1
    assert lib.qimm_status_string(0) == b"ok"
    assert lib.qimm_status_string(3) == b"unsupported GGML type"


def test_null_arguments_return_codes():
    lib = qimm.load()
    assert lib.qimm_ctx_create(0, None) == 1
    assert lib.qimm_ctx_destroy(None) == 1
    assert lib.qimm_weight_free(None) == 1
    assert lib.qimm_kv_destroy(None) == 1
    assert lib.qimm_block_destroy(None) == 1
    assert lib.qimm_last_error(None) == b"null context"


def test_ctx_create_without_gpu_fails_cleanly():
    torch = pytest.importorskip("torch")
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    h = C.c_void_p()
    rc = qimm.load().qimm_ctx_create(0, C.byref(h))
    assert rc != 0 and not h.value


@pytest.mark.parametrize("t,m,n,k,route", BF16_ROWS_CASES)
def test_bf16_rows_cases_take_the_paths_they_name(t, m, n, k, route):
    """The GPU cases of the kernel over bf16 rows run that kernel, in the shares of K, tiles
    and tail that each is there for, on 256 compute units."""
    assert bf16_rows_route(t, m, n, k, 256) == (True, route)


def test_plan_of_mixed_tiles_follows_the_rounds():
    """The tiles of 256 tokens that the plan picks, against a plan that places the tiles round
    by round (the estimate of qgemm_bf16.hip, 256 compute units): odd and large token counts,
    few and many weight tiles."""
    cus = 256

    def round_us(steps, small, wgs):
        f = min(1.0, wgs / cus)
        return 6.0 + steps * (0.61 + 0.26 * f if small else 1.08 + 0.42 * f)

    def span(steps, n1, n2):
        c1, c2 = round_us(steps, False, n1 + n2), round_us(steps, True, n1 + n2)
        late, t0 = n1 % cus, n1 // cus * c1
        t1, x, y = t0 + c1, 0, 0
        while x * (cus - late) + y * late < n2:
            if late == 0 or t0 + (x + 1) * c2 <= t1 + (y + 1) * c2:
                x += 1
            else:
                y += 1
        return max(t1 + y * c2 if late else t0, t0 + x * c2)

    for n, k in ((24576, 4096), (12288, 4096), (4096, 12288), (9216, 3072)):
        for m in (2304, 2817, 3072, 3289, 4095, 4097, 4352, 5000, 6889, 8448, 9001, 13799):
            full, nt, steps = (m + 255) // 256, n // 256, k // 64
            best, us = full, span(steps, full * nt, 0)
            for h in range(full):
                t = span(steps, h * nt, (m - 256 * h + 127) // 128 * nt)
                if t < us * 0.995:
                    best, us = h, t
            r = qimm.qmatmul_route(qimm.Q4_K if k != 12288 else qimm.Q6_K, n, k, m, cus)
            assert r.kernel == qimm.GEMM_BF16_ROWS
            if r.tail == 0:
                assert r.large_tiles == best, (n, k, m)


def test_plan_of_many_tokens_is_quick():
    """A plan is made at each launch: its cost grows with the tokens at most (it used to place
    every round of tiles, 9 ms at 200000 tokens)."""
    import time
    qimm.qmatmul_route(qimm.Q4_K, 24576, 4096, 4096, 256)
    t = min(_timed(lambda: qimm.qmatmul_route(qimm.Q4_K, 24576, 4096, 200000, 256), time) for _ in range(5))
    assert t < 1e-3, t


def _timed(f, time):
    t0 = time.perf_counter()
    f()
    return time.perf_counter() - t0


def test_bench_counts_the_weight_bytes_the_kernels_read():
    """bench.py's weight bytes and traffic are those of the kernels that run: the bf16 rows at
    the block step's 4096 tokens, the codes at 16; no traffic figure of another kernel."""
    import bench
    import synth
    n, k = 2 * bench.MLP, bench.HID
    assert bench.weight_read(qimm, synth, synth.Q4_K, n, k, bench.S_IMG, 256) == (2 * n * k, qimm.GEMM_BF16_ROWS)
    assert bench.weight_read(qimm, synth, synth.Q4_K, n, k, 16, 256) == (n * k // 256 * 144, qimm.GEMM_STREAM)
    t = bench.measured_traffic("gate_up", "qgemm_bf16_kernel")
    assert t and t["bytes"] > 2 * n * k
    assert bench.measured_traffic("gate_up", "no_such_kernel") is None


def test_qmatmul_route_codes():
    lib = qimm.load()
    r = qimm.GemmRoute()
    assert lib.qimm_qmatmul_route(qimm.Q4_K, 256, 256, 1, 100, 256, None) == 1
    assert lib.qimm_qmatmul_route(qimm.Q4_K, 256, 256, 1, 0, 256, C.byref(r)) == 1
    assert lib.qimm_qmatmul_route(qimm.Q4_K, 96, 256, 1, 100, 256, C.byref(r)) == 2
    assert lib.qimm_qmatmul_route(7, 256, 256, 1, 100, 256, C.byref(r)) == 3
    # few rows stream the codes; without bf16 rows many rows decode in 256 x 256 tiles
    assert qimm.qmatmul_route(qimm.Q4_K, 4096, 4096, 16, 256).kernel == qimm.GEMM_STREAM
    assert qimm.qmatmul_route(qimm.Q4_K, 4096, 4096, 4352, 256).kernel == qimm.GEMM_BF16_ROWS
    assert qimm.qmatmul_route(qimm.Q4_K, 4096, 4096, 4352, 256, bf16_rows=False).kernel == qimm.GEMM_WIDE
    # so do quantized weights of short K with rows: they are not left to the decoding kernels
    for t, m, n, k in ((qimm.Q8_0, 3072, 12288, 128), (qimm.Q8_0, 8448, 8192, 256), (qimm.Q4_K, 16384, 8192, 256)):
        assert qimm.qmatmul_route(t, n, k, m, 256).kernel == qimm.GEMM_BF16_ROWS
    # bf16-stored ones take the four-wave kernel there
    assert qimm.qmatmul_route(qimm.BF16, 12288, 128, 3072, 256).kernel == qimm.GEMM_LARGE
    # float weights are bf16 rows themselves
    assert qimm.qmatmul_route(qimm.BF16, 4096, 4096, 4352, 256, bf16_rows=False).kernel == qimm.GEMM_BF16_ROWS
