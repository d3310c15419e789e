"""The rule that sends large products to 256 x 256 tiles and to slices of k
(csrc/gemm_split.hpp), compiled for the host: the sizes of the GPU tests of those kernels run on
the kernel and in the slices that they are there for (256 compute units), and slices cover k
without an empty one."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

import test_gpu_gemm_ksplit
import test_gpu_gemm_wide

SRC = Path(__file__).resolve().parent / "host" / "gemm_split_host.cpp"
PREC = {"f64": 0, "f32": 1, "bf16x3": 2}


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host C++ compiler")
    out = tmp_path_factory.mktemp("gs") / "gemm_split_host.so"
    subprocess.run([gxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-o", str(out), str(SRC)], check=True)
    return C.CDLL(str(out))


def route(lib, prec, M, N, K):
    """(kernel, slices) of a product whose operands can be loaded as vectors."""
    split = K >= 1024
    wide = lib.wide_slices(256, PREC[prec], M, N, K, int(split))
    if wide:
        return "wide", wide
    return "tiles", lib.ksplit_wanted(256, PREC[prec], M, N, K) if split else 1


def test_wide_sizes_take_the_wide_kernel(lib):
    for prec in ("f32", "bf16x3"):
        for M, N, K in test_gpu_gemm_wide.SIZES:
            assert route(lib, prec, M, N, K) == route(lib, prec, M, N, (K + 3) // 4 * 4) == ("wide", 1)
        for (M, N, K), want in test_gpu_gemm_wide.SLICED.items():
            assert route(lib, prec, M, N, K) == route(lib, prec, M, N, (K + 3) // 4 * 4) == want[prec]
    # both kernels, and a last slice that ends inside a k-step
    for prec in ("f32", "bf16x3"):
        sliced = [(K, w[prec][1]) for (M, N, K), w in test_gpu_gemm_wide.SLICED.items()
                  if w[prec][0] == "wide" and w[prec][1] > 1]
        assert any((K - (s - 1) * lib.slice_width(K, s)) % 32 for K, s in sliced)
    for M, N, K in test_gpu_gemm_wide.SAME_BITS:
        assert route(lib, "f32", M, N, K) == ("wide", 1)


def test_ksplit_sizes_split(lib):
    for (M, N, K), want in test_gpu_gemm_ksplit.SLICES.items():
        for prec in PREC:
            assert route(lib, prec, M, N, K) == ("tiles", want[prec])


def test_slices_cover_k(lib):
    for s in range(2, 7):
        for K in list(range(512 * s, 512 * s + 200)) + [2 ** 22 - 1, 2 ** 22]:
            w = lib.slice_width(K, s)
            assert w % 64 == 0 and (s - 1) * w < K <= s * w
