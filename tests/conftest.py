import ctypes as C
import importlib
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a gfx950 device (run on the GPU box)")


@pytest.fixture(scope="session")
def O():
    import oracle
    return oracle


@pytest.fixture(scope="session")
def tfq():
    return importlib.import_module("transformers-fusion_amd")


@pytest.fixture(scope="session")
def gpu(tfq):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    tfq.init(0)
    return torch.device("cuda:0")


class Plan(C.Structure):
    """A plan of the integer tile kernel; shape 4: tiles of 32 x 32, K over the wavefronts of a workgroup."""
    _fields_ = [("shape", C.c_int), ("ksplit", C.c_int), ("rows", C.c_int), ("launches", C.c_int), ("us", C.c_double)]


class Rules:
    """The rules by which the library chooses kernels (tests/plan_driver.cpp): a matrix's format and sizes in, no GPU needed."""
    ANY = (1 << 63) - 1  # scratch of any size
    SOLO = 4

    def __init__(self, tfq):
        tfq.lib()
        path = os.path.join(ROOT, "tests", "libplan_driver.so")
        if not os.path.exists(path):
            pytest.fail("tests/libplan_driver.so is missing: run __graft_entry__.build()")
        self._tfq, self._d = tfq, C.CDLL(path)
        matrix = [C.c_int, C.c_int64, C.c_int64, C.c_int, C.c_int]
        self._d.drv_gemm_exact_plans.argtypes = matrix + [C.c_size_t, C.c_int, C.c_int, C.POINTER(Plan), C.POINTER(Plan)]
        self._d.drv_gemm_takes_exact.argtypes = matrix + [C.c_size_t]
        self._d.drv_mlp_pairs.argtypes = matrix
        self._d.drv_gemm_scratch_bytes.argtypes = matrix
        self._d.drv_gemm_scratch_bytes.restype = C.c_size_t
        self._d.drv_gemv_rows_scratch_bytes.argtypes = matrix + [C.POINTER(C.c_size_t)]
        self._d.drv_gemv_rows_scratch_bytes.restype = C.c_size_t

    def _args(self, fmt, N, K, f32, M):
        return self._tfq.lib().tfq_format_id(fmt.encode()), N, K, self._tfq.F32 if f32 else self._tfq.BF16, M

    def plans(self, fmt, N, K, f32, M, scratch=ANY, matrices=1):
        """(all plans of the integer tile kernel, the one that is taken)"""
        buf, taken = (Plan * 128)(), Plan()
        n = self._d.drv_gemm_exact_plans(*self._args(fmt, N, K, f32, M), scratch, matrices, 128, buf, taken)
        assert 0 < n <= 128
        return buf[:n], taken

    def product(self, fmt, N, K, f32, M, scratch=None):
        """The plan of Weight.gemv (up to sixteen rows) or Weight.gemm, with the scratch that it asks for unless one is given; None
        where another kernel serves."""
        if scratch is None:
            scratch = self.rows_scratch(fmt, N, K, f32, M)[0] if M <= 16 else self._d.drv_gemm_scratch_bytes(*self._args(fmt, N, K, f32, M))
        if not self._d.drv_gemm_takes_exact(*self._args(fmt, N, K, f32, M), scratch):
            return None
        return self.plans(fmt, N, K, f32, M, scratch)[1]

    def pair(self, fmt, F, D, f32, B, scratch):
        """The plan of gate and up in tfq_mlp_step with `scratch` bytes for it; None where they are not one launch of this kernel."""
        return self.plans(fmt, F, D, f32, B, scratch, 2)[1] if self._d.drv_mlp_pairs(*self._args(fmt, F, D, f32, B)) else None

    def rows_scratch(self, fmt, N, K, f32, B):
        """Scratch of up to sixteen rows: (what the kernel that serves uses, what the decode kernels use)"""
        decode = C.c_size_t()
        return self._d.drv_gemv_rows_scratch_bytes(*self._args(fmt, N, K, f32, B), decode), decode.value


@pytest.fixture(scope="session")
def rules(tfq):
    return Rules(tfq)
