"""Reductions of a few slices over many outputs: odd column counts, outputs written by rows and by columns."""
import numpy as np
import pytest

from approxtrain_amd import ApproxMulLut, functors
from oracle import cpu
from tests.gpu_util import assert_close_sum_abs, dev, host, lut32
from tests.util import lut_path

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(1000, 515, 513), (513, 515, 1000), (700, 2049, 301), (301, 2049, 700),
                                   (1025, 640, 64), (1000, 1000, 65)])
@pytest.mark.parametrize("trans", [(False, False), (True, False), (False, True)])
def test_shallow_slices(m, k, n, trans):
    rng = np.random.default_rng(m + k + n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    lut = ApproxMulLut(lut_path("MBM", 3))
    ga, gb = dev(np.ascontiguousarray(a.T if trans[0] else a)), dev(np.ascontiguousarray(b.T if trans[1] else b))
    out = host(functors.gemm(lut, ga, gb, trans_a=trans[0], trans_b=trans[1]))
    table = lut32("MBM", 3)
    # slices added in another order than one ascending chain: the bound every split reduction is held to
    assert_close_sum_abs(out, cpu.gemm(table, 3, a, b, threads=16), cpu.gemm_abs(table, 3, a, b, threads=16), 1e-5)
