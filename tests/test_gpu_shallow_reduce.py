"""Reductions of a few slices over many outputs: odd column counts, outputs written by rows and by columns."""
import ctypes as C

import numpy as np
import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from approxtrain_amd import ApproxMulLut, functors, load_library
from oracle import cpu
from tests.gpu_util import assert_close_sum_abs, dev, host, lut32
from tests.util import lut_path

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(1000, 515, 513), (513, 515, 1000), (700, 2049, 301), (301, 2049, 700),
                                   (1025, 640, 64), (1000, 1000, 65)])
@pytest.mark.parametrize("trans", [(False, False), (True, False), (False, True)])
def test_shallow_slices(m, k, n, trans):
    # (sizes on both sides of the rules: the first two are cut into two slices, the others deeper or too small)
    rng = np.random.default_rng(m + k + n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    lut = ApproxMulLut(lut_path("MBM", 3))
    ga, gb = dev(np.ascontiguousarray(a.T if trans[0] else a)), dev(np.ascontiguousarray(b.T if trans[1] else b))
    out = host(functors.gemm(lut, ga, gb, trans_a=trans[0], trans_b=trans[1]))
    table = lut32("MBM", 3)
    # slices added in another order than one ascending chain: the bound every split reduction is held to
    assert_close_sum_abs(out, cpu.gemm(table, 3, a, b, threads=16), cpu.gemm_abs(table, 3, a, b, threads=16), 1e-5)


ENGINE_LDS_TABLE = 1


def _reductions(call):
    """The call's result and the names of the reductions that it launched."""
    out = call()  # (once before: a handle's first call)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        out = call()
        torch.cuda.synchronize()
    names = [e.name for e in p.events() if "kernel(" in e.name or "kernel<" in e.name]
    if not any("lutgemm_kernel" in n for n in names):
        pytest.skip("no kernel activity recorded")
    return out, [n.split("splitk_reduce_")[1].split("_kernel")[0] for n in names if "splitk_reduce_" in n]


def _handles(kind="MBM", m=3):
    lib = load_library()
    split, whole = ApproxMulLut(lut_path(kind, m)), ApproxMulLut(lut_path(kind, m))
    for lut in (split, whole):
        lib.amsim_lut_set_engine(lut.handle, ENGINE_LDS_TABLE)
    lib.amsim_lut_set_split_k(whole.handle, 0)
    return split, whole


def _in_slices(whole, a, b, chunks, rows_from, rows_to, along_m):
    """The product's rows (columns, unless along_m) rows_from .. rows_to, as whole products over slices of the
    reduction (one ascending chain per output each) added in slice order."""
    part = slice(rows_from, rows_to)
    a, b = (a[..., part, :], b) if along_m else (a, b[..., part])
    total = None
    for k0 in range(0, a.shape[-1], 32 * chunks):
        s = functors.gemm(whole, a[..., k0:k0 + 32 * chunks].contiguous(), b[..., k0:k0 + 32 * chunks, :].contiguous())
        total = s if total is None else total + s
    return total


@pytest.mark.parametrize("m,k,n,batch,along,slices,tail,kernel", [
    (1446, 232, 1539, 1, "rows", 2, 0, "shallow"), (2083, 260, 870, 1, "rows", 3, 0, "shallow"),
    (936, 484, 877, 1, "rows", 4, 0, "shallow"), (716, 500, 218, 5, "rows", 4, 0, "shallow"),
    (2655, 68, 2331, 1, "rows", 1, 3, "shallow"), (1203, 100, 1694, 3, "rows", 1, 4, "shallow"),
    (1223, 228, 1540, 1, "cols", 2, 0, "turn"), (1388, 268, 1016, 1, "cols", 3, 0, "turn"),
    (369, 488, 1868, 1, "cols", 4, 0, "turn"), (656, 484, 498, 2, "cols", 4, 0, "turn"),
    (2258, 100, 2791, 1, "cols", 1, 2, "turn"), (388, 100, 2755, 5, "cols", 1, 4, "turn"),
    # outputs along the rows, too few of them for the turn: two tiles of rows, one of 6 and of 59 rows
    (1998, 68, 2630, 1, "cols", 1, 3, "shallow"), (323, 72, 2747, 5, "cols", 1, 3, "shallow"),
])
def test_slices_are_added_in_order(m, k, n, batch, along, slices, tail, kernel):
    """Bit for bit: whole products over the planner's slices, added in slice order, then bias and ReLU."""
    split, whole = _handles()
    info = (C.c_int64 * 8)()
    assert load_library().amsim_gemm_plan_info(0, 0, m, n, k, batch, info) == 0
    # (reduction slices inside a workgroup would sum in another order: none of these)
    assert info[1] == 1 and info[2] == slices and info[5] == tail
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    lead = () if batch == 1 else (batch,)
    a, b = (torch.randn(lead + s, device="cuda", generator=gen) for s in ((m, k), (k, n)))
    along_m = along == "rows"
    rows, axis = (m, -2) if along_m else (n, -1)
    parts = [_in_slices(whole, a, b, info[3], 0, info[4], along_m)]
    if tail:
        parts.append(_in_slices(whole, a, b, info[6], info[4], rows, along_m))
    else:
        assert info[4] == rows
    want = torch.cat(parts, axis)
    got, names = _reductions(lambda: functors.gemm(split, a, b))
    assert names == [kernel]
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    if batch == 1:
        bias = torch.randn(n, device="cuda", generator=gen)
        got, names = _reductions(lambda: functors.denseam(split, a, b, bias=bias, activation="relu"))
        assert names == [kernel] and torch.equal(got, (want + bias).relu())


def test_mapped_outputs():
    """Residue classes of a strided convolution's input gradient, each reduced into its own pixels."""
    split, whole = _handles()
    gen = torch.Generator(device="cuda").manual_seed(9)
    dy = torch.randn((4, 28, 28, 128), device="cuda", generator=gen)
    w = torch.randn((3, 3, 65, 128), device="cuda", generator=gen)
    call = lambda lut, w, dy: functors.convam_input_grad(lut, (4, 56, 56, 65), w, dy, (2, 2), "SAME")
    got, names = _reductions(lambda: call(split, w, dy))
    assert names == ["shallow"] * 4
    # the table's products of absolute values are the products' absolute values
    assert_close_sum_abs(host(got), host(call(whole, w, dy)), host(call(whole, w.abs(), dy.abs())), 1e-5)
