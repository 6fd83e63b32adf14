"""The column-stage kernels' real products: couplings symmetric in the pair (l, m) take only the
Re products (a prefix of the Raman lines), others the Im products too; a pair whose two slots differ
in parity (the reference-CPU decode) lies in both parity segments. Against the FP64 oracle at the
bars of the short runs (1e-12; mixed precision 1e-6), at the mode counts where the step table, the
coefficient groups and the wavefronts' shares change (one product to 256, odd and even)."""
import copy

import numpy as np
import pytest

import oracle_binding as ob
from gpu_util import note, require_device
from mm_propagation_amd import _capi, configs
from mm_propagation_amd.batch import MultimodePropagationBatch, SolverGroup
from mm_propagation_amd.problem import NonZeroValue
from mm_propagation_amd.solver import Context, MultimodePropagationGPU_RamanOFF, MultimodePropagationGPU_RamanON

pytestmark = pytest.mark.gpu

FP64, MIXED = _capi.MMP_PRECISION_FP64, _capi.MMP_PRECISION_MIXED


def unsymmetric(sp):
    """The same index structure with one coupling Q^(0)_{k,l,m}, l != m, changed."""
    out = copy.deepcopy(sp)
    q = out.coupling_coefficients[0]
    i = next(i for i, e in enumerate(q) if e.index[1] != e.index[2])
    q.resetValue(i, 0.5 * q.getNonZeroValue(i).value)
    return out


@pytest.mark.parametrize("precision,flags", [(FP64, 0), (MIXED, 0), (MIXED, _capi.MMP_FLAG_NO_MATRIX_CORES)])
@pytest.mark.parametrize("M,coupling,decode", [(1, "symmetric", 1), (2, "k_le_l", 0), (3, "unsymmetric", 1), (4, "k_le_l", 0),
                                               (5, "k_le_l", 0), (5, "symmetric", 1), (6, "unsymmetric", 1), (6, "k_le_l", 0),
                                               (7, "mirror", 1), (9, "k_le_l", 0), (11, "unsymmetric", 1), (16, "unsymmetric", 1)])
def test_products_against_oracle(M, coupling, decode, precision, flags):
    require_device()
    sp = configs.grin_fiber(M=M, nt=4096, symmetric=coupling in ("symmetric", "unsymmetric"), mirror=coupling == "mirror",
                            power_range=(1.0, 100.0), seed=3)
    if coupling == "unsymmetric":
        sp = unsymmetric(sp)
    note(f"case products M={M} {coupling} decode={decode} precision={precision} flags={flags}")
    s = MultimodePropagationGPU_RamanON(sp, pair_decode=decode, precision=precision, flags=flags)
    s.computeLawsonRK(5)
    got = s.getResult()
    s.close()
    o = ob.Oracle(sp, pair_decode=decode, n_threads=16)
    o.compute_lawson_rk(5)
    err = configs.rel_l2_per_mode(got, o.get_result())
    o.close()
    assert np.all(err <= (1e-12 if precision == FP64 else 1e-6)), err


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("M", [3, 6, 10])
def test_a_general_fiber_joins_a_symmetric_batch(M, precision):
    """Loading the first fiber that needs the Im products changes the batch's plan (lines, steps and
    coefficients) under its graph and its group's: the other fibers keep their arithmetic bit for
    bit, and every fiber equals itself alone."""
    require_device()
    sps = [configs.grin_fiber(M=M, nt=4096, fiber_length=0.5 + 0.1 * i, seed=20 + i, symmetric=True) for i in range(3)]
    general = unsymmetric(configs.grin_fiber(M=M, nt=4096, fiber_length=0.9, seed=31, symmetric=True))
    note(f"case general fiber into a symmetric batch M={M} precision={precision}")
    ctx = Context(0)
    b = MultimodePropagationBatch(sps, pair_decode=1, precision=precision, ctx=ctx)
    other = MultimodePropagationGPU_RamanON(sps[1], pair_decode=1, precision=precision, ctx=Context(0))
    g = SolverGroup([b, other], ctx)
    g.advance(5)
    b.load(1, general)
    for _ in range(2):
        g.advance(17)
    steps = [39, 34, 39]
    for f, sp in enumerate([sps[0], general, sps[2]]):
        s = MultimodePropagationGPU_RamanON(sp, pair_decode=1, precision=precision)
        s.computeLawsonRK(steps[f])
        assert np.array_equal(b.result(f), s.getResult()), f
        s.close()
    s = MultimodePropagationGPU_RamanON(sps[1], pair_decode=1, precision=precision)
    s.computeLawsonRK(39)
    assert np.array_equal(other.getResult(), s.getResult())
    s.close()
    g.close()
    b.close()
    other.close()


def odd_coupling(sp):
    """One more nonzero, at odd k + l - m - p: the couplings have no parity structure left."""
    out = copy.deepcopy(sp)
    q = out.coupling_coefficients[0]
    q.addNonZeroValue(NonZeroValue((0, 1, 0), 0.3 * q.getNonZeroValue(0).value))
    return out


@pytest.mark.parametrize("raman", [True, False])
@pytest.mark.parametrize("M,nt,coupling", [(1, 256, "symmetric"), (2, 1024, "k_le_l"), (4, 512, "odd"), (5, 1024, "unsymmetric"),
                                           (8, 2048, "symmetric"), (9, 1024, "unsymmetric"), (16, 256, "odd"),
                                           (17, 1024, "symmetric"), (17, 256, "odd"), (20, 512, "unsymmetric"),
                                           (32, 256, "symmetric"), (33, 256, "symmetric")])
def test_separate_gather_against_oracle(M, nt, coupling, raman):
    """The separate passes' gather at its smallest and largest tables: one chunk and several, one to
    four groups of modes, 4, 2 and 1 products a step; beyond 16 coefficients per product and mode the sparse
    gather serves (odd couplings of 17 modes, 33 modes)."""
    require_device()
    sp = configs.grin_fiber(M=M, nt=nt, symmetric=coupling != "k_le_l", power_range=(1.0, 100.0), seed=5)
    if coupling == "unsymmetric":
        sp = unsymmetric(sp)
    if coupling == "odd":
        sp = odd_coupling(sp)
    note(f"case separate gather M={M} nt={nt} {coupling} raman={raman}")
    cls = MultimodePropagationGPU_RamanON if raman else MultimodePropagationGPU_RamanOFF
    s = cls(sp, pair_decode=1)
    s.computeLawsonRK(3)
    got = s.getResult()
    s.close()
    o = ob.Oracle(sp, raman=raman, pair_decode=1, n_threads=16)
    o.compute_lawson_rk(3)
    err = configs.rel_l2_per_mode(got, o.get_result())
    o.close()
    assert np.all(err <= 1e-12), err


def test_a_general_fiber_joins_a_large_symmetric_batch():
    """At 6 modes and 2048 columns the gather takes two columns per workgroup on the 11 lines of
    symmetric couplings; all 18 lines pass its LDS, so the load changes the workgroups too."""
    require_device()
    sps = [configs.grin_fiber(M=6, nt=4096, fiber_length=0.5 + 0.01 * i, seed=20 + i, symmetric=True) for i in range(32)]
    general = unsymmetric(configs.grin_fiber(M=6, nt=4096, fiber_length=0.9, seed=61, symmetric=True))
    note("case general fiber into a large symmetric batch")
    b = MultimodePropagationBatch(sps, pair_decode=1)
    b.advance(3)
    b.load(31, general)
    b.advance(3)
    for f, sp, steps in ((0, sps[0], 6), (30, sps[30], 6), (31, general, 3)):
        s = MultimodePropagationGPU_RamanON(sp, pair_decode=1)
        s.computeLawsonRK(steps)
        assert np.array_equal(b.result(f), s.getResult()), f
        s.close()
    b.close()


@pytest.mark.parametrize("M,nt,coupling", [(1, 4096, "symmetric"), (2, 8192, "k_le_l"), (3, 4096, "unsymmetric"), (4, 4096, "odd"),
                                           (5, 4096, "unsymmetric"), (6, 65536, "symmetric"), (7, 4096, "mirror"),
                                           (9, 4096, "unsymmetric"), (10, 4096, "odd"), (16, 4096, "unsymmetric")])
def test_kerr_column_kernel_against_oracle(M, nt, coupling):
    """Without Raman the whole column side of a stage is one kernel: odd and even modes (the zero field
    row), one product to 256, coefficients in LDS and read ahead, one chunk and several; and the separate
    passes on the same fiber."""
    require_device()
    sp = configs.grin_fiber(M=M, nt=nt, symmetric=coupling in ("symmetric", "unsymmetric", "odd"), mirror=coupling == "mirror",
                            power_range=(1.0, 100.0), seed=9)
    if coupling == "unsymmetric":
        sp = unsymmetric(sp)
    if coupling == "odd":
        sp = odd_coupling(sp)
    note(f"case kerr columns M={M} nt={nt} {coupling}")
    o = ob.Oracle(sp, raman=False, pair_decode=1, n_threads=16)
    o.compute_lawson_rk(3)
    want = o.get_result()
    o.close()
    for flags in (0, _capi.MMP_FLAG_SEPARATE_COLUMNS):
        s = MultimodePropagationGPU_RamanOFF(sp, pair_decode=1, flags=flags)
        s.computeLawsonRK(3)
        err = configs.rel_l2_per_mode(s.getResult(), want)
        s.close()
        assert np.all(err <= 1e-12), (flags, err)
