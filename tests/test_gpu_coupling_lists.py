"""Coupling lists other than the full ones of the workloads: pairs that are there one way only and
no parity structure. Against the FP64 oracle at the bars of the short runs (1e-12; mixed precision 1e-6)."""
import copy

import numpy as np
import pytest

import oracle_binding as ob
from gpu_util import note, require_device
from mm_propagation_amd import _capi, configs
from mm_propagation_amd.batch import MultimodePropagationBatch, SolverGroup
from mm_propagation_amd.problem import Sparse3DArray
from mm_propagation_amd.solver import Context, MultimodePropagationGPU_RamanOFF, MultimodePropagationGPU_RamanON

pytestmark = pytest.mark.gpu

FP64, MIXED = _capi.MMP_PRECISION_FP64, _capi.MMP_PRECISION_MIXED


def with_lists(sp, entries):
    """sp with Q^(p) from entries(p): (k, l, m) indices; values SR u, u ~ U(-0.5, 1)."""
    rng = np.random.default_rng(11)
    out = copy.deepcopy(sp)
    out.coupling_coefficients = [Sparse3DArray([(k, l, m, configs.SR * float(rng.uniform(-0.5, 1.0))) for k, l, m in entries(p)])
                                 for p in range(sp.n_modes)]
    return out


def partial_pairs(sp, both):
    """Every pair (l, m): the first `both` cross pairs both ways, the other ones l < m only, and
    no parity structure (two neighbouring k each)."""
    M = sp.n_modes
    cross = [(a, b) for a in range(M) for b in range(a + 1, M)]

    def entries(p):
        out = []
        for i, (a, b) in enumerate(cross):
            out += [((p + i) % M, a, b), ((p + i + 1) % M, a, b)]
            if i < both:
                out.append(((p + i) % M, b, a))
        return out + [(p, a, a) for a in range(M)]

    return with_lists(sp, entries)


def full(sp, symmetric, seed=11):
    """Every (k, l, m): no parity structure; symmetric: equal values at (l, m) and (m, l)."""
    out = with_lists(sp, lambda p: [(k, l, m) for k in range(sp.n_modes) for l in range(sp.n_modes) for m in range(sp.n_modes)])
    rng = np.random.default_rng(seed)
    for q in out.coupling_coefficients:
        values = configs.SR * rng.uniform(-0.5, 1.0, (sp.n_modes,) * 3)
        for i, e in enumerate(q):
            k, l, m = e.index
            q.resetValue(i, values[(k, min(l, m), max(l, m)) if symmetric else (k, l, m)])
    return out


def check(solver, sp, steps, decode, bar):
    solver.computeLawsonRK(steps)
    got = solver.getResult()
    o = ob.Oracle(sp, raman=solver.raman, pair_decode=decode, n_threads=16)
    o.compute_lawson_rk(steps)
    err = configs.rel_l2_per_mode(got, o.get_result())
    o.close()
    assert np.all(err <= bar), err


@pytest.mark.parametrize("flags", [0, _capi.MMP_FLAG_NO_MATRIX_CORES])
@pytest.mark.parametrize("M,both", [(10, 20), (13, 24), (14, 20), (16, 16)])
def test_later_chunks_with_more_lines_than_the_first(M, both, flags):
    """Mixed precision bounds a chunk by its slots (M^2 coefficients each): the first chunk holds lines of
    two slots, `both` of them, the next ones lines of one slot, up to 30, and so wavefronts that had no line before."""
    require_device()
    sp = partial_pairs(configs.grin_fiber(M=M, nt=4096, power_range=(1.0, 100.0), seed=3), both)
    note(f"case later chunks M={M} both={both} flags={flags}")
    s = MultimodePropagationGPU_RamanON(sp, precision=MIXED, flags=flags)
    assert s.info()["gather_chunks"] > 1
    check(s, sp, 5, 1, 1e-6)
    s.close()


@pytest.mark.parametrize("raman", [True, False])
@pytest.mark.parametrize("M", [5, 6, 7])
def test_full_lists_without_parity_structure(M, raman):
    """At 6 modes all 36 products' 18 lines, 19 steps of coefficients and sigma in rows of its own pass the 64 KB
    of the FP64 column gather's workgroup."""
    require_device()
    sp = full(configs.grin_fiber(M=M, nt=4096, power_range=(1.0, 100.0), seed=3), symmetric=False)
    cls = MultimodePropagationGPU_RamanON if raman else MultimodePropagationGPU_RamanOFF
    for decode in (0, 1):
        note(f"case full list M={M} raman={raman} decode={decode}")
        s = cls(sp, pair_decode=decode)
        check(s, sp, 5, decode, 1e-12)
        s.close()


@pytest.mark.parametrize("fibers", [3, 32])
def test_a_general_fiber_joins_a_symmetric_batch_without_parity_structure(fibers):
    """6 modes: 11 lines before the load and 18 after; every fiber equals itself alone bit for bit (32 fibers:
    2048 columns, two a workgroup before)."""
    require_device()
    base = [configs.grin_fiber(M=6, nt=4096, fiber_length=0.5 + 0.01 * i, seed=20 + i, power_range=(1.0, 100.0)) for i in range(3)]
    sps = [full(sp, symmetric=True, seed=i) for i, sp in enumerate(base)]
    general = full(base[0], symmetric=False, seed=9)
    note(f"case general fiber into a symmetric batch without parity, {fibers} fibers")
    b = MultimodePropagationBatch([sps[i % 3] for i in range(fibers)])
    b.advance(3)
    b.load(1, general)
    b.advance(3)
    for f, sp, steps in ((0, sps[0], 6), (2, sps[2], 6), (1, general, 3)):
        s = MultimodePropagationGPU_RamanON(sp)
        s.computeLawsonRK(steps)
        assert np.array_equal(b.result(f), s.getResult()), f
        s.close()
    b.close()


def one_k_per_pair(sp):
    """Every pair (l, m), one coupling each, with the parity structure."""
    M = sp.n_modes
    return with_lists(sp, lambda p: [((p + l + m) % 2, l, m) for l in range(M) for m in range(M)])


def every_k(sp):
    """The same pairs in the same order with all their couplings of the parity structure."""
    M = sp.n_modes
    return with_lists(sp, lambda p: [(k, l, m) for l in range(M) for m in range(M) for k in range((p + l + m) % 2, M, 2)])


def other_fiber(sp, lists):
    """Another length, pulse width, Raman share, field and couplings; the same structure."""
    out = lists(configs.grin_fiber(M=sp.n_modes, nt=sp.nt, fiber_length=0.7, t0=0.15, seed=8, power_range=(1.0, 100.0)))
    out.raman_proportion = 0.25
    return out


@pytest.mark.parametrize("M,nt,precision,raman", [(2, 1024, MIXED, True), (5, 1024, MIXED, False), (13, 512, MIXED, True),
                                                  (20, 256, MIXED, False), (20, 512, FP64, True), (33, 256, FP64, True),
                                                  (16, 4096, FP64, False)])
def test_a_loaded_fiber_brings_its_couplings(M, nt, precision, raman):
    """A solver of one fiber on the separate passes: the fiber loaded into it, with fewer, more and other couplings,
    equals itself alone bit for bit, also stepped by a group that was there before."""
    require_device()
    base = configs.grin_fiber(M=M, nt=nt, power_range=(1.0, 100.0), seed=4)
    first, few, many = every_k(base), other_fiber(base, one_k_per_pair), other_fiber(base, every_k)
    ctx = Context(0)
    b = MultimodePropagationBatch([first], raman=raman, precision=precision, ctx=ctx)
    other = MultimodePropagationBatch([first], raman=raman, precision=precision, ctx=Context(0))
    g = SolverGroup([b, other], ctx)
    g.advance(3)
    steps = 0
    for sp in (few, many, few):
        note(f"case load M={M} nt={nt} precision={precision} raman={raman}")
        b.load(0, sp)
        g.advance(4)
        steps += 4
        alone = MultimodePropagationBatch([sp], raman=raman, precision=precision)
        alone.advance(4)
        assert np.array_equal(b.result(0), alone.result(0))
        alone.close()
    untouched = MultimodePropagationBatch([first], raman=raman, precision=precision)
    untouched.advance(3 + steps)
    assert np.array_equal(other.result(0), untouched.result(0))
    for x in (g, b, other, untouched):
        x.close()


@pytest.mark.parametrize("raman", [True, False])
@pytest.mark.parametrize("M,nt,lists", [(12, 1024, "own"), (13, 1024, "own"), (13, 4096, "one"), (16, 4096, "own"), (16, 1024, "one"),
                                        (16, 4096, "full"), (20, 1024, "own"), (20, 1024, "one"), (32, 256, "one")])
def test_lists_on_both_sides_of_the_gathers_choice(M, nt, lists, raman):
    """FP64 on the separate passes (and without Raman the column kernel): self pairs alone, one coupling a pair
    and the full list, on either side of the line between the sparse sum and the products."""
    require_device()
    sp = configs.grin_fiber(M=M, nt=nt, power_range=(1.0, 100.0), seed=6)
    if lists != "full":
        sp = with_lists(sp, lambda p: [(p, l, l) for l in range(M)]) if lists == "own" else one_k_per_pair(sp)
    cls = MultimodePropagationGPU_RamanON if raman else MultimodePropagationGPU_RamanOFF
    note(f"case gather choice M={M} nt={nt} lists={lists} raman={raman}")
    s = cls(sp)
    check(s, sp, 3, 1, 1e-12)
    s.close()


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("M,fibers", [(1, 17), (1, 32), (2, 16), (2, 32), (2, 64), (3, 32), (4, 16), (5, 16), (6, 16), (6, 64),
                                      (8, 32), (13, 9)])
def test_gather_forms_of_large_grids(M, fibers, symmetric):
    """FP64 batches on 576 to 4096 columns: one, two and four columns a workgroup, four and eight wavefronts. Every
    fiber equals itself alone (one column, eight or 12 wavefronts) bit for bit."""
    require_device()
    sps = [configs.grin_fiber(M=M, nt=4096, fiber_length=0.5 + 0.01 * i, seed=50 + i, symmetric=symmetric, power_range=(1.0, 100.0))
           for i in range(3)]
    note(f"case gather forms M={M} fibers={fibers} symmetric={symmetric}")
    b = MultimodePropagationBatch([sps[i % 3] for i in range(fibers)])
    b.advance(4)
    for i, sp in enumerate(sps):
        s = MultimodePropagationGPU_RamanON(sp)
        s.advance(4)
        want = s.getResult()
        for f in (i, i + (fibers - 1 - i) // 3 * 3):  # its first and its last copy
            assert np.array_equal(b.result(f), want), f
        s.close()
    b.close()


@pytest.mark.parametrize("M,nt", [(1, 65536), (4, 32768), (5, 32768), (7, 32768), (13, 32768)])
def test_column_kernel_without_raman_on_large_grids(M, nt):
    """512 and 1024 columns: eight wavefronts up to 4 modes on the first, four else."""
    require_device()
    sp = configs.grin_fiber(M=M, nt=nt, power_range=(1.0, 100.0), seed=12)
    note(f"case columns without Raman M={M} nt={nt}")
    s = MultimodePropagationGPU_RamanOFF(sp)
    check(s, sp, 2, 1, 1e-12)
    s.close()
