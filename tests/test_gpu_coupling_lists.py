"""Coupling lists other than the full ones of the workloads: pairs that are there one way only and
no parity structure. Against the FP64 oracle at the bars of the short runs (1e-12; mixed precision 1e-6)."""
import copy

import numpy as np
import pytest

import oracle_binding as ob
from gpu_util import note, require_device
from mm_propagation_amd import _capi, configs
from mm_propagation_amd.problem import Sparse3DArray
from mm_propagation_amd.solver import MultimodePropagationGPU_RamanON

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
