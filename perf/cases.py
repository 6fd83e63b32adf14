"""Timed cases of the propagation library: what its users have it do, through its public entry
points, over the range the library takes (1 to 20 modes, 2^8 to 2^16 samples, FP64 and mixed
precision, the three tableaux, Raman on and off, symmetric and general coupling lists, one fiber,
batches and groups).

A pass starts every fiber from its initial field (set_state), takes `steps` steps and returns the
physical fields, as a driver does between two outputs; a one-shot case makes the whole call from
the parameters. Real runs take 500 to 20000 steps between a start and an output; `steps` is cut so
that a pass stays in the milliseconds, and the initial powers (1 to 100 W) keep every field finite.
"""
import math

import numpy as np
import torch

from mm_propagation_amd import _capi, configs
from mm_propagation_amd.batch import MultimodePropagationBatch, SolverGroup
from mm_propagation_amd.solver import (Context, MultimodePropagationGPU_RamanOFF, MultimodePropagationGPU_RamanON,
                                       default_context, solve_static)

FP64, MIXED = _capi.MMP_PRECISION_FP64, _capi.MMP_PRECISION_MIXED


def _case(name, kind, modes, nt, steps, mixed, order=4, raman=True, coupling="symmetric", fibers=1, **more):
    c = {"kind": kind, "modes": modes, "nt": nt, "steps": steps, "mixed": mixed, "order": order, "raman": raman,
         "coupling": coupling, "fibers": fibers}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: the smoke run's two-mode Gaussian on 1024 samples (launch bound)
        _case("two_mode_1024", "advance", 2, 1024, 100, False, coupling="two_mode"),
        # the reference drivers' loop: the two-mode Gaussian with outputs on the way (n_save)
        _case("two_mode_snapshots", "snapshots", 2, 4096, 200, False, coupling="two_mode", saves=5),
        # a short solve in one call without device allocation (serving loops, hosts that forbid it)
        _case("three_mode_one_shot", "static", 3, 4096, 64, True),
        # the RamanOFF class (Kerr only) on the six-mode graded-index fiber
        _case("six_mode_kerr_only", "advance", 6, 16384, 80, False, raman=False),
        # the plain FP64 solver on the six-mode graded-index fiber, with its energy monitored
        _case("six_mode_fp64", "advance", 6, 16384, 100, False, energy=True),
        # a coupling list without index symmetry (k <= l rule) and the reference's pair decode, order 6
        _case("five_mode_general_rk6", "advance", 5, 8192, 37, False, order=6, coupling="k_le_l"),
        # the 11-stage tableau in mixed precision
        _case("four_mode_rk8_mixed", "advance", 4, 32768, 20, True, order=8),
        # ten modes on the largest grid, mixed precision
        _case("ten_mode_65536_mixed", "advance", 10, 65536, 60, True),
        # the largest single fiber of a serving mix
        _case("fifteen_mode_65536_mixed", "advance", 15, 65536, 20, True),
        # more modes than the column-stage kernels take
        _case("twenty_mode_fp64", "advance", 20, 4096, 6, False),
        # many fibers of one shape in one launch (parameter sweeps)
        _case("batch_six_mode", "batch", 6, 16384, 120, True, fibers=19, energy=True),
        # fibers of several shapes stepped together: 8 x 3 modes, 6 x 6 modes, 4 x 10 modes
        _case("group_mixed_shapes", "group", 10, 16384, 100, True, fibers=18),
    ]


def _shapes(case):
    """(modes, samples, fibers) of every batch of the case."""
    M, nt, F = case["modes"], case["nt"], case["fibers"]
    if case["kind"] != "group":
        return [(M, nt, F)]
    # the largest shape, a middle one and a small one, more fibers the smaller they are
    big = max(1, F * 2 // 9)
    mid = max(1, F // 3)
    small = max(1, F - big - mid)
    return [(max(2, M // 3), max(4096, nt // 4), small), (max(2, M * 6 // 10), max(4096, nt // 2), mid), (M, nt, big)]


def _stages(case):
    return {8: 11, 6: 7}.get(case["order"], 4)


def _cost(case):
    """About the time of a pass, to hold drawn cases below the largest listed one."""
    per_step = 0.
    for M, nt, F in _shapes(case):
        per_step += F * nt * (M * 60. + M * M * 20. + (M ** 4 if M > 16 else M ** 3) * 0.5)
    return _stages(case) * case["steps"] * (per_step + 2e7)


def draw(rng):
    kind = rng.choice(["advance", "advance", "advance", "snapshots", "static", "batch", "group"])
    mixed = rng.random() < 0.5
    coupling = rng.choice(["symmetric", "symmetric", "symmetric", "mirror", "k_le_l"])
    raman = rng.random() < 0.8
    order = rng.choice([4, 4, 4, 6, 8])
    fibers = 1
    if kind in ("batch", "group"):
        M = rng.randint(2, 12)
        nt = 2 ** rng.randint(12, 15)
        fibers = rng.randint(3, 24)
        raman, order = True, 4
    elif kind == "static":
        M, nt = rng.randint(1, 6), 2 ** rng.randint(8, 13)
    else:
        M = max(1, min(20, int(round(math.exp(rng.uniform(0., math.log(20.5)))))))
        nt = 2 ** rng.randint(8, 16)
        if M > 16:
            nt = min(nt, 4096)
    c = _case(None, kind, M, nt, rng.randint(5, 150), mixed, order, raman, coupling, fibers)
    if kind == "snapshots":
        c["saves"] = min(c["steps"], rng.randint(2, 5))
        c["steps"] -= c["steps"] % c["saves"]
    if rng.random() < 0.3 and kind in ("advance", "batch"):
        c["energy"] = True
    limit = 0.5 * max(_cost(x) for x in listed())
    while _cost(c) > limit and c["steps"] > 5:
        c["steps"] -= max(1, c["steps"] // 8)
        if kind == "snapshots":
            c["steps"] = max(c["saves"], c["steps"] - c["steps"] % c["saves"])
    while _cost(c) > limit and c["fibers"] > 3:
        c["fibers"] -= 1
    while _cost(c) > limit and c["nt"] > 4096:
        c["nt"] //= 2
    return c


def _decode(case):
    return _capi.MMP_PAIRS_REFERENCE_CPU if case["coupling"] in ("two_mode", "k_le_l") else _capi.MMP_PAIRS_PHYSICAL


def _params(case, M, nt, seed):
    if case["coupling"] == "two_mode":
        sp = configs.two_mode_gaussian(nt=nt, method_order=case["order"])
        rng = np.random.default_rng(seed)
        sp.initial_fields = np.stack([configs.gaussian(nt, sp.time_window, 0.1, float(np.exp(rng.uniform(0., math.log(100.)))),
                                                       float(rng.uniform(0., 2. * math.pi))) for _ in range(2)])
        return sp
    return configs.grin_fiber(M=M, nt=nt, n_steps=20000, seed=seed, method_order=case["order"], power_range=(1.0, 100.0),
                              symmetric=case["coupling"] == "symmetric", mirror=case["coupling"] == "mirror")


def _all_params(case, seed):
    """The parameters of every fiber, per batch of the case."""
    out, k = [], 0
    for M, nt, F in _shapes(case):
        out.append([_params(case, M, nt, 1000 * seed + k + f) for f in range(F)])
        k += F
    return out


def prepare(case, seed):
    params = _all_params(case, seed)
    precision = MIXED if case["mixed"] else FP64
    st = {"case": case, "precision": precision, "params": params}
    if case["kind"] == "static":
        default_context()
        return st
    if case["kind"] in ("batch", "group"):
        group = case["kind"] == "group"
        # members of a group on streams of their own: parallel branches of its graph
        st["solvers"] = [MultimodePropagationBatch(sps, pair_decode=_decode(case), precision=precision,
                                                   ctx=Context(0) if group else default_context()) for sps in params]
        st["psi"] = [[s.state(f)[0] for f in range(s.F)] for s in st["solvers"]]
        if group:
            st["group"] = SolverGroup(st["solvers"], Context(0))
        return st
    cls = MultimodePropagationGPU_RamanON if case["raman"] else MultimodePropagationGPU_RamanOFF
    st["solver"] = cls(params[0][0], pair_decode=_decode(case), precision=precision)
    st["psi"] = st["solver"].get_state()[0]
    return st


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "static":
        return {"field": solve_static(state["params"][0][0], case["steps"], raman=case["raman"], pair_decode=_decode(case),
                                      precision=state["precision"])}
    if kind in ("batch", "group"):
        for s, psis in zip(state["solvers"], state["psi"]):
            for f, psi in enumerate(psis):
                s.set_state(f, psi)
        if kind == "group":
            state["group"].advance(case["steps"])
        else:
            state["solvers"][0].advance(case["steps"])
        out = {"field": [s.result(f) for s in state["solvers"] for f in range(s.F)]}
        if case.get("energy"):
            out["energy"] = [s.energy(f) for s in state["solvers"] for f in range(s.F)]
        return out
    s = state["solver"]
    s.set_state(state["psi"])
    if kind == "snapshots":
        fields, z = s.propagate_snapshots(case["steps"], case["saves"], resumable=True)
        return {"field": fields, "z": z}
    s.advance(case["steps"])
    out = {"field": s.getResult()}
    if case.get("energy"):
        out["energy"] = s.energy()
    return out


def _real_pairs(case, M):
    """Real products Re and Im U_a conj(U_b) the coupling needs (only Re where it is symmetric)."""
    return M * (M + 1) // 2 if case["coupling"] == "symmetric" else M * M


def work(case):
    """Per step and stage the transforms (5 n log2 n), the pair products' convolutions (two real
    ones per complex transform) and the coupling sums over the real products (half of the mode
    pairs by parity for the graded-index lists); the field and the operator read once and the
    result written once."""
    flops = bytes_ = 0.
    for M, nt, F in _shapes(case):
        fft = 5. * nt * math.log2(nt)
        pr = _real_pairs(case, M)
        stage = 2 * M * fft + 40. * M * nt
        if case["raman"]:
            stage += pr * (fft + 8. * nt)
        stage += nt * (pr * M * M / 2. * 2. + M * M * 4.)
        flops += F * _stages(case) * case["steps"] * stage
        # the field read, Im L read, every output field written
        bytes_ += F * M * nt * (16. + 8. + 16. * case.get("saves", 1))
    return {"bytes": bytes_, "flops": flops}


# --- the same in 64 bits with plain torch -----------------------------------------------------
def _tableau(order):
    """(a, b, c) of the classic fourth-order, the seven-stage sixth-order (nu = 1) and the
    eleven-stage eighth-order Runge-Kutta methods."""
    r = math.sqrt(21.)
    if order == 8:
        a = [[], [1 / 2], [1 / 4, 1 / 4], [1 / 7, (-7 + 3 * r) / 98, (21 - 5 * r) / 49],
             [(11 - r) / 84, 0, (18 - 4 * r) / 63, (21 + r) / 252],
             [(5 - r) / 48, 0, (9 - r) / 36, (-231 - 14 * r) / 360, (63 + 7 * r) / 80],
             [(10 + r) / 42, 0, (-432 - 92 * r) / 315, (633 + 145 * r) / 90, (-504 - 115 * r) / 70, (63 + 13 * r) / 35],
             [1 / 14, 0, 0, 0, (14 + 3 * r) / 126, (13 + 3 * r) / 63, 1 / 9],
             [1 / 32, 0, 0, 0, (91 + 21 * r) / 576, 11 / 72, (-385 + 75 * r) / 1152, (63 - 13 * r) / 128],
             [1 / 14, 0, 0, 0, 1 / 9, (-733 + 147 * r) / 2205, (515 - 111 * r) / 504, (-51 + 11 * r) / 56, (132 - 28 * r) / 245],
             [0, 0, 0, 0, (-42 - 7 * r) / 18, (-18 - 28 * r) / 45, (-273 + 53 * r) / 72, (301 - 53 * r) / 72,
              (28 + 28 * r) / 45, (49 + 7 * r) / 18]]
        b = [1 / 20, 0, 0, 0, 0, 0, 0, 49 / 180, 16 / 45, 49 / 180, 1 / 20]
        c = [0, 1 / 2, 1 / 2, (7 - r) / 14, (7 - r) / 14, 1 / 2, (7 + r) / 14, (7 + r) / 14, 1 / 2, (7 - r) / 14, 1]
        return a, b, c
    if order == 6:
        a = [[], [1], [3 / 8, 1 / 8], [8 / 27, 2 / 27, 8 / 27],
             [(-21 - 9 * r) / 392, -8 * (7 + r) / 392, 48 * (7 + r) / 392, -3 * (21 + r) / 392],
             [-5 * (231 - 51 * r) / 1960, -40 * (7 - r) / 1960, 320 * r / 1960, 3 * (21 - 121 * r) / 1960,
              392 * (6 - r) / 1960],
             [15 * (22 - 7 * r) / 180, 120 / 180, -40 * (5 + 7 * r) / 180, 63 * (2 + 3 * r) / 180, -14 * (49 - 9 * r) / 180,
              70 * (7 + r) / 180]]
        b = [9 / 180, 0, 64 / 180, 0, 49 / 180, 49 / 180, 9 / 180]
        c = [0, 1, 1 / 2, 2 / 3, (7 + r) / 14, (7 - r) / 14, 1]
        return a, b, c
    return [[], [1 / 2], [0, 1 / 2], [0, 0, 1]], [1 / 6, 1 / 3, 1 / 3, 1 / 6], [0, 1 / 2, 1 / 2, 1]


class _Exact:
    """One fiber: the Lawson-Runge-Kutta scheme of the interaction picture in complex128."""

    def __init__(self, sp, case, dev):
        M, nt = sp.n_modes, sp.nt
        self.sp, self.M, self.nt = sp, M, nt
        beta = np.array(sp.dispersion_coefficients)
        t0 = sp.pulse_width
        ld = t0 * t0 / np.abs(beta[:, 2]).max()
        entries = [[(e.index[0], e.index[1], e.index[2], e.value) for e in q] for q in sp.coupling_coefficients]
        qmax = max(abs(e[3]) for q in entries for e in q)
        gamma = sp.nonlinearity_const
        self.conv = math.sqrt(abs(gamma) * ld) * math.sqrt(qmax)
        self.isgn = 1j if gamma >= 0 else -1j
        t_final = sp.time_window / t0
        self.dt = t_final / nt
        self.h = sp.fiber_length / ld / sp.n_steps
        k = np.arange(nt)
        alpha = 2. * math.pi / t_final * np.where(k <= nt // 2, k, k - nt)
        lam = np.zeros((M, nt))
        for o in range(beta.shape[1]):
            lam += (beta[:, o] * ld / t0 ** o)[:, None] * (-1.) ** o / math.factorial(o) * alpha ** o * (-1. if o == 2 else 1.)
        self.lam = torch.tensor(lam, device=dev)
        codes = {}
        for q in entries:
            for _, l, m, _v in q:
                codes.setdefault(l + m * M, len(codes))
        keys = list(codes) if _decode(case) == _capi.MMP_PAIRS_PHYSICAL else list(range(len(codes)))
        self.a = torch.tensor([x % M for x in keys], device=dev)
        self.b = torch.tensor([x // M for x in keys], device=dev)
        qd = np.zeros((M * M, len(codes)))
        for p, q in enumerate(entries):
            for kk, l, m, v in q:
                qd[p * M + kk, codes[l + m * M]] += v / qmax
        self.q = torch.tensor(qd, device=dev)
        self.raman = case["raman"]
        self.kv, self.kr = (1. - sp.raman_proportion, sp.raman_proportion * t0) if self.raman else (1., 0.)
        self.hr = torch.fft.fft(torch.tensor(sp.raman_response, device=dev).to(torch.complex128)) * self.dt
        self.psi = torch.fft.fft(torch.tensor(sp.initial_fields * self.conv, device=dev))
        self.a_rk, self.b_rk, self.c_rk = _tableau(case["order"])
        self.n = 0

    def nonlinear(self, u):
        v = u[self.a] * u[self.b].conj()
        x = self.kv * v
        if self.raman:
            x = x + self.kr * torch.fft.ifft(torch.fft.fft(v) * self.hr)
        w = torch.complex(self.q @ x.real.contiguous(), self.q @ x.imag.contiguous()).view(self.M, self.M, self.nt)
        return self.isgn * torch.fft.fft((w * u[None]).sum(1))

    def advance(self, steps):
        for _ in range(steps):
            ns, acc = [], self.psi
            e_c = {c: torch.exp(1j * (self.lam * ((self.n + c) * self.h))) for c in set(self.c_rk)}
            for i in range(len(self.b_rk)):
                x = self.psi
                for j, aij in enumerate(self.a_rk[i]):
                    if aij:
                        x = x + (aij * self.h) * ns[j]
                e = e_c[self.c_rk[i]]
                n = e.conj() * self.nonlinear(torch.fft.ifft(e * x))
                ns.append(n)
                if self.b_rk[i]:
                    acc = acc + (self.b_rk[i] * self.h) * n
            self.psi = acc
            self.n += 1

    def _field(self):
        return torch.fft.ifft(torch.exp(1j * (self.lam * (self.n * self.h))) * self.psi) / self.conv

    def field(self):
        return self._field().cpu().numpy()

    def energy(self):
        return (self._field().abs() ** 2).sum(1).cpu().numpy() * (self.sp.time_window / self.nt)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if _cost(case) > (8e11 if dev == "cuda" else 4e9):
        return None
    fibers = [_Exact(sp, case, dev) for sps in _all_params(case, seed) for sp in sps]
    if case["kind"] == "snapshots":
        x, fields = fibers[0], []
        for _ in range(case["saves"]):
            x.advance(case["steps"] // case["saves"])
            fields.append(x.field())
        z = (np.arange(case["saves"]) + 1.) / case["saves"] * x.sp.fiber_length
        return {"field": np.stack(fields), "z": z}
    for x in fibers:
        x.advance(case["steps"])
    many = case["kind"] in ("batch", "group")
    out = {"field": [x.field() for x in fibers] if many else fibers[0].field()}
    if case.get("energy"):
        out["energy"] = [x.energy() for x in fibers] if many else fibers[0].energy()
    return out
