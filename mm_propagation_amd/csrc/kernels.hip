// kernels.hip -- gfx950 kernels of the Lawson-Runge-Kutta propagation step.
//
// One RK stage i of a step is, in the four-step layout of kernels.h:
//   row_head(i)        rows: finish N_{i-1} (row DFT of sigma, conj(E) phase,
//                      RK accumulate) and build E_i * (psi + h sum a_ij N_j),
//                      then the inverse row DFT
//   col_inverse        columns: inverse column DFT -> U (time domain)
//   col_pairs_forward  columns: pair products of U, forward column DFT   (Raman on)
//   row_raman          rows: DFT, multiply by the Raman spectrum, inverse DFT
//   col_inverse        columns: -> Raman-convolved pair products (time domain)
//   gather             samples: Kerr + Raman sum sigma_p
//   col_forward        columns: forward column DFT of sigma
// and row_head(s) closes the step. The state psi is kept as its spectrum, so the
// reference's F^-1 F round trips between stages vanish (exact algebra; results
// differ from the reference by rounding only).
#include "kernels.h"

#include <hip/hip_ext.h>

#include <mutex>
#include <type_traits>

namespace mmp {

thread_local LaunchEvents g_launch_events;

// Every launch goes through hipExtLaunchKernelGGL so that, when g_launch_events is set, the
// dispatch itself records its start and stop (no separate event packets around the kernel).
#define MMP_LAUNCH(KERNEL, GRID, BLOCK, SHMEM, STREAM, ...)                                               \
  hipExtLaunchKernelGGL(KERNEL, GRID, BLOCK, SHMEM, STREAM, g_launch_events.start, g_launch_events.stop, 0, \
                        __VA_ARGS__)

// ---------------------------------------------------------------------------
// configuration of the row and column passes
// ---------------------------------------------------------------------------
template <int L>
struct RowCfg {
  static constexpr int T = L / 8;                  // lanes per row
  static constexpr int G = T >= 64 ? 1 : 64 / T;   // rows per workgroup
  static constexpr int THREADS = G * T;            // 64 (128 for rows of 1024)
  static constexpr int SLOTS = LineSlots<L, 1>::value;
};

// Column passes: a workgroup transforms CB neighbouring columns of G lines.
// CB = 8 reads whole 128 B lines; CB = 4 or 2 gives more workgroups for small
// problems (the LDS layout is then padded to keep lanes on distinct banks).
template <int L, int CB>
struct ColCfg {
  static constexpr int T = L / 8;                               // lanes per column line
  static constexpr int G = (CB * T >= 64) ? 1 : 64 / (CB * T);  // lines per workgroup
  static constexpr int THREADS = G * CB * T;
  static constexpr int PAD = CB < 8 ? 1 : 0;
  static constexpr int SLOTS = LineSlots<L, PAD>::value;        // per column
};

// Block ids are dealt round-robin to the 8 XCDs; remap them so that consecutive
// logical blocks (neighbouring columns) run on one XCD and share its L2.
__device__ __forceinline__ int xcd_block(int bid, int nb) {
  if (nb % 8) return bid;
  return (bid % 8) * (nb / 8) + bid / 8;
}

// Streaming store for arrays the next kernel reads (it runs on other XCDs, whose L2s do not
// share lines with this one).
template <class T>
__device__ __forceinline__ void store_stream(cpx<T>* p, cpx<T> v) {
  if constexpr (sizeof(T) == 4) {
    // one 8-byte store per FP32 value (p is 8-byte aligned: cpx<float> is)
    const unsigned long long bits =
        (unsigned long long)__float_as_uint(v.re) | ((unsigned long long)__float_as_uint(v.im) << 32);
    __builtin_nontemporal_store(bits, reinterpret_cast<unsigned long long*>(p));
  } else {
    __builtin_nontemporal_store(v.re, &p->re);
    __builtin_nontemporal_store(v.im, &p->im);
  }
}
// The same in FP64 only: FP32 stores of the column kernels measured slower streamed.
template <class T>
__device__ __forceinline__ void store_stream64(cpx<T>* p, cpx<T> v) {
  if constexpr (std::is_same<T, double>::value) store_stream(p, v);
  else *p = v;
}

__device__ __forceinline__ cd phase(double imL, double tau) {
  double s, c;
  sincos(imL * tau, &s, &c);
  return {c, s};
}

// ---------------------------------------------------------------------------
// row stage head
// ---------------------------------------------------------------------------
// E <- E * E1 with the reference's rounding (no FMA contraction), so stored
// tables stay bit-identical to src/MultimodePropagation_CPU.cpp:41.
__device__ __forceinline__ cd cmul_exact(cd a, cd b) {
  return {__dsub_rn(__dmul_rn(a.re, b.re), __dmul_rn(a.im, b.im)),
          __dadd_rn(__dmul_rn(a.re, b.im), __dmul_rn(a.im, b.re))};
}

// RE: Lawson factors computed from Im L and the fiber's z (HeadArgs::recompute_e) instead of
// read from the tables; they are formed where they are used, so no table registers stay live.
// ST: stage i's argument takes stashed N_j (the tableaux beyond RK4). In FP64 two of them are requested
// together, since each trip to memory is exposed (a lone fiber's head has one wavefront per SIMD at
// most), and RK4 runs without that code: 5 modes, NT = 8192, sixth order 176.2 -> 164.6 us per step, RK4
// of two modes 71.2 -> 70.2. The table-free form has no registers for two (its second wavefront per SIMD
// would go), and without the loop its batched heads measured 3 % slower, so it keeps one form.
template <int L, class W, bool RE, bool ST>
__global__ void __launch_bounds__(RowCfg<L>::THREADS) k_row_head(Geometry g, const cpx<W>* __restrict__ rowtw, HeadArgs a, Batch b) {
  using C = RowCfg<L>;
  using cw = cpx<W>;
  __shared__ cw smem[C::G * C::SLOTS];
  const int tid = threadIdx.x;
  const int gl = tid / C::T, t = tid % C::T;
  const int row = blockIdx.x * C::G + gl;
  const bool valid = row < g.M * g.N1;
  const size_t base = valid ? (size_t)row * g.N2 + t : t;  // (lanes without a row: in bounds, not stored)
  cw* sm = smem + gl * C::SLOTS;
  const size_t MN = (size_t)g.M * g.N;
  // fiber blockIdx.y of the batch: its arrays and scalars
  const int fib = blockIdx.y;
  const FiberParams fp = b.fp[fib];
  if (!fp.live) return;  // uniform over the workgroup
  const double* __restrict__ hc = b.coef + ((size_t)fib * b.nheads + a.head) * kHeadCoef;  // uniform
  cd* __restrict__ psi_hat = a.psi_hat + fib * b.sf;
  cd* __restrict__ accp = a.acc + fib * b.sf;
  cd* __restrict__ stash = a.stash ? a.stash + fib * b.ss : nullptr;
  cd* __restrict__ e_prev = a.e_prev ? a.e_prev + fib * b.se : nullptr;
  const cd* __restrict__ e_cur = a.e_cur ? a.e_cur + fib * b.se : nullptr;
  const cd* __restrict__ e1p = a.e1 ? a.e1 + fib * b.sf : nullptr;
  const double* __restrict__ imLp = a.imL ? a.imL + fib * b.sf : nullptr;
  const cw* __restrict__ ysig = static_cast<const cw*>(a.ysig) + fib * b.sf;
  cw* __restrict__ yout = static_cast<cw*>(a.yout) + fib * b.sf;
  LineTw<L, W> lt;
  load_line_tw<L>(lt, rowtw, t);

  // issue every load this lane needs before the first barrier
  cw v[8];
  cd x[8], accb[8];
  cd ep[RE ? 1 : 8], ec[RE ? 1 : 8], e1[RE ? 1 : 8];  // Lawson tables (not RE)
  double lam[RE ? 8 : 1];                              // Im L (RE)
  const cd zero = {0., 0.};
  const bool want_cur = !a.final_stage || a.chain_next;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const size_t idx = base + i * C::T;
    if constexpr (RE) lam[i] = valid ? imLp[idx] : 0.;
    v[i] = (valid && a.has_prev) ? ysig[idx] : cw{0, 0};
    if constexpr (!RE) ep[i] = (valid && a.has_prev) ? e_prev[idx] : zero;
    const cd psi = (valid && (a.prev_is_first || !a.final_stage)) ? psi_hat[idx] : zero;
    const cd accin = (valid && a.has_prev && !a.prev_is_first) ? accp[idx] : zero;
    accb[i] = a.prev_is_first ? psi : accin;  // the step result so far
    x[i] = psi;                               // stage i's argument (not the final stage)
    if constexpr (!RE) {
      e1[i] = (valid && a.update_prev) ? e1p[idx] : zero;
      ec[i] = (valid && want_cur) ? e_cur[idx] : zero;
    }
  }
  // RE: E_{i-1} = exp(i Im L (n + c_{i-1}) h), E_i = exp(i Im L (n + c_i) h) with n the steps
  // taken before this one (one rounding of the distance, where z sums h step by step); the
  // close head's block 0 advances the count in this kernel, so it reads n from n0 (recorded by
  // stage head 1) and its chained next stage 0 is at n + 1
  // (both at one distance, as in a stage that repeats c or a close with c_{s-1} = 1: E_{i-1}
  // serves both, applied to the stage product as soon as that is formed)
  double tp = 0., tc = 0.;
  bool same = false;
  if constexpr (RE) {
    const double n = a.final_stage ? b.st[fib].n0 : (double)b.st[fib].steps;  // uniform
    tp = (n + a.c_prev) * fp.h;
    tc = ((a.final_stage ? n + 1.0 : n) + a.c_cur) * fp.h;
    same = a.has_prev && want_cur && tp == tc;
    if (a.set_n0 && blockIdx.x == 0 && threadIdx.x == 0) b.st[fib].n0 = n;
  }
  if (a.final_stage && a.advance_z && blockIdx.x == 0 && threadIdx.x == 0) {
    b.st[fib].z += fp.h;  // z += h (repeated FP64 addition)
    b.st[fib].steps += 1;
  }
  // stage i's argument psi + sum_j a_ij h N_j over j < i in increasing j: the stashed N_j now,
  // N_{i-1} (the largest j, from this head's transform) last
  if constexpr (ST) {
    int e = 0;
    if constexpr (!RE) {
#pragma unroll 1
      for (; e + 2 <= a.n_stash; e += 2) {
        const cd* n0 = stash + (size_t)a.a_idx[e] * MN + base;
        const cd* n1 = stash + (size_t)a.a_idx[e + 1] * MN + base;
        cd t0[8], t1[8];
#pragma unroll
        for (int i = 0; i < 8; i++) t0[i] = n0[i * C::T];
#pragma unroll
        for (int i = 0; i < 8; i++) t1[i] = n1[i * C::T];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = cadd(cadd(x[i], cscale(t0[i], hc[1 + e])), cscale(t1[i], hc[2 + e]));
      }
    }
#pragma unroll 1
    for (; e < a.n_stash; e++) {
      const cd* n0 = stash + (size_t)a.a_idx[e] * MN + base;
      cd t0[8];
#pragma unroll
      for (int i = 0; i < 8; i++) t0[i] = n0[i * C::T];
#pragma unroll
      for (int i = 0; i < 8; i++) x[i] = cadd(x[i], cscale(t0[i], hc[1 + e]));
    }
  }
  // the Lawson table of stage i-1 moves on by E1 (it is not read again in this step)
  if constexpr (!RE) {
    if (a.has_prev && a.update_prev && valid) {
#pragma unroll
      for (int i = 0; i < 8; i++) store_stream(e_prev + base + i * C::T, cmul_exact(ep[i], e1[i]));
    }
  }
  if (a.has_prev) {
    const double bh = hc[0];
    const double cprev = a.prev_term ? hc[a.n_a] : 0.;
    line_fft<L, -1, 1, 1>(v, sm, lt, t);
    bool finite = true;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const size_t idx = base + i * C::T;
      cd epi;
      if constexpr (RE) epi = phase(lam[i], tp);
      else epi = ep[i];
      const cd y = cmulc(widen(v[i]), epi);         // sigma_hat * conj(E_{i-1})
      const cd nh = {-y.im * fp.sgn, y.re * fp.sgn};  // * (i sgn) = N_{i-1}
      cd acc = accb[i];
      if (a.b_prev != 0.) acc = cadd(acc, cscale(nh, bh));
      finite = finite && __builtin_isfinite(acc.re) && __builtin_isfinite(acc.im);
      if (valid) {
        if (a.final_stage) store_stream(psi_hat + idx, acc);
        else store_stream(accp + idx, acc);
        if (a.stash_prev) store_stream(stash + (size_t)a.prev_stage * MN + idx, nh);
      }
      if (a.final_stage) x[i] = acc;  // chain_next: stage 0 of the next step from the new psi_hat
      else if (a.prev_term) x[i] = cadd(x[i], cscale(nh, cprev));
      if constexpr (RE) {
        if (same) x[i] = cmul(epi, x[i]);  // E_i x_i
      }
    }
    // a state that is no longer finite stays so: the fiber is parked (every lane that sees it
    // stores the same values), its later kernels skip it and its z and step count stop here
    if (a.final_stage && valid && !finite) {
      b.st[fib].halted = 1u;
      b.fp[fib].live = 0u;
    }
  }
  if (a.final_stage && !a.chain_next) return;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    cd ex;  // E_i x_i
    if constexpr (RE) ex = same ? x[i] : cmul(phase(lam[i], tc), x[i]);
    else ex = cmul(ec[i], x[i]);
    v[i] = narrow<W>(cscale(ex, a.scale_cur));
  }
  line_fft<L, 1, 1, 1>(v, sm, lt, t);
  if (valid) {
#pragma unroll
    for (int i = 0; i < 8; i++) store_stream(yout + base + i * C::T, v[i]);
  }
}

// ---------------------------------------------------------------------------
// column passes
// ---------------------------------------------------------------------------
struct ColIdx {
  int c, t, gl, cb, lg;
};

// lane -> (column c, line lane t, line gl) and block -> (column block cb, line group lg)
template <int L, int CB>
__device__ __forceinline__ ColIdx col_index(int ncb) {
  using C = ColCfg<L, CB>;
  const int tid = threadIdx.x;
  const int lb = xcd_block(blockIdx.x, gridDim.x);
  return {tid % CB, (tid / CB) % C::T, tid / (CB * C::T), lb % ncb, lb / ncb};
}

// inverse column DFT: in = spectral-side rows (k1), out = time domain, times scale, divided by divisor
template <int L, int CB, class W>
__global__ void __launch_bounds__(256) k_col_inverse(Geometry g, const cpx<W>* __restrict__ coltw,
                                                     const cpx<W>* __restrict__ fourtw, const cpx<W>* in,
                                                     cpx<W>* out, int lines, double scale, double divisor) {
  using C = ColCfg<L, CB>;
  using cw = cpx<W>;
  __shared__ cw smem[C::G * C::SLOTS * CB];
  const ColIdx ix = col_index<L, CB>(g.N2 / CB);
  const int q = ix.lg * C::G + ix.gl;
  const int n2 = ix.cb * CB + ix.c;
  const bool valid = q < lines;
  const size_t base = (size_t)(valid ? q : 0) * g.N + n2;
  cw* sm = smem + ix.gl * C::SLOTS * CB + ix.c;
  LineTw<L, W> lt;
  load_line_tw<L>(lt, coltw, ix.t);
  cw v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int k1 = ix.t + i * C::T;
    v[i] = valid ? cmulc(in[base + (size_t)k1 * g.N2], fourtw[n2 * k1]) : cw{0, 0};
  }
  line_fft<L, 1, CB, C::PAD>(v, sm, lt, ix.t);
  if (valid) {
    const W sc = (W)scale, dv = (W)divisor;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int n1 = ix.t + i * C::T;
      cw x = cscale(v[i], sc);
      if (divisor != 1.0) x = {x.re / dv, x.im / dv};
      out[base + (size_t)n1 * g.N2] = x;
    }
  }
}

// forward column DFT + four-step twiddle: in = time domain, out = spectral-side rows
template <int L, int CB, class W>
__global__ void __launch_bounds__(256) k_col_forward(Geometry g, const cpx<W>* __restrict__ coltw,
                                                     const cpx<W>* __restrict__ fourtw, const cpx<W>* in,
                                                     cpx<W>* out, int lines) {
  using C = ColCfg<L, CB>;
  using cw = cpx<W>;
  __shared__ cw smem[C::G * C::SLOTS * CB];
  const ColIdx ix = col_index<L, CB>(g.N2 / CB);
  const int q = ix.lg * C::G + ix.gl;
  const int n2 = ix.cb * CB + ix.c;
  const bool valid = q < lines;
  const size_t base = (size_t)(valid ? q : 0) * g.N + n2;
  cw* sm = smem + ix.gl * C::SLOTS * CB + ix.c;
  LineTw<L, W> lt;
  load_line_tw<L>(lt, coltw, ix.t);
  cw v[8], w4[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int n1 = ix.t + i * C::T;
    v[i] = valid ? in[base + (size_t)n1 * g.N2] : cw{0, 0};
    w4[i] = fourtw[n2 * n1];  // index k1 = n1 after the transform
  }
  line_fft<L, -1, CB, C::PAD>(v, sm, lt, ix.t);
  if (valid) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int k1 = ix.t + i * C::T;
      out[base + (size_t)k1 * g.N2] = cmul(v[i], w4[i]);
    }
  }
}

// forward column DFT of one real line (the Raman response), FP64 only
template <int L, int CB, class W>
__global__ void __launch_bounds__(256) k_col_forward_real(Geometry g, const cd* __restrict__ coltw,
                                                          const cd* __restrict__ fourtw, const double* __restrict__ in,
                                                          cd* __restrict__ out) {
  using C = ColCfg<L, CB>;
  __shared__ cd smem[C::G * C::SLOTS * CB];
  const ColIdx ix = col_index<L, CB>(g.N2 / CB);
  const bool valid = ix.lg * C::G + ix.gl < 1;
  const int n2 = ix.cb * CB + ix.c;
  cd* sm = smem + ix.gl * C::SLOTS * CB + ix.c;
  LineTw<L> lt;
  load_line_tw<L>(lt, coltw, ix.t);
  cd v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int n1 = ix.t + i * C::T;
    v[i] = valid ? cd{in[(size_t)n1 * g.N2 + n2], 0.} : cd{0., 0.};
  }
  line_fft<L, -1, CB, C::PAD>(v, sm, lt, ix.t);
  if (valid) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int k1 = ix.t + i * C::T;
      out[(size_t)k1 * g.N2 + n2] = cmul(v[i], fourtw[n2 * k1]);
    }
  }
}

// pair products of the time-domain fields U (two real products a line), then forward column DFT
template <int L, int CB, class W>
__global__ void __launch_bounds__(256) k_col_pairs_forward(Geometry g, const cpx<W>* __restrict__ coltw,
                                                           const cpx<W>* __restrict__ fourtw,
                                                           const cpx<W>* __restrict__ U, cpx<W>* __restrict__ out,
                                                           int lines, const uint2* __restrict__ line_prod) {
  using C = ColCfg<L, CB>;
  using cw = cpx<W>;
  __shared__ cw smem[C::G * C::SLOTS * CB];
  const ColIdx ix = col_index<L, CB>(g.N2 / CB);
  const int q = ix.lg * C::G + ix.gl;
  const int n2 = ix.cb * CB + ix.c;
  const bool valid = q < lines;
  const int qq = valid ? q : 0;
  const uint2 d = line_prod[qq];
  const cw* const a0 = U + (size_t)(d.x & 255u) * g.N;
  const cw* const b0 = U + (size_t)((d.x >> 8) & 255u) * g.N;
  const cw* const a1 = U + (size_t)(d.y & 255u) * g.N;
  const cw* const b1 = U + (size_t)((d.y >> 8) & 255u) * g.N;
  const bool im0 = (d.x >> 16) & 1u, im1 = (d.y >> 16) & 1u, has1 = !((d.y >> 17) & 1u);
  const bool same = !((d.x ^ d.y) & 0xffffu);  // both parts of one pair's product
  cw* sm = smem + ix.gl * C::SLOTS * CB + ix.c;
  LineTw<L, W> lt;
  load_line_tw<L>(lt, coltw, ix.t);
  cw v[8], w4[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int n1 = ix.t + i * C::T;
    const size_t tt = (size_t)n1 * g.N2 + n2;
    cw x = {0, 0};
    if (valid) {
      const cw x0 = cmulc(a0[tt], b0[tt]);
      cw x1 = x0;
      if (has1 && !same) x1 = cmulc(a1[tt], b1[tt]);
      x = {im0 ? x0.im : x0.re, has1 ? (im1 ? x1.im : x1.re) : (W)0};
    }
    v[i] = x;
    w4[i] = fourtw[n2 * n1];
  }
  line_fft<L, -1, CB, C::PAD>(v, sm, lt, ix.t);
  if (valid) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int k1 = ix.t + i * C::T;
      out[(size_t)q * g.N + (size_t)k1 * g.N2 + n2] = cmul(v[i], w4[i]);
    }
  }
}

// ---------------------------------------------------------------------------
// row passes
// ---------------------------------------------------------------------------
template <int L>
__global__ void __launch_bounds__(RowCfg<L>::THREADS) k_row_forward(Geometry g, const cd* __restrict__ rowtw, cd* __restrict__ data,
                                                    int lines) {
  using C = RowCfg<L>;
  __shared__ cd smem[C::G * C::SLOTS];
  const int tid = threadIdx.x;
  const int gl = tid / C::T, t = tid % C::T;
  const int row = blockIdx.x * C::G + gl;
  const bool valid = row < lines * g.N1;
  const size_t base = valid ? (size_t)row * g.N2 : 0;  // rows of consecutive lines are contiguous
  cd* sm = smem + gl * C::SLOTS;
  LineTw<L> lt;
  load_line_tw<L>(lt, rowtw, t);
  cd v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = valid ? data[base + t + i * C::T] : cd{0., 0.};
  line_fft<L, -1, 1, 1>(v, sm, lt, t);
  if (valid) {
#pragma unroll
    for (int i = 0; i < 8; i++) data[base + t + i * C::T] = v[i];
  }
}

// optional phase exp(i ImL z) (the reference's exp(L z)), then inverse row DFT
template <int L>
__global__ void __launch_bounds__(RowCfg<L>::THREADS) k_row_inverse_phase(Geometry g, const cd* __restrict__ rowtw,
                                                          const cd* __restrict__ in, cd* __restrict__ out,
                                                          const double* __restrict__ imL,
                                                          const StepState* __restrict__ st, int use_phase) {
  using C = RowCfg<L>;
  __shared__ cd smem[C::G * C::SLOTS];
  const int tid = threadIdx.x;
  const int gl = tid / C::T, t = tid % C::T;
  const int row = blockIdx.x * C::G + gl;
  const bool valid = row < g.M * g.N1;
  const size_t base = valid ? (size_t)row * g.N2 : 0;
  cd* sm = smem + gl * C::SLOTS;
  const double z = st->z;
  LineTw<L> lt;
  load_line_tw<L>(lt, rowtw, t);
  cd v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const size_t idx = base + t + i * C::T;
    cd x = valid ? in[idx] : cd{0., 0.};
    if (use_phase && valid) x = cmul(x, phase(imL[idx], z));
    v[i] = x;
  }
  line_fft<L, 1, 1, 1>(v, sm, lt, t);
  if (valid) {
#pragma unroll
    for (int i = 0; i < 8; i++) out[base + t + i * C::T] = v[i];
  }
}

// Raman convolution in the spectral rows: DFT, * H * hscale, inverse DFT (in place)
template <int L, class W>
__global__ void __launch_bounds__(RowCfg<L>::THREADS) k_row_raman(Geometry g, const cpx<W>* __restrict__ rowtw,
                                                  cpx<W>* __restrict__ data, int lines,
                                                  const cpx<W>* __restrict__ hspec, Batch b) {
  using C = RowCfg<L>;
  using cw = cpx<W>;
  __shared__ cw smem[C::G * C::SLOTS];
  const int fib = blockIdx.y;
  if (!b.fp[fib].live) return;  // uniform over the workgroup
  data += fib * b.sl;
  hspec += fib * b.sh;
  const double hscale = b.fp[fib].dt;
  const int tid = threadIdx.x;
  const int gl = tid / C::T, t = tid % C::T;
  const int row = blockIdx.x * C::G + gl;
  const bool valid = row < lines * g.N1;
  const size_t base = valid ? (size_t)row * g.N2 : 0;
  const size_t hbase = valid ? (size_t)(row % g.N1) * g.N2 : 0;
  cw* sm = smem + gl * C::SLOTS;
  LineTw<L, W> lt;
  load_line_tw<L>(lt, rowtw, t);
  cw v[8], hs[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    v[i] = valid ? data[base + t + i * C::T] : cw{0, 0};
    hs[i] = hspec[hbase + t + i * C::T];
  }
  line_fft<L, -1, 1, 1>(v, sm, lt, t);
  const W hsc = (W)hscale;
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = cscale(cmul(v[i], hs[i]), hsc);
  line_fft<L, 1, 1, 1>(v, sm, lt, t);
  if (valid) {
#pragma unroll
    for (int i = 0; i < 8; i++) data[base + t + i * C::T] = v[i];
  }
}

// Raman row pass of the column-stage step: the arithmetic of k_row_raman, with R consecutive
// rows of one line per workgroup (n1 .. n1 + R - 1), its lines read from `in` and stored to
// `out` in column order (sample (n1, n2) of a line at n2 * N1 + n1). The rows are staged in
// LDS as [n2][R + 1] on the way in and out, so that every load and store moves runs of R
// consecutive samples; the column kernels on either side (the pair pass writing the lines,
// the gather reading them) then move each column of a line as one contiguous run instead of
// N1 samples N2 apart. R is the
// largest of 16 (FP32) or 8 (FP64), halved as needed, that keeps the workgroup within 512
// threads and 50 KB of LDS: measured on one MI355X, wider workgroups lose more to occupancy
// than the longer runs gain (FP64 rows of 1024: R = 2 60 us, R = 4 83 us; FP32 rows of 1024:
// R = 4 21.7 us, R = 8 27.4 us; FP32 rows of 256: R = 16 111 us, R = 8 131 us).
template <int L, class W>
constexpr int raman_cols_rows() {
  constexpr int slots = LineSlots<L, 1>::value;
  int r = std::is_same<W, float>::value ? 16 : 8;
  while (r > 1) {
    const int lds = (r * slots > L * (r + 1) ? r * slots : L * (r + 1)) * (int)sizeof(cpx<W>);
    if (r * (L / 8) <= 512 && lds <= 51200) break;
    r /= 2;
  }
  return r;
}
template <int L, class W>
struct RamanColsCfg {
  static constexpr int T = L / 8;                              // lanes per row
  static constexpr int R = raman_cols_rows<L, W>();            // rows per workgroup
  static constexpr int THREADS = R * T;
  static constexpr bool WAVE = T <= 64;                        // each row inside one wavefront
  static constexpr int SLOTS = LineSlots<L, 1>::value;
  static constexpr int FFT = R * SLOTS;                        // transform rows
  static constexpr int STAGE = L * (R + 1);                    // [n2][R + 1] staging
  static constexpr int LDS = FFT > STAGE ? FFT : STAGE;
};

template <int L, class W>
__global__ void __launch_bounds__((RamanColsCfg<L, W>::THREADS)) k_row_raman_cols(Geometry g, const cpx<W>* __restrict__ rowtw,
                                                                            const cpx<W>* __restrict__ in,
                                                                            cpx<W>* __restrict__ out,
                                                                            const cpx<W>* __restrict__ hspec, Batch b,
                                                                            int in_cols) {
  using C = RamanColsCfg<L, W>;
  using cw = cpx<W>;
  __shared__ cw smem[C::LDS];
  const int fib = blockIdx.y;
  if (!b.fp[fib].live) return;  // uniform over the workgroup
  in += fib * b.sl;
  out += fib * b.sl;
  hspec += fib * b.sh;
  const double hscale = b.fp[fib].dt;
  const int tid = threadIdx.x;
  const int r = tid / C::T, t = tid % C::T;
  // R divides N1: the rows share one line. In FP32 neighbouring row groups run on one XCD, so
  // the parts of a cache line that several of them store meet in one L2 (measured: rows of 1024
  // 23.7 -> 21.7 us); FP64 runs of 8 rows already fill 128-byte lines, and there the plain
  // order measured slightly faster (rows of 256: 5.09 vs 5.21 us)
  // Where those FP32 runs fill whole 128-byte lines (R = 16) the blocks take the lines fastest
  // instead, so the blocks on one XCD share row groups and read only those rows of the Raman
  // spectrum (every XCD reading all of it fetched the spectrum 8 times from HBM)
  const int blk = std::is_same<W, float>::value ? xcd_block(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  int row0 = blk * C::R;
  if constexpr (std::is_same<W, float>::value && C::R * sizeof(cw) >= 128) {
    const int nl = (int)gridDim.x * C::R / g.N1;  // lines of the launch
    if (gridDim.x % 8 == 0) row0 = (blk % nl) * g.N1 + (blk / nl) * C::R;
  }
  const int line = row0 / g.N1, n10 = row0 % g.N1, n1 = n10 + r;
  const size_t cbase = (size_t)line * g.N + n10;  // the R rows' first sample in column order
  const size_t hbase = (size_t)n1 * g.N2;
  cw* sm = smem + r * C::SLOTS;
  cw v[8], hs[8];
  if (in_cols) {  // uniform branch: lines in column order, staged through LDS
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int e = tid + k * C::THREADS;  // R * L = 8 * THREADS samples
      const int rr = e % C::R, n2 = e / C::R;
      smem[n2 * (C::R + 1) + rr] = in[cbase + (size_t)n2 * g.N1 + rr];
    }
  } else {  // lines in row order: each row read directly
    const size_t rbase = (size_t)line * g.N + (size_t)n1 * g.N2;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = in[rbase + t + i * C::T];
  }
#pragma unroll
  for (int i = 0; i < 8; i++) hs[i] = hspec[hbase + t + i * C::T];
  LineTw<L, W> lt;
  load_line_tw<L>(lt, rowtw, t);
  if (in_cols) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = smem[(t + i * C::T) * (C::R + 1) + r];
    __syncthreads();  // the staging area becomes the rows' transform slots
  }
  line_fft<L, -1, 1, 1, W, C::WAVE>(v, sm, lt, t);
  const W hsc = (W)hscale;
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = cscale(cmul(v[i], hs[i]), hsc);
  line_fft<L, 1, 1, 1, W, C::WAVE>(v, sm, lt, t);
  __syncthreads();  // every row's transform is done with its LDS row before the staging reuses it
#pragma unroll
  for (int i = 0; i < 8; i++) smem[(t + i * C::T) * (C::R + 1) + r] = v[i];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int e = tid + k * C::THREADS;  // R * L = 8 * THREADS staged samples
    const int rr = e % C::R, n2 = e / C::R;
    if constexpr (C::R * sizeof(cw) >= 128) store_stream(out + cbase + (size_t)n2 * g.N1 + rr, smem[n2 * (C::R + 1) + rr]);
    else out[cbase + (size_t)n2 * g.N1 + rr] = smem[n2 * (C::R + 1) + rr];
  }
}

// ---------------------------------------------------------------------------
// Kerr + Raman gather over a tile of 64 consecutive samples:
//   X_slot = kv * U_a conj(U_b) + kr * VR_slot        (slot mix, into LDS)
//   sigma_p = sum over the nonzeros (k, slot, q) of Q^(p):  q * X_slot * U_k
// One wavefront per mode p (lanes = samples; wavefronts of blockIdx.y's groups take turns where the
// modes are more), so the nonzero loop and its metadata loads are uniform; nonzeros are sorted by slot
// so consecutive ones reuse X. Slots are staged through LDS in chunks when M + P exceeds the tile.
// ---------------------------------------------------------------------------
// sum += q_e * X[slot_e - s0] * U[k_e] over the nonzeros [e0, e1) for this lane's sample.
// e0, e1 and s0 are wave-uniform. Xs and Us point at the lane's sample in LDS rows of
// `stride` values. Lane l loads nonzero eb + l; v_readlane broadcasts it, eight at a
// time, so the sixteen LDS reads of a batch are in flight together. The products are
// added in nonzero order.
// Broadcast lane j's coefficient (kept as its bit pattern in one or two ints) to the wave.
struct QBits {
  int lo, hi;
};
__device__ __forceinline__ QBits q_bits(double v) { return {__double2loint(v), __double2hiint(v)}; }
__device__ __forceinline__ QBits q_bits(float v) { return {__float_as_int(v), 0}; }
template <class W>
__device__ __forceinline__ W q_lane(QBits b, int j) {
  if constexpr (sizeof(W) == 8)
    return __hiloint2double(__builtin_amdgcn_readlane(b.hi, j), __builtin_amdgcn_readlane(b.lo, j));
  else
    return __int_as_float(__builtin_amdgcn_readlane(b.lo, j));
}

template <class W>
__device__ __forceinline__ cpx<W> gather_sum(cpx<W> sum, const uint32_t* __restrict__ kslot, const W* __restrict__ q,
                                             uint32_t e0, uint32_t e1, int s0, const cpx<W>* Xs, const cpx<W>* Us,
                                             int stride, int lane) {
  constexpr int B = 8;
  for (uint32_t eb = e0; eb < e1; eb += 64) {
    const uint32_t mine = eb + lane;
    const uint32_t ks = mine < e1 ? kslot[mine] : 0u;
    const QBits qb = q_bits(mine < e1 ? q[mine] : (W)0);
    const int cnt = (int)min(64u, e1 - eb);
    int j = 0;
    for (; j + B <= cnt; j += B) {
      cpx<W> xs[B], us[B];
      W qs[B];
#pragma unroll
      for (int u = 0; u < B; u++) {
        const uint32_t ksj = (uint32_t)__builtin_amdgcn_readlane((int)ks, j + u);
        qs[u] = q_lane<W>(qb, j + u);
        xs[u] = Xs[((int)(ksj >> 8) - s0) * stride];
        us[u] = Us[(int)(ksj & 255u) * stride];
      }
#pragma unroll
      for (int u = 0; u < B; u++) sum = cadd(sum, cscale(cmul(xs[u], us[u]), qs[u]));
    }
    for (; j < cnt; j++) {
      const uint32_t ksj = (uint32_t)__builtin_amdgcn_readlane((int)ks, j);
      const W qj = q_lane<W>(qb, j);
      sum = cadd(sum, cscale(cmul(Xs[((int)(ksj >> 8) - s0) * stride], Us[(int)(ksj & 255u) * stride]), qj));
    }
  }
  return sum;
}

// Slot mixes of a 64-sample tile into LDS: X[s - s0][j] = kv U_a conj(U_b) + kr VR_s[t0 + j]
// for slots [s0, s0 + ns). Every Raman value a lane needs is loaded before any is used, so
// the loads overlap instead of each waiting for the previous one.
template <class W>
__device__ __forceinline__ void slot_mix_tile(const GatherArgs& a, const Geometry& g, const cpx<W>* __restrict__ VR,
                                              const cpx<W>* Ush, cpx<W>* Xsh, int s0, int ns, int t0, int tid,
                                              int NTHR) {
  using cw = cpx<W>;
  constexpr int TS = 64, R = 16;
  const int total = ns * TS;
  const W kv = (W)a.kv, kr = (W)a.kr;
  for (int base = 0; base < total; base += R * NTHR) {
    cw r[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int e = base + tid + i * NTHR;
      r[i] = {0, 0};
      // e / 64 is the same for the whole wavefront (e = base + 64 * wave + lane + i * NTHR)
      const int sl = __builtin_amdgcn_readfirstlane(s0 + e / TS);
      if (a.raman && e < total) r[i] = VR[(size_t)a.slot_line[sl] * g.N + t0 + e % TS];
    }
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int e = base + tid + i * NTHR;
      if (e >= total) break;
      const int sl = __builtin_amdgcn_readfirstlane(s0 + e / TS), j = e % TS;
      const cw V = cmulc(Ush[a.slot_a[sl] * TS + j], Ush[a.slot_b[sl] * TS + j]);
      cw X = cscale(V, kv);
      if (a.raman) {
        cw vr;
        switch (a.slot_kind[sl]) {
          case kDirect: vr = r[i]; break;
          case kConj: vr = cconj(r[i]); break;
          case kRe: vr = {r[i].re, 0}; break;
          default: vr = {r[i].im, 0}; break;
        }
        X = cadd(X, cscale(vr, kr));
      }
      Xsh[e] = X;
    }
  }
}

constexpr int kGatherTS = 64;
constexpr int kGatherMaxPW = 8;  // modes per wavefront

void gather_plan(int M, int P, int& cap, int& chunk) {
  cap = 0;
  chunk = 0;
  const int caps[2] = {4096, 8192};
  for (int c : caps) {
    const int room = c / kGatherTS - M;
    if (room <= 0) continue;
    if (room >= P || c == 8192) {
      cap = c;
      chunk = room < P ? room : P;
      return;
    }
  }
}

template <int CAP, class W>
__global__ void __launch_bounds__(512) k_gather(Geometry g, const cpx<W>* __restrict__ U,
                                                const cpx<W>* __restrict__ VR, cpx<W>* __restrict__ sigma,
                                                GatherArgs a) {
  using cw = cpx<W>;
  __shared__ cw sh[CAP];
  constexpr int TS = kGatherTS;
  const int M = g.M;
  const W* __restrict__ qv = static_cast<const W*>(a.q);
  cw* Ush = sh;            // [M][TS]
  cw* Xsh = sh + M * TS;   // [chunk][TS]
  const int t0 = blockIdx.x * TS;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int lane = tid % TS, nwaves = nthr / TS, ny = gridDim.y;
  const int wave = __builtin_amdgcn_readfirstlane(tid / TS);  // wave-uniform for the compiler
#pragma unroll 4
  for (int e = tid; e < M * TS; e += nthr) Ush[e] = U[(size_t)(e / TS) * g.N + t0 + e % TS];
  cw acc[kGatherMaxPW];
#pragma unroll
  for (int r = 0; r < kGatherMaxPW; r++) acc[r] = {0, 0};
  for (int c = 0; c < a.n_chunks; c++) {
    const int s0 = c * a.chunk;
    const int ns = min(a.chunk, a.n_slots - s0);
    __syncthreads();  // Ush loaded / previous chunk consumed
    slot_mix_tile(a, g, VR, Ush, Xsh, s0, ns, t0, tid, nthr);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kGatherMaxPW; r++) {
      const int p = wave + (r * ny + blockIdx.y) * nwaves;
      if (p >= M) break;
      const uint32_t* co = a.coff + (size_t)p * (a.n_chunks + 1) + c;
      acc[r] = gather_sum(acc[r], a.kslot, qv, co[0], co[1], s0, Xsh + lane, Ush + lane, TS, lane);
    }
  }
#pragma unroll
  for (int r = 0; r < kGatherMaxPW; r++) {
    const int p = wave + (r * ny + blockIdx.y) * nwaves;
    if (p >= M) break;
    sigma[(size_t)p * g.N + t0 + lane] = acc[r];
  }
}

// ---------------------------------------------------------------------------
// Column-stage kernels (N1 = 64, M <= 16; with Raman, and C2 in FP64 also without). One workgroup of 256 lanes
// or more owns one column n2, or a few neighbouring ones, and does every column-side step of a stage there, with
// the column of each field and Raman line held in LDS between the steps:
//   C1  inverse column DFT of the M fields -> U (HBM, column order, and LDS) -> pair
//       products -> forward column DFT of the Raman lines -> conv (row order, or column
//       order on large grids; the Raman row pass reads them so and writes column order)
//   C2  inverse column DFT of the Raman lines (column order; kept in LDS) -> dense Kerr +
//       Raman gather of the 64 samples, forming each slot mix X_s on the way -> forward
//       column DFT of sigma -> yout; without Raman the inverse column DFT of the fields takes the lines' place
// Column order: sample (n1, n2) of an array at n2 * N1 + n1, so that a column is one
// contiguous run of N1 samples.
// Lanes form 32 line slots of 8 lanes; a round transforms up to 32 lines.
// ---------------------------------------------------------------------------
constexpr int kColStageL = 64;       // column length the column-stage kernels take
constexpr int kColStageMaxM = 16;    // modes kept in registers by the gather
// LDS limits of one chunk, by mode count: a few modes have few lines and small coupling
// blocks, and a small LDS footprint lets more workgroups share a CU (batched fibers)
constexpr int colstage_lines_cap(int M) { return M <= 4 ? 16 : (M <= 6 ? 24 : 40); }  // Raman lines
// FP32: coupling coefficients held in LDS
constexpr int colstage_qcap(int M) { return M <= 4 ? 1024 : (M <= 6 ? 2048 : (M <= 10 ? 4096 : 8192)); }
// of those, prefetched into registers before the chunk's barrier (the rest go straight to LDS):
// what a small tensor needs in all (up to 4 modes: 512, up to 6: 1024, parity-compact), 4096
// where the registers allow it (7 to 12 modes), else 2048
constexpr int colstage_qpre(int M) { return M <= 4 ? 512 : (M <= 6 ? 1024 : (M <= 12 ? 4096 : 2048)); }
constexpr int kColStageSCap = 128;   // slots of one chunk
constexpr int kColStageRS = LineSlots<kColStageL, 1>::value;  // LDS row stride of a line (72)
// LDS rows for the lines of a chunk: every wavefront of a round transforms 8 line slots, so
// the rows cover the chunk's lines rounded up to 8
constexpr int colstage_rows(int M) { return (colstage_lines_cap(M) + 7) / 8 * 8; }

struct ColStageCfg {
  static constexpr int L = kColStageL;
  static constexpr int T = L / 8;                      // 8 lanes per line
  static constexpr int NL = 256 / T;                   // 32 line slots per round
  static constexpr int SLOTS = LineSlots<L, 1>::value;  // 72
  static constexpr int FFT = NL * SLOTS;               // 2304
};

int colstage_max_modes() { return kColStageMaxM; }

// Columns per FP64 C2 workgroup: one, two up to 6 modes (a wavefront pair per column; at 7 and 8 modes two were
// 4 and 7 % slower than one on every grid, beyond the lines do not fit), four up to 2 modes (beyond they do not fit)
constexpr int kColStageMaxM2 = 6, kColStageMaxM4 = 2;
bool colstage_cols_ok(int M, int cols) {
  return cols == 1 || (cols == 2 && M <= kColStageMaxM2) || (cols == 4 && M <= kColStageMaxM4);
}
int colstage_lines_per_chunk(int M) { return colstage_lines_cap(M); }
int colstage_coefficients_per_chunk(int M) { return colstage_qcap(M); }
int colstage_slots_per_chunk() { return kColStageSCap; }
// FP32: 8-wavefront gather workgroups up to 12 modes (beyond, the registers of a 512-lane
// workgroup would spill)
constexpr bool wide_gather(int M) { return M <= 12; }
bool colstage_wide_ok(int M) { return wide_gather(M); }

// C1 over CW neighbouring columns per workgroup, the column block's Raman lines dealt to
// `groups` workgroups (each transforms every field of the block, group 0 stores them to U).
// Lanes are ordered column-fastest, tid = (row_job * 8 + t) * CW + c, so every global access
// of a wavefront reads or writes runs of CW consecutive samples of one row: with one column
// per workgroup each lane's sample sits in a cache line of its own and the pass is bound by
// the L2 request rate, not by HBM. The arithmetic of every line is the same for any CW and
// groups, so the results are too.
template <class W, int CW>
__global__ void __launch_bounds__(256) k_colstage_fields_pairs(Geometry g, const cpx<W>* __restrict__ coltw,
                                                               const cpx<W>* __restrict__ fourtw,
                                                               const cpx<W>* __restrict__ yin, cpx<W>* __restrict__ U,
                                                               cpx<W>* __restrict__ conv, int n_lines,
                                                               const uint2* __restrict__ line_prod, double scale,
                                                               Batch b, int groups, int conv_cols) {
  using F = ColStageCfg;
  using cw = cpx<W>;
  constexpr int L = F::L;
  constexpr int JL = F::NL / CW;  // field or line rows per round: 32 jobs = JL rows x CW columns
  static_assert(CW == 1 || CW == 2 || CW == 4, "columns per workgroup");
  extern __shared__ __align__(16) unsigned char c1_lds[];
  cw* sh = reinterpret_cast<cw*>(c1_lds);  // [32 jobs][SLOTS] transform rows, then [M][L][CW] fields
  const int fib = blockIdx.y;
  if (!b.fp[fib].live) return;  // uniform over the workgroup
  yin += fib * b.sf;
  U += fib * b.sf;
  conv += fib * b.sl;
  cw* Ush = sh + F::FFT;
  const int tid = threadIdx.x;
  const int c = tid % CW, t = (tid / CW) % F::T, jl = tid / (F::T * CW);
  const int blk = xcd_block(blockIdx.x, gridDim.x);  // the groups of a column block are neighbours
  const int grp = blk % groups;
  const int n2 = (blk / groups) * CW + c;
  const int lpg = (n_lines + groups - 1) / groups;
  const int lbeg = grp * lpg < n_lines ? grp * lpg : n_lines;
  const int lend = lbeg + lpg < n_lines ? lbeg + lpg : n_lines;
  cw* fsm = sh + (jl * CW + c) * F::SLOTS;
  cw w4[8], v[8];
  LineTw<L, W> lt;
  const int wave_jl0 = __builtin_amdgcn_readfirstlane(tid / 64) * (64 / (F::T * CW));  // first row job of this wavefront
  // the first round's field samples are requested before the twiddles, and the first round's
  // line descriptors with them (each later round's during the round before); wavefronts without a
  // field or line load nothing (see C2)
  if (wave_jl0 < g.M) {
    const size_t base = (size_t)(jl < g.M ? jl : g.M - 1) * g.N + n2;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = yin[base + (size_t)(t + i * F::T) * g.N2];
  }
  uint2 d_n = line_prod[lbeg + jl < n_lines ? lbeg + jl : n_lines - 1];
  if (wave_jl0 < (lend - lbeg > g.M ? lend - lbeg : g.M)) {
    load_line_tw<L>(lt, coltw, t);
#pragma unroll
    for (int i = 0; i < 8; i++) w4[i] = fourtw[n2 * (t + i * F::T)];
  }
  const W sc = (W)scale;
  for (int r0 = 0; r0 < g.M; r0 += JL) {
    const int q = r0 + jl;
    const bool valid = q < g.M;
    const size_t base = (size_t)(valid ? q : g.M - 1) * g.N + n2;
    if (r0 + wave_jl0 >= g.M) continue;  // no field of this wavefront in the round
    if (r0 > 0) {
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = yin[base + (size_t)(t + i * F::T) * g.N2];
    }
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = cmulc(v[i], w4[i]);
    line_fft<L, 1, 1, 1, W, true>(v, fsm, lt, t);
    if (valid) {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int n1 = t + i * F::T;
        const cw x = cscale(v[i], sc);
        if (grp == 0) store_stream64(U + (size_t)q * g.N + (size_t)n2 * L + n1, x);  // column order, for the gather
        Ush[(q * L + n1) * CW + c] = x;
      }
    }
  }
  __syncthreads();
  for (int r0 = lbeg; r0 < lend; r0 += JL) {
    const int q = r0 + jl;
    const bool valid = q < lend;
    if (r0 + wave_jl0 >= lend) continue;  // no line of this wavefront in this round or later
    const uint2 d = d_n;
    d_n = line_prod[q + JL < n_lines ? q + JL : n_lines - 1];
    const int i0 = (int)(d.x & 255u) * L * CW + c, j0 = (int)((d.x >> 8) & 255u) * L * CW + c;
    const int i1 = (int)(d.y & 255u) * L * CW + c, j1 = (int)((d.y >> 8) & 255u) * L * CW + c;
    const bool im0 = (d.x >> 16) & 1u, im1 = (d.y >> 16) & 1u, has1 = !((d.y >> 17) & 1u);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int o = (t + i * F::T) * CW;
      const cw x0 = cmulc(Ush[i0 + o], Ush[j0 + o]), x1 = cmulc(Ush[i1 + o], Ush[j1 + o]);
      v[i] = {im0 ? x0.im : x0.re, has1 ? (im1 ? x1.im : x1.re) : (W)0};
    }
    line_fft<L, -1, 1, 1, W, true>(v, fsm, lt, t);
    if (valid) {
      if (conv_cols) {  // column order (uniform branch)
        const size_t base = (size_t)q * g.N + (size_t)n2 * L;
#pragma unroll
        for (int i = 0; i < 8; i++) store_stream64(conv + base + t + i * F::T, cmul(v[i], w4[i]));
      } else {
        const size_t base = (size_t)q * g.N + n2;
#pragma unroll
        for (int i = 0; i < 8; i++) store_stream64(conv + base + (size_t)(t + i * F::T) * g.N2, cmul(v[i], w4[i]));
      }
    }
  }
}

// Coupling coefficients of the vector gather: 16 to a register (pair), those of mode p for
// G = 16 / QP consecutive products, QP each (the QROW coefficients padded to 4, 8 or 16). Lane l of
// each row of 16 lanes holds the l-th, and an FMAC takes its coefficient by DPP row broadcast: no
// scalar load or LDS read per coefficient. A step is one such register for every mode; the steps go
// through the segments in order, and a group of products that two segments share has a step in
// each, the other segment's products with zeros.
constexpr int coef_pad(int q) { return q <= 4 ? 4 : (q <= 8 ? 8 : 16); }
int colstage_coef_pad(int M, bool parity) { return coef_pad(parity ? (M + 1) / 2 : M); }

// B[k] += c[N + k] x for k < Q, c[n] being lane n of each row of 16 lanes. The s_nop covers the two
// wait states a DPP operand needs after a VALU write of it (a register copy that the compiler may
// place before the block).
#define MMP_BC(OP, K, N) "\n\t" OP " %" #K ", %[c], %[x] row_newbcast:%c[" #N "] row_mask:0xf bank_mask:0xf"
#define MMP_FMAC_BCAST(OP)                                                                                             \
  if constexpr (Q == 1)                                                                                                \
    asm("s_nop 1" MMP_BC(OP, 0, n0) : "+v"(B[0]) : [c] "v"(c), [x] "v"(x), [n0] "n"(N));                               \
  if constexpr (Q == 2)                                                                                                \
    asm("s_nop 1" MMP_BC(OP, 0, n0) MMP_BC(OP, 1, n1)                                                                  \
        : "+v"(B[0]), "+v"(B[1])                                                                                       \
        : [c] "v"(c), [x] "v"(x), [n0] "n"(N), [n1] "n"(N + 1));                                                       \
  if constexpr (Q == 3)                                                                                                \
    asm("s_nop 1" MMP_BC(OP, 0, n0) MMP_BC(OP, 1, n1) MMP_BC(OP, 2, n2)                                                \
        : "+v"(B[0]), "+v"(B[1]), "+v"(B[2])                                                                           \
        : [c] "v"(c), [x] "v"(x), [n0] "n"(N), [n1] "n"(N + 1), [n2] "n"(N + 2));                                      \
  if constexpr (Q >= 4)                                                                                                \
    asm("s_nop 1" MMP_BC(OP, 0, n0) MMP_BC(OP, 1, n1) MMP_BC(OP, 2, n2) MMP_BC(OP, 3, n3)                              \
        : "+v"(B[0]), "+v"(B[1]), "+v"(B[2]), "+v"(B[3])                                                               \
        : [c] "v"(c), [x] "v"(x), [n0] "n"(N), [n1] "n"(N + 1), [n2] "n"(N + 2), [n3] "n"(N + 3));
template <int Q, int N>
__device__ __forceinline__ void fmac_bcast(double* B, double c, double x) {
  static_assert(Q >= 1 && N + Q <= 16, "coefficients of one register");
  MMP_FMAC_BCAST("v_fmac_f64_dpp")
  if constexpr (Q > 4) fmac_bcast<Q - 4, N + 4>(B + 4, c, x);
}
#undef MMP_FMAC_BCAST
#undef MMP_BC

// Steps of the vector gather whose coefficients pass through registers on their way to LDS (up to 6 modes): every
// product once, and a shared group per further segment. Pairs whose slots differ in parity lie in two segments
// and add steps (16 at 6 modes under the reference pair decode, where this is 12): those go straight to LDS.
constexpr int steps_cap(int M, bool parity) {
  const int G = 16 / coef_pad(parity ? (M + 1) / 2 : M);
  return (M * M + G - 1) / G + 3;
}
// sigma in rows of its own (one barrier less) where one column's LDS has room for them beside the lines of
// all products: up to 6 modes with the parity structure, up to 5 without (6 modes: 18 lines in 24 rows and 19
// steps would take 65,792 bytes; sigma in the lines' rows leaves 51,968)
constexpr bool own_sigma(int M, int cols, bool parity) { return cols == 1 && M <= (parity ? 6 : 5); }
// LDS of the products' C2: field rows (whole wavefronts of line slots, so that the transform of sigma has its
// rows there), the rows of a chunk's lines, sigma's (in the lines' place where they are not its own), and up to 6 modes
// the steps' coefficients.
template <int M, int COLS, bool PAR>
struct C2Cfg {
  static constexpr int UR = (M + 7) / 8 * 8;
  static constexpr int STEPS = steps_cap(M, PAR);
  static __host__ __device__ size_t q_offset(int lines) {
    const int jw = 8 / COLS, rows = (lines + jw - 1) / jw * jw, sig = 2 * M;
    return (size_t)(UR + (OWN ? rows + sig : (rows > sig ? rows : sig))) * COLS * kColStageRS * sizeof(cd);
  }
  static constexpr bool OWN = own_sigma(M, COLS, PAR);
  // vector form with two wavefronts per mode and column, one for each parity class
  template <int NW>
  static constexpr bool cs() { return PAR && M <= 6 && NW / COLS >= 2 * M; }
};
size_t colstage_products_lds_bytes(int M, int cols, int lines, int steps, bool parity) {
  const int jw = 8 / cols, rows = (lines + jw - 1) / jw * jw, sig = 2 * M;
  const bool own = own_sigma(M, cols, parity);
  return (size_t)((M + 7) / 8 * 8 + (own ? rows + sig : (rows > sig ? rows : sig))) * cols * kColStageRS * sizeof(cd) +
         (M <= 6 ? ((size_t)M * steps + 4) * 16 * sizeof(double) : 0);  // (+ 4: steps read ahead)
}

// B[kk] += over the G = 16 / QP products of one coefficient register
template <int QROW, int QP, int I = 0>
__device__ __forceinline__ void group_fmac(double* B, double c, const double* x) {
  fmac_bcast<QROW, I * QP>(B, c, x[I]);
  if constexpr ((I + 1) * QP < 16) group_fmac<QROW, QP, I + 1>(B, c, x);
}

// The vector gather's steps over the products [xc0, xc1) of one chunk, for the modes
// p = sub + j WPC < M of this wavefront and the sample of this lane: B[p][kk] per segment, then
// acc (even parity class) or acc2 (odd) += U_k B. Xc: the sample in the chunk's first X row (rows of
// RS reals, the two products of a line together, COLS columns per line); Uc: in field row 0. The
// coefficients come from LDS (QL) or by `coefs`, PD steps ahead. CS: parity class `cls` only.
template <int QROW, int NP, int PD, int WPC, int COLS, int RS, bool PAR, bool QL, bool CS, class Coefs, int PQ,
          int P2>
__device__ __forceinline__ void product_sums(const ProductArgs& fa, const double* Qsh, const double* Xc, const cd* Uc, int xc0,
                                             int xc1, int M, int sub, int cls, bool busy, int lane, int& step,
                                             uint32_t& sdesc, double (&cq)[PQ][NP], const Coefs& coefs, cd (&acc)[NP],
                                             cd (&acc2)[P2]) {
  constexpr int QP = coef_pad(QROW), G = 16 / QP;
  auto xrow = [&](int x) { return ((x >> 1) * COLS * 2 + (x & 1)) * RS; };  // of product xc0 + x
  double B[NP][QROW];
#pragma unroll
  for (int j = 0; j < NP; j++)
#pragma unroll
    for (int kk = 0; kk < QROW; kk++) B[j][kk] = 0.;
  // PD steps with their coefficients in PD fixed registers, each loaded again for the step PD
  // further on as soon as it is used
  // lane i: step i of its 64: offset of its X values (G products of one line, or of two neighbouring
  // ones) in place of its first product (steps of other chunks: any valid place)
  uint32_t sx = 0;
  auto describe = [&]() {
    const int x = (int)(sdesc & 0xffffu);
    sx = (sdesc & 0xf0000000u) | (uint32_t)xrow(x >= xc0 && x < xc1 ? x - xc0 : 0);
  };
  describe();
  double xv[PD][G], cl[PD][NP];
  uint32_t sd[PD];
  const double* ql[NP];  // QL: step's coefficients
#pragma unroll
  for (int j = 0; j < NP; j++)
    ql[j] = Qsh + ((sub + j * WPC < M ? sub + j * WPC : 0) * fa.stride + step) * 16 + (lane & 15);
  auto operands = [&](int s, int u, int qo) {
    if constexpr (!QL) {  // (QL: fewer than 64 steps)
      if (s > 0 && (s & 63) == 0) {
        sdesc = fa.steps[s + lane];
        describe();
      }
    }
    sd[u] = __builtin_amdgcn_readlane(sx, QL ? s : s & 63);
    const double* xs = Xc + (sd[u] & 0xfffffffu);
#pragma unroll
    for (int i = 0; i < G; i++) xv[u][i] = xs[xrow(i)];
    if constexpr (QL) {
#pragma unroll
      for (int j = 0; j < NP; j++) cl[u][j] = ql[j][qo];
    }
  };
#pragma unroll
  for (int u = 0; u < PD; u++) operands(step + u, u, u * 16);
  // (CS: wavefronts beyond the modes' and classes with no product have nothing to sum)
  bool more = !CS || (busy && (cls ? fa.odd_step < fa.n_steps : fa.odd_step > 0));
#pragma unroll 1
  while (more) {
#pragma unroll
    for (int u = 0; u < PD; u++) {
      const uint32_t sdu = sd[u];
#pragma unroll
      for (int j = 0; j < NP; j++) group_fmac<QROW, QP>(B[j], QL ? cl[u][j] : cq[QL ? 0 : u][j], xv[u]);
      if constexpr (!QL) coefs(step + PD, cq[u]);
      operands(step + PD, u, (PD + u) * 16);  // (past the last step: any valid place)
      step++;
      if (!(sdu >> 31)) continue;
      // the segment (or the chunk's part of it) is complete
      const int sg = (sdu >> 28) & 3u;
#pragma unroll
      for (int j = 0; j < NP; j++) {
        const int par = PAR ? ((sub + j * WPC + sg) & 1) : 0;
        cd sum = {0, 0};
#pragma unroll
        for (int kk = 0; kk < QROW; kk++) {
          sum = cadd(sum, cscale(Uc[((PAR ? 2 * kk : kk) + par) * COLS * RS], B[j][kk]));
          B[j][kk] = 0.;
        }
        if (sg >= 2) sum = {-sum.im, sum.re};
        if constexpr (!CS && PAR) {  // (selects of values: of places would put the sums in scratch memory)
          const bool odd = sg & 1;
          const cd even = cadd(acc[j], sum), odds = cadd(acc2[CS || !PAR ? 0 : j], sum);
          acc[j] = {odd ? acc[j].re : even.re, odd ? acc[j].im : even.im};
          cd& o = acc2[CS || !PAR ? 0 : j];
          o = {odd ? odds.re : o.re, odd ? odds.im : o.im};
        } else {
          acc[j] = cadd(acc[j], sum);
        }
      }
      more = ((sdu >> 30) & 1u) && !(CS && !cls && step == fa.odd_step);
      if (!more) break;
    }
#pragma unroll
    for (int j = 0; j < NP; j++) ql[j] += PD * 16;
  }
}

// C2 over COLS neighbouring columns per workgroup. Lanes are ordered column-fastest as in C1, each
// line transform runs inside one wavefront, in place in its padded LDS row, and wavefronts without
// a line skip it. Each line's row is then mixed into its two real products' slot mixes
// X = kv Re|Im(U_a conj U_b) + kr (the line's real|imaginary part), in its place (two X rows of RS
// reals), by whole wavefronts. NW / COLS wavefronts then sum each column: wavefront `sub` of a column
// takes the modes p = sub, sub + NW / COLS, ... (product_sums). The sum over the products runs in
// their order whatever NW and COLS are.
// Bound by latency for one fiber (a workgroup per CU or two: loads, line transform, mix, sums and
// transform follow one another), by the FP64 units from 10 modes on. Summing complex slots took 18 Raman lines
// instead of 11 at 6 modes and 4 to 5 times the coupling sums. Whole step on one MI355X, before and after: 6 modes,
// NT = 16384, RK4 111.5 -> 101.7 us; 2 modes, NT = 4096 71.1 -> 68.3 us; 5 modes without the
// symmetric couplings (all products), NT = 8192, sixth order 164.6 -> 165.2 us (the one form kept).
// Without Raman (RAMAN = false) the whole column side of a stage is this one kernel: it takes the fields
// themselves from `U` (row order; the same array as yout: a workgroup reads and writes its own columns only),
// transforms them in their LDS rows, and the products have no line: 8 launches of 5-8 us an RK4 step in place
// of 16, 6 modes, NT = 16384 78.7 -> 50.6 us per step. Bound by latency and its column access.
template <int M, int NW, int COLS, bool PAR, bool RAMAN>
__global__ void __launch_bounds__(NW * 64) k_colstage_products(
    Geometry g, const cd* __restrict__ coltw, const cd* __restrict__ fourtw, const cd* U,
    const cd* __restrict__ conv, cd* yout, ProductArgs fa, const double* __restrict__ Qp, double scale, Batch b) {
  using C2 = C2Cfg<M, COLS, PAR>;
  const int fib = blockIdx.y;
  const FiberParams fp = b.fp[fib];
  if (!fp.live) return;  // uniform over the workgroup
  U += fib * b.sf;
  yout += fib * b.sf;
  conv += fib * b.sl;
  constexpr int L = kColStageL, T = L / 8, RS = kColStageRS, UR = C2::UR;
  constexpr int NT = NW * 64;
  constexpr int JL = NT / (T * COLS);  // lines of every column per round
  constexpr int JW = 64 / (T * COLS);  // of which one wavefront holds
  constexpr int WPC = NW / COLS;       // wavefronts per column
  constexpr int QROW = PAR ? (M + 1) / 2 : M;  // coefficients per product and mode p
  constexpr int UIN = (M * COLS * L + NT - 1) / NT;
  static_assert(M >= 1 && M <= kColStageMaxM && JW >= 1 && WPC >= 1 && JL >= M, "modes or columns out of range");
  extern __shared__ __align__(16) unsigned char c2_lds[];
  cd* const Ush = reinterpret_cast<cd*>(c2_lds);  // field rows [UR][COLS] (zeros beyond M); transform rows of sigma
  cd* const Rsh = Ush + UR * COLS * RS;           // line rows [lines][COLS], then their X rows; then sigma
  double* const Xsh = reinterpret_cast<double*>(Rsh);
  double* const Qsh = reinterpret_cast<double*>(c2_lds + C2::q_offset(fa.max_chunk_lines));  // coefficients (QL)
  cd* const Ssh = C2::OWN ? Rsh + (fa.max_chunk_lines + 7) / 8 * 8 * RS : Rsh;  // sigma rows
  const int tid = threadIdx.x;
  const int c = tid % COLS, t = (tid / COLS) % T, jl = tid / (T * COLS);
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int n20 = xcd_block(blockIdx.x, gridDim.x) * COLS, n2 = n20 + c;
  // The first chunk's lines, the field samples and the coefficients are requested before anything
  // waits on memory, each by the wavefronts that use it only: the vector memory pipe takes a
  // wavefront's 16-byte loads at 64 bytes a cycle, and eight wavefronts loading every twiddle kept
  // a lone workgroup's first line waiting for 3000 cycles.
  cd v[8], uin[UIN], w4[8];
  LineTw<L, double> lt;
  int l0 = 0, l1 = fa.first_lines;
  if (wave * JW < (RAMAN ? l1 : M)) {
    const int last = (RAMAN ? l1 : M) - 1, q = jl < last ? jl : last;  // lanes without a line read the last one's
    const size_t base = (size_t)q * g.N + (RAMAN ? (size_t)n2 * L : (size_t)n2);
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = RAMAN ? conv[base + t + i * T] : U[base + (size_t)(t + i * T) * g.N2];
  }
  if constexpr (RAMAN) {
#pragma unroll
    for (int r = 0; r < UIN; r++) {
      const int e = tid + r * NT;
      if (wave * 64 + r * NT < M * COLS * L)  // (whole wavefronts)
        uin[r] = U[(size_t)(e / (COLS * L)) * g.N + (size_t)n20 * L + e % (COLS * L)];
    }
  }
  if (wave * JW < (RAMAN && l1 > M ? l1 : M)) {
    load_line_tw<L>(lt, coltw, t);
#pragma unroll
    for (int i = 0; i < 8; i++) w4[i] = fourtw[n2 * (t + i * T)];
  }
  const int col = wave % COLS, sub = wave / COLS;  // column of this wavefront's sums, its place there
  // with two wavefronts per mode each takes one parity class (CS), else a wavefront takes the modes
  // sub, sub + WPC, ... in both; the classes' sums are added last either way
  constexpr bool CS = C2::template cs<NW>();
  constexpr int NP = CS ? 1 : (M + WPC - 1) / WPC;  // modes of this wavefront
  const int cls = CS && sub >= M ? 1 : 0, sub0 = CS ? (sub < M ? sub : (sub < 2 * M ? sub - M : 0)) : sub;
  constexpr int QP = coef_pad(QROW), G = 16 / QP;   // products per coefficient register
  // the steps' coefficients go through LDS where all of them fit (up to 6 modes), else
  // each wavefront reads its modes' ahead of use, from cache lines requested here
  constexpr bool QL = M <= 6;
  constexpr int PD = QL ? 2 : 4;          // steps read ahead
  const double* qf = Qp + fib * b.sq + (lane & 15);
  auto coefs = [&](int s, double (&q)[NP]) {  // step s's coefficients of this wavefront's modes
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const int p = sub0 + j * WPC < M ? sub0 + j * WPC : 0;
      q[j] = qf[((size_t)p * fa.stride + (s < fa.stride ? s : 0)) * 16];
    }
  };
  constexpr int QIN = QL ? (M * C2::STEPS * 16 + NT - 1) / NT : 1;
  double cq[QL ? 1 : PD][NP], qin[QIN], touch[QL ? 1 : NP];
  uint32_t sdesc = fa.steps[lane];
  {
    if constexpr (QL) {
      const int last = M * fa.stride * 16 - 1;
#pragma unroll
      for (int r = 0; r < QIN; r++)
        if (wave * 64 + r * NT <= last) qin[r] = Qp[fib * b.sq + (tid + r * NT < last ? tid + r * NT : last)];
    } else {
#pragma unroll
      for (int u = 0; u < PD; u++) coefs(u, cq[u]);
#pragma unroll
      for (int j = 0; j < NP; j++) {
        const int p = sub0 + j * WPC < M ? sub0 + j * WPC : 0, e = lane * (128 / (int)sizeof(double));
        touch[j] = Qp[fib * b.sq + (size_t)p * fa.stride * 16 + (e < fa.stride * 16 ? e : 0)];
      }
    }
  }
  if constexpr (RAMAN) {
#pragma unroll
    for (int r = 0; r < UIN; r++) {
      const int e = tid + r * NT;
      if (wave * 64 + r * NT < M * COLS * L) Ush[(e / L) * RS + e % L] = uin[r];
    }
    // the field row after the last one, which the coupling rows of an odd number of modes read with
    // zero coefficients
    constexpr int UZ = M % 2 && PAR ? M + 1 : M;
    for (int e = M * COLS * L + tid; e < UZ * COLS * L; e += NT) Ush[(e / L) * RS + e % L] = cd{0, 0};
  } else if (wave * JW < M) {
    // the fields; the lanes beyond the last one leave zero rows (whole wavefronts: up to UR rows)
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = cmulc(v[i], w4[i]);
    cd* row = Ush + (jl * COLS + c) * RS;
    line_fft<L, 1, 1, 1, double, true>(v, row, lt, t);
#pragma unroll
    for (int i = 0; i < 8; i++) row[t + i * T] = jl < M ? cscale(v[i], scale) : cd{0, 0};
  }
  if constexpr (QL) {
#pragma unroll
    for (int r = 0; r < QIN; r++)
      if (tid + r * NT < M * fa.stride * 16) Qsh[tid + r * NT] = qin[r];
    for (int e = tid + QIN * NT; e < M * fa.stride * 16; e += NT) Qsh[e] = Qp[fib * b.sq + e];
  }
  const double sc = scale, kv = fp.kv, kr = fp.kr;
  cd acc[NP], acc2[CS || !PAR ? 1 : NP];  // sums of the even (CS: its own) and of the odd parity class
#pragma unroll
  for (int p = 0; p < NP; p++) acc[p] = {0, 0};
#pragma unroll
  for (int p = 0; p < (CS || !PAR ? 1 : NP); p++) acc2[p] = {0, 0};
  int step = cls ? fa.odd_step : 0;  // steps taken
  for (int ch = 0; ch < fa.n_chunks; ch++) {
    if (ch > 0) {
      __syncthreads();  // X rows of the previous chunk consumed
      l0 = l1;
      l1 = (int)fa.chunk_line[ch + 1];
      sdesc = fa.steps[(step & ~63) + lane];
      if constexpr (!QL) {
#pragma unroll
        for (int u = 0; u < PD; u++) coefs(step + u, cq[u]);
      }
    }
    // lane i: the products of the wavefront's i-th (line, column) row to mix
    // (without lines: to an even number, as a step of four products may read the row after the last one,
    // times zero; the lines' rows fill up whole wavefronts)
    const int rows = (RAMAN ? l1 - l0 : (l1 - l0 + 1) / 2 * 2) * COLS, nrow = (l1 - l0) * COLS;
    const uint2 dl = fa.line_prod[l0 + (wave + NW * lane < nrow ? (wave + NW * lane) / COLS : 0)];
    for (int r0 = l0; RAMAN && r0 < l1; r0 += JL) {
      if (r0 + wave * JW >= l1) break;  // no line of this wavefront in the round
      const int q = r0 + jl;
      const bool valid = q < l1;
      if (ch > 0 || r0 > l0) {
        const size_t base = (size_t)(valid ? q : l1 - 1) * g.N + (size_t)n2 * L;
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = conv[base + t + i * T];
      }
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = cmulc(v[i], w4[i]);
      cd* row = Rsh + ((q - l0) * COLS + c) * RS;
      line_fft<L, 1, 1, 1, double, true>(v, row, lt, t);
#pragma unroll
      for (int i = 0; i < 8; i++) row[t + i * T] = v[i];
    }
    __syncthreads();  // the lines' and the fields' rows
    // slot mixes, a row at a time by whole wavefronts (lane = sample): the two products of a line
    // take the place of its samples
#pragma unroll 1
    for (int i = 0, r = wave; r < rows; i++, r += NW) {
      const uint32_t d0 = __builtin_amdgcn_readlane(dl.x, i), d1 = __builtin_amdgcn_readlane(dl.y, i);
      const cd* uc = Ush + (COLS > 1 ? r % COLS : 0) * RS + lane;
      const cd V0 = cmulc(uc[(d0 & 255u) * COLS * RS], uc[((d0 >> 8) & 255u) * COLS * RS]);
      const cd V1 = cmulc(uc[(d1 & 255u) * COLS * RS], uc[((d1 >> 8) & 255u) * COLS * RS]);
      double* x0 = Xsh + r * 2 * RS + lane;
      if constexpr (RAMAN) {
        const cd vr = Rsh[r * RS + lane];
        x0[0] = kv * ((d0 >> 16) & 1u ? V0.im : V0.re) + kr * (vr.re * sc);
        x0[RS] = kv * ((d1 >> 16) & 1u ? V1.im : V1.re) + kr * (vr.im * sc);
      } else {
        x0[0] = kv * ((d0 >> 16) & 1u ? V0.im : V0.re);
        x0[RS] = kv * ((d1 >> 16) & 1u ? V1.im : V1.re);
      }
    }
    if constexpr (!QL) {
#pragma unroll
      for (int j = 0; j < NP; j++) asm volatile("" ::"v"(touch[j]));
    }
    __syncthreads();
    const int xc0 = 2 * l0, xc1 = 2 * l1 < fa.n_products ? 2 * l1 : fa.n_products;  // products of the chunk
    const double* const Xc = Xsh + col * 2 * RS + lane;  // this lane's sample of the chunk's first X row
    const cd* const Uc = Ush + col * RS + lane;     // this lane's sample of field k: Uc[k * COLS * RS]
    product_sums<QROW, NP, PD, WPC, COLS, RS, PAR, QL, CS>(fa, Qsh, Xc, Uc, xc0, xc1, M, sub0, cls, sub < 2 * M, lane, step,
                                                           sdesc, cq, coefs, acc, acc2);
  }
  if constexpr (!C2::OWN) __syncthreads();  // every lane done with the X rows, whose place sigma takes
  // sigma rows [modes][COLS]; CS: a set for each parity class
  constexpr int SETS = CS ? 2 : 1;
#pragma unroll
  for (int j = 0; j < NP; j++) {
    if (CS ? sub < 2 * M : sub + j * WPC < M)
      Ssh[((sub + j * WPC) * COLS + col) * RS + lane] = !CS && PAR ? cadd(acc[j], acc2[CS || !PAR ? 0 : j]) : acc[j];
  }
  __syncthreads();
  if (wave * JW < M) {
    const int q = jl;
    const bool valid = q < M;
    const cd* in = Ssh + ((valid ? q : 0) * COLS + c) * RS;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      v[i] = in[t + i * T];
      if constexpr (SETS == 2) v[i] = cadd(v[i], in[M * COLS * RS + t + i * T]);
    }
    line_fft<L, -1, 1, 1, double, true>(v, Ush + (q * COLS + c) * RS, lt, t);
    if (valid) {
      const size_t base = (size_t)q * g.N + n2;
#pragma unroll
      for (int i = 0; i < 8; i++) store_stream64(yout + base + (size_t)(t + i * T) * g.N2, cmul(v[i], w4[i]));
    }
  }
}

// ---------------------------------------------------------------------------
// The separate column passes' gather in FP64, on the same real products: a workgroup takes a tile of
// 64 samples (lane = sample) and a group of modes, a wavefront per mode; the chunk's X rows are mixed by
// whole wavefronts, then each wavefront sums its mode, segment by segment (the steps of a segment take
// consecutive products, so no step table is read).
// ---------------------------------------------------------------------------
// More groups of modes give more wavefronts, and each group mixes the tile's X rows again: groups of at most
// eight. LDS holds the field rows and as many lines' X rows as 64 KB take; a chunk's Raman rows are requested
// before the sums of the chunk before. Bound by latency (a chain of steps whose coefficients come from
// the L2). Whole step on one MI355X against the sparse sum (one slot entry after the other, up to 20 modes 708 us a
// launch, now 25) or the dense slot blocks: 20 modes, NT = 4096 2995 -> 251 us; 6 modes, NT = 16384
// without Raman 93.0 -> 78.7 us; 2 modes, NT = 1024 113.0 -> 107.6 us. Of it at 20 modes: step table as in
// C2 336 us, steps by segment 272, loads kept in place 260, Raman rows ahead 251.
constexpr int kProductsTS = 64, kProductsMaxWaves = 8;
// (16 coefficients of a product and mode fill the register; field rows beyond 32 leave the chunks few lines)
bool gather_products_ok(int M, bool parity) { return M >= 1 && M <= 32 && (parity ? (M + 1) / 2 : M) <= 16; }
static int products_field_rows(int M, bool parity) { return parity ? M + (M & 1) : M; }
int gather_products_lines(int M, bool parity) {
  return ((int)(kColStageLds / (kProductsTS * sizeof(cd))) - products_field_rows(M, parity)) & ~1;
}

// One segment's part of a chunk for mode p: B[kk] = sum over the products [x, x + G ns) of this lane's sample
// (xs: that of product x, rows of TS) and the coefficients from step `step` on, PD steps ahead in PD fixed
// registers; the steps past the last one read any valid place.
template <int QROW, int PD, int TS>
__device__ __forceinline__ void segment_products(double (&B)[QROW], const double* __restrict__ q, int step, int last_step,
                                                 const double* xs, int ns, int lane) {
  constexpr int QP = coef_pad(QROW), G = 16 / QP;
  double cq[PD], xv[PD][G];
  auto load = [&](int s, int u) {
    const int sq = step + s < last_step ? step + s : last_step, sx = s < ns ? s : ns - 1;
    cq[u] = (q + (size_t)sq * 16)[lane & 15];
#pragma unroll
    for (int i = 0; i < G; i++) xv[u][i] = xs[(sx * G + i) * TS];
  };
#pragma unroll
  for (int u = 0; u < PD; u++) load(u, u);
#pragma unroll
  for (int kk = 0; kk < QROW; kk++) B[kk] = 0.;
  int s = 0;
#pragma unroll 1
  for (; s + PD <= ns; s += PD) {
#pragma unroll
    for (int u = 0; u < PD; u++) {
      group_fmac<QROW, QP>(B, cq[u], xv[u]);
      load(s + PD + u, u);
      __builtin_amdgcn_sched_barrier(0);  // (else all PD loads end up behind the last step, each round a latency)
    }
  }
#pragma unroll
  for (int u = 0; u < PD - 1; u++)
    if (s + u < ns) group_fmac<QROW, QP>(B, cq[u], xv[u]);
}

template <int QROW, bool PAR>
__global__ void __launch_bounds__(kProductsMaxWaves * 64) k_gather_products(
    Geometry g, const cd* __restrict__ U, const cd* __restrict__ VR, cd* __restrict__ sigma, ProductArgs fa,
    const double* __restrict__ Qp, Batch b, int raman, int field_rows) {
  constexpr int TS = kProductsTS, PD = 8, R = 8, G = 16 / coef_pad(QROW);
  extern __shared__ __align__(16) unsigned char gp_lds[];
  cd* const Ush = reinterpret_cast<cd*>(gp_lds);                       // [field_rows][TS], zeros beyond M
  double* const Xsh = reinterpret_cast<double*>(Ush + field_rows * TS);  // [2 lines of a chunk][TS]
  const int M = g.M;
  const int t0 = blockIdx.x * TS;
  const int tid = threadIdx.x, lane = tid % TS, waves = blockDim.x / TS;
  const int wave = __builtin_amdgcn_readfirstlane(tid / TS);
  const int p = blockIdx.y * waves + wave;  // this wavefront's mode
  const double kv = b.fp[0].kv, kr = raman ? b.fp[0].kr : 0.;
  const double* const q = Qp + (size_t)(p < M ? p : 0) * fa.stride * 16;
  // a chunk's first Raman rows of this wavefront are requested before the sums of the chunk before
  cd vr[R];
  uint2 d[R];
  auto request = [&](int l, int l1) {
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int r = l + i * waves < l1 ? l + i * waves : l1 - 1;
      d[i] = fa.line_prod[r];
      vr[i] = raman ? VR[(size_t)r * g.N + t0 + lane] : cd{0, 0};
    }
  };
  request(wave, (int)fa.chunk_line[1]);
#pragma unroll 4
  for (int r = wave; r < field_rows; r += waves)
    Ush[r * TS + lane] = r < M ? U[(size_t)r * g.N + t0 + lane] : cd{0, 0};
  cd acc = {0, 0}, acc2 = {0, 0};  // sums of the even and of the odd parity class
  int step = 0;
  for (int ch = 0; ch < fa.n_chunks; ch++) {
    const int l0 = (int)fa.chunk_line[ch], l1 = (int)fa.chunk_line[ch + 1];
    __syncthreads();  // the fields' rows / X rows of the previous chunk consumed
    // (a step of four products may read the row after the chunk's last one, times zero)
    const int lend = l0 + (l1 - l0 + 1) / 2 * 2;
#pragma unroll 1
    for (int l = l0 + wave; l < lend; l += R * waves) {
      if (l > l0 + wave) request(l, l1);
#pragma unroll
      for (int i = 0; i < R; i++) {
        if (l + i * waves >= lend) break;
        const cd V0 = cmulc(Ush[(d[i].x & 255u) * TS + lane], Ush[((d[i].x >> 8) & 255u) * TS + lane]);
        const cd V1 = cmulc(Ush[(d[i].y & 255u) * TS + lane], Ush[((d[i].y >> 8) & 255u) * TS + lane]);
        double* x0 = Xsh + (l + i * waves - l0) * 2 * TS + lane;
        x0[0] = kv * ((d[i].x >> 16) & 1u ? V0.im : V0.re) + kr * vr[i].re;
        x0[TS] = kv * ((d[i].y >> 16) & 1u ? V1.im : V1.re) + kr * vr[i].im;
      }
    }
    if (ch + 1 < fa.n_chunks) request(l1 + wave, (int)fa.chunk_line[ch + 2]);
    __syncthreads();
    if (p < M) {
      const int xc0 = 2 * l0, xc1 = 2 * l1 < fa.n_products ? 2 * l1 : fa.n_products;  // products of the chunk
#pragma unroll
      for (int j = 0; j < (PAR ? 4 : 2); j++) {  // segments in the order of their steps
        const int sg = PAR ? (j == 1 ? 2 : (j == 2 ? 1 : j)) : 2 * j;
        const int xb = fa.seg_b[sg] > xc0 ? fa.seg_b[sg] : xc0, xe = fa.seg_e[sg] < xc1 ? fa.seg_e[sg] : xc1;
        if (xb >= xe) continue;
        const int x = xb / G * G, ns = (xe - x + G - 1) / G;
        double B[QROW];
        segment_products<QROW, PD, TS>(B, q, step, fa.stride - 1, Xsh + (x - xc0) * TS + lane, ns, lane);
        step += ns;
        const cd* const Uc = Ush + (PAR ? (p + sg) & 1 : 0) * TS + lane;
        cd sum = {0, 0};
#pragma unroll
        for (int kk = 0; kk < QROW; kk++) sum = cadd(sum, cscale(Uc[(PAR ? 2 * kk : kk) * TS], B[kk]));
        if (sg >= 2) sum = {-sum.im, sum.re};
        cd& a = sg & 1 ? acc2 : acc;
        a = cadd(a, sum);
      }
    }
  }
  if (p < M) sigma[(size_t)p * g.N + t0 + lane] = PAR ? cadd(acc, acc2) : acc;
}

// ---------------------------------------------------------------------------
// C2 in FP32 (mixed precision): complex slots X_s and complex Raman lines
// ---------------------------------------------------------------------------
// 4-wavefront FP32 gathers of 7 to 10 modes also come in a variant held to 168 VGPRs, so
// that three workgroups share a CU (their LDS is under 50 KB); it reads the coupling rows in
// 64-byte groups to make room, and spills at most 12 dwords. Measured on one MI355X it pays
// for large grids only: batched M = 10, NT = 16384 x 36 fibers 563 -> 480 us, M = 8 x 16
// fibers 125 -> 102 us; one fiber at NT = 65536 (1024 workgroups) 65 -> 67 us. Beyond 10
// modes (and without parity blocks at 10) the bound spills hundreds of bytes per lane.
constexpr bool hi_occupancy(int M, bool parity) { return M >= 7 && (M <= 9 || (M == 10 && parity)); }
bool colstage_hi_occupancy_ok(int M, bool parity) { return hi_occupancy(M, parity); }

// The slot sums on the matrix cores (MF, FP32): per sample, B[p][k] = sum over slots s of
// Qd[s][p][k] X_s is a real-by-complex matrix product with the rows (p, k) of one coupling parity
// class, the slots of that class as the inner dimension and the samples (real and imaginary parts
// as two products) as the columns; sigma_p = sum_k U_k B[p][k] follows per sample. One
// v_mfma_f32_32x32x2_f32 takes 32 rows, two slots and 32 samples. Rows are ordered so that the
// two lane halves of a 32 x 32 result hold the same modes p: the row of (p, kk) is
// 8 (u / 4) + 4 (kk % 2) + u % 4 with u = p * KHH + kk / 2 (KHH = ceil(QROW / 2), QROW the
// coefficients per row p), so an accumulator register r of tile t holds u = 16 t + r in both
// halves, and only k depends on the half. Tiles: ceil(M * KHH / 16), up to four. With one or two
// tiles each wavefront holds all of them (32 or 64 accumulator registers per lane) and takes every
// other pair of slots; with three or four the wavefront pairs split the tiles (two each) and every
// wavefront takes every pair, forming its slots' X twice over the workgroup.
template <int M, bool PAR>
struct MfmaRows {
  static constexpr int QROW = PAR ? (M + 1) / 2 : M;
  static constexpr int KHH = (QROW + 1) / 2;
  static constexpr int RT = (M * KHH + 15) / 16;
  static constexpr bool TSPLIT = RT > 2;      // the wavefront pairs split the tiles
  static constexpr int TPW = TSPLIT ? 2 : RT;  // tiles per wavefront
};
template <int M, bool PAR>
constexpr bool kColStageMfma = M >= 4 && MfmaRows<M, PAR>::RT <= 4;
bool colstage_matrix_cores_ok(int M, bool parity) {
  if (M < 4 || M > kColStageMaxM) return false;
  const int qrow = parity ? (M + 1) / 2 : M, khh = (qrow + 1) / 2;
  return (M * khh + 15) / 16 <= 4;
}
typedef float mfma_acc_t __attribute__((ext_vector_type(16)));

// NW wavefronts (4, or 8 when M <= 6); each line transform runs inside one wavefront,
// in place in its padded LDS row, and wavefronts without a line skip it. With MF (4 wavefronts,
// FP32) the slot sums run on the matrix cores: wavefront w takes the samples 32 (w % 2) .. + 31
// and, with up to two 32-row tiles, every other pair of its parity class's slots (from pair
// w / 2); with three or four tiles, tiles 2 (w / 2) and 2 (w / 2) + 1 over every pair.
template <int M, int NW, bool PAR, bool HI = false, bool MF = false>
__global__ void __launch_bounds__(NW * 64, HI ? 3 : (MF ? (MfmaRows<M, PAR>::RT == 1 ? 3 : 2) : 1)) k_colstage_raman_gather(Geometry g, const cf* __restrict__ coltw,
                                                                   const cf* __restrict__ fourtw,
                                                                   const cf* __restrict__ U,
                                                                   const cf* __restrict__ conv,
                                                                   cf* __restrict__ yout, SlotArgs fa, const float* __restrict__ Qd,
                                                                   double scale, Batch b) {
  const int fib = blockIdx.y;
  const FiberParams fp = b.fp[fib];
  if (!fp.live) return;  // uniform over the workgroup
  U += fib * b.sf;
  yout += fib * b.sf;
  conv += fib * b.sl;
  Qd += fib * b.sq;
  constexpr int L = kColStageL, T = L / 8, RS = kColStageRS;
  constexpr int NT = NW * 64;
  constexpr int JOBS = NT / T;  // line slots per round
  constexpr int KH = (M + 1) / 2;
  constexpr int MM = PAR ? M * KH : M * M;  // coupling coefficients per slot
  constexpr int UR = (M + 7) / 8 * 8;  // field rows, rounded up to whole wavefronts of lines
  constexpr int UIN = (M * L + NT - 1) / NT;
  // Raman line rows of a chunk, or the NW partial sums of M modes after the gather
  constexpr int RCAP = colstage_rows(M) * RS > NW * M * L ? colstage_rows(M) * RS : NW * M * L;
  static_assert(M >= 1 && M <= kColStageMaxM, "modes out of range");
  static_assert(!MF || (NW == 4 && !HI && kColStageMfma<M, PAR>), "matrix-core gather: 4 wavefronts");
  __shared__ cf Ush[UR * RS];   // field rows; sigma rows after the gather
  __shared__ cf Rsh[RCAP];      // Raman line rows of the chunk; partial sums after the gather
  __shared__ float Qsh[colstage_qcap(M)];  // [slots of the chunk][M][M] coupling blocks
  __shared__ uint32_t Msh[kColStageSCap];  // slot metadata of the chunk
  // MF: the chunk's slots of each parity class in order (metadata, offset in the chunk), and
  // their counts
  __shared__ uint2 Lsh[MF ? 2 * kColStageSCap : 1];
  __shared__ int Nsh[2];
  const int tid = threadIdx.x;
  const int job = tid / T, t = tid % T;
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int n2 = xcd_block(blockIdx.x, gridDim.x);
  // the first chunk's lines, this lane's field samples, coupling blocks and slot metadata are
  // all requested before anything waits on memory
  cf v[8], uin[UIN];
  // (each by the wavefronts that use it only: see the products' C2)
  int l0 = 0, l1 = fa.first_lines, s0 = 0, s1 = fa.first_slots;
  LineTw<L, float> lt;
  cf w4[8];
  if (wave * (64 / T) < l1) {
    const size_t base = (size_t)(job < l1 ? job : l1 - 1) * g.N + (size_t)n2 * L;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = conv[base + t + i * T];
  }
#pragma unroll
  for (int r = 0; r < UIN; r++) {
    const int e = tid + r * NT;
    if (wave * 64 + r * NT < M * L) uin[r] = U[(size_t)(e / L) * g.N + (size_t)n2 * L + e % L];
  }
  constexpr int QIN = colstage_qpre(M) / NT;
  float qin[QIN];
  uint32_t min_ = 0;
#pragma unroll
  for (int r = 0; r < QIN; r++) {
    const int e = tid + r * NT;
    qin[r] = e < (s1 - s0) * MM ? Qd[(size_t)s0 * MM + e] : 0.f;
  }
  if (tid < s1 - s0) min_ = fa.slot_meta[s0 + tid];
  // (a later chunk may hold more lines than the first one: its limit is on slots, one or two a line)
  if (wave * (64 / T) < (fa.max_chunk_lines > M ? fa.max_chunk_lines : M)) {
    load_line_tw<L>(lt, coltw, t);
#pragma unroll
    for (int i = 0; i < 8; i++) w4[i] = fourtw[n2 * (t + i * T)];
  }
#pragma unroll
  for (int r = 0; r < UIN; r++) {
    const int e = tid + r * NT;
    if (wave * 64 + r * NT < M * L) Ush[(e / L) * RS + e % L] = uin[r];
  }
  const float sc = (float)scale, kv = (float)fp.kv, kr = (float)fp.kr;
  cf u[MF ? 1 : M], acc[M];
#pragma unroll
  for (int p = 0; p < M; p++) acc[p] = {0, 0};
  // MF: this lane's sample and lane half, and the coupling offset of its A-operand row in each
  // tile and parity class (-1: a padding row, zero)
  const int hh = lane >> 5;
  const int smp = MF ? 32 * (wave & 1) + (lane & 31) : lane;
  using MR = MfmaRows<M, PAR>;
  const int tg = MR::TSPLIT ? (wave >> 1) : 0;  // this wavefront's tile group (tiles TPW tg .. TPW tg + TPW - 1)
  int aoff[2][MF ? MR::TPW : 1];
  if constexpr (MF) {
#pragma unroll
    for (int cc = 0; cc < 2; cc++)
#pragma unroll
      for (int j = 0; j < MR::TPW; j++) {
        const int t = MR::TPW * tg + j;
        const int R = 32 * t + (lane & 31);
        const int uu = 4 * (R >> 3) + (R & 3);
        const int p = uu / MR::KHH, kk = 2 * (uu % MR::KHH) + ((R >> 2) & 1);
        const int k = PAR ? 2 * kk + ((p + cc) & 1) : kk;
        aoff[cc][j] = (t < MR::RT && p < M && kk < MR::QROW && k < M) ? p * MR::QROW + kk : -1;
      }
  }
  for (int c = 0; c < fa.n_chunks; c++) {
    if (c > 0) {
      __syncthreads();  // Rsh, Qsh and Msh of the previous chunk consumed
      l0 = l1;
      l1 = (int)fa.chunk_line[c + 1];
      s0 = s1;
      s1 = (int)fa.chunk_slot[c + 1];
#pragma unroll
      for (int r = 0; r < QIN; r++) {
        const int e = tid + r * NT;
        qin[r] = e < (s1 - s0) * MM ? Qd[(size_t)s0 * MM + e] : 0.f;
      }
      if (tid < s1 - s0) min_ = fa.slot_meta[s0 + tid];
    }
#pragma unroll
    for (int r = 0; r < QIN; r++) Qsh[tid + r * NT] = qin[r];
    for (int e = QIN * NT + tid; e < (s1 - s0) * MM; e += NT) Qsh[e] = Qd[(size_t)s0 * MM + e];
    if (tid < s1 - s0) Msh[tid] = min_;
    if constexpr (MF) {
      // the class lists: wavefronts 0 and 1 hold the chunk's slots 0..63 and 64..127 (at most
      // kColStageSCap = 128); wavefront 1 also reads the metadata of slots 0..63 for their counts
      if (tid < 128) {
        const int ns = s1 - s0, ln = tid % 64;
        const bool has = tid < ns;
        const int cls = PAR ? (int)((min_ >> 18) & 1u) : 0;
        const uint64_t own1 = __ballot(has && cls == 1), own0 = __ballot(has && cls == 0);
        uint64_t lo1 = own1, lo0 = own0;  // class masks of slots 0..63
        if (tid >= 64) {
          const bool has_lo = ln < ns;
          const uint32_t m = has_lo ? fa.slot_meta[s0 + ln] : 0u;
          const int cl = PAR ? (int)((m >> 18) & 1u) : 0;
          lo1 = __ballot(has_lo && cl == 1);
          lo0 = __ballot(has_lo && cl == 0);
        }
        const uint64_t below = ln ? (~0ull >> (64 - ln)) : 0ull;
        const int pos = cls ? (tid >= 64 ? __popcll(lo1) : 0) + __popcll(own1 & below)
                            : (tid >= 64 ? __popcll(lo0) : 0) + __popcll(own0 & below);
        if (has) Lsh[cls * kColStageSCap + pos] = make_uint2(min_, (uint32_t)tid);
        if (tid == 64) {
          Nsh[0] = __popcll(lo0) + __popcll(own0);
          Nsh[1] = __popcll(lo1) + __popcll(own1);
        }
      }
    }
    for (int r0 = l0; r0 < l1; r0 += JOBS) {
      const int q = r0 + job;
      const bool valid = q < l1;
      if (r0 + wave * (64 / T) >= l1) continue;  // no line of this wavefront in the round
      if (c > 0 || r0 > l0) {
        const size_t base = (size_t)(valid ? q : l1 - 1) * g.N + (size_t)n2 * L;
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = conv[base + t + i * T];
      }
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = cmulc(v[i], w4[i]);
      cf* row = Rsh + (q - l0) * RS;
      line_fft<L, 1, 1, 1, float, true>(v, row, lt, t);
      if (valid) {
#pragma unroll
        for (int i = 0; i < 8; i++) row[t + i * T] = cscale(v[i], sc);
      }
    }
    __syncthreads();
    if constexpr (!MF) {
      if (c == 0) {
#pragma unroll
        for (int k = 0; k < M; k++) u[k] = Ush[k * RS + lane];
      }
    }
    // slot s mixes kv U_a conj(U_b) with its Raman line read as is, conjugated, or by real or
    // imaginary part; everything but the sample is wave-uniform and read from LDS by broadcast.
    // With parity-structured blocks each wavefront passes over its slots once per parity, so
    // the parity is a compile-time constant of the loop body (no per-slot selects).
    auto slot_pass = [&](auto par_c) {
      constexpr int par = decltype(par_c)::value;
      // each slot's metadata is read from LDS one slot ahead of its use
      uint32_t meta_next = s0 + wave < s1 ? Msh[wave] : 0u;
      for (int sl = s0 + wave; sl < s1; sl += NW) {
        const uint32_t meta = __builtin_amdgcn_readfirstlane(meta_next);  // wave-uniform
        meta_next = sl + NW < s1 ? Msh[sl + NW - s0] : 0u;
        if (PAR && (int)((meta >> 18) & 1u) != par) continue;
        const int pa = meta & 255u, pb = (meta >> 8) & 255u, kind = (meta >> 16) & 3u, line = (int)(meta >> 19);
        const float* qb = Qsh + (sl - s0) * MM;
        const cf r = Rsh[(line - l0) * RS + lane];
        const cf V = cmulc(Ush[pa * RS + lane], Ush[pb * RS + lane]);
        cf vr;
        switch (kind) {
          case kDirect: vr = r; break;
          case kConj: vr = cconj(r); break;
          case kRe: vr = {r.re, 0}; break;
          default: vr = {r.im, 0}; break;
        }
        const cf X = cadd(cscale(V, kv), cscale(vr, kr));
        cf y[M];
#pragma unroll
        for (int k = 0; k < M; k++) y[k] = cmul(X, u[k]);
        // the block's rows in groups of about 224 bytes (128 beyond 10 modes, whose
        // registers are fuller; 64 in the 168-VGPR variant): each group's LDS reads are issued together (the scheduling
        // barrier keeps them ahead of their uses), so one LDS latency is exposed per group
        // rather than one per pair of coefficients
        constexpr int QROW = PAR ? KH : M;  // coefficients per row p
        constexpr int QGB = HI ? 64 : (M > 10 ? 128 : 224);
        constexpr int PG = (int)(QGB / sizeof(float)) / QROW > 0 ? (int)(QGB / sizeof(float)) / QROW : 1;
#pragma unroll
        for (int p0 = 0; p0 < M; p0 += PG) {
          float qv[PG * QROW];
#pragma unroll
          for (int e = 0; e < PG * QROW; e++) qv[e] = p0 * QROW + e < M * QROW ? qb[p0 * QROW + e] : 0.f;
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int pp = 0; pp < PG; pp++) {
            const int p = p0 + pp;
            if (p >= M) break;
            cf tsum = acc[p];
            if constexpr (PAR) {
              // only k with (p + k) % 2 == the slot's parity: q[p][kk] belongs to k = 2 kk + ((p + par) % 2)
#pragma unroll
              for (int kk = 0; kk < KH; kk++) {
                const int k = 2 * kk + ((p + par) & 1);
                if (k < M) tsum = cadd(tsum, cscale(y[k], qv[pp * QROW + kk]));
              }
            } else {
#pragma unroll
              for (int k = 0; k < M; k++) tsum = cadd(tsum, cscale(y[k], qv[pp * QROW + k]));
            }
            acc[p] = tsum;
          }
        }
      }
    };
    // the matrix-core form: per parity class, the pairs of its slots in the chunk through the
    // 32 x 32 x 2 products, then sigma_p += U_k B[p][k] for this lane's sample
    auto mf_pass = [&](auto cls_c) {
      constexpr int cc = decltype(cls_c)::value;
      const int n = Nsh[cc];
      const int npairs = (n + 1) >> 1;
      constexpr int TPW = MR::TPW;
      constexpr int PSTEP = MR::TSPLIT ? 1 : 2;  // pairs between a wavefront's consecutive pairs
      mfma_acc_t ar[TPW], ai[TPW];
#pragma unroll
      for (int t = 0; t < TPW; t++) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          ar[t][r] = 0.f;
          ai[t][r] = 0.f;
        }
      }
      // the operands of pair pi (this lane's slot 2 pi + hh: X at its sample and its A-operand
      // coefficients; zeros past the class's last slot), built one pair ahead of its products so
      // that their LDS reads overlap the matrix-core work of the pair before; the slot's
      // descriptor (metadata, offset in the chunk) is read one pair before that
      auto descriptor = [&](int pi) { return Lsh[cc * kColStageSCap + (2 * pi + hh < n ? 2 * pi + hh : 0)]; };
      auto operands = [&](int pi, uint2 d, float& xre, float& xim, float (&qa)[TPW]) {
        // past the last slot: slot 0's data (finite) times zero, so that no branch splits the reads
        const float hm = 2 * pi + hh < n ? 1.f : 0.f;
        const uint32_t meta = d.x;
        const int x = (int)d.y;
        const int pa = meta & 255u, pb = (meta >> 8) & 255u, kind = (meta >> 16) & 3u, line = (int)(meta >> 19);
        const cf r = Rsh[(line - l0) * RS + smp];
        const cf ua = Ush[pa * RS + smp], ub = Ush[pb * RS + smp];
#pragma unroll
        for (int t = 0; t < TPW; t++) {
          const int o = aoff[cc][t];
          qa[t] = Qsh[x * MM + (o >= 0 ? o : 0)] * (o >= 0 ? hm : 0.f);
        }
        const cf V = cmulc(ua, ub);
        const float vre = kind == kIm ? r.im : r.re;
        const float vim = kind == kDirect ? r.im : (kind == kConj ? -r.im : 0.f);
        xre = (kv * V.re + kr * vre) * hm;
        xim = (kv * V.im + kr * vim) * hm;
      };
      int pi = MR::TSPLIT ? 0 : (wave >> 1);
      float xre, xim, qa[TPW];
      uint2 dn = {0u, 0u};
      if (n > 0) {
        operands(pi, descriptor(pi), xre, xim, qa);
        dn = descriptor(pi + PSTEP);
      }
#pragma nounroll
      for (; pi < npairs; pi += PSTEP) {  // wave-uniform
        float nre, nim, nqa[TPW];
        const uint2 d2 = dn;
        dn = descriptor(pi + 2 * PSTEP);
        operands(pi + PSTEP, d2, nre, nim, nqa);
#pragma unroll
        for (int t = 0; t < TPW; t++) {
          if (MR::TSPLIT && TPW * tg + t >= MR::RT) continue;  // wave-uniform: a tile of the group absent
          ar[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(qa[t], xre, ar[t], 0, 0, 0);
          ai[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(qa[t], xim, ai[t], 0, 0, 0);
        }
        xre = nre;
        xim = nim;
#pragma unroll
        for (int t = 0; t < TPW; t++) qa[t] = nqa[t];
      }
      // accumulator register r of tile t holds u = 16 t + r: mode p = u / KHH, and k from the
      // half; the tile group is a compile-time constant of each epilogue instance
      auto epilogue = [&](auto tg_c) {
        constexpr int TG = decltype(tg_c)::value;
#pragma unroll
        for (int j = 0; j < TPW; j++) {
          const int t = TPW * TG + j;
          if (t >= MR::RT) break;
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int uu = 16 * t + r;
            const int p = uu / MR::KHH;
            if (p < M) {
              const int kk0 = 2 * (uu % MR::KHH);
              const int kA = PAR ? 2 * kk0 + ((p + cc) & 1) : kk0;
              const int kB = PAR ? kA + 2 : kA + 1;
              // U_k of this lane's half from its LDS row (a padding row's products are zero: any
              // field row serves)
              const int row = kA >= M ? 0 : (kB < M ? kA + (kB - kA) * hh : kA);
              const cf uk = Ush[row * RS + smp];
              acc[p] = cadd(acc[p], cmul(uk, cf{ar[j][r], ai[j][r]}));
            }
          }
        }
      };
      if constexpr (!MR::TSPLIT) {
        epilogue(std::integral_constant<int, 0>{});
      } else {
        if (tg == 0) epilogue(std::integral_constant<int, 0>{});
        else epilogue(std::integral_constant<int, 1>{});
      }
      // the sums are taken here, so that the accumulators of one class are free before the next
      // class's products start (otherwise the compiler sinks them past those and spills)
#pragma unroll
      for (int p = 0; p < M; p++) asm volatile("" : "+v"(acc[p].re), "+v"(acc[p].im));
    };
    if constexpr (MF) {
      mf_pass(std::integral_constant<int, 0>{});
      if constexpr (PAR) mf_pass(std::integral_constant<int, 1>{});
    } else {
      slot_pass(std::integral_constant<int, 0>{});
      if constexpr (PAR) slot_pass(std::integral_constant<int, 1>{});
    }
  }
  __syncthreads();  // every lane done with Ush and Rsh
  // NW partial sums of every mode and sample (MF: one per pair parity, or tile group, and lane half)
  const int part = MF ? 2 * (wave >> 1) + hh : wave;
#pragma unroll
  for (int p = 0; p < M; p++) Rsh[(part * M + p) * L + smp] = acc[p];
  __syncthreads();
  for (int e = tid; e < M * L; e += NT) {
    const int p = e / L, j = e % L;
    cf tsum = Rsh[p * L + j];
#pragma unroll
    for (int w = 1; w < NW; w++) tsum = cadd(tsum, Rsh[(w * M + p) * L + j]);
    Ush[p * RS + j] = tsum;
  }
  __syncthreads();
  if (wave * (64 / T) < M) {
    const int q = job;
    const bool valid = q < M;
    cf* row = Ush + q * RS;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = valid ? row[t + i * T] : cf{0, 0};
    line_fft<L, -1, 1, 1, float, true>(v, row, lt, t);
    if (valid) {
      const size_t base = (size_t)q * g.N + n2;
#pragma unroll
      for (int i = 0; i < 8; i++) store_stream64(yout + base + (size_t)(t + i * T) * g.N2, cmul(v[i], w4[i]));
    }
  }
}

// ---------------------------------------------------------------------------
// Dense-block Kerr + Raman gather for M <= 16 modes, 64 samples per workgroup:
//   sigma_p = sum over slots s of  sum_k Qd[s][p][k] * X_s * U_k
// Each lane keeps its sample's U_k (all k) and sigma_p (all p) in registers; X_s
// comes from LDS (one read per slot) and the M x M block Qd[s] (zeros included)
// from scalar loads. The four wavefronts take every fourth slot and their
// partial sums are added in wavefront order at the end.
// ---------------------------------------------------------------------------
constexpr int kDenseCap = 4096;  // complex LDS values (64 KB)

int dense_gather_chunk(int M) {
  if (M < 1 || M > 16) return 0;
  const int room = kDenseCap / 64 - M;
  return room >= 4 * M ? room : 0;
}

template <int M>
__global__ void __launch_bounds__(256) k_gather_dense(Geometry g, const cf* __restrict__ U,
                                                      const cf* __restrict__ VR, cf* __restrict__ sigma,
                                                      GatherArgs a, const float* __restrict__ Qd, int chunk) {
  __shared__ cf sh[kDenseCap];
  constexpr int TS = 64;
  cf* Ush = sh;           // [M][TS]
  cf* Xsh = sh + M * TS;  // [chunk][TS]; reused for the partial sums
  const int t0 = blockIdx.x * TS;
  const int tid = threadIdx.x, lane = tid % TS;
  const int wave = __builtin_amdgcn_readfirstlane(tid / TS);
#pragma unroll 4
  for (int e = tid; e < M * TS; e += 256) Ush[e] = U[(size_t)(e / TS) * g.N + t0 + e % TS];
  __syncthreads();
  cf u[M], acc[M];
#pragma unroll
  for (int k = 0; k < M; k++) {
    u[k] = Ush[k * TS + lane];
    acc[k] = {0, 0};
  }
  for (int s0 = 0; s0 < a.n_slots; s0 += chunk) {
    const int ns = min(chunk, a.n_slots - s0);
    __syncthreads();  // previous chunk consumed
    slot_mix_tile(a, g, VR, Ush, Xsh, s0, ns, t0, tid, 256);
    __syncthreads();
    for (int sl = s0 + wave; sl < s0 + ns; sl += 4) {
      const cf X = Xsh[(sl - s0) * TS + lane];
      const float* qb = Qd + (size_t)sl * M * M;
      cf y[M];
#pragma unroll
      for (int k = 0; k < M; k++) y[k] = cmul(X, u[k]);
#pragma unroll
      for (int p = 0; p < M; p++) {
        cf t = acc[p];
#pragma unroll
        for (int k = 0; k < M; k++) t = cadd(t, cscale(y[k], qb[p * M + k]));
        acc[p] = t;
      }
    }
  }
  __syncthreads();  // X consumed: the region takes the partial sums
#pragma unroll
  for (int p = 0; p < M; p++) Xsh[(wave * M + p) * TS + lane] = acc[p];
  __syncthreads();
  for (int e = tid; e < M * TS; e += 256) {
    const int p = e / TS, j = e % TS;
    cf t = Xsh[p * TS + j];
#pragma unroll
    for (int w = 1; w < 4; w++) t = cadd(t, Xsh[(w * M + p) * TS + j]);
    sigma[(size_t)p * g.N + t0 + j] = t;
  }
}

// per-mode energy sum_j |A_p,j|^2 * dt; one workgroup per mode, fixed reduction order
__global__ void __launch_bounds__(256) k_energy(Geometry g, const cd* __restrict__ f, double* __restrict__ out,
                                                double dt) {
  __shared__ double red[256];
  const int p = blockIdx.x;
  double s = 0.;
  for (int j = threadIdx.x; j < g.N; j += 256) {
    const cd x = f[(size_t)p * g.N + j];
    s += x.re * x.re + x.im * x.im;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[p] = red[0] * dt;
}

// Per-mode photon number of a spectral state in four-step order (S[k1*N2 + k2] holds bin
// k = k1 + N1*k2): out[p] = scale * sum_k |S_p[k]|^2 / (omega0 - dalpha * k_signed), k_signed = k
// for k <= N/2, else k - N (the reference's frequency grid, src/MultimodePropagation.cpp:171-175).
// One workgroup per mode, fixed reduction order; FP64 throughout.
__global__ void __launch_bounds__(256) k_photon_number(Geometry g, const cd* __restrict__ S, double* __restrict__ out,
                                                       double omega0, double dalpha, double scale) {
  __shared__ double red[256];
  const int p = blockIdx.x;
  double s = 0.;
  for (int idx = threadIdx.x; idx < g.N; idx += 256) {
    const int k1 = idx / g.N2, k2 = idx - k1 * g.N2;
    const int k = k1 + g.N1 * k2;
    const int ks = k <= g.N / 2 ? k : k - g.N;
    const cd x = S[(size_t)p * g.N + idx];
    s += (x.re * x.re + x.im * x.im) / (omega0 - dalpha * (double)ks);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[p] = red[0] * scale;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
#define MMP_DISPATCH_L(Lv, FN, ...)                        \
  switch (Lv) {                                            \
    case 8: return FN<8>(__VA_ARGS__);                     \
    case 16: return FN<16>(__VA_ARGS__);                   \
    case 32: return FN<32>(__VA_ARGS__);                   \
    case 64: return FN<64>(__VA_ARGS__);                   \
    case 128: return FN<128>(__VA_ARGS__);                 \
    case 256: return FN<256>(__VA_ARGS__);                 \
    case 512: return FN<512>(__VA_ARGS__);                 \
    case 1024: return FN<1024>(__VA_ARGS__);               \
    default: return hipErrorInvalidValue;                  \
  }

// column lengths: N1 <= 64 for every supported nt (the split keeps rows within 1024)
#define MMP_DISPATCH_COL_LW(Lv, FN, W, ...)                \
  switch (Lv) {                                            \
    case 8: return FN<8, W>(__VA_ARGS__);                  \
    case 16: return FN<16, W>(__VA_ARGS__);                \
    case 32: return FN<32, W>(__VA_ARGS__);                \
    case 64: return FN<64, W>(__VA_ARGS__);                \
    default: return hipErrorInvalidValue;                  \
  }

#define MMP_DISPATCH_LW(Lv, FN, W, ...)                    \
  switch (Lv) {                                            \
    case 8: return FN<8, W>(__VA_ARGS__);                  \
    case 16: return FN<16, W>(__VA_ARGS__);                \
    case 32: return FN<32, W>(__VA_ARGS__);                \
    case 64: return FN<64, W>(__VA_ARGS__);                \
    case 128: return FN<128, W>(__VA_ARGS__);              \
    case 256: return FN<256, W>(__VA_ARGS__);              \
    case 512: return FN<512, W>(__VA_ARGS__);              \
    case 1024: return FN<1024, W>(__VA_ARGS__);            \
    default: return hipErrorInvalidValue;                  \
  }

template <int L, class W>
static hipError_t row_head_impl(const Geometry& g, const Twiddles& tw, const HeadArgs& a, const Batch& b, int F,
                                hipStream_t s) {
  using C = RowCfg<L>;
  const int rows = g.M * g.N1;
  dim3 grid((rows + C::G - 1) / C::G, F);
  // FP32 work arrays (mixed precision) take the table-free form, FP64 ones the tables
  constexpr bool RE = std::is_same<W, float>::value;
  if ((a.recompute_e != 0) != RE) return hipErrorInvalidValue;
#define MMP_HEAD(ST) MMP_LAUNCH((k_row_head<L, W, RE, ST>), grid, dim3(C::THREADS), 0, s, g, TwOf<W>::row(tw), a, b)
  if constexpr (RE) {
    MMP_HEAD(true);
  } else {
    if (a.n_stash > 0) MMP_HEAD(true);
    else MMP_HEAD(false);
  }
#undef MMP_HEAD
  return hipGetLastError();
}
template <class W>
hipError_t launch_row_head(const Geometry& g, const Twiddles& tw, const HeadArgs& a, const Batch& b, int F,
                           hipStream_t s) {
  if (F < 1 || F > 65535) return hipErrorInvalidValue;
  MMP_DISPATCH_LW(g.N2, row_head_impl, W, g, tw, a, b, F, s);
}

// Column-block width: 8 when that already gives >= 256 workgroups, else 4, else 2.
template <int L>
static int pick_cb(const Geometry& g, int lines) {
  const int cbs[3] = {8, 4, 2};
  for (int cb : cbs) {
    const int T = L / 8;
    const int G = (cb * T >= 64) ? 1 : 64 / (cb * T);
    const int blocks = (g.N2 / cb) * ((lines + G - 1) / G);
    if (blocks >= 256 || cb == 2) return cb;
  }
  return 2;
}

template <int L, int CB>
static dim3 col_grid(const Geometry& g, int lines) {
  using C = ColCfg<L, CB>;
  return dim3((g.N2 / CB) * ((lines + C::G - 1) / C::G));
}

#define MMP_COL_LAUNCH(KERNEL, LINES, ...)                                                                      \
  switch (pick_cb<L>(g, LINES)) {                                                                               \
    case 8: MMP_LAUNCH((KERNEL<L, 8, W>), (col_grid<L, 8>(g, LINES)), (dim3(ColCfg<L, 8>::THREADS)), 0, s, \
                               __VA_ARGS__); break;                                                            \
    case 4: MMP_LAUNCH((KERNEL<L, 4, W>), (col_grid<L, 4>(g, LINES)), (dim3(ColCfg<L, 4>::THREADS)), 0, s, \
                               __VA_ARGS__); break;                                                            \
    default: MMP_LAUNCH((KERNEL<L, 2, W>), (col_grid<L, 2>(g, LINES)), (dim3(ColCfg<L, 2>::THREADS)), 0,  \
                                s, __VA_ARGS__); break;                                                        \
  }                                                                                                             \
  return hipGetLastError();

template <int L, class W>
static hipError_t col_inverse_impl(const Geometry& g, const Twiddles& tw, const cpx<W>* in, cpx<W>* out, int lines,
                                   double scale, double divisor, hipStream_t s) {
  MMP_COL_LAUNCH(k_col_inverse, lines, g, TwOf<W>::col(tw), TwOf<W>::four(tw), in, out, lines, scale, divisor)
}
template <class W>
hipError_t launch_col_inverse(const Geometry& g, const Twiddles& tw, const cpx<W>* in, cpx<W>* out, int lines,
                              double scale, double divisor, hipStream_t s) {
  MMP_DISPATCH_COL_LW(g.N1, col_inverse_impl, W, g, tw, in, out, lines, scale, divisor, s);
}

template <int L, class W>
static hipError_t col_forward_impl(const Geometry& g, const Twiddles& tw, const cpx<W>* in, cpx<W>* out, int lines,
                                   hipStream_t s) {
  MMP_COL_LAUNCH(k_col_forward, lines, g, TwOf<W>::col(tw), TwOf<W>::four(tw), in, out, lines)
}
template <class W>
hipError_t launch_col_forward(const Geometry& g, const Twiddles& tw, const cpx<W>* in, cpx<W>* out, int lines,
                              hipStream_t s) {
  MMP_DISPATCH_COL_LW(g.N1, col_forward_impl, W, g, tw, in, out, lines, s);
}

template <int L, class W>
static hipError_t col_forward_real_impl(const Geometry& g, const Twiddles& tw, const double* in, cd* out,
                                        hipStream_t s) {
  MMP_COL_LAUNCH(k_col_forward_real, 1, g, tw.coltw, tw.fourtw, in, out)
}
hipError_t launch_col_forward_real(const Geometry& g, const Twiddles& tw, const double* in, cd* out,
                                   hipStream_t s) {
  MMP_DISPATCH_COL_LW(g.N1, col_forward_real_impl, double, g, tw, in, out, s);
}

template <int L, class W>
static hipError_t col_pairs_forward_impl(const Geometry& g, const Twiddles& tw, const cpx<W>* U, cpx<W>* out,
                                         int lines, const uint2* line_prod, hipStream_t s) {
  MMP_COL_LAUNCH(k_col_pairs_forward, lines, g, TwOf<W>::col(tw), TwOf<W>::four(tw), U, out, lines, line_prod)
}
template <class W>
hipError_t launch_col_pairs_forward(const Geometry& g, const Twiddles& tw, const cpx<W>* U, cpx<W>* out, int lines,
                                    const uint2* line_prod, hipStream_t s) {
  MMP_DISPATCH_COL_LW(g.N1, col_pairs_forward_impl, W, g, tw, U, out, lines, line_prod, s);
}

template <int L>
static hipError_t row_forward_impl(const Geometry& g, const Twiddles& tw, cd* data, int lines, hipStream_t s) {
  using C = RowCfg<L>;
  const int rows = lines * g.N1;
  MMP_LAUNCH(k_row_forward<L>, dim3((rows + C::G - 1) / C::G), dim3(C::THREADS), 0, s, g, tw.rowtw, data,
                     lines);
  return hipGetLastError();
}
hipError_t launch_row_forward(const Geometry& g, const Twiddles& tw, cd* data, int lines, hipStream_t s) {
  MMP_DISPATCH_L(g.N2, row_forward_impl, g, tw, data, lines, s);
}

template <int L>
static hipError_t row_inverse_phase_impl(const Geometry& g, const Twiddles& tw, const cd* in, cd* out,
                                         const double* imL, const StepState* st, int use_phase, hipStream_t s) {
  using C = RowCfg<L>;
  const int rows = g.M * g.N1;
  MMP_LAUNCH(k_row_inverse_phase<L>, dim3((rows + C::G - 1) / C::G), dim3(C::THREADS), 0, s, g, tw.rowtw,
                     in, out, imL, st, use_phase);
  return hipGetLastError();
}
hipError_t launch_row_inverse_phase(const Geometry& g, const Twiddles& tw, const cd* in, cd* out,
                                    const double* imL, const StepState* st, int use_phase, hipStream_t s) {
  MMP_DISPATCH_L(g.N2, row_inverse_phase_impl, g, tw, in, out, imL, st, use_phase, s);
}

template <int L, class W>
static hipError_t row_raman_impl(const Geometry& g, const Twiddles& tw, cpx<W>* data, int lines, const cpx<W>* hspec,
                                 const Batch& b, int F, hipStream_t s) {
  using C = RowCfg<L>;
  const int rows = lines * g.N1;
  MMP_LAUNCH((k_row_raman<L, W>), dim3((rows + C::G - 1) / C::G, F), dim3(C::THREADS), 0, s, g,
                     TwOf<W>::row(tw), data, lines, hspec, b);
  return hipGetLastError();
}
template <class W>
hipError_t launch_row_raman(const Geometry& g, const Twiddles& tw, cpx<W>* data, int lines, const cpx<W>* hspec,
                            const Batch& b, int F, hipStream_t s) {
  if (F < 1 || F > 65535) return hipErrorInvalidValue;
  MMP_DISPATCH_LW(g.N2, row_raman_impl, W, g, tw, data, lines, hspec, b, F, s);
}

template <int L, class W>
static hipError_t row_raman_cols_impl(const Geometry& g, const Twiddles& tw, const cpx<W>* in, cpx<W>* out, int lines,
                                      const cpx<W>* hspec, const Batch& b, int F, int in_cols, hipStream_t s) {
  using C = RamanColsCfg<L, W>;
  if (g.N1 % C::R) return hipErrorInvalidValue;
  MMP_LAUNCH((k_row_raman_cols<L, W>), dim3(lines * g.N1 / C::R, F), dim3(C::THREADS), 0, s, g, TwOf<W>::row(tw), in,
             out, hspec, b, in_cols);
  return hipGetLastError();
}
template <class W>
hipError_t launch_row_raman_cols(const Geometry& g, const Twiddles& tw, const cpx<W>* in, cpx<W>* out, int lines,
                                 const cpx<W>* hspec, const Batch& b, int F, int in_cols, hipStream_t s) {
  if (F < 1 || F > 65535 || lines < 1 || in == out) return hipErrorInvalidValue;
  MMP_DISPATCH_LW(g.N2, row_raman_cols_impl, W, g, tw, in, out, lines, hspec, b, F, in_cols, s);
}

template <class W>
hipError_t launch_gather(const Geometry& g, const cpx<W>* U, const cpx<W>* VR, cpx<W>* sigma, const GatherArgs& a,
                         hipStream_t s) {
  if (g.N % kGatherTS) return hipErrorInvalidValue;
  int waves = g.M < 8 ? g.M : 8;
  if ((g.M + waves - 1) / waves > kGatherMaxPW) return hipErrorInvalidValue;
  // A wavefront sums its modes one after the other, so small grids deal the modes to groups of workgroups,
  // up to one mode a wavefront, while tiles x groups stay within 512 in FP32 (two workgroups a CU) and 256 in FP64
  // (one: up to 128 KB of LDS each). Beyond that each group's own slot mix, and its reading of every field, cost
  // more than it gives. Steps on one MI355X, us with one group and with the rule's. Mixed: 20 modes, NT = 1024 (16
  // tiles) 2307 -> 1174, NT = 4096 2392 -> 1223; 32 modes, NT = 4096 15423 -> 4310; 14 modes, NT = 1024 835 -> 527;
  // 18 modes, NT = 16384 (256 tiles) 2002 -> 1644 with two, 1873 with three; 20 modes, NT = 65536 (1024 tiles)
  // 8222, two groups 8546; a tenth of the list or less gains too (20 modes, NT = 16384 590 -> 494) or stays. FP64,
  // 20 modes without parity structure, a tenth of the list: NT = 4096 679 -> 353 (three groups of 64 tiles), NT =
  // 8192 693 -> 516 with two (598 with three), NT = 16384 748 with one, 854 with two; self pairs alone, NT = 16384
  // 133 with one, 145 with two.
  const int tiles = g.N / kGatherTS;
  const int resident = sizeof(W) == 8 ? 256 : 512;
  int groups = (g.M + waves - 1) / waves;
  while (groups > 1 && tiles * groups > resident) groups--;
  dim3 grid(g.N / kGatherTS, groups), block(kGatherTS * waves);
  if (a.cap == 4096) MMP_LAUNCH((k_gather<4096, W>), grid, block, 0, s, g, U, VR, sigma, a);
  else if (a.cap == 8192) MMP_LAUNCH((k_gather<8192, W>), grid, block, 0, s, g, U, VR, sigma, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

template <int QROW, bool PAR>
static hipError_t gather_products_impl(const Geometry& g, const cd* U, const cd* VR, cd* sigma, const ProductArgs& fa,
                                       const double* Qp, const Batch& b, int raman, hipStream_t s) {
  const int rows = products_field_rows(g.M, PAR);
  const size_t lds = (size_t)(rows + (fa.max_chunk_lines + 1) / 2 * 2) * kProductsTS * sizeof(cd);
  if (lds > kColStageLds) return hipErrorInvalidValue;
  const int groups = (g.M + kProductsMaxWaves - 1) / kProductsMaxWaves;
  int waves = (g.M + groups - 1) / groups;
  if (waves < 4) waves = 4;  // (the X rows are mixed by all)
  MMP_LAUNCH((k_gather_products<QROW, PAR>), dim3(g.N / kProductsTS, groups), dim3(waves * 64), lds, s, g, U, VR, sigma, fa,
             Qp, b, raman, rows);
  return hipGetLastError();
}
#define MMP_GATHER_PRODUCTS_CASE(QV)                                                                    \
  case QV:                                                                                              \
    return fa.parity ? gather_products_impl<QV, true>(g, U, VR, sigma, fa, Qp, b, raman, s)             \
                     : gather_products_impl<QV, false>(g, U, VR, sigma, fa, Qp, b, raman, s);
hipError_t launch_gather_products(const Geometry& g, const cd* U, const cd* VR, cd* sigma, const ProductArgs& fa,
                                  const double* Qp, const Batch& b, int raman, hipStream_t s) {
  if (g.N % kProductsTS || !gather_products_ok(g.M, fa.parity) || fa.n_chunks < 1 || fa.max_chunk_lines < 1 ||
      fa.n_products > 2 * fa.n_lines || fa.n_steps < 1 || fa.n_steps > fa.stride || (raman && !VR))
    return hipErrorInvalidValue;
  switch (fa.parity ? (g.M + 1) / 2 : g.M) {
    MMP_GATHER_PRODUCTS_CASE(1) MMP_GATHER_PRODUCTS_CASE(2) MMP_GATHER_PRODUCTS_CASE(3) MMP_GATHER_PRODUCTS_CASE(4)
    MMP_GATHER_PRODUCTS_CASE(5) MMP_GATHER_PRODUCTS_CASE(6) MMP_GATHER_PRODUCTS_CASE(7) MMP_GATHER_PRODUCTS_CASE(8)
    MMP_GATHER_PRODUCTS_CASE(9) MMP_GATHER_PRODUCTS_CASE(10) MMP_GATHER_PRODUCTS_CASE(11) MMP_GATHER_PRODUCTS_CASE(12)
    MMP_GATHER_PRODUCTS_CASE(13) MMP_GATHER_PRODUCTS_CASE(14) MMP_GATHER_PRODUCTS_CASE(15) MMP_GATHER_PRODUCTS_CASE(16)
    default: return hipErrorInvalidValue;
  }
}

size_t colstage_pairs_lds_bytes(int M, int columns, bool mixed) {
  return (size_t)(ColStageCfg::FFT + M * kColStageL * columns) * (mixed ? sizeof(cf) : sizeof(cd));
}

// Measured on one MI355X (M = 2..15, NT = 4096..65536, 1 to 36 fibers): four columns per
// workgroup took the pass from 0.6-1.5 TB/s to 2-3.4 TB/s; eight gained nothing over four
// (twice the LDS, lower occupancy). Line groups fill the CUs when the column blocks alone are
// too few, but each group transforms every field again, so a group keeps at least 4 lines of the general count.
// FP64 with couplings symmetric in the pair runs about half of those (11 of 18 at 6 modes: groups of 2 and 3);
// groups planned on the lines that run measured the same within 1 % over 232 forms (NT = 4096, us per step: 4
// modes 72.7 as planned and 73.8, 6 modes 80.7 and 81.5, 13 modes 164 and 158), so one layout serves
// the fiber whatever its couplings and whichever fibers join it.
void colstage_pairs_plan(int M, int N2, int n_lines, int F, bool mixed, int& columns, int& groups) {
  columns = 1;
  for (int cw : {4, 2})
    if (N2 % cw == 0 && colstage_pairs_lds_bytes(M, cw, mixed) <= kColStagePairsLds) {
      columns = cw;
      break;
    }
  groups = 1;
  while ((long)(N2 / columns) * F * groups < 512 && groups * 2 * 4 <= n_lines) groups *= 2;
}

template <class W>
hipError_t launch_colstage_fields_pairs(const Geometry& g, const Twiddles& tw, const cpx<W>* yin, cpx<W>* U,
                                        cpx<W>* conv, const uint2* line_prod, int n_lines, double scale,
                                        const Batch& b, int F, int columns, int groups, int conv_cols, hipStream_t s) {
  if (g.N1 != kColStageL || g.M < 1 || g.M > kColStageMaxM || F < 1 || F > 65535 || n_lines < 1) return hipErrorInvalidValue;
  if (columns < 1 || g.N2 % columns || groups < 1 || groups > n_lines) return hipErrorInvalidValue;
  const size_t lds = colstage_pairs_lds_bytes(g.M, columns, std::is_same<W, float>::value);
  if (lds > kColStagePairsLds) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(g.N2 / columns * groups), F);
  switch (columns) {
    case 1: MMP_LAUNCH((k_colstage_fields_pairs<W, 1>), grid, dim3(256), lds, s, g, TwOf<W>::col(tw),
                       TwOf<W>::four(tw), yin, U, conv, n_lines, line_prod, scale, b, groups, conv_cols); break;
    case 2: MMP_LAUNCH((k_colstage_fields_pairs<W, 2>), grid, dim3(256), lds, s, g, TwOf<W>::col(tw),
                       TwOf<W>::four(tw), yin, U, conv, n_lines, line_prod, scale, b, groups, conv_cols); break;
    case 4: MMP_LAUNCH((k_colstage_fields_pairs<W, 4>), grid, dim3(256), lds, s, g, TwOf<W>::col(tw),
                       TwOf<W>::four(tw), yin, U, conv, n_lines, line_prod, scale, b, groups, conv_cols); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// C2 in FP64, on the real products
template <int M, int NW, int COLS, bool PAR, bool RAMAN>
static hipError_t c2_launch(const Geometry& g, const Twiddles& tw, const cd* U, const cd* conv, cd* yout,
                            const ProductArgs& fa, const double* Qp, double scale, const Batch& b, int F, hipStream_t s) {
  const size_t lds = colstage_products_lds_bytes(M, COLS, fa.max_chunk_lines, fa.stride, PAR);
  if (g.N2 % COLS || lds > kColStageLds) return hipErrorInvalidValue;
  MMP_LAUNCH((k_colstage_products<M, NW, COLS, PAR, RAMAN>), dim3(g.N2 / COLS, F), dim3(NW * 64), lds, s, g, tw.coltw,
             tw.fourtw, U, conv, yout, fa, Qp, scale, b);
  return hipGetLastError();
}
template <int M, bool PAR, bool RAMAN>
static hipError_t c2_variant(const Geometry& g, const Twiddles& tw, const cd* U, const cd* conv, cd* yout,
                             const ProductArgs& fa, const double* Qp, double scale, const Batch& b, int F, hipStream_t s) {
  if constexpr (RAMAN && M <= kColStageMaxM4) {  // (without Raman one fiber's columns: one a workgroup)
    if (fa.cols == 4) return c2_launch<M, 4, 4, PAR, RAMAN>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
  }
  if constexpr (RAMAN && M <= kColStageMaxM2) {
    if (fa.cols == 2) return c2_launch<M, 4, 2, PAR, RAMAN>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
  }
  if (fa.cols != 1) return hipErrorInvalidValue;
  if constexpr (PAR && (M == 5 || M == 6)) {
    if (fa.waves == 12) {
      if (fa.n_chunks != 1) return hipErrorInvalidValue;
      return c2_launch<M, 12, 1, PAR, RAMAN>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
    }
  }
  if (fa.waves == 8 && M <= 4 && PAR && fa.n_chunks != 1) return hipErrorInvalidValue;
  if (fa.waves == 8) return c2_launch<M, 8, 1, PAR, RAMAN>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
  return c2_launch<M, 4, 1, PAR, RAMAN>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
}
template <int M>
static hipError_t c2_form(const Geometry& g, const Twiddles& tw, const cd* U, const cd* conv, cd* yout, const ProductArgs& fa,
                          const double* Qp, double scale, const Batch& b, int F, hipStream_t s) {
  if (conv) return fa.parity ? c2_variant<M, true, true>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s)
                             : c2_variant<M, false, true>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
  return fa.parity ? c2_variant<M, true, false>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s)
                   : c2_variant<M, false, false>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
}
#define MMP_PRODUCTS_CASE(MV) \
  case MV: return c2_form<MV>(g, tw, U, conv, yout, fa, Qp, scale, b, F, s);
hipError_t launch_colstage_products(const Geometry& g, const Twiddles& tw, const cd* U, const cd* conv, cd* yout,
                                    const ProductArgs& fa, const double* Qp, double scale, const Batch& b, int F,
                                    hipStream_t s) {
  if (g.N1 != kColStageL || F < 1 || F > 65535) return hipErrorInvalidValue;
  if (fa.n_chunks < 1 || fa.max_chunk_lines < 1 || fa.max_chunk_lines > colstage_lines_per_chunk(g.M) ||
      fa.first_lines > fa.max_chunk_lines || fa.n_products > 2 * fa.n_lines || fa.stride < 1 || fa.n_steps > fa.stride)
    return hipErrorInvalidValue;
  switch (g.M) {
    MMP_PRODUCTS_CASE(1) MMP_PRODUCTS_CASE(2) MMP_PRODUCTS_CASE(3) MMP_PRODUCTS_CASE(4) MMP_PRODUCTS_CASE(5)
    MMP_PRODUCTS_CASE(6) MMP_PRODUCTS_CASE(7) MMP_PRODUCTS_CASE(8) MMP_PRODUCTS_CASE(9) MMP_PRODUCTS_CASE(10)
    MMP_PRODUCTS_CASE(11) MMP_PRODUCTS_CASE(12) MMP_PRODUCTS_CASE(13) MMP_PRODUCTS_CASE(14) MMP_PRODUCTS_CASE(15)
    MMP_PRODUCTS_CASE(16)
    default: return hipErrorInvalidValue;
  }
}

// C2 in FP32, on the complex slots
#define MMP_COLSTAGE_GO(MV, NWV, PARV, ...)                                                                        \
  MMP_LAUNCH((k_colstage_raman_gather<MV, NWV, PARV __VA_ARGS__>), dim3(g.N2, F), dim3(NWV * 64), 0, s, g,  \
             tw.coltw32, tw.fourtw32, U, conv, yout, fa, Qd, scale, b);                                            \
  break;
#define MMP_COLSTAGE_LAUNCH(MV, PARV)                                                                              \
  if constexpr (kColStageMfma<MV, PARV>)                                                                           \
    if (fa.waves == 4 && fa.matrix_cores) {                                                                        \
      MMP_COLSTAGE_GO(MV, 4, PARV, , false, true)                                                                  \
    }                                                                                                              \
  if constexpr (hi_occupancy(MV, PARV))                                                                            \
    if (fa.waves == 4 && fa.hi_occupancy) {                                                                        \
      MMP_COLSTAGE_GO(MV, 4, PARV, , true)                                                                         \
    }                                                                                                              \
  if constexpr (wide_gather(MV))                                                                                   \
    if (fa.waves == 8) {                                                                                           \
      MMP_COLSTAGE_GO(MV, 8, PARV)                                                                                 \
    }                                                                                                              \
  MMP_COLSTAGE_GO(MV, 4, PARV)
#define MMP_COLSTAGE_CASE(MV)                                                                                      \
  case MV:                                                                                                         \
    if (fa.parity) {                                                                                               \
      MMP_COLSTAGE_LAUNCH(MV, true)                                                                                \
    } else {                                                                                                       \
      MMP_COLSTAGE_LAUNCH(MV, false)                                                                               \
    }
hipError_t launch_colstage_raman_gather(const Geometry& g, const Twiddles& tw, const cf* U, const cf* conv, cf* yout,
                                        const SlotArgs& fa, const float* Qd, double scale, const Batch& b, int F,
                                        hipStream_t s) {
  if (g.N1 != kColStageL || F < 1 || F > 65535) return hipErrorInvalidValue;
  const int block = fa.parity ? g.M * ((g.M + 1) / 2) : g.M * g.M;
  if (fa.n_chunks < 1 || fa.max_chunk_lines < 1 || fa.max_chunk_lines > colstage_lines_per_chunk(g.M) ||
      fa.max_chunk_slots < 1 || fa.max_chunk_slots > colstage_slots_per_chunk() ||
      fa.max_chunk_slots * block > colstage_coefficients_per_chunk(g.M))
    return hipErrorInvalidValue;
  switch (g.M) {
    MMP_COLSTAGE_CASE(1) MMP_COLSTAGE_CASE(2) MMP_COLSTAGE_CASE(3) MMP_COLSTAGE_CASE(4) MMP_COLSTAGE_CASE(5)
    MMP_COLSTAGE_CASE(6) MMP_COLSTAGE_CASE(7) MMP_COLSTAGE_CASE(8) MMP_COLSTAGE_CASE(9) MMP_COLSTAGE_CASE(10)
    MMP_COLSTAGE_CASE(11) MMP_COLSTAGE_CASE(12) MMP_COLSTAGE_CASE(13) MMP_COLSTAGE_CASE(14) MMP_COLSTAGE_CASE(15)
    MMP_COLSTAGE_CASE(16)
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

#define MMP_DENSE_CASE(MV)                                                                                     \
  case MV:                                                                                                      \
    MMP_LAUNCH((k_gather_dense<MV>), dim3(g.N / 64), dim3(256), 0, s, g, U, VR, sigma, a, Qd, chunk);           \
    break;

hipError_t launch_gather_dense(const Geometry& g, const cf* U, const cf* VR, cf* sigma, const GatherArgs& a, const float* Qd,
                               hipStream_t s) {
  const int chunk = dense_gather_chunk(g.M);
  if (!chunk || g.N % 64) return hipErrorInvalidValue;
  switch (g.M) {
    MMP_DENSE_CASE(1) MMP_DENSE_CASE(2) MMP_DENSE_CASE(3) MMP_DENSE_CASE(4) MMP_DENSE_CASE(5) MMP_DENSE_CASE(6)
    MMP_DENSE_CASE(7) MMP_DENSE_CASE(8) MMP_DENSE_CASE(9) MMP_DENSE_CASE(10) MMP_DENSE_CASE(11) MMP_DENSE_CASE(12)
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

__global__ void __launch_bounds__(256) k_narrow(const cd* __restrict__ in, cf* __restrict__ out, size_t n) {
  for (size_t j = (size_t)blockIdx.x * 256 + threadIdx.x; j < n; j += (size_t)gridDim.x * 256)
    out[j] = narrow<float>(in[j]);
}

}  // namespace mmp

// Device memory of the no-allocation entry point (mmp_solve_static): every device array of one
// solve is carved from this array, so the call needs no hipMalloc. One copy per device, held
// until the process ends; its host-side name is not a device address (the address comes from
// hipGetSymbolAddress, once per device, in static_scratch_resolve).
static __device__ __align__(256) unsigned char scratch[mmp::kStaticScratchBytes];

namespace mmp {

namespace {
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kStaticScratchDevices] = {};
}  // namespace

hipError_t static_scratch_resolve(int device) {
  if (device < 0 || device >= kStaticScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[device]) return hipSuccess;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  g_scratch_ptr[device] = p;
  return hipSuccess;
}

void* static_scratch(int device) {
  if (device < 0 || device >= kStaticScratchDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  return g_scratch_ptr[device];
}

hipError_t launch_narrow(const cd* in, cf* out, size_t n, hipStream_t s) {
  const size_t blocks = (n + 255) / 256;
  MMP_LAUNCH(k_narrow, dim3((unsigned)(blocks < 4096 ? (blocks ? blocks : 1) : 4096)), dim3(256), 0, s, in,
                     out, n);
  return hipGetLastError();
}

hipError_t launch_energy(const Geometry& g, const cd* fields, double* out, double dt, hipStream_t s) {
  MMP_LAUNCH(k_energy, dim3(g.M), dim3(256), 0, s, g, fields, out, dt);
  return hipGetLastError();
}

hipError_t launch_photon_number(const Geometry& g, const cd* spectra, double* out, double omega0, double dalpha,
                                double scale, hipStream_t s) {
  if (g.N1 * g.N2 != g.N || g.M < 1) return hipErrorInvalidValue;
  MMP_LAUNCH(k_photon_number, dim3(g.M), dim3(256), 0, s, g, spectra, out, omega0, dalpha, scale);
  return hipGetLastError();
}

#define MMP_INSTANTIATE_W(W)                                                                                        \
  template hipError_t launch_row_head<W>(const Geometry&, const Twiddles&, const HeadArgs&, const Batch&, int,    \
                                         hipStream_t);                                                             \
  template hipError_t launch_col_inverse<W>(const Geometry&, const Twiddles&, const cpx<W>*, cpx<W>*, int, double, \
                                            double, hipStream_t);                                                 \
  template hipError_t launch_col_forward<W>(const Geometry&, const Twiddles&, const cpx<W>*, cpx<W>*, int,         \
                                            hipStream_t);                                                         \
  template hipError_t launch_col_pairs_forward<W>(const Geometry&, const Twiddles&, const cpx<W>*, cpx<W>*, int,   \
                                                  const uint2*, hipStream_t);                                     \
  template hipError_t launch_row_raman<W>(const Geometry&, const Twiddles&, cpx<W>*, int, const cpx<W>*,           \
                                          const Batch&, int, hipStream_t);                                         \
  template hipError_t launch_gather<W>(const Geometry&, const cpx<W>*, const cpx<W>*, cpx<W>*, const GatherArgs&,  \
                                       hipStream_t);                                                              \
  template hipError_t launch_row_raman_cols<W>(const Geometry&, const Twiddles&, const cpx<W>*, cpx<W>*, int,         \
                                               const cpx<W>*, const Batch&, int, int, hipStream_t);                 \
  template hipError_t launch_colstage_fields_pairs<W>(const Geometry&, const Twiddles&, const cpx<W>*, cpx<W>*,     \
                                                      cpx<W>*, const uint2*, int, double, const Batch&, int, int,  \
                                                      int, int, hipStream_t);
MMP_INSTANTIATE_W(double)
MMP_INSTANTIATE_W(float)

}  // namespace mmp
