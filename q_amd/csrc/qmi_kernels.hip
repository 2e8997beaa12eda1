// HIP kernels of the MI355X qdyn step (gfx950, wave64).
//
// Bulk nonbonded work runs over neighbour rows, one wave per cluster of 8
// molecules or atoms: lane l takes every eighth entry of row l/8 and
// accumulates the gradient of that row's member only ("owner computes": each
// unordered pair is evaluated from both sides), so no per-pair atomics are
// needed.  The q-atoms are taken one after the other by waves of 64 waters or
// solute atoms.  Sums go to int64 fixed point, into buffers that a kernel
// owns or the shared gradient, and the integrator adds them.  Rows are built
// with the reference's FP64 group cut-off tests, so the set of interacting
// pairs equals the reference pair lists.  Pair arithmetic is FP32; energy
// terms on energy steps, LRF, bonded terms, restraints, leapfrog and SHAKE
// run in FP64.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "qmi_device.h"
#include "qmi_kernels.h"

namespace qmi {

// ------------------------------------------------------------ helpers --
// index of the calling wave in the grid (blocks are whole waves), read from
// the first lane so the compiler keeps it, and the list loads it indexes, in
// scalar registers
__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
}

__device__ __forceinline__ long long fix(double v, double scale) { return __double2ll_rn(v * scale); }

// 1/sqrt(a) for the FP64 energy terms: the FP32 hardware estimate (relative
// error below 2^-22) and one FP64 Newton step, which squares it to below
// 1e-12
__device__ __forceinline__ double rsqrt_e(double r2) {
  const double h = 0.5 * r2;
  const double y = (double)__builtin_amdgcn_rsqf((float)r2);
  return fma(y, fma(-(h * y), y, 0.5), y);
}
// FP32 1/sqrt of a squared interatomic distance: the hardware instruction
// alone.  rsqrtf wraps the same instruction in a rescaling for denormal
// arguments (a compare and two selects); the squared distance of a listed
// pair is never that small, and on normal arguments both return the same bits
__device__ __forceinline__ float rsq_r2(float r2) { return __builtin_amdgcn_rsqf(r2); }
// 1/a for the Q-atom energy terms, as rsqrt_e: the FP32 hardware estimate
// and one FP64 Newton step (relative error below 1e-12; a is a sum of
// powers of interatomic distances, well inside the FP32 range)
__device__ __forceinline__ double rcp_e(double a) {
  const double y = (double)__builtin_amdgcn_rcpf((float)a);
  return fma(y, fma(-a, y, 1.0), y);
}

__device__ __forceinline__ void add_grad(long long* f, int atom, double gx, double gy, double gz) {
  atomicAdd((unsigned long long*)&f[3 * atom + 0], (unsigned long long)fix(gx, kFScale));
  atomicAdd((unsigned long long*)&f[3 * atom + 1], (unsigned long long)fix(gy, kFScale));
  atomicAdd((unsigned long long*)&f[3 * atom + 2], (unsigned long long)fix(gz, kFScale));
}
// the gradient of one atom from a per-atom pass, summed in the lane's own
// fixed-point registers
__device__ __forceinline__ void atom_grad(long long acc[3], double gx, double gy, double gz) {
  acc[0] += fix(gx, kFScale);
  acc[1] += fix(gy, kFScale);
  acc[2] += fix(gz, kFScale);
}

__device__ __forceinline__ void add_energy(WinState* ws, int w, int slot, double e) {
  if (e != 0.0) atomicAdd((unsigned long long*)&ws[w].E[slot], (unsigned long long)fix(e, kEScale));
}

// ------------------------------------------------ cross-lane sums --
// Partner values without the LDS crossbar: DPP moves inside rows of 16
// lanes and the gfx950 permlane swaps between rows.  Every sum below is a
// butterfly whose step k adds the value of lane l ^ m_k; at each step the
// values are already uniform over the lane groups of the earlier steps, so
// a DPP pattern that lands in the right group reads the same value as the
// xor partner (row_ror:8 for m = 8, row_ror:4 for m = 4 once the values are
// symmetric under l ^ 8, row_half_mirror for m = 4 once they are uniform over
// quads).  The sums are therefore the same, bit for bit, as the butterflies
// over __shfl_xor.  All 64 lanes must be active.
constexpr int kDppXor1 = 0xB1;      // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;      // quad_perm [2,3,0,1]
constexpr int kDppRor4 = 0x124;     // row_ror:4
constexpr int kDppRor8 = 0x128;     // row_ror:8
constexpr int kDppHalfMirror = 0x141;
template <int CTRL>
__device__ __forceinline__ unsigned dpp_u(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
// the value of lane l ^ 16 (row swap) and of lane l ^ 32 (half swap)
__device__ __forceinline__ unsigned xor16_u(unsigned v) {
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return (threadIdx.x & 16) ? r[0] : r[1];
}
__device__ __forceinline__ unsigned xor32_u(unsigned v) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return (threadIdx.x & 32) ? r[0] : r[1];
}
// the same moves for 32- and 64-bit values: M is a DPP control, or 16 / 32
// for the row and half swaps
template <int M>
__device__ __forceinline__ unsigned mv_u(unsigned v) {
  if constexpr (M == 16) return xor16_u(v);
  else if constexpr (M == 32) return xor32_u(v);
  else return dpp_u<M>(v);
}
template <int M>
__device__ __forceinline__ float mv(float v) { return __builtin_bit_cast(float, mv_u<M>(__builtin_bit_cast(unsigned, v))); }
template <int M>
__device__ __forceinline__ int mv(int v) { return (int)mv_u<M>((unsigned)v); }
template <int M>
__device__ __forceinline__ unsigned long long mv(unsigned long long v) {
  return (unsigned long long)mv_u<M>((unsigned)v) | ((unsigned long long)mv_u<M>((unsigned)(v >> 32)) << 32);
}
template <int M>
__device__ __forceinline__ long long mv(long long v) { return (long long)mv<M>((unsigned long long)v); }
template <int M>
__device__ __forceinline__ double mv(double v) {
  return __builtin_bit_cast(double, mv<M>(__builtin_bit_cast(unsigned long long, v)));
}

// sum over the wave: partners l^32, l^16, l^8, l^4, l^2, l^1
template <class T>
__device__ __forceinline__ T wave_sum_t(T v) {
  v += mv<32>(v);
  v += mv<16>(v);
  v += mv<kDppRor8>(v);
  v += mv<kDppRor4>(v);
  v += mv<kDppXor2>(v);
  v += mv<kDppXor1>(v);
  return v;
}
__device__ __forceinline__ double wave_sum(double v) { return wave_sum_t(v); }
// integer forms: exact, so the order of the sums does not matter
__device__ __forceinline__ long long wave_sum_i(long long v) { return wave_sum_t(v); }
// sum over the 8 lanes that share lane>>3: partners l^1, l^2, l^4
template <class T>
__device__ __forceinline__ T row8_sum_t(T v) {
  v += mv<kDppXor1>(v);
  v += mv<kDppXor2>(v);
  v += mv<kDppHalfMirror>(v);
  return v;
}
// sum over the 8 lanes that share lane&7: partners l^8, l^16, l^32
template <class T>
__device__ __forceinline__ T col8_sum_t(T v) {
  v += mv<kDppRor8>(v);
  v += mv<16>(v);
  v += mv<32>(v);
  return v;
}
__device__ __forceinline__ void add_grad_fix(long long* f, int atom, long long gx, long long gy, long long gz) {
  atomicAdd((unsigned long long*)&f[3 * atom + 0], (unsigned long long)gx);
  atomicAdd((unsigned long long*)&f[3 * atom + 1], (unsigned long long)gy);
  atomicAdd((unsigned long long*)&f[3 * atom + 2], (unsigned long long)gz);
}
__device__ __forceinline__ void add_energy_fix(WinState* ws, int w, int slot, long long e) {
  if (e != 0) atomicAdd((unsigned long long*)&ws[w].E[slot], (unsigned long long)e);
}
// energy of a term into slot `slot` of window w: each lane's term goes to
// fixed point, then lanes of a wave that agree on (w, slot) are summed and
// added with one atomic.  The integer sums are exact, so the result does not
// depend on which terms share a wave (it is the same for a window alone or
// batched with others).
__device__ __forceinline__ void wave_energy(WinState* ws, int w, int slot, double e, bool valid) {
  const unsigned long long vm = __ballot(valid);
  if (vm == 0ull) return;
  const int first = __ffsll((long long)vm) - 1;
  const int key = valid ? w * E_NSLOT + slot : -1;
  const int key0 = __builtin_amdgcn_readlane(key, first);   // first is uniform over the wave
  const bool uniform = __ballot(valid && key != key0) == 0ull;
  const long long ef = valid ? fix(e, kEScale) : 0ll;
  if (uniform) {
    const long long sum = wave_sum_i(ef);
    if ((int)(threadIdx.x & 63) == first) add_energy_fix(ws, w, slot, sum);
  } else if (valid) {
    add_energy_fix(ws, w, slot, ef);
  }
}

__device__ __forceinline__ double row8_sum(double v) { return row8_sum_t(v); }

// ------------------------------------------------------ step control --
// The gradient array is zero between steps and evaluations: the kernel that
// completes a gradient (k_integrate, k_atom_terms<false>) takes it and clears
// it.
__device__ __forceinline__ bool window_runs(const WinState& s) {
  return s.istep < s.stop_at && !s.shake_fail && !s.list_overflow;
}
// flags and energy accumulators at the start of the MD step s.istep
__device__ __forceinline__ void begin_step(WinState& s, const WinDev& W) {
  s.active = window_runs(s) ? 1 : 0;
  s.wpol_acc = s.active;
  s.list_now = (s.istep % W.nbcycle) == 0;
  s.energy_now = (W.iene > 0 && s.istep % W.iene == 0 && s.istep > 0) || (W.iout > 0 && s.istep % W.iout == 0) ? 1 : 0;
  if (s.energy_now)
    for (int k = 0; k < E_NSLOT; ++k) s.E[k] = 0;
}

// start of a run's first step (eval 0; later steps are begun by k_temperature)
// or of an evaluation, one thread per window.  eval 1: energy evaluation; 2:
// forces only (timing runs); 3: the energy evaluation after
// the last step of a run (md.f90:4207-4208), which is a pot_energy call of
// the run for windows that completed; a window stopped by a failure is left
// as it is.
__global__ void k_begin(Dev d, int eval, int rebuild) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.nwin) return;
  WinState& s = d.ws[i];
  const WinDev& W = d.win[i];
  if (!eval) {
    begin_step(s, W);
    return;
  }
  s.active = eval != 3 || !(s.shake_fail || s.list_overflow);
  s.list_now = rebuild;
  s.energy_now = eval != 2 ? 1 : 0;
  s.wpol_acc = eval == 3 && s.istep >= W.nsteps ? 1 : 0;
  if (s.energy_now)
    for (int k = 0; k < E_NSLOT; ++k) s.E[k] = 0;
}

// dynamic Q-atom lists (nbqplist / nbqwlist, md.f90:7875-7964, 8066-8118): at
// a list update, an atom is in the lists while the switching atom of its
// group (the oxygen of its water) lies within the q_atom cut-off of the Q
// centre; the static lists cover every candidate, and the q kernels test
// this flag
__global__ void k_qin(Dev d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.ntot || d.qref[i] < 0) return;
  const WinState& s = d.ws[d.wid[i]];
  if (!s.active || !s.list_now) return;
  const WinDev& W = d.win[d.wid[i]];
  const int r = d.qref[i];
  const double dx = __dsub_rn(d.x[3 * r], W.xpcent[0]), dy = __dsub_rn(d.x[3 * r + 1], W.xpcent[1]),
               dz = __dsub_rn(d.x[3 * r + 2], W.xpcent[2]);
  d.qin[i] = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz)) <= W.rcq2 ? 1 : 0;
}

// EVB off-diagonal elements at the step's starting coordinates (offdiag,
// md.f90:12911-12937), into the step's ring slot; the ring is read for steps
// the window ran, so a stopped window's slot goes unread
__global__ void k_offdiag(Dev d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.noffd_all) return;
  const WinState& s = d.ws[d.offd_win[i]];
  const int2 kl = d.offd_kl[i];
  const double dx = d.x[3 * kl.y] - d.x[3 * kl.x], dy = d.x[3 * kl.y + 1] - d.x[3 * kl.x + 1],
               dz = d.x[3 * kl.y + 2] - d.x[3 * kl.x + 2];
  const double r = sqrt(dx * dx + dy * dy + dz * dz);
  const double2 p = d.offd_par[i];
  double* o = &d.o_ring[((size_t)((s.istep - s.ring_base) % d.ring_n) * d.noffd_all + i) * 2];
  o[0] = p.x * exp(-p.y * r);
  o[1] = r;
}

// charge-group centres (cgp_centers, md.f90:1000-1019) and cluster bounding
// spheres, at list-update steps
__global__ void k_centres(Dev d, int ngrp_total) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ngrp_total) return;
  int w = d.g_win[g];
  if (!d.ws[w].active || !d.ws[w].list_now) return;
  double c[3] = {0, 0, 0};
  int n = d.g_n[g], f0 = d.g_first[g];
  for (int k = 0; k < n; ++k) {
    int a = d.g_atoms[f0 + k];
    c[0] += d.x[3 * a]; c[1] += d.x[3 * a + 1]; c[2] += d.x[3 * a + 2];
  }
  for (int k = 0; k < 3; ++k) d.g_cent[3 * g + k] = c[k] / (double)(float)n;
  for (int k = 0; k < 20; ++k) d.g_lrf[20 * g + k] = 0.0;
}

__global__ void k_bounds(Dev d, int nwc_total, int nsc_total) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nwc_total + nsc_total) return;
  bool water = c < nwc_total;
  int cl = water ? c : c - nwc_total;
  int w = water ? d.wc_win[cl] : d.sc_win[cl];
  if (!d.ws[w].active || !d.ws[w].list_now) return;
  // member records (switching-atom position and flag), then the sphere
  double4* cm = (water ? d.wc_cm : d.sc_cm) + (size_t)cl * kCl;
  double cx = 0, cy = 0, cz = 0;
  int n = 0;
  for (int k = 0; k < kCl; ++k) {
    int a = water ? d.wc_o[cl * kCl + k] : d.sc_a[cl * kCl + k];
    if (a < 0) { cm[k] = make_double4(0, 0, 0, -1.0); continue; }
    int sw = water ? a : d.g_sw[d.grp[a]];
    const double px = d.x[3 * sw], py = d.x[3 * sw + 1], pz = d.x[3 * sw + 2];
    cm[k] = make_double4(px, py, pz, (d.aflag[sw] & 1) ? 1.0 : 0.0);
    cx += px; cy += py; cz += pz;
    ++n;
  }
  if (n > 0) { cx /= n; cy /= n; cz /= n; }
  double r = 0;
  for (int k = 0; k < kCl; ++k) {
    const double4 m = cm[k];
    if (m.w < 0.0) continue;
    double dx = m.x - cx, dy = m.y - cy, dz = m.z - cz;
    r = fmax(r, sqrt(dx * dx + dy * dy + dz * dz));
  }
  double* bs = water ? &d.wc_bs[4 * cl] : &d.sc_bs[4 * cl];
  bs[0] = cx; bs[1] = cy; bs[2] = cz; bs[3] = n > 0 ? r : -1.0;
}

// ------------------------------------------------- neighbour rows --
__device__ __forceinline__ int special_type(const Dev& d, int i, int j) {
  // 1 = excluded pair, 2 = 1-4 pair, 0 = normal (listex/list14 and the long
  // lists of topo.f90, as nbpplist checks them, md.f90:5256-5294)
  const int2 r = d.sp_rng[i];
  if (j < r.x || j > r.y) return 0;   // outside the partners' index range
  int s0 = d.sp_start[i], s1 = d.sp_start[i + 1];
  for (int k = s0; k < s1; ++k)
    if (d.sp_j[k] == j) return d.sp_t[k];
  return 0;
}

// Pair-list build (nbwwlist/nbpwlist/nbpplist without LRF bookkeeping,
// md.f90:8370-8556, 6864-7068, 5448-5700): one wave per i-cluster.  Candidate
// j-clusters come from the bounding spheres of the switching atoms; for each
// candidate, lane (a, b) applies the reference's exact FP64 group test to
// member a of the i-cluster and member b of the j-cluster, and the passing
// members are appended, in j order, to row a.
template <int TT>
__device__ __forceinline__ void build_row(const Dev& d, int wave) {
  const int lane = threadIdx.x & 63;
  const RowList L = d.rl[TT];
  if (wave >= L.nicl) return;
  const int ic = wave;
  constexpr bool iw = (TT == T_WW || TT == T_WP);
  constexpr bool jw = (TT == T_WW || TT == T_PW);
  const int w = iw ? d.wc_win[ic] : d.sc_win[ic];
  const WinState& st = d.ws[w];
  if (!st.active || !st.list_now) return;
  const WinDev& W = d.win[w];
  const int j0 = jw ? W.wc_off : W.sc_off;
  const int nj = jw ? W.nwc : W.nsc;
  const double rc2 = (TT == T_WW) ? W.rcww2 : (TT == T_PP) ? W.rcpp2 : W.rcpw2;
  const double rc = sqrt(rc2);
  const double* bi = iw ? &d.wc_bs[4 * ic] : &d.sc_bs[4 * ic];
  const int a = lane >> 3, b = lane & 7;
  const int row = ic * kCl + a;
  const int ea = iw ? d.wc_o[ic * kCl + a] : d.sc_a[ic * kCl + a];
  const double4 mi = (iw ? d.wc_cm : d.sc_cm)[ic * kCl + a];
  const bool a_ok = mi.w == 0.0;
  const double4* cmj = jw ? d.wc_cm : d.sc_cm;
  const int* memj = jw ? d.wc_o : d.sc_a;
  int cnt = 0;  // entries of row a (the same in the 8 lanes of the row)
  for (int base = 0; base < nj && bi[3] >= 0.0; base += 64) {
    bool cand = false;
    if (base + lane < nj) {
      const double* bj = jw ? &d.wc_bs[4 * (j0 + base + lane)] : &d.sc_bs[4 * (j0 + base + lane)];
      const double dx = bi[0] - bj[0], dy = bi[1] - bj[1], dz = bi[2] - bj[2];
      const double dc = sqrt(dx * dx + dy * dy + dz * dz);
      cand = bj[3] >= 0.0 && dc - bi[3] - bj[3] <= rc + 1e-3;
    }
    unsigned long long cb = __ballot(cand);
    // candidates in j order; the next one's member record is loaded while
    // the current one is tested
    int k = cb ? __ffsll((long long)cb) - 1 : 0;
    double4 mb = make_double4(0, 0, 0, -1.0);
    int eb = -1;
    if (cb) { mb = cmj[(size_t)(j0 + base + k) * kCl + b]; eb = memj[(j0 + base + k) * kCl + b]; }
    while (cb) {
      cb &= cb - 1ull;
      const int kn = cb ? __ffsll((long long)cb) - 1 : k;
      const double4 mn = cmj[(size_t)(j0 + base + kn) * kCl + b];
      const int en = memj[(j0 + base + kn) * kCl + b];
      bool keep = false;
      int sp = 0;
      if (a_ok && mb.w == 0.0 && !(TT == T_WW && ea == eb) && !(TT == T_PP && ea == eb)) {
        if (TT == T_PP) sp = special_type(d, ea, eb);
        if (sp != 1) {
#pragma clang fp contract(off)
          const double dx = __dsub_rn(mi.x, mb.x), dy = __dsub_rn(mi.y, mb.y), dz = __dsub_rn(mi.z, mb.z);
          keep = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz)) <= rc2;
        }
      }
      const unsigned long long kb = __ballot(keep);
      const unsigned rowbits = (unsigned)((kb >> (8 * a)) & 0xffull);
      if (keep) {
        const int idx = cnt + __popc(rowbits & ((1u << b) - 1u));
        // entries name the member's place in the slot coordinates
        const int jc = j0 + base + k;
        const int ev = jw ? xw_at(jc, b, 0) : (jc * kCl + b) | (TT == T_PP && sp == 2 ? kRow14 : 0);
        if (idx < L.cap) L.ent[(size_t)row * L.cap + idx] = ev;
      }
      cnt += __popc(rowbits);
      k = kn;
      mb = mn;
      eb = en;
    }
  }
  if (b == 0) {
    L.cnt[row] = cnt < L.cap ? cnt : L.cap;
    if (cnt > L.cap) d.ws[w].list_overflow = 1;
  }
}

// all four kinds of rows in one launch, the longest-running first
__global__ void __launch_bounds__(256) k_build_rows(Dev d) {
  int wave = wave_id();
  const int np = (d.rl[T_PP].nicl + 3) & ~3, nw = (d.rl[T_WW].nicl + 3) & ~3;   // whole blocks of each kind
  if (wave < np) return build_row<T_PP>(d, wave);
  wave -= np;
  if (wave < nw) return build_row<T_WW>(d, wave);
  wave -= nw;
  if (wave < nw) return build_row<T_WP>(d, wave);
  wave -= nw;
  if (wave < np) return build_row<T_PW>(d, wave);
}

constexpr int kUnroll = 4;   // row entries per pass of the pair kernels
// the number of chunks of 8 entries the wave must walk: the longest row
__device__ __forceinline__ int row_chunks(int n) {
  int m = n;
  m = max(m, mv<kDppRor8>(m));
  m = max(m, mv<16>(m));
  m = max(m, mv<32>(m));
  return (m + kCl - 1) / kCl;
}

// FP32 pair expressions with their rounding spelled out: which products of a
// sum the compiler fuses differs from kernel to kernel and with what stands
// beside them, and the gradient's last bits, and with them a trajectory,
// should not change when a kernel is reorganised.
// squared distance
__device__ __forceinline__ float r2_f(float dx, float dy, float dz) {
#pragma clang fp contract(off)
  return __builtin_fmaf(dz, dz, __builtin_fmaf(dx, dx, dy * dy));
}
// dv = r2inv (-qq rinv - 12 va + 6 vb), the product with va or, CHARGE, with
// the charges fused
template <bool CHARGE>
__device__ __forceinline__ float pair_dv(float r2inv, float rinv, float qq, float va, float vb) {
#pragma clang fp contract(off)
  const float t = CHARGE ? __builtin_fmaf(qq, -rinv, -(12.f * va)) : __builtin_fmaf(va, -12.f, -(qq * rinv));
  return r2inv * __builtin_fmaf(6.f, vb, t);
}

// the gradient of a row's member: the sums over the row's 8 lanes, lane b
// holding component b in fixed point (lo) and every lane component 8 (hi)
struct RowGrad {
  long long lo = 0, hi = 0;
  template <int N>
  __device__ __forceinline__ void add(const float* g, int b) {
    if constexpr (N == 3) {
      const double x = row8_sum((double)g[0]), y = row8_sum((double)g[1]), z = row8_sum((double)g[2]);
      lo += fix(b == 0 ? x : b == 1 ? y : z, kFScale);
    } else {
      // each step halves the components a lane sums: after the step with
      // lane l ^ m a lane holds those whose index agrees with its own in the
      // bit m (the step of 4 by the mirrored lane, which differs in that bit)
      const bool b4 = b & 4, b1 = b & 1, b2 = b & 2;
      double s4[4], s2[2];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        s4[k] = (double)(b4 ? g[k + 4] : g[k]) + (double)mv<kDppHalfMirror>(b4 ? g[k] : g[k + 4]);
#pragma unroll
      for (int k = 0; k < 2; ++k)
        s2[k] = (b1 ? s4[2 * k + 1] : s4[2 * k]) + mv<kDppXor1>(b1 ? s4[2 * k] : s4[2 * k + 1]);
      lo += fix((b2 ? s2[1] : s2[0]) + mv<kDppXor2>(b2 ? s2[0] : s2[1]), kFScale);
      hi += fix(row8_sum((double)g[8]), kFScale);
    }
  }
};

// --------------------------------------------------- nonbonded rows --
// Lane (a, b) of the wave for i-cluster ic evaluates entries b, b+8, ... of
// row a and accumulates the gradient of its i-member only (each pair is
// evaluated from both sides); the 8 lanes of a row are then reduced and
// added once.
// water-water: 9 interactions per molecule pair (nonbond_ww_spc, md.f90:11823-12047;
// W3, a 3-atom solvent: LJ on all nine, nonbond_3atomsolvent, 12317-12591).
// The energy sums run only on energy steps: EN selects the form of the
// loop for the wave's window (uniform over the wave).
template <bool EN, bool W3>
__device__ __forceinline__ void ww_impl(const Dev& d, int wave, RowGrad& rg) {
  const int lane = threadIdx.x & 63;
  const RowList L = d.rl[T_WW];
  if (wave >= L.nicl) return;
  const int ic = wave;
  const int w = d.wc_win[ic];
  const WinState& st = d.ws[w];
  if (!st.active) return;
  const WinDev& W = d.win[w];
  const int a = lane >> 3, b = lane & 7;
  const int row = ic * kCl + a;
  const int n = L.cnt[row];   // none for an empty member
  const int nch = row_chunks(n);
  const int xa = xw_at(ic, a, 0);
  float3 pi[3];
  for (int k = 0; k < 3; ++k) {
    const float4 q = d.xw[xa + kCl * k];
    pi[k] = make_float3(q.x, q.y, q.z);
  }
  const float q0 = W.crg_w[0], q1 = W.crg_w[1], q2 = W.crg_w[2];
  const float qq[3][3] = {{q0 * q0, q0 * q1, q0 * q2}, {q1 * q0, q1 * q1, q1 * q2}, {q2 * q0, q2 * q1, q2 * q2}};
  const float A = W.ww_a, B = W.ww_b;
  constexpr bool en = EN;
  float g[9];
  for (int k = 0; k < 9; ++k) g[k] = 0.f;
  double eel = 0.0, evdw = 0.0;
  // energy steps: the energy terms in FP64 from the FP64 coordinates, as
  // nonbond_ww_spc / nonbond_3atomsolvent evaluate them
  double xi[9];
  if (en)
    for (int k = 0; k < 3; ++k) {
      const double4 q = d.xwd[xa + kCl * k];
      xi[3 * k] = q.x; xi[3 * k + 1] = q.y; xi[3 * k + 2] = q.z;
    }
  const int* ent = L.ent + (size_t)row * L.cap + b;
  // one site of a neighbouring cluster's members is one line of xw, so the 8
  // lanes of a row mostly read one line a load.  The next entry and its
  // coordinates are loaded while the current one is evaluated (entries past
  // the row end read place 0 and are skipped; the table has kCl entries
  // beyond its last row)
  const int e0 = ent[0];
  unsigned ob_next = b < n ? e0 : 0;
  float4 nx[3];
  for (int s = 0; s < 3; ++s) nx[s] = (d.xw + ob_next)[kCl * s];
  for (int t = 0; t < nch; ++t) {
    const int k = t * kCl + b;
    const unsigned ob = ob_next;
    float3 pj[3];
    for (int s = 0; s < 3; ++s) pj[s] = make_float3(nx[s].x, nx[s].y, nx[s].z);
    {
      const int e = ent[(t + 1) * kCl];
      ob_next = k + kCl < n ? e : 0;
      for (int s = 0; s < 3; ++s) nx[s] = (d.xw + ob_next)[kCl * s];
    }
    if (k >= n) continue;
    // each unordered pair counted once, from the row with the lower slot: a
    // row's entries ascend in slot order, so the counted ones are a suffix
    // of the row and the 8 rows of the wave (consecutive slots) switch at
    // nearly the same place, which keeps the FP64 block from diverging
    const bool cnt = en && xa < (int)ob;
    if (cnt) {
      double xj[9];
      for (int m = 0; m < 3; ++m) {
        const double4 q = (d.xwd + ob)[kCl * m];
        xj[3 * m] = q.x; xj[3 * m + 1] = q.y; xj[3 * m + 2] = q.z;
      }
      for (int p = 0; p < 3; ++p)
        for (int q = 0; q < 3; ++q) {
          const double dx = xj[3 * q] - xi[3 * p], dy = xj[3 * q + 1] - xi[3 * p + 1],
                       dz = xj[3 * q + 2] - xi[3 * p + 2];
          const double rinv = rsqrt_e(dx * dx + dy * dy + dz * dz);
          eel += (double)qq[p][q] * rinv;
          if (W3 || (p == 0 && q == 0)) {
            const double r2i = rinv * rinv, r6 = r2i * r2i * r2i;
            const double a_ = W3 ? W.ww3_ad[3 * p + q] : W.ww_ad, b_ = W3 ? W.ww3_bd[3 * p + q] : W.ww_bd;
            evdw += a_ * r6 * r6 - b_ * r6;
          }
        }
    }
    for (int p = 0; p < 3; ++p) {
      for (int q = 0; q < 3; ++q) {
        float dx = pj[q].x - pi[p].x, dy = pj[q].y - pi[p].y, dz = pj[q].z - pi[p].z;
        // (the force-only loop sums the squares of an oxygen's distances from x)
        const float r2 = !EN && q == 0 ? r2_f(dy, dx, dz) : r2_f(dx, dy, dz);
        float rinv = rsq_r2(r2);
        float r2inv = rinv * rinv;
        float dv;
        if (W3 || (p == 0 && q == 0)) {
          float r6 = r2inv * r2inv * r2inv;
          const float a_ = W3 ? W.ww3_a[3 * p + q] : A, b_ = W3 ? W.ww3_b[3 * p + q] : B;
          dv = pair_dv<W3>(r2inv, rinv, qq[p][q], a_ * r6 * r6, b_ * r6);
        } else {
          dv = r2inv * (-(qq[p][q] * rinv));
        }
        g[3 * p + 0] = __builtin_fmaf(-dx, dv, g[3 * p + 0]);
        g[3 * p + 1] = __builtin_fmaf(-dy, dv, g[3 * p + 1]);
        g[3 * p + 2] = __builtin_fmaf(-dz, dv, g[3 * p + 2]);
      }
    }
  }
  rg.add<9>(g, b);
  if (en) {
    eel = wave_sum(eel);
    evdw = wave_sum(evdw);
    if (lane == 0) { add_energy(d.ws, w, E_WW_EL, eel); add_energy(d.ws, w, E_WW_VDW, evdw); }
  }
}

// solute atom - water: LJ on O (on all three sites for a 3-atom solvent),
// Coulomb on all three sites (nonbond_pw, md.f90:10631-10682).  WATER_SIDE: rows are waters and entries solute atoms
// (W<-P); otherwise rows are solute atoms and entries water slots (P<-W),
// which also counts the energies.
template <bool WATER_SIDE, bool EN, bool W3>
__device__ __forceinline__ void pw_impl(const Dev& d, int wave, RowGrad& rg) {
  const int lane = threadIdx.x & 63;
  const RowList L = d.rl[WATER_SIDE ? T_WP : T_PW];
  if (wave >= L.nicl) return;
  const int ic = wave;
  const int w = WATER_SIDE ? d.wc_win[ic] : d.sc_win[ic];
  const WinState& st = d.ws[w];
  if (!st.active) return;
  const WinDev& W = d.win[w];
  const int a = lane >> 3, b = lane & 7;
  const int row = ic * kCl + a;
  const int n = L.cnt[row];   // none for an empty member
  const int nch = row_chunks(n);
  const float4* xs = d.xw + 3 * (size_t)d.nwslot;   // the solute slots
  float4 pi[3];
  float2 ljs = make_float2(0, 0);
  if (WATER_SIDE) {
    for (int k = 0; k < 3; ++k) pi[k] = d.xw[xw_at(ic, a, k)];
  } else {
    pi[0] = xs[row];
    ljs = *(const float2*)&d.sljp[row];
  }
  constexpr bool en = EN && !WATER_SIDE;
  constexpr bool wat3 = W3;
  float g[9];
  for (int k = 0; k < 9; ++k) g[k] = 0.f;
  double eel = 0.0, evdw = 0.0;
  // energy steps: the energy terms in FP64 from the FP64 coordinates and
  // LJ columns, as nonbond_pw / nonbond_3atomsolvent evaluate them
  double4 xd = make_double4(0, 0, 0, 0);
  double Ad[3] = {0, 0, 0}, Bd[3] = {0, 0, 0};
  if (en) {
    xd = d.xwd[3 * (size_t)d.nwslot + row];
    const double4 tl = d.sljd[row];
    for (int k = 0; k < (wat3 ? 3 : 1); ++k)
      lj_ab(tl.x, tl.y, k == 0 ? W.aO1d : W.awd[k], k == 0 ? W.bO1d : W.bwd[k], W.arith, &Ad[k], &Bd[k]);
  }
  const int* ent = L.ent + (size_t)row * L.cap + b;
  // kUnroll entries per pass, loads first (as in pp_impl)
  auto rows = [&](auto AR) {
    constexpr bool arith = AR;
    for (int t0 = 0; t0 < nch; t0 += kUnroll) {
      unsigned e[kUnroll];
      bool v[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        v[u] = (t0 + u) * kCl + b < n;
        const int le = ent[(t0 + u) * kCl];
        e[u] = v[u] ? le : 0;
      }
      float4 ld[kUnroll][3];
      float2 lt[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        if (WATER_SIDE) {
          ld[u][0] = xs[e[u]];
          lt[u] = *(const float2*)&d.sljp[e[u]];
        } else {
          const float4* xe = d.xw + e[u];
          ld[u][0] = xe[0]; ld[u][1] = xe[kCl]; ld[u][2] = xe[2 * kCl];
        }
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const float4 ps = WATER_SIDE ? ld[u][0] : pi[0];
        const float2 lj = WATER_SIDE ? lt[u] : ljs;
        if (!v[u]) continue;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const float4 pw = WATER_SIDE ? pi[k] : ld[u][k];
          // dx = x(water atom) - x(solute atom), as nonbond_pw with i solute, j water
          const float dx = pw.x - ps.x, dy = pw.y - ps.y, dz = pw.z - ps.z;
          const float rinv = rsq_r2(r2_f(dx, dy, dz)), r2inv = rinv * rinv;
          const float qq = ps.w * pw.w;
          float dv;
          if (k == 0 || wat3) {
            const float r6 = r2inv * r2inv * r2inv;
            float A, B;
            lj_ab(lj.x, lj.y, k == 0 ? W.aO1 : W.aw[k], k == 0 ? W.bO1 : W.bw[k], arith, &A, &B);
            dv = pair_dv<!W3 && !en>(r2inv, rinv, qq, A * r6 * r6, B * r6);
          } else {
            dv = r2inv * (-(qq * rinv));
          }
          if (en) {
            const double4 xa = (d.xwd + e[u])[kCl * k];   // the water atom, FP64
            const double ddx = xa.x - xd.x, ddy = xa.y - xd.y, ddz = xa.z - xd.z;
            const double rinv_d = rsqrt_e(ddx * ddx + ddy * ddy + ddz * ddz);
            eel += (double)qq * rinv_d;
            if (k == 0 || wat3) {
              const double r2i = rinv_d * rinv_d, r6d = r2i * r2i * r2i;
              evdw += Ad[k] * r6d * r6d - Bd[k] * r6d;
            }
          }
          const float sd = WATER_SIDE ? dv : -dv;
          const int o = WATER_SIDE ? 3 * k : 0;
          g[o] = __builtin_fmaf(sd, dx, g[o]);
          g[o + 1] = __builtin_fmaf(sd, dy, g[o + 1]);
          g[o + 2] = __builtin_fmaf(sd, dz, g[o + 2]);
        }
      }
    }
  };
  if (W.arith) rows(std::true_type{});
  else rows(std::false_type{});
  rg.add<WATER_SIDE ? 9 : 3>(g, b);
  if (en) {
    eel = wave_sum(eel);
    evdw = wave_sum(evdw);
    if (lane == 0) { add_energy(d.ws, w, E_PW_EL, eel); add_energy(d.ws, w, E_PW_VDW, evdw); }
  }
}

// solute-solute (nonbond_pp, md.f90:10387-10491): 1-4 pairs use the third
// LJ column and the el14 scale
template <bool EN>
__device__ __forceinline__ void pp_impl(const Dev& d, int wave, RowGrad& rg) {
  const int lane = threadIdx.x & 63;
  const RowList L = d.rl[T_PP];
  if (wave >= L.nicl) return;
  const int ic = wave;
  const int w = d.sc_win[ic];
  const WinState& st = d.ws[w];
  if (!st.active) return;
  const WinDev& W = d.win[w];
  const int a = lane >> 3, b = lane & 7;
  const int row = ic * kCl + a;
  const int n = L.cnt[row];   // none for an empty member
  const int nch = row_chunks(n);
  const float4* xs = d.xw + 3 * (size_t)d.nwslot;      // the solute slots
  const double4* xsd = d.xwd + 3 * (size_t)d.nwslot;
  const float4 pi = xs[row], li = d.sljp[row];
  constexpr bool en = EN;
  float g0 = 0.f, g1 = 0.f, g2 = 0.f;
  double eel = 0.0, evdw = 0.0;
  // energy steps: the energy terms in FP64 from the FP64 coordinates and LJ
  // columns, as nonbond_pp evaluates them
  double4 xd = make_double4(0, 0, 0, 0), tli = make_double4(0, 0, 0, 0);
  if (en) {
    xd = xsd[row];
    tli = d.sljd[row];
  }
  const int* ent = L.ent + (size_t)row * L.cap + b;
  // kUnroll entries per pass: all their loads are issued before the
  // arithmetic (a row's capacity is a multiple of the entries of a pass, so
  // they need no branch); entries past the row end read atom 0 and are
  // masked, and the sums run in entry order as in a plain loop.  The LJ
  // columns of a 1-4 pair are the second half of the atom's record.
  auto rows = [&](auto AR) {
    constexpr bool arith = AR;
    const float lx = li.x, ly = li.y, l14x = li.z, l14y = li.w;
    for (int t = 0; t < nch; t += kUnroll) {
      unsigned e[kUnroll];
      bool v[kUnroll], is14[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        v[u] = (t + u) * kCl + b < n;
        const int ld = ent[(t + u) * kCl];
        const int eu = v[u] ? ld : 0;
        is14[u] = (eu & kRow14) != 0;
        e[u] = eu & ~kRow14;
      }
      float4 pj[kUnroll];
      float2 lj[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        pj[u] = xs[e[u]];
        lj[u] = ((const float2*)d.sljp)[2ull * e[u] + is14[u]];
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const float dx = pj[u].x - pi.x, dy = pj[u].y - pi.y, dz = pj[u].z - pi.z;
        const float rinv = rsq_r2(r2_f(dx, dy, dz)), r2inv = rinv * rinv;
        const float r6 = r2inv * r2inv * r2inv;
        const float vel = (pi.w * pj[u].w) * rinv * (is14[u] ? W.el14 : 1.f);
        float aa, bb;
        lj_ab(is14[u] ? l14x : lx, is14[u] ? l14y : ly, lj[u].x, lj[u].y, arith, &aa, &bb);
        const float va = r6 * r6 * aa, vb = r6 * bb;
        const float dv = r2inv * __builtin_fmaf(6.f, vb, __builtin_fmaf(va, -12.f, -vel));
        if (!v[u]) continue;
        g0 = __builtin_fmaf(-dx, dv, g0); g1 = __builtin_fmaf(-dy, dv, g1); g2 = __builtin_fmaf(-dz, dv, g2);
        // each pair counted once, from the row with the lower slot (a suffix
        // of the row, as for the waters)
        if (en && row < (int)e[u]) {
          const double4 xj = xsd[e[u]], tlj = d.sljd[e[u]];
          const double ddx = xj.x - xd.x, ddy = xj.y - xd.y, ddz = xj.z - xd.z;
          const double rinv_d = rsqrt_e(ddx * ddx + ddy * ddy + ddz * ddz);
          const double r2i = rinv_d * rinv_d, r6d = r2i * r2i * r2i;
          double ad, bd;
          double vd = (double)(pi.w * pj[u].w) * rinv_d;
          if (is14[u]) {
            vd *= W.el14d;
            lj_ab(tli.z, tli.w, tlj.z, tlj.w, arith, &ad, &bd);
          } else {
            lj_ab(tli.x, tli.y, tlj.x, tlj.y, arith, &ad, &bd);
          }
          eel += vd;
          evdw += ad * r6d * r6d - bd * r6d;
        }
      }
    }
  };
  if (W.arith) rows(std::true_type{});
  else rows(std::false_type{});
  const float g[3] = {g0, g1, g2};
  rg.add<3>(g, b);
  if (en) {
    eel = wave_sum(eel);
    evdw = wave_sum(evdw);
    if (lane == 0) { add_energy(d.ws, w, E_PP_EL, eel); add_energy(d.ws, w, E_PP_VDW, evdw); }
  }
}

// The rows of one i-cluster, a wave each: k_wrow the water-water and
// water<-solute rows of a water cluster, k_srow the solute<-water and
// solute<-solute rows of a solute cluster.  The gradient of the cluster's
// members is stored in the row buffer (Dev::grow), which the integrator adds:
// atomics on the shared gradient array go past the XCDs' L2s to memory, at
// about 22 per ns for the whole GPU, and were most of what these kernels
// spent.  64-window ladder, force-only, alone: water rows 58 + 67 us as two
// kernels with atomics, 89 as one with stores, 85 with 82 -> 57 instructions a
// water<-solute entry; solute rows 34 + 55, 74, then 70 with 70 -> 41 a solute
// pair.  They are bound by VALU issue (about 75 %) and the gathers' return path
// (76 %): with four floats loaded a water atom where three are used, the water
// rows take 10 us more.
// W3: the instance for windows with a 3-atom solvent (launched only when
// there are any); each instance skips the other windows' rows.
// EK: the instance launched on steps where some window computes energies
// (it also serves that step's other windows); the instance without energy
// terms keeps the smaller register footprint of the force-only loop.
// PART (k_wrow): 1 water-water rows alone, 2 water<-solute rows alone, added
// to what part 1 stored (for timing them), 3 both.
template <bool W3, bool EK, int PART>
__device__ __forceinline__ void wrow_wave(const Dev& d, int wave) {
  if (wave >= d.rl[T_WW].nicl) return;
  const int w = d.wc_win[wave];
  if ((d.win[w].wat3 != 0) != W3 || !d.ws[w].active) return;
  RowGrad rg;
  if (PART & 1) {
    if (EK && d.ws[w].energy_now) ww_impl<EK, W3>(d, wave, rg);
    else ww_impl<false, W3>(d, wave, rg);
  }
  if (PART & 2) pw_impl<true, false, W3>(d, wave, rg);
  const int lane = threadIdx.x & 63, b = lane & 7, row = wave * kCl + (lane >> 3);
  long long* o = d.grow + 9 * (size_t)row;
  if (PART == 2) rg.lo += o[b];
  o[b] = rg.lo;
  if (b == 0) o[8] = PART == 2 ? o[8] + rg.hi : rg.hi;
}
template <bool W3, bool EK, int PART>
__global__ void __launch_bounds__(256) k_wrow(Dev d) {
  wrow_wave<W3, EK, PART>(d, wave_id());
}

template <bool W3, bool EK>
__device__ __forceinline__ void srow_wave(const Dev& d, int wave) {
  if (wave >= d.rl[T_PP].nicl) return;
  const int w = d.sc_win[wave];
  if ((d.win[w].wat3 != 0) != W3 || !d.ws[w].active) return;
  RowGrad rg;
  if (EK && d.ws[w].energy_now) {
    pw_impl<false, EK, W3>(d, wave, rg);
    pp_impl<EK>(d, wave, rg);
  } else {
    pw_impl<false, false, W3>(d, wave, rg);
    pp_impl<false>(d, wave, rg);
  }
  const int lane = threadIdx.x & 63, b = lane & 7, row = wave * kCl + (lane >> 3);
  if (b < 3) d.grow[9 * (size_t)d.nwslot + 3 * row + b] = rg.lo;
}
template <bool W3, bool EK>
__global__ void __launch_bounds__(256) k_srow(Dev d) {
  srow_wave<W3, EK>(d, wave_id());
}

// ---- q-atoms against water (nonbond_qw_spc, md.f90:11302-11411; 3-atom
// solvent nonbond_qw_3atom, 11545-11670) and against solute atoms
// (nonbond_qp_qvdw / nonbond_qp, 11138-11204, 10980-11045), all states;
// gradients are lambda-weighted over states.
//
// One block per 64 consecutive cluster slots (one water or solute atom per
// lane): its waves take the window's q-atoms in chunks of up to 16, whose
// coordinates and parameters are the same for every lane and come through
// scalar loads.  The q-atoms of a chunk are members 4h .. 4h+3 (h its half) of
// four consecutive q-clusters, taken member by member: FP32 sums run over the
// four clusters and go to fixed point, as do the reactions on a q-atom, summed
// in FP32 over a cluster's 8 lanes; what is added up beyond that are integers,
// so the gradient depends on neither the batch nor the split into chunks.  The
// waves' sums are added in LDS and stored in the q row buffer (Dev::gq), which
// the integrator adds; the reactions take one atomic per chunk.  On energy steps
// the same pass adds the per-state energies in FP64.
//
// Bound by VALU issue (about 150 instructions per 64 pairs with water and
// two states).  As 8 x 8 tiles with both sides gathered per lane, the q-atom
// records cost a texture-address gather each (58 cycles a wave-load), the
// reactions went through memory to a gather kernel, and the energies were two
// more kernels.  Chunks of 16: four waves hold the 50 q-atoms of a ligand.
// (With a wave per chunk and an atomic per component the kernel took 157 us
// for the 64-window ladder, all of it atomics.)  64-window ladder, force-only:
// water 86 + solute 39 + gather 9 us as tiles, now 35 + 40 (31 + 39 when sums
// beyond the four clusters are FP64, but then their last bits depend on the split).
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
// (12 va - 6 vb) ratio
__device__ __forceinline__ float lj_f(float va, float vb, float ratio) {
#pragma clang fp contract(off)
  return __builtin_fmaf(12.f, va, -(6.f * vb)) * ratio;
}
// dv + r2inv (-q r - t) lam
__device__ __forceinline__ float dv_f(float dv, float r2inv, float q, float r, float t, float lam) {
#pragma clang fp contract(off)
  return __builtin_fmaf(r2inv * __builtin_fmaf(-q, r, -t), lam, dv);
}
typedef const float __attribute__((address_space(4))) * ConstF;    // read with scalar loads
typedef const double __attribute__((address_space(4))) * ConstD;
typedef const int __attribute__((address_space(4))) * ConstI;

constexpr int kQWaves = 4;
// the block's work item: window, first slot, slots (at most 64)
__device__ __forceinline__ int4 q_item(const int4* work, int block) {
  const ConstI k = (ConstI)(const int*)work + 4 * (size_t)block;
  return make_int4(k[0], k[1], k[2], k[3]);
}
// the sums of an item's waves of the N components of its slots into out[N *
// slot + k]; s: LDS of N * 64 * kQWaves integers for the group of kQWaves waves.
// Every thread of the block calls it; a group without an item has 0 slots.
template <int N>
__device__ __forceinline__ void q_store(const long long* acc, int slots, long long* out, long long* s) {
  constexpr int kStride = N * 64;
  const int lane = threadIdx.x & 63, wv = (threadIdx.x >> 6) % kQWaves, t = threadIdx.x % (64 * kQWaves);
#pragma unroll
  for (int k = 0; k < N; ++k) s[wv * kStride + k * 64 + lane] = acc[k];
  __syncthreads();
  for (int i = t; i < N * slots; i += 64 * kQWaves) {
    const long long* p = s + (i % N) * 64 + i / N;
    out[i] = (p[0] + p[kStride]) + (p[2 * kStride] + p[3 * kStride]);
  }
}

// The q-atoms' gradients of a chunk: add() takes each lane's reaction on the
// chunk's q-atom j (-r is its gradient), flush() adds them.  Every lane calls
// both.
struct QReaction {
  long long v[2] = {0, 0};   // lane (k, c): component c of q-atoms k and k + 8
  __device__ __forceinline__ void add(int j, float x, float y, float z) {
    x = row8_sum_t(x);
    y = row8_sum_t(y);
    z = row8_sum_t(z);
    const int c = threadIdx.x & 7;
    const long long t = col8_sum_t(fix(-(double)(c == 0 ? x : c == 1 ? y : z), kFScale));
    if ((int)((threadIdx.x >> 3) & 7) == (j & 7)) v[j >> 3] = t;
  }
  // slot0: q-cluster slot of the chunk's first q-atom (j = 4 member + cluster)
  __device__ __forceinline__ void flush(const Dev& d, int slot0, int q_left) const {
    const int c = threadIdx.x & 7, k = (threadIdx.x >> 3) & 7;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int j = k + 8 * h, m = kCl * (j & 3) + (j >> 2);
      if (c < 3 && m < q_left)
        atomicAdd((unsigned long long*)&d.f[3 * (size_t)d.qc_atom[slot0 + m] + c], (unsigned long long)v[h]);
    }
  }
};

// NS: number of states, or 0 to read it from the window
template <bool W3, bool EN, int NS>
__device__ __forceinline__ void qw_impl(const Dev& d, const WinDev& W, const int4 wk, long long acc[9]) {
  const int lane = threadIdx.x & 63, w = wk.x;
  const int S = NS ? NS : W.S;
  const bool qvdw = W.qvdw;
  const int slot = wk.y + (lane < wk.z ? lane : 0);
  const int ow = lane < wk.z ? d.wc_o[slot] : -1;
  const bool on = ow >= 0 && d.qw_on[slot] && d.qin[ow];   // the lane's water is in the Q lists
  float4 pw[3];
  const int xa = xw_at(slot / kCl, slot % kCl, 0);
  for (int k = 0; k < 3; ++k) pw[k] = d.xw[xa + kCl * k];
  double pd[9];
  if (EN)
    for (int k = 0; k < 3; ++k) {
      const double4 t = d.xwd[xa + kCl * k];
      pd[3 * k] = t.x; pd[3 * k + 1] = t.y; pd[3 * k + 2] = t.z;
    }
  float lam[kMaxS];
  for (int s = 0; s < kMaxS; ++s) lam[s] = s < S ? (float)W.lambda[s] : 0.f;
  const ConstF xq = (ConstF)(const float*)d.xq, par = (ConstF)(const float*)d.qcw_par, sct = (ConstF)d.qcw_sc;
  const ConstF parh = (ConstF)(const float*)d.qcw_h;
  const ConstD pare = (ConstD)(const double*)d.qcw_e, xd = (ConstD)d.x;
  const ConstI qat = (ConstI)d.qc_atom;
  constexpr int NLJ = W3 ? 3 : 1;
  double eel[kMaxS] = {}, evdw[kMaxS] = {};
  for (int ch = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) % kQWaves); ch < W.nqch; ch += kQWaves) {
    const int q0 = (ch >> 1) * 4 * kCl + (ch & 1) * 4;   // the chunk's first q-atom
    const int slot0 = W.qc_off * kCl + q0;
    QReaction react;
#pragma unroll 1
    for (int mb = 0; mb < 4; ++mb) {
      if (q0 + mb >= W.nq) break;
      float g[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int u = 0; u < 4; ++u) {
        if (q0 + kCl * u + mb >= W.nq) break;
        const int m = slot0 + kCl * u + mb;
        const float qx = xq[4 * m], qy = xq[4 * m + 1], qz = xq[4 * m + 2];
        float rx = 0.f, ry = 0.f, rz = 0.f;
        if (on) {
          float dxv[3], dyv[3], dzv[3], r2v[3];
  #pragma unroll
          for (int k = 0; k < 3; ++k) {
            dxv[k] = pw[k].x - qx; dyv[k] = pw[k].y - qy; dzv[k] = pw[k].z - qz;
            r2v[k] = r2_f(dxv[k], dyv[k], dzv[k]);
          }
          const float rO = rsq_r2(r2v[0]), r2O = rO * rO;
          const float rH1 = rsq_r2(r2v[1]), r2H1 = rH1 * rH1;
          const float rH2 = rsq_r2(r2v[2]), r2H2 = rH2 * rH2;
          const float r6hc = r2v[0] * r2v[0] * r2v[0];
          float dvO = 0.f, dvH1 = 0.f, dvH2 = 0.f;
  #pragma unroll
          for (int s = 0; s < (NS ? NS : kMaxS); ++s) {
            if (!NS && s >= S) break;
            // A, B with the oxygen, the charge products with oxygen and
            // hydrogen, the soft-core term
            const ConstF P = par + 4 * ((size_t)m * kMaxS + s);
            const float pa = P[0], pb = P[1], po = P[2], ph = P[3];
            float va, vb, ratio = 1.f;
            if (qvdw) {
              const float inv = rcp(r6hc + sct[(size_t)m * kMaxS + s]);
              va = pa * inv * inv;
              vb = pb * inv;
              ratio = r6hc * inv;
            } else {
              const float r6 = r2O * r2O * r2O;
              va = pa * r6 * r6;
              vb = pb * r6;
            }
            dvO = dv_f(dvO, r2O, po, rO, lj_f(va, vb, ratio), lam[s]);
            if (W3) {
              // 3-atom solvent: LJ and soft-core on the hydrogens too, and their
              // own charges (md.f90:11620-11640)
  #pragma unroll
              for (int k = 1; k < 3; ++k) {
                const ConstF H = parh + 4 * (((size_t)m * kMaxS + s) * 2 + k - 1);
                const float r2k = r2v[k], r2ik = k == 1 ? r2H1 : r2H2, rk = k == 1 ? rH1 : rH2;
                const float r6k = r2k * r2k * r2k;
                float vak, vbk, ratk = 1.f;
                if (qvdw) {
                  const float inv = rcp(r6k + H[3]);
                  vak = H[0] * inv * inv;
                  vbk = H[1] * inv;
                  ratk = r6k * inv;
                } else {
                  const float r6i = r2ik * r2ik * r2ik;
                  vak = H[0] * r6i * r6i;
                  vbk = H[1] * r6i;
                }
                float& dvk = k == 1 ? dvH1 : dvH2;
                dvk = dv_f(dvk, r2ik, H[2], rk, lj_f(vak, vbk, ratk), lam[s]);
              }
            } else {
              dvH1 = __builtin_fmaf(-(r2H1 * (ph * rH1)), lam[s], dvH1);
              dvH2 = __builtin_fmaf(-(r2H2 * (ph * rH2)), lam[s], dvH2);
            }
          }
          const float dv[3] = {dvO, dvH1, dvH2};
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            g[3 * k] = __builtin_fmaf(dv[k], dxv[k], g[3 * k]);
            g[3 * k + 1] = __builtin_fmaf(dv[k], dyv[k], g[3 * k + 1]);
            g[3 * k + 2] = __builtin_fmaf(dv[k], dzv[k], g[3 * k + 2]);
          }
          rx = __builtin_fmaf(dvH2, dxv[2], W3 ? __builtin_fmaf(dvH1, dxv[1], dvO * dxv[0])
                                               : __builtin_fmaf(dvO, dxv[0], dvH1 * dxv[1]));
          ry = __builtin_fmaf(dvH2, dyv[2], __builtin_fmaf(dvO, dyv[0], dvH1 * dyv[1]));
          rz = __builtin_fmaf(dvH2, dzv[2], __builtin_fmaf(dvO, dzv[0], dvH1 * dzv[1]));
          if (EN) {
            const ConstD qd = xd + 3 * (size_t)qat[m];
            double rinv[3], r6[NLJ];
  #pragma unroll
            for (int k = 0; k < 3; ++k) {
              const double dx = pd[3 * k] - qd[0], dy = pd[3 * k + 1] - qd[1], dz = pd[3 * k + 2] - qd[2];
              const double r2 = dx * dx + dy * dy + dz * dz;
              rinv[k] = rsqrt_e(r2);
              if (k < NLJ) r6[k < NLJ ? k : 0] = r2 * r2 * r2;
            }
  #pragma unroll
            for (int s = 0; s < (NS ? NS : kMaxS); ++s) {
              if (!NS && s >= S) break;
  #pragma unroll
              for (int k = 0; k < 3; ++k) {
                const ConstD E = pare + 4 * (((size_t)m * kMaxS + s) * 3 + k);   // A, B, soft-core, charge product
                eel[s] += E[3] * rinv[k];
                if (k < NLJ) {
                  const double inv = rcp_e(r6[k < NLJ ? k : 0] + E[2]);
                  evdw[s] += E[0] * inv * inv - E[1] * inv;
                }
              }
            }
          }
        }
        react.add(4 * mb + u, rx, ry, rz);
      }
      for (int k = 0; k < 9; ++k) acc[k] += fix((double)g[k], kFScale);
    }
    react.flush(d, slot0, W.nq - q0);
  }
  if (EN)
#pragma unroll
    for (int s = 0; s < (NS ? NS : kMaxS); ++s) {
      if (!NS && s >= S) break;
      const long long e1 = wave_sum_i(fix(eel[s], kEScale)), e2 = wave_sum_i(fix(evdw[s], kEScale));
      if (lane == 0) {
        add_energy_fix(d.ws, w, E_QW0 + 2 * s, e1);
        add_energy_fix(d.ws, w, E_QW0 + 2 * s + 1, e2);
      }
    }
}

// the work item of a group of kQWaves waves (past the last item: nothing but
// the barrier).  W3: the instance for 3-atom solvent windows; EK: the instance
// of steps where some window computes energies
template <bool W3, bool EK>
__device__ __forceinline__ void qw_group(const Dev& d, int item, long long* s) {
  long long acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  int4 wk = make_int4(0, 0, 0, 0);
  if (item < d.nqw_work) {
    wk = q_item(d.qw_work, item);
    const WinDev& W = d.win[wk.x];
    if (!d.ws[wk.x].active || (W.wat3 != 0) != W3) {
      wk.z = 0;
    } else {
      const bool en = EK && d.ws[wk.x].energy_now;
      if (W.S == 2) {
        if (en) qw_impl<W3, EK, 2>(d, W, wk, acc);
        else qw_impl<W3, false, 2>(d, W, wk, acc);
      } else {
        if (en) qw_impl<W3, EK, 0>(d, W, wk, acc);
        else qw_impl<W3, false, 0>(d, W, wk, acc);
      }
    }
  }
  q_store<9>(acc, wk.z, d.gq + 9 * (size_t)wk.y, s);
}
template <bool W3, bool EK>
__global__ void __launch_bounds__(64 * kQWaves) k_qw(Dev d) {
  __shared__ long long s[9 * 64 * kQWaves];
  qw_group<W3, EK>(d, blockIdx.x, s);
}

template <bool EN, int NS>
__device__ __forceinline__ void qp_impl(const Dev& d, const WinDev& W, const int4 wk, long long acc[3]) {
  const int lane = threadIdx.x & 63, w = wk.x;
  const int S = NS ? NS : W.S;
  const bool qvdw = W.qvdw, arith = W.arith;
  const float el14 = W.el14;
  const int slot = wk.y + (lane < wk.z ? lane : 0);
  const int pa = lane < wk.z ? d.sc_a[slot] : -1;
  const bool on = pa >= 0 && d.qp_on[slot] && d.qin[pa];   // the lane's solute atom is in the Q lists
  const int ia = pa >= 0 ? pa : W.ao;
  const float4 pj = d.x32[ia], lj = d.sljp[slot];
  const int iacj = d.iac[ia];
  double xj[3];
  double4 tlj = make_double4(0, 0, 0, 0);
  if (EN) {
    for (int c = 0; c < 3; ++c) xj[c] = d.x[3 * (size_t)ia + c];
    tlj = d.sljd[slot];
  }
  float lam[kMaxS];
  for (int s = 0; s < kMaxS; ++s) lam[s] = s < S ? (float)W.lambda[s] : 0.f;
  const ConstF xq = (ConstF)(const float*)d.xq, qlj = (ConstF)(const float*)(d.q_lj + W.qs_off);
  const ConstF qcr = (ConstF)(d.q_crg + W.qs_off);
  const ConstD xd = (ConstD)d.x, qljd = (ConstD)(d.q_ljd + 4 * (size_t)W.qs_off);
  const ConstI qat = (ConstI)d.qc_atom;
  const float* sct = d.q_sc + W.qsc_off + (size_t)iacj * S;
  const double* scd = d.q_scd + W.qsc_off + (size_t)iacj * S;
  double eel[kMaxS] = {}, evdw[kMaxS] = {};
  for (int ch = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) % kQWaves); ch < W.nqch; ch += kQWaves) {
    const int q0 = (ch >> 1) * 4 * kCl + (ch & 1) * 4;   // the chunk's first q-atom
    const int slot0 = W.qc_off * kCl + q0;
    // 1-4 pairs with the chunk's q-atoms, bit j for q-atom j
    const unsigned m14 = d.qp14[W.qp14_off + (size_t)(slot - W.sc_off * kCl) * W.nqch + ch];
    QReaction react;
#pragma unroll 1
    for (int mb = 0; mb < 4; ++mb) {
      if (q0 + mb >= W.nq) break;
      float g0 = 0.f, g1 = 0.f, g2 = 0.f;
#pragma unroll 1
      for (int u = 0; u < 4; ++u) {
        const int iq = q0 + kCl * u + mb;
        if (iq >= W.nq) break;
        const int m = slot0 + kCl * u + mb, j = 4 * mb + u;
        const float qx = xq[4 * m], qy = xq[4 * m + 1], qz = xq[4 * m + 2];
        float rx = 0.f, ry = 0.f, rz = 0.f;
        if (on) {
          const bool is14 = (m14 >> j) & 1u;
          const float dx = pj.x - qx, dy = pj.y - qy, dz = pj.z - qz;
          const float r2 = r2_f(dx, dy, dz);
          const float rinv = rsq_r2(r2), r2inv = rinv * rinv;
          const float r6hc = r2 * r2 * r2;
          float dv = 0.f;
  #pragma unroll
          for (int s = 0; s < (NS ? NS : kMaxS); ++s) {
            if (!NS && s >= S) break;
            const ConstF ql = qlj + 4 * (iq * S + s);
            const float qc = qcr[iq * S + s];
            float aLJ, bLJ;
            if (is14) lj_ab((float)ql[2], (float)ql[3], lj.z, lj.w, arith, &aLJ, &bLJ);
            else lj_ab((float)ql[0], (float)ql[1], lj.x, lj.y, arith, &aLJ, &bLJ);
            float vel = (qc * pj.w) * rinv;
            if (is14) vel *= el14;
            float va, vb, ratio = 1.f;
            if (qvdw) {
              const float inv = rcp(r6hc + sct[(size_t)iq * W.natyps * S + s]);
              va = aLJ * inv * inv;
              vb = bLJ * inv;
              ratio = r6hc * inv;
            } else {
              const float r6 = r2inv * r2inv * r2inv;
              va = aLJ * r6 * r6;
              vb = bLJ * r6;
            }
            // (the charge term's factors are rounded one by one: el14 comes between)
            dv = __builtin_fmaf(r2inv * __builtin_fmaf(-ratio, lj_f(va, vb, 1.f), -vel), lam[s], dv);
          }
          g0 = __builtin_fmaf(dv, dx, g0); g1 = __builtin_fmaf(dv, dy, g1); g2 = __builtin_fmaf(dv, dz, g2);
          rx = dv * dx; ry = dv * dy; rz = dv * dz;
          if (EN) {
            const ConstD qd = xd + 3 * (size_t)qat[m];
            const double ex = xj[0] - qd[0], ey = xj[1] - qd[1], ez = xj[2] - qd[2];
            const double rr = ex * ex + ey * ey + ez * ez;
            const double ri = rsqrt_e(rr), r6 = rr * rr * rr;
            const double ta = is14 ? tlj.z : tlj.x, tb = is14 ? tlj.w : tlj.y;
  #pragma unroll
            for (int s = 0; s < (NS ? NS : kMaxS); ++s) {
              if (!NS && s >= S) break;
              double vel = (double)(qcr[iq * S + s] * pj.w) * ri;
              if (is14) vel *= W.el14d;
              eel[s] += vel;
              const ConstD ql = qljd + 4 * (iq * S + s);
              double aLJ, bLJ;
              lj_ab(is14 ? (double)ql[2] : (double)ql[0], is14 ? (double)ql[3] : (double)ql[1], ta, tb, arith, &aLJ, &bLJ);
              const double inv = rcp_e(r6 + (qvdw ? scd[(size_t)iq * W.natyps * S + s] : 0.0));
              evdw[s] += aLJ * inv * inv - bLJ * inv;
            }
          }
        }
        react.add(j, rx, ry, rz);
      }
      atom_grad(acc, (double)g0, (double)g1, (double)g2);
    }
    react.flush(d, slot0, W.nq - q0);
  }
  if (EN)
#pragma unroll
    for (int s = 0; s < (NS ? NS : kMaxS); ++s) {
      if (!NS && s >= S) break;
      const long long e1 = wave_sum_i(fix(eel[s], kEScale)), e2 = wave_sum_i(fix(evdw[s], kEScale));
      if (lane == 0) {
        add_energy_fix(d.ws, w, E_Q0 + 8 * s + 6, e1);
        add_energy_fix(d.ws, w, E_Q0 + 8 * s + 7, e2);
      }
    }
}

template <bool EK>
__device__ __forceinline__ void qp_group(const Dev& d, int item, long long* s) {
  long long acc[3] = {0, 0, 0};
  int4 wk = make_int4(0, 0, 0, 0);
  if (item < d.nqp_work) {
    wk = q_item(d.qp_work, item);
    const WinDev& W = d.win[wk.x];
    if (!d.ws[wk.x].active) {
      wk.z = 0;
    } else {
      const bool en = EK && d.ws[wk.x].energy_now;
      if (W.S == 2) {
        if (en) qp_impl<EK, 2>(d, W, wk, acc);
        else qp_impl<false, 2>(d, W, wk, acc);
      } else {
        if (en) qp_impl<EK, 0>(d, W, wk, acc);
        else qp_impl<false, 0>(d, W, wk, acc);
      }
    }
  }
  q_store<3>(acc, wk.z, d.gq + 9 * (size_t)d.nwslot + 3 * (size_t)wk.y, s);
}
template <bool EK>
__global__ void __launch_bounds__(64 * kQWaves) k_qp(Dev d) {
  __shared__ long long s[3 * 64 * kQWaves];
  qp_group<EK>(d, blockIdx.x, s);
}

// q-q and q-(bonded neighbour) pairs (nonbond_qq, md.f90:10763-10868).
// Forces: one wave per atom over the atom's pairs of every state (each pair
// from both sides), FP32 from the packed record of the pair, summed in fixed
// point over the wave, with one atomic per component.  As per-pair slots and
// a gather it was two kernels in a row, 14 us for the 64-window ladder and 11
// us (of an 86 us step) for one window.
__device__ __forceinline__ void qq_atom(const Dev& d, int k) {
  const int atom = d.qqg_atom[k], lane = threadIdx.x & 63;
  const int w = d.wid[atom];
  if (!d.ws[w].active) return;   // uniform over the wave
  const WinDev& W = d.win[w];
  const float4 pi = d.x32[atom];
  long long gx = 0, gy = 0, gz = 0;
  const int m1 = d.qqg_start[k + 1];
  for (int m = d.qqg_start[k] + lane; m < m1; m += 64) {
#pragma clang fp contract(off)
    const float4 p = d.qqg_ent[2 * (size_t)m], r = d.qqg_ent[2 * (size_t)m + 1];
    const float q = p.x, es = p.y, aLJ = p.z, bLJ = p.w, sc = r.x;
    const int j = __float_as_int(r.y), fl = __float_as_int(r.z);   // partner; state, LJ code 3, exponential
    const float4 pj = d.x32[j];
    const float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
    const float r2 = r2_f(dx, dy, dz);
    const float r4 = r2 * r2, r6hc = r2 * r4;
    const float r2inv = 1.f / r2, ri = sqrtf(r2inv);
    float vel = q * ri * es;
    if (fl & 8) vel *= W.el14;
    float t;
    if (fl & 16) {
      const float va = aLJ * expf(-bLJ / ri);
      t = -vel - bLJ * va / ri;
    } else {
      const float r6 = 1.f / __builtin_fmaf(r2, r4, sc);
      t = __builtin_fmaf(-r6, r6hc * __builtin_fmaf(aLJ * (r6 * r6), 12.f, -6.f * (bLJ * r6)), -vel);
    }
    const float dv = r2inv * t * (float)W.lambda[fl & 7];
    gx += fix(-(double)(dv * dx), kFScale);
    gy += fix(-(double)(dv * dy), kFScale);
    gz += fix(-(double)(dv * dz), kFScale);
  }
  gx = wave_sum_i(gx);
  gy = wave_sum_i(gy);
  gz = wave_sum_i(gz);
  if (lane < 3)
    atomicAdd((unsigned long long*)&d.f[3 * (size_t)atom + lane], (unsigned long long)(lane == 0 ? gx : lane == 1 ? gy : gz));
}

// energies of q-q pair k and its state, FP64 (energy steps); k past the last
// pair does nothing.  Every lane of the wave must call it.
__device__ __forceinline__ void qq_energy(const Dev& d, int k) {
  bool valid = false;
  int w = 0, s = 0, base = 6;
  double e_el = 0.0, e_vdw = 0.0;
  if (k < d.nqq) {
    w = d.qq_win[k];
    const WinState& st = d.ws[w];
    if (st.active && st.energy_now) {
      valid = true;
      const WinDev& W = d.win[w];
      const int4 e = d.qq_ij[k];
      s = d.qq_st[k];
      const int i = d.q_atom[W.q_off + e.x], j = e.y, jq = e.z, iLJ = e.w;
      const float2 qq = d.qq_q[k];
      // qi qj is exact in FP64, as the reference's real(8) product
      const double qi = (double)qq.x, qj = (double)qq.y;
      const double2 ab = d.qq_ab[k];
      const double ddx = d.x[3 * j] - d.x[3 * i], ddy = d.x[3 * j + 1] - d.x[3 * i + 1],
                   ddz = d.x[3 * j + 2] - d.x[3 * i + 2];
      const double rr2 = ddx * ddx + ddy * ddy + ddz * ddz;
      e_el = qi * qj * rsqrt_e(rr2) * (double)d.qq_es[k];
      if (iLJ == 3) e_el *= W.el14d;
      if (W.qvdw && jq && iLJ == 2) {
        e_vdw = ab.x * exp(-ab.y * sqrt(rr2));
      } else {
        const double inv = rcp_e(rr2 * rr2 * rr2 + (double)d.qq_sc[k]);
        e_vdw = ab.x * inv * inv - ab.y * inv;
      }
      base = jq ? 4 : 6;  // qq or qp slot
    }
  }
  wave_energy(d.ws, w, E_Q0 + 8 * s + base, e_el, valid);
  wave_energy(d.ws, w, E_Q0 + 8 * s + base + 1, e_vdw, valid);
}

// waves of the q-q work: one per atom, then on energy steps one per 64 pairs
template <bool EK>
__device__ __forceinline__ void qq_wave(const Dev& d, int wave) {
  if (wave < d.nqqg) qq_atom(d, wave);
  else if (EK) qq_energy(d, (wave - d.nqqg) * 64 + (int)(threadIdx.x & 63));
}
template <bool EK>
__global__ void __launch_bounds__(256) k_qq(Dev d) {
  qq_wave<EK>(d, wave_id());
}
static int qq_waves(const Dev& d, bool energy) { return d.nqqg + (energy ? (d.nqq + 63) / 64 : 0); }
static void launch_qq(const Dev& d, hipStream_t s, bool energy) {
  if (!d.nqq) return;
  const int nb = (qq_waves(d, energy) * 64 + 255) / 256;
  if (energy) k_qq<true><<<nb, 256, 0, s>>>(d);
  else k_qq<false><<<nb, 256, 0, s>>>(d);
}

// ------------------------------------------------------------- LRF --
// LRF expansions (the phi sums of the list builders, e.g. nbpplist_lrf,
// md.f90:5589-5700): for every target charge group g, the Taylor terms about
// its centre of all charges of groups h whose switching atoms lie beyond the
// cut-off and within the LRF radius.
// Pack: the switching atom of every group (x, y, z, excluded) and the
// non-q atoms of every group (x, y, z, charge), contiguous per group.
__global__ void __launch_bounds__(256) k_lrf_pack(Dev d) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < d.ngrp_all) {
    const int w = d.g_win[k];
    if (d.ws[w].active && d.ws[w].list_now && d.win[w].use_lrf) {
      const int sw = d.g_sw[k];
      d.ls_sw[k] = make_double4(d.x[3 * sw], d.x[3 * sw + 1], d.x[3 * sw + 2], (d.aflag[sw] & 1) ? 1.0 : 0.0);
    }
  }
  if (k < d.nls) {
    const int at = d.ls_atom[k];
    const int w = d.wid[at];
    if (d.ws[w].active && d.ws[w].list_now && d.win[w].use_lrf)
      d.ls_xq[k] = make_double4(d.x[3 * at], d.x[3 * at + 1], d.x[3 * at + 2], (double)d.x32[at].w);
  }
}

__device__ __forceinline__ double r2_pos(double ax, double ay, double az, double bx, double by, double bz) {
#pragma clang fp contract(off)
  const double dx = __dsub_rn(ax, bx), dy = __dsub_rn(ay, by), dz = __dsub_rn(az, bz);
  return __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
}

// Taylor terms of one source charge q at d = x(source) - centre: potential,
// field, field gradient and its derivative (the sums of nbpw/nbww lists with
// LRF, md.f90:5589-5700), with the shared factors hoisted.  The terms of the
// form u - f0 (diagonal of the gradient) and u - g d (derivative) are split:
// acc takes the u parts and aux the sums of f0 and of g d_x, g d_y, g d_z,
// which lrf_finish subtracts once.  Which products are fused is spelled out, as
// for the FP32 pairs.  SET: kLrfLow the potential, field and gradient (acc 0..9),
// kLrfHigh the derivative (acc 10..19), or both.
// (The derivatives of 1/r are traceless, so 16 of the 20 sums and r^2 would do,
// with 45 FP64 instructions a source for 55.  But r^2 times the squared
// reciprocal root is 1 only to the root's 1e-12, and with the sums' other last
// bits the gradient moves by a quantum now and then, and with it a trajectory.)
constexpr int kLrfLow = 1, kLrfHigh = 2, kLrfSums = 20;
template <int SET>
__device__ __forceinline__ void lrf_add(double acc[kLrfSums], double aux[4], double q, double dx, double dy, double dz) {
#pragma clang fp contract(off)
  const double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
  const double ir = rsqrt_e(r2);
  const double ir2 = ir * ir;
  const double qr = q * ir;            // q / r
  const double f0 = qr * ir2;          // q / r^3
  const double f1 = 3.0 * f0 * ir2;    // 3 q / r^5
  if constexpr (SET & kLrfLow) {
    acc[0] = fma(q, ir, acc[0]);
    acc[1] = fma(-f0, dx, acc[1]); acc[2] = fma(-f0, dy, acc[2]); acc[3] = fma(-f0, dz, acc[3]);
    const double ax = f1 * dx, ay = f1 * dy;
    acc[4] = fma(ax, dx, acc[4]); acc[5] = fma(ax, dy, acc[5]); acc[6] = fma(ax, dz, acc[6]);
    acc[7] = fma(ay, dy, acc[7]); acc[8] = fma(ay, dz, acc[8]); acc[9] = fma(f1 * dz, dz, acc[9]);
    aux[0] = fma(qr, ir2, aux[0]);
  }
  if constexpr (SET & kLrfHigh) {
    // f2 (5 d_a d_b d_c - r2 (delta_ab d_c + delta_ac d_b + delta_bc d_a))
    const double f2 = -f1 * ir2;       // -3 q / r^7
    const double c5 = 5.0 * f2, g = f2 * r2;
    const double px = c5 * dx, py = c5 * dy;
    const double xx = px * dx, yy = py * dy, zz = c5 * dz * dz;
    acc[10] = fma(xx, dx, acc[10]); acc[11] = fma(xx, dy, acc[11]); acc[12] = fma(xx, dz, acc[12]);
    acc[13] = fma(yy, dx, acc[13]); acc[14] = fma(px * dy, dz, acc[14]); acc[15] = fma(zz, dx, acc[15]);
    acc[16] = fma(yy, dy, acc[16]); acc[17] = fma(yy, dz, acc[17]); acc[18] = fma(zz, dy, acc[18]);
    acc[19] = fma(zz, dz, acc[19]);
    aux[1] = fma(g, dx, aux[1]); aux[2] = fma(g, dy, aux[2]); aux[3] = fma(g, dz, aux[3]);
  }
}
template <int SET>
__device__ __forceinline__ void lrf_finish(double acc[kLrfSums], const double aux[4]) {
#pragma clang fp contract(off)
  if constexpr (SET & kLrfLow) {
    acc[4] -= aux[0]; acc[7] -= aux[0]; acc[9] -= aux[0];
  }
  if constexpr (SET & kLrfHigh) {
    acc[10] = fma(-3.0, aux[1], acc[10]); acc[11] -= aux[2]; acc[12] -= aux[3];
    acc[13] -= aux[1]; acc[15] -= aux[1];
    acc[16] = fma(-3.0, aux[2], acc[16]); acc[17] -= aux[3]; acc[18] -= aux[2];
    acc[19] = fma(-3.0, aux[3], acc[19]);
  }
}

// Build: one lane per target group; a block is a wave, which takes 64 consecutive
// targets and one of kLrfParts parts of the window's source groups.  The sources
// are the same for all lanes, so they are read into scalar registers.  Every wave
// sums its sources in index order and k_lrf_reduce adds the parts in theirs, so
// the sums depend on neither batch nor scheduling.
//
// Bound by the FP64 rate for many windows (55 instructions a source at one per 4
// cycles, 1.2 of the 2.0 ms that the 64-window ladder's 820 M take; blocks of
// 256 threads 2.3 ms) and by latency for few, whose waves are fewer than the
// SIMDs.  Those take SPLIT: two waves for one, each with one of the sums' two
// sets, the next group's record and first three sources loaded while the current
// ones are summed, three sources at a time.  One ligand-in-water window 132 us
// without, 68 with; one protein window 310 and 189; the ladder 2005 and 3035 (the
// common factors are formed twice).
constexpr int kLrfSplitMost = 1024;   // waves without SPLIT, one a SIMD: 5, 7, 9 small windows (720, 1008, 1296)
                                      // 153, 172, 176 us without and 119, 160, 194 with
template <int SET>
__device__ __forceinline__ void lrf_wave(const Dev& d, int4 lw) {
  constexpr bool kAhead = SET != (kLrfLow | kLrfHigh);
  const WinDev& W = d.win[lw.x];
  const int lane = threadIdx.x & 63;
  const int g = lw.y + lane;
  bool g_ok = lane < lw.z;
  double4 sg = make_double4(0, 0, 0, 1);
  double cx = 0, cy = 0, cz = 0;
  bool gw = false;
  if (g_ok) {
    sg = d.ls_sw[g];
    g_ok = sg.w == 0.0;
    gw = (g - W.g_off) >= W.ngrp_solute;
    cx = d.g_cent[3 * g]; cy = d.g_cent[3 * g + 1]; cz = d.g_cent[3 * g + 2];
  }
  const double rclrf2 = W.rclrf2;
  double acc[kLrfSums], aux[4] = {0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < kLrfSums; ++k) acc[k] = 0.0;
  // (wave-uniform: kept in scalar registers, with what they index)
  const int h_beg = __builtin_amdgcn_readfirstlane(W.g_off + (int)(((long long)lw.w * W.ngrp) / kLrfParts));
  const int h_end = __builtin_amdgcn_readfirstlane(W.g_off + (int)(((long long)(lw.w + 1) * W.ngrp) / kLrfParts));
  const int h_sol = __builtin_amdgcn_readfirstlane(min(max(W.g_off + W.ngrp_solute, h_beg), h_end));
  const ConstD sw = (ConstD)(const double*)d.ls_sw, xq = (ConstD)(const double*)d.ls_xq;
  const ConstI nn = (ConstI)d.ls_n;
  // the groups' sources are consecutive
  int f = __builtin_amdgcn_readfirstlane(h_beg < h_end ? d.ls_first[h_beg] : 0);
  // in range of the group whose switching atom is at s (a target is within the
  // cut-off of itself)
  auto in_range = [&](double x, double y, double z, double excluded, double rc2) {
    const double r2g = r2_pos(sg.x, sg.y, sg.z, x, y, z);
    return excluded == 0.0 && g_ok && !(r2g <= rc2) && !(r2g > rclrf2);
  };
  double hs[4], a[12];
  int n = 0;
  if (kAhead && h_beg < h_end) {
    n = nn[h_beg];
    for (int k = 0; k < 4; ++k) hs[k] = sw[4 * (size_t)h_beg + k];
    for (int k = 0; k < 12; ++k) a[k] = xq[4 * (size_t)f + k];
  }
#pragma unroll 1
  for (int seg = 0; seg < 2; ++seg) {
    // cut-off against a solute, then against a water source group
    const double rc2 = seg ? (gw ? W.rcww2 : W.rcpw2) : (gw ? W.rcpw2 : W.rcpp2);
    const int h1 = seg ? h_end : h_sol;
#pragma unroll 1
    for (int h = seg ? h_sol : h_beg; h < h1; ++h) {
      if constexpr (kAhead) {
        // (the last group loads itself again)
        const int hn = h + 1 < h_end ? h + 1 : h, fn = h + 1 < h_end ? f + n : f, n1 = nn[hn];
        double hs1[4], a1[12];
        for (int k = 0; k < 4; ++k) hs1[k] = sw[4 * (size_t)hn + k];
        for (int k = 0; k < 12; ++k) a1[k] = xq[4 * (size_t)fn + k];
        if (in_range(hs[0], hs[1], hs[2], hs[3], rc2)) {
          if (n == 3) {
#pragma unroll
            for (int k = 0; k < 3; ++k) lrf_add<SET>(acc, aux, a[4 * k + 3], a[4 * k] - cx, a[4 * k + 1] - cy, a[4 * k + 2] - cz);
          } else {
            for (int k = 0; k < n; ++k) {
              const ConstD b = xq + 4 * (size_t)(f + k);
              lrf_add<SET>(acc, aux, b[3], b[0] - cx, b[1] - cy, b[2] - cz);
            }
          }
        }
        f = fn;
        n = n1;
        for (int k = 0; k < 4; ++k) hs[k] = hs1[k];
        for (int k = 0; k < 12; ++k) a[k] = a1[k];
      } else {
        const int m = nn[h];
        const ConstD s = sw + 4 * (size_t)h;
        if (in_range(s[0], s[1], s[2], s[3], rc2)) {
#pragma unroll 1
          for (int k = 0; k < m; ++k) {
            const ConstD b = xq + 4 * (size_t)(f + k);
            lrf_add<SET>(acc, aux, b[3], b[0] - cx, b[1] - cy, b[2] - cz);
          }
        }
        f += m;
      }
    }
  }
  if (!g_ok) return;
  lrf_finish<SET>(acc, aux);
  double* out = d.g_lrf_part + kLrfSums * ((size_t)lw.w * d.ngrp_all + g);
  for (int k = SET & kLrfLow ? 0 : 10; k < (SET & kLrfHigh ? kLrfSums : 10); ++k) out[k] = acc[k];
}
template <bool SPLIT>
__global__ void __launch_bounds__(64, 4) k_lrf_build(Dev d) {
  const int4 lw = q_item(d.lrf_work, SPLIT ? blockIdx.x >> 1 : blockIdx.x);   // window, first target group, count, source part
  if (!d.ws[lw.x].active || !d.ws[lw.x].list_now || !d.win[lw.x].use_lrf) return;
  if (!SPLIT) lrf_wave<kLrfLow | kLrfHigh>(d, lw);
  else if (blockIdx.x & 1) lrf_wave<kLrfHigh>(d, lw);
  else lrf_wave<kLrfLow>(d, lw);
}

// sum of the source parts in part order, one thread per (group, term)
__global__ void __launch_bounds__(256) k_lrf_reduce(Dev d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kLrfSums * d.ngrp_all) return;
  const int g = i / kLrfSums, w = d.g_win[g];
  if (!d.ws[w].active || !d.ws[w].list_now || !d.win[w].use_lrf || d.ls_sw[g].w != 0.0) return;
  double v = 0.0;
  for (int p = 0; p < kLrfParts; ++p) v += d.g_lrf_part[(size_t)p * kLrfSums * d.ngrp_all + i];
  d.g_lrf[i] = v;
}

// Evaluation per atom (lrf_taylor, md.f90:3646-3712), FP64.
__device__ __forceinline__ void lrf_taylor_atom(const Dev& d, int i, long long* acc) {
  bool on = false;
  int w = 0;
  double e = 0.0;
  if (i < d.ntot) {
    w = d.wid[i];
    const WinState& st = d.ws[w];
    const WinDev& W = d.win[w];
    on = st.active && W.use_lrf && !(d.aflag[i] & (1 | 8));  // not excluded, not a q-atom
    if (on) {
      const int g = d.grp[i];
      const double* p = &d.g_lrf[20 * g];
      const double r0 = d.g_cent[3 * g] - d.x[3 * i], r1 = d.g_cent[3 * g + 1] - d.x[3 * i + 1],
                   r2 = d.g_cent[3 * g + 2] - d.x[3 * i + 2];
      const double xx = p[4], xy = p[5], xz = p[6], yy = p[7], yz = p[8], zz = p[9];
      const double t_xxx = p[10], t_xxy = p[11], t_xxz = p[12], t_xyy = p[13], t_xyz = p[14], t_xzz = p[15],
                   t_yyy = p[16], t_yyz = p[17], t_yzz = p[18], t_zzz = p[19];
      const double vij = p[0] + p[1] * r0 + p[2] * r1 + p[3] * r2 + 0.5 * (xx * r0 + xy * r1 + xz * r2) * r0 +
                         0.5 * (xy * r0 + yy * r1 + yz * r2) * r1 + 0.5 * (xz * r0 + yz * r1 + zz * r2) * r2;
      const double f0 = p[1] + xx * r0 + xy * r1 + xz * r2 + 0.5 * (t_xxx * r0 + t_xxy * r1 + t_xxz * r2) * r0 +
                        0.5 * (t_xxy * r0 + t_xyy * r1 + t_xyz * r2) * r1 +
                        0.5 * (t_xxz * r0 + t_xyz * r1 + t_xzz * r2) * r2;
      const double f1 = p[2] + xy * r0 + yy * r1 + yz * r2 + 0.5 * (t_xxy * r0 + t_xyy * r1 + t_xyz * r2) * r0 +
                        0.5 * (t_xyy * r0 + t_yyy * r1 + t_yyz * r2) * r1 +
                        0.5 * (t_xyz * r0 + t_yyz * r1 + t_yzz * r2) * r2;
      const double f2 = p[3] + xz * r0 + yz * r1 + zz * r2 + 0.5 * (t_xxz * r0 + t_xyz * r1 + t_xzz * r2) * r0 +
                        0.5 * (t_xyz * r0 + t_yyz * r1 + t_yzz * r2) * r1 +
                        0.5 * (t_xzz * r0 + t_yzz * r1 + t_zzz * r2) * r2;
      const double q = (double)d.x32[i].w;
      atom_grad(acc, -q * f0, -q * f1, -q * f2);
      e = 0.5 * q * vij;
      on = st.energy_now;
    }
  }
  wave_energy(d.ws, w, E_LRF, e, on);
}

// ---------------------------------------------------------- bonded --
__device__ __forceinline__ void torsion_geom(const double* x, int i, int j, int k, int l, double* phi,
                                             double* scp_out, double dp[12]) {
  double rji[3], rjk[3], rkl[3], rnj[3], rnk[3];
  for (int c = 0; c < 3; ++c) {
    rji[c] = x[3 * i + c] - x[3 * j + c];
    rjk[c] = x[3 * k + c] - x[3 * j + c];
    rkl[c] = x[3 * l + c] - x[3 * k + c];
  }
  rnj[0] = rji[1] * rjk[2] - rji[2] * rjk[1];
  rnj[1] = rji[2] * rjk[0] - rji[0] * rjk[2];
  rnj[2] = rji[0] * rjk[1] - rji[1] * rjk[0];
  rnk[0] = -rjk[1] * rkl[2] + rjk[2] * rkl[1];
  rnk[1] = -rjk[2] * rkl[0] + rjk[0] * rkl[2];
  rnk[2] = -rjk[0] * rkl[1] + rjk[1] * rkl[0];
  double bj2inv = 1.0 / (rnj[0] * rnj[0] + rnj[1] * rnj[1] + rnj[2] * rnj[2]);
  double bk2inv = 1.0 / (rnk[0] * rnk[0] + rnk[1] * rnk[1] + rnk[2] * rnk[2]);
  double bjinv = sqrt(bj2inv), bkinv = sqrt(bk2inv);
  double scp = (rnj[0] * rnk[0] + rnj[1] * rnk[1] + rnj[2] * rnk[2]) * (bjinv * bkinv);
  if (scp > 1.0) scp = 1.0;
  else if (scp < -1.0) scp = -1.0;
  double ph = acos(scp);
  double sg = rjk[0] * (rnj[1] * rnk[2] - rnj[2] * rnk[1]) + rjk[1] * (rnj[2] * rnk[0] - rnj[0] * rnk[2]) +
              rjk[2] * (rnj[0] * rnk[1] - rnj[1] * rnk[0]);
  if (sg < 0) ph = -ph;
  double f1 = sin(ph);
  if (fabs(f1) < 1.e-12) f1 = 1.e-12;
  f1 = -1.0 / f1;
  double di[3], dl[3];
  for (int c = 0; c < 3; ++c) {
    di[c] = f1 * (rnk[c] * (bjinv * bkinv) - scp * rnj[c] * bj2inv);
    dl[c] = f1 * (rnj[c] * (bjinv * bkinv) - scp * rnk[c] * bk2inv);
  }
  double rki[3], rlj[3];
  for (int c = 0; c < 3; ++c) { rki[c] = rji[c] - rjk[c]; rlj[c] = -rjk[c] - rkl[c]; }
  dp[0] = rjk[1] * di[2] - rjk[2] * di[1];
  dp[1] = rjk[2] * di[0] - rjk[0] * di[2];
  dp[2] = rjk[0] * di[1] - rjk[1] * di[0];
  dp[3] = rki[1] * di[2] - rki[2] * di[1] + rkl[1] * dl[2] - rkl[2] * dl[1];
  dp[4] = rki[2] * di[0] - rki[0] * di[2] + rkl[2] * dl[0] - rkl[0] * dl[2];
  dp[5] = rki[0] * di[1] - rki[1] * di[0] + rkl[0] * dl[1] - rkl[1] * dl[0];
  dp[6] = rlj[1] * dl[2] - rlj[2] * dl[1] - rji[1] * di[2] + rji[2] * di[1];
  dp[7] = rlj[2] * dl[0] - rlj[0] * dl[2] - rji[2] * di[0] + rji[0] * di[2];
  dp[8] = rlj[0] * dl[1] - rlj[1] * dl[0] - rji[0] * di[1] + rji[1] * di[0];
  dp[9] = rjk[1] * dl[2] - rjk[2] * dl[1];
  dp[10] = rjk[2] * dl[0] - rjk[0] * dl[2];
  dp[11] = rjk[0] * dl[1] - rjk[1] * dl[0];
  *phi = ph;
  *scp_out = scp;
}

template <class Sink>
__device__ __forceinline__ void put4(const Sink& put, const int4& a, double dv, const double dp[12]) {
  put(a.x, 0, dv * dp[0], dv * dp[1], dv * dp[2]);
  put(a.y, 1, dv * dp[3], dv * dp[4], dv * dp[5]);
  put(a.z, 2, dv * dp[6], dv * dp[7], dv * dp[8]);
  put(a.w, 3, dv * dp[9], dv * dp[10], dv * dp[11]);
}

// angle (md.f90:814-901): energy and the gradient factors di, dk of the end
// atoms (the middle atom takes -(di + dk)); dv = fk * (theta - theta0)
__device__ __forceinline__ void angle_geom(const double* x, int i, int j, int k, double fk, double ang0, double* e,
                                           double* dv, double di[3], double dk[3]) {
  double rji[3], rjk[3];
  for (int c = 0; c < 3; ++c) { rji[c] = x[3 * i + c] - x[3 * j + c]; rjk[c] = x[3 * k + c] - x[3 * j + c]; }
  const double bji2inv = 1.0 / (rji[0] * rji[0] + rji[1] * rji[1] + rji[2] * rji[2]);
  const double bjk2inv = 1.0 / (rjk[0] * rjk[0] + rjk[1] * rjk[1] + rjk[2] * rjk[2]);
  const double bjiinv = sqrt(bji2inv), bjkinv = sqrt(bjk2inv);
  double scp = (rji[0] * rjk[0] + rji[1] * rjk[1] + rji[2] * rjk[2]) * bjiinv * bjkinv;
  if (scp > 1.0) scp = 1.0;
  else if (scp < -1.0) scp = -1.0;
  const double angv = acos(scp);
  const double da = angv - ang0;
  *e = 0.5 * fk * da * da;
  *dv = fk * da;
  double f1 = sin(angv);
  if (fabs(f1) < 1.e-12) f1 = -1.e12;
  else f1 = -1.0 / f1;
  for (int c = 0; c < 3; ++c) {
    di[c] = f1 * (rjk[c] * bjiinv * bjkinv - scp * rji[c] * bji2inv);
    dk[c] = f1 * (rji[c] * bjiinv * bjkinv - scp * rjk[c] * bjk2inv);
  }
}


// One bonded term t of the flat term index (bonds, angles, torsions,
// impropers, then the q-bonds, q-angles, q-torsions and q-impropers), its
// gradient handed to `put` per term atom (the atom and its place in the term)
// and its energy to put.energy; t past the last term does nothing.  Every lane
// of the wave must call it (the energy goes through a wave sum).
template <class Sink>
__device__ __forceinline__ void bonded_term(const Dev& d, int t, const Sink& put) {
  const int n1 = d.nbond, n2 = n1 + d.nang, n3 = n2 + d.ntor, n4 = n3 + d.nimp;
  const int n5 = n4 + d.nqb, n6 = n5 + d.nqa, n7 = n6 + d.nqt, n8 = n7 + d.nqi;
  const double* x = d.x;
  bool valid = false;
  int w = 0, eslot = 0;
  double e = 0.0;
  if (t < n1) {  // bond (md.f90:954-997)
    w = d.b_win[t];
    if (d.ws[w].active) {
      const int2 ij = d.b_ij[t];
      const double2 p = d.b_par[t];
      double r[3];
      for (int c = 0; c < 3; ++c) r[c] = x[3 * ij.y + c] - x[3 * ij.x + c];
      const double bl = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
      const double db = bl - p.y;
      const double dv = p.x * db / bl;
      put(ij.x, 0, -r[0] * dv, -r[1] * dv, -r[2] * dv);
      put(ij.y, 1, r[0] * dv, r[1] * dv, r[2] * dv);
      valid = true;
      e = 0.5 * p.x * db * db;
      eslot = d.b_solv[t] ? E_W_BOND : E_P_BOND;
    }
  } else if (t < n2) {  // angle (+ Urey-Bradley for CHARMM, md.f90:904-951)
    const int a = t - n1;
    w = d.a_win[a];
    if (d.ws[w].active) {
      const int4 ijk = d.a_ijk[a];
      const double4 p = d.a_par[a];
      double dv, di[3], dk[3];
      angle_geom(x, ijk.x, ijk.y, ijk.z, p.x, p.y, &e, &dv, di, dk);
      double gi[3], gk[3];
      for (int c = 0; c < 3; ++c) { gi[c] = dv * di[c]; gk[c] = dv * dk[c]; }
      double gj[3] = {-dv * (di[0] + dk[0]), -dv * (di[1] + dk[1]), -dv * (di[2] + dk[2])};
      if (d.urey[w] && p.z > 0.0) {
        double r[3];
        for (int c = 0; c < 3; ++c) r[c] = x[3 * ijk.z + c] - x[3 * ijk.x + c];
        const double dik = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
        const double ru = dik - p.w;
        e += p.z * ru * ru;
        const double du = 2 * p.z * ru / dik;
        for (int c = 0; c < 3; ++c) { gk[c] += du * r[c]; gi[c] -= du * r[c]; }
      }
      put(ijk.x, 0, gi[0], gi[1], gi[2]);
      put(ijk.y, 1, gj[0], gj[1], gj[2]);
      put(ijk.z, 2, gk[0], gk[1], gk[2]);
      valid = true;
      eslot = d.a_solv[a] ? E_W_ANG : E_P_ANG;
    }
  } else if (t < n3) {  // torsion (md.f90:14793-14907)
    const int a = t - n2;
    w = d.t_win[a];
    if (d.ws[w].active) {
      const int4 q = d.t_ijkl[a];
      const float4 p = d.t_par[a];  // fk, rmult, deltor, paths (1/paths)
      double phi, scp, dp[12];
      torsion_geom(x, q.x, q.y, q.z, q.w, &phi, &scp, dp);
      const double arg = (double)p.y * phi - (double)p.z;
      e = (double)p.x * (1.0 + cos(arg)) * (double)p.w;
      const double dv = -(double)p.y * (double)p.x * sin(arg) * (double)p.w;
      put4(put, q, dv, dp);
      valid = true;
      eslot = d.t_solv[a] ? E_W_TOR : E_P_TOR;
    }
  } else if (t < n4) {  // improper: harmonic (1677-1786) or periodic (1789-1897)
    const int a = t - n3;
    w = d.i_win[a];
    if (d.ws[w].active) {
      const int4 q = d.i_ijkl[a];
      const float2 p = d.i_par[a];
      double phi, scp, dp[12];
      torsion_geom(x, q.x, q.y, q.z, q.w, &phi, &scp, dp);
      double dv;
      if (d.i_kind[w] == 2) {
        const double arg = 2 * phi - (double)p.y;
        e = (double)p.x * (1 + cos(arg));
        dv = -2 * (double)p.x * sin(arg);
      } else {
        const double pi = (double)(4.0f * atanf(1.0f));
        double arg = phi - (double)p.y;
        arg = arg - 2. * pi * round(arg / (2. * pi));
        dv = (double)p.x * arg;
        e = 0.5 * dv * arg;
      }
      put4(put, q, dv, dp);
      valid = true;
      eslot = d.i_solv[a] ? E_W_IMP : E_P_IMP;
    }
  } else if (t < n5) {  // q-bond, Morse + harmonic (md.f90:14060-14114)
    const int a = t - n4;
    const int2 ws2 = d.qb_ws[a];
    w = ws2.x;
    const int s = ws2.y;
    if (d.ws[w].active) {
      const double lam = d.win[w].lambda[s];
      const int2 ij = d.qb_ij[a];
      const double4 p = d.qb_par[a];  // Dmz, amz, r0, fk
      double r[3];
      for (int c = 0; c < 3; ++c) r[c] = x[3 * ij.y + c] - x[3 * ij.x + c];
      const double bl = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
      const double db = bl - p.z;
      const double fexp = exp(-p.y * db);
      e = p.x * (fexp * fexp - 2. * fexp) + 0.5 * p.w * db * db;
      const double dv = (2. * p.x * p.y * (fexp - fexp * fexp) + p.w * db) * lam / bl;
      put(ij.x, 0, -dv * r[0], -dv * r[1], -dv * r[2]);
      put(ij.y, 1, dv * r[0], dv * r[1], dv * r[2]);
      valid = true;
      eslot = E_Q0 + 8 * s + 0;
    }
  } else if (t < n6) {  // q-angle (md.f90:13896-13988)
    const int a = t - n5;
    const int2 ws2 = d.qa_ws[a];
    w = ws2.x;
    const int s = ws2.y;
    if (d.ws[w].active) {
      const int4 ijk = d.qa_ijk[a];
      const double2 p = d.qa_par[a];
      const int i = ijk.x, j = ijk.y, k = ijk.z;
      double rji[3], rjk[3];
      for (int c = 0; c < 3; ++c) { rji[c] = x[3 * i + c] - x[3 * j + c]; rjk[c] = x[3 * k + c] - x[3 * j + c]; }
      const double bji = sqrt(rji[0] * rji[0] + rji[1] * rji[1] + rji[2] * rji[2]);
      const double bjk = sqrt(rjk[0] * rjk[0] + rjk[1] * rjk[1] + rjk[2] * rjk[2]);
      double scp = (rji[0] * rjk[0] + rji[1] * rjk[1] + rji[2] * rjk[2]) / (bji * bjk);
      if (scp > 1.0) scp = 1.0;
      if (scp < -1.0) scp = -1.0;
      const double ang = acos(scp);
      const double da = ang - p.y;
      e = 0.5 * p.x * da * da;
      const double dv = p.x * da * d.win[w].lambda[s];
      double f1 = sin(ang);
      if (fabs(f1) < 1.e-12) f1 = 1.e-12;
      f1 = -1.0 / f1;
      double di[3], dk[3];
      for (int c = 0; c < 3; ++c) {
        di[c] = f1 * (rjk[c] / (bji * bjk) - scp * rji[c] / (bji * bji));
        dk[c] = f1 * (rji[c] / (bji * bjk) - scp * rjk[c] / (bjk * bjk));
      }
      put(i, 0, dv * di[0], dv * di[1], dv * di[2]);
      put(j, 1, -dv * (di[0] + dk[0]), -dv * (di[1] + dk[1]), -dv * (di[2] + dk[2]));
      put(k, 2, dv * dk[0], dv * dk[1], dv * dk[2]);
      valid = true;
      eslot = E_Q0 + 8 * s + 1;
    }
  } else if (t < n8) {  // q-torsion (14262-14403) / q-improper (14117-14258)
    const bool tors = t < n7;
    const int a = tors ? t - n6 : t - n7;
    const int2 ws2 = tors ? d.qt_ws[a] : d.qi_ws[a];
    w = ws2.x;
    const int s = ws2.y;
    if (d.ws[w].active) {
      const int4 q = tors ? d.qt_ijkl[a] : d.qi_ijkl[a];
      double phi, scp, dp[12];
      torsion_geom(x, q.x, q.y, q.z, q.w, &phi, &scp, dp);
      const double lam = d.win[w].lambda[s];
      double dv;
      if (tors) {
        const double4 p = d.qt_par[a];  // fk, rmult, deltor
        const double arg = p.y * phi - p.z;
        e = p.x * (1.0 + cos(arg));
        dv = -p.y * p.x * sin(arg) * lam;
      } else {
        const double pi = (double)(4.0f * atanf(1.0f));
        const double2 p = d.qi_par[a];  // fk, imp0
        double arg = phi - p.y;
        arg = arg - 2. * pi * round(arg / (2. * pi));
        dv = p.x * arg;
        e = 0.5 * dv * arg;
        dv = dv * lam;
      }
      put4(put, q, dv, dp);
      valid = true;
      eslot = E_Q0 + 8 * s + (tors ? 2 : 3);
    }
  }
  put.energy(eslot, e, valid);
}

// Bonded terms in tiles: a block takes the terms of one tile (of one window,
// consecutive by their first atom, at most kBondTileTerms of them, grouped by
// kind so that waves run one kind) and sums their gradients in LDS, per atom
// of the tile's span, and on energy steps their energies, with integer
// atomics; then one atomic add per atom and component goes to the gradient
// and one per energy.  An atom outside the span (a term that reaches further
// than kBondSpan atoms) goes to the gradient directly.
// The term's gradients are recorded per term atom (pos 0..3, a constant at
// each call site, so the record stays in registers) and added to the tile's
// LDS sums after the term, in one loop for every kind.
// Bound by the latency of the terms' FP64 functions and gathers: 64-window
// ladder 33 us alone, force-only or with energies.  On energy steps the terms
// used to write a slot per term atom for a gather kernel (300 MB of traffic, 70
// us alone), because tiles added every term's energy with a global atomic.
struct TermRec {
  int k[4];
  long long g[4][3];
};
struct TileSink {
  TermRec* rec;
  unsigned long long* e;   // LDS energies by slot, or null
  __device__ void operator()(int atom, int pos, double gx, double gy, double gz) const {
    rec->k[pos] = atom;
    rec->g[pos][0] = fix(gx, kFScale);
    rec->g[pos][1] = fix(gy, kFScale);
    rec->g[pos][2] = fix(gz, kFScale);
  }
  // as wave_energy, into LDS
  __device__ void energy(int slot, double v, bool valid) const {
    if (!e) return;   // uniform over the block
    const unsigned long long vm = __ballot(valid);
    if (vm == 0ull) return;
    const int first = __ffsll((long long)vm) - 1;
    const int slot0 = __builtin_amdgcn_readlane(valid ? slot : -1, first);
    const long long ef = valid ? fix(v, kEScale) : 0ll;
    if (__ballot(valid && slot != slot0) == 0ull) {
      const long long sum = wave_sum_i(ef);
      if ((int)(threadIdx.x & 63) == first) atomicAdd(&e[slot0], (unsigned long long)sum);
    } else if (valid) {
      atomicAdd(&e[slot], (unsigned long long)ef);
    }
  }
};

__device__ __forceinline__ void bonded_tile(const Dev& d, int tile, unsigned long long* s_acc, unsigned long long* s_e) {
  const int4 tl = d.btile[tile];   // first entry, terms, first atom, atoms spanned
  const int w = d.wid[tl.z];
  if (!d.ws[w].active) return;     // uniform over the block
  const bool en = d.ws[w].energy_now;
  for (int m = threadIdx.x; m < 3 * tl.w; m += blockDim.x) s_acc[m] = 0ull;
  if ((int)threadIdx.x < E_NSLOT) s_e[threadIdx.x] = 0ull;
  __syncthreads();
  for (int k0 = 0; k0 < tl.y; k0 += blockDim.x) {
    const int k = k0 + (int)threadIdx.x;
    TermRec rec;
#pragma unroll
    for (int p = 0; p < 4; ++p) rec.k[p] = -1;
    bonded_term(d, k < tl.y ? d.btile_terms[tl.x + k] : 0x7fffffff, TileSink{&rec, en ? s_e : nullptr});
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (rec.k[p] < 0) continue;
      const int l = rec.k[p] - tl.z;
      if (l >= 0 && l < kBondSpan) {
        for (int c = 0; c < 3; ++c) atomicAdd(&s_acc[3 * l + c], (unsigned long long)rec.g[p][c]);
      } else {
        add_grad_fix(d.f, rec.k[p], rec.g[p][0], rec.g[p][1], rec.g[p][2]);
      }
    }
  }
  __syncthreads();
  for (int m = threadIdx.x; m < 3 * tl.w; m += blockDim.x)
    if (s_acc[m]) atomicAdd((unsigned long long*)&d.f[3 * (size_t)tl.z + m], s_acc[m]);
  if (en && (int)threadIdx.x < E_NSLOT) add_energy_fix(d.ws, w, threadIdx.x, (long long)s_e[threadIdx.x]);
}
__global__ void __launch_bounds__(256) k_bonded(Dev d) {
  __shared__ unsigned long long s_acc[3 * kBondSpan], s_e[E_NSLOT];
  bonded_tile(d, blockIdx.x, s_acc, s_e);
}

// fixed/shell restraints (fix_shell, md.f90:1414-1450) and the radial
// solvent restraint (restrain_solvent, 14910-14957), per atom
__device__ __forceinline__ void restr_atom(const Dev& d, int i, long long* acc) {
  int w = 0;
  bool en = false, is_fix = false, is_shell = false, is_rad = false;
  double e_fs = 0.0, e_rad = 0.0;
  if (i < d.ntot) {
    w = d.wid[i];
    const WinState& st = d.ws[w];
    const WinDev& W = d.win[w];
    if (st.active) {
      en = st.energy_now;
      const uint8_t fl = d.aflag[i];
      if (fl & 3) {
        const double fk = (fl & 1) ? 200.0 : W.fk_pshell;
        double dr[3];
        for (int c = 0; c < 3; ++c) dr[c] = d.x[3 * i + c] - d.xtop[3 * i + c];
        atom_grad(acc, fk * dr[0], fk * dr[1], fk * dr[2]);
        e_fs = 0.5 * fk * (dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
        is_fix = fl & 1;
        is_shell = fl & 2;
      }
      const int li = i - W.ao;
      if (li >= W.nat_solute && ((li - W.nat_solute) % 3) == 0 && !(fl & 1)) {
        const double shift = (W.fk_wsphere != 0.) ? sqrt((double)0.001986f * st.tfree / W.fk_wsphere) : 0.0;
        double dr[3];
        for (int c = 0; c < 3; ++c) dr[c] = d.x[3 * i + c] - W.xwcent[c];
        const double b = sqrt(dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
        const double db = b - (W.rwat - shift);
        double dv;
        if (db > 0) {
          e_rad = 0.5 * W.fk_wsphere * db * db - W.dwmz;
          dv = W.fk_wsphere * db / b;
        } else if (b > 0.0) {
          const double fexp = exp(W.awmz * db);
          e_rad = W.dwmz * (fexp * fexp - 2. * fexp);
          dv = -2. * W.dwmz * W.awmz * (fexp - fexp * fexp) / b;
        } else {
          dv = 0.0;
        }
        atom_grad(acc, dv * dr[0], dv * dr[1], dv * dr[2]);
        is_rad = true;
      }
    }
  }
  wave_energy(d.ws, w, E_FIX, e_fs, en && is_fix);
  wave_energy(d.ws, w, E_SHELL, e_fs, en && is_shell);
  wave_energy(d.ws, w, E_RAD, e_rad, en && is_rad);
}

// the per-atom terms of a step in one pass: LRF evaluation, then the
// fixed, shell and solvent restraints (one thread per atom; every lane
// reaches the wave energy sums of both).  STORE: the atom's sum of them is
// stored in fterm, which k_integrate adds to the gradient (an MD step, where
// it runs beside the pair kernels); else it completes the gradient of an
// evaluation as the integrator does, after every other kernel
template <bool STORE>
__device__ __forceinline__ void atom_terms(const Dev& d, int i) {
  long long g[3] = {0, 0, 0};
  lrf_taylor_atom(d, i, g);
  restr_atom(d, i, g);
  if (i >= d.ntot || !d.ws[d.wid[i]].active) return;   // (a stopped window keeps its last gradient, which is in fterm)
  if (STORE) {
    for (int c = 0; c < 3; ++c) d.fterm[3 * i + c] = g[c];
  } else {
    const int r = d.rslot[i];
    for (int c = 0; c < 3; ++c) {
      if (r >= 0) g[c] += d.grow[3 * (size_t)r + c] + d.gq[3 * (size_t)r + c];
      d.fterm[3 * i + c] = g[c] + d.f[3 * i + c];
      d.f[3 * i + c] = 0;
    }
  }
}
template <bool STORE>
__global__ void __launch_bounds__(256) k_atom_terms(Dev d) {
  atom_terms<STORE>(d, blockIdx.x * blockDim.x + threadIdx.x);
}

// p_restrain (md.f90:12940-13274): one wave per restraint record.
// Sequence and wall records walk their atom range across the lanes; the
// centre forms first reduce the mean displacement over the block.
// State-dependent records (position, distance, angle) add their energy to
// every state (ipsi 0) or to state ipsi, whose lambda weights the force.
__device__ __forceinline__ void state_restraint_energy(const Dev& d, int w, const WinDev& W, int ipsi, double e) {
  if (ipsi == 0) {
    for (int s = 0; s < W.S; ++s) add_energy(d.ws, w, E_QR0 + s, e);
    if (W.S == 0) add_energy(d.ws, w, E_PROT, e);
  } else {
    add_energy(d.ws, w, E_QR0 + ipsi - 1, e);
  }
}

__device__ __forceinline__ void prestr_wave(const Dev& d, int r) {
  if (r >= d.nrst) return;
  const int4 kwij = d.rs_kwij[r];
  const int kind = kwij.x, w = kwij.y, i0 = kwij.z, j0 = kwij.w;
  if (!d.ws[w].active) return;
  const bool en = d.ws[w].energy_now;
  const WinDev& W = d.win[w];
  const int2 kf = d.rs_kf[r];
  const double* P = &d.rs_par[8 * r];
  const int lane = threadIdx.x & 63;
  if (kind == R_SEQ_ATOMS || kind == R_WALL) {
    double e = 0.0;
    for (int a = i0 + lane; a <= j0; a += 64) {
      if (!((d.aflag[a] & 4) || kf.y == 1)) continue;   // heavy atoms, or all with the H flag
      if (kind == R_SEQ_ATOMS) {
        const double fk = P[0];
        double dr[3];
        for (int c = 0; c < 3; ++c) dr[c] = d.x[3 * a + c] - d.xtop[3 * a + c];
        e += 0.5 * fk * (dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
        add_grad(d.f, a, fk * dr[0], fk * dr[1], fk * dr[2]);
      } else {
        const double fk = P[1], aM = P[2], dM = P[3];
        double dr[3];
        for (int c = 0; c < 3; ++c) dr[c] = d.x[3 * a + c] - W.xwcent[c];
        const double b = sqrt(dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
        const double db = b - P[0];
        double dv;
        if (db > 0.) {
          e += 0.5 * fk * db * db - dM;
          dv = fk * db / b;
        } else {
          const double fexp = exp(aM * db);
          e += dM * (fexp * fexp - 2. * fexp);
          dv = -2. * dM * aM * (fexp - fexp * fexp) / b;
        }
        add_grad(d.f, a, dv * dr[0], dv * dr[1], dv * dr[2]);
      }
    }
    if (en) {
      e = wave_sum(e);
      if (lane == 0) add_energy(d.ws, w, E_PROT, e);
    }
    return;
  }
  if (kind == R_SEQ_GEOM || kind == R_SEQ_MASS) {
    const bool mw = kind == R_SEQ_MASS;
    double sx = 0, sy = 0, sz = 0, sm = 0;
    for (int a = i0 + lane; a <= j0; a += 64) {
      if (!((d.aflag[a] & 4) || kf.y == 1)) continue;
      const double m = mw ? d.mass[a] : 1.0;
      sx += (d.x[3 * a] - d.xtop[3 * a]) * m;
      sy += (d.x[3 * a + 1] - d.xtop[3 * a + 1]) * m;
      sz += (d.x[3 * a + 2] - d.xtop[3 * a + 2]) * m;
      sm += m;
    }
    sx = wave_sum(sx); sy = wave_sum(sy); sz = wave_sum(sz); sm = wave_sum(sm);
    if (!(sm > 0.0)) return;
    const double fk = P[0];
    const double dr[3] = {sx / sm, sy / sm, sz / sm};
    if (en && lane == 0) add_energy(d.ws, w, E_PROT, 0.5 * fk * (dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]));
    for (int a = i0 + lane; a <= j0; a += 64) {
      if (!((d.aflag[a] & 4) || kf.y == 1)) continue;
      if (mw) {
        add_grad(d.f, a, fk * dr[0], fk * dr[1], fk * dr[2]);
      } else {
        // geometric centre: force scaled by mass / 12.010 (a default-real literal)
        const double sc = d.mass[a] / (double)12.010f;
        add_grad(d.f, a, fk * dr[0] * sc, fk * dr[1] * sc, fk * dr[2] * sc);
      }
    }
    return;
  }
  if (lane != 0) return;
  const int ipsi = kf.y;
  const double wgt = ipsi != 0 ? W.lambda[ipsi - 1] : 1.0;
  if (kind == R_POS) {
    double dr[3];
    for (int c = 0; c < 3; ++c) dr[c] = d.x[3 * i0 + c] - P[c];
    const double e = 0.5 * P[3] * dr[0] * dr[0] + 0.5 * P[4] * dr[1] * dr[1] + 0.5 * P[5] * dr[2] * dr[2];
    add_grad(d.f, i0, P[3] * dr[0] * wgt, P[4] * dr[1] * wgt, P[5] * dr[2] * wgt);
    if (en) state_restraint_energy(d, w, W, ipsi, e);
  } else if (kind == R_DIST) {
    double dr[3];
    for (int c = 0; c < 3; ++c) dr[c] = d.x[3 * j0 + c] - d.x[3 * i0 + c];
    const double b = sqrt(dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
    double db;
    if (b < P[0]) db = b - P[0];
    else if (b > P[1]) db = b - P[1];
    else return;
    const double dv = wgt * P[2] * db / b;
    add_grad(d.f, j0, dr[0] * dv, dr[1] * dv, dr[2] * dv);
    add_grad(d.f, i0, -dr[0] * dv, -dr[1] * dv, -dr[2] * dv);
    if (en) state_restraint_energy(d, w, W, ipsi, 0.5 * P[2] * db * db);
  } else if (kind == R_ANGLE) {
    const int k0 = kf.x;
    double a[3], c[3];
    for (int q = 0; q < 3; ++q) {
      a[q] = d.x[3 * i0 + q] - d.x[3 * j0 + q];
      c[q] = d.x[3 * k0 + q] - d.x[3 * j0 + q];
    }
    const double r2ij = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
    const double r2jk = c[0] * c[0] + c[1] * c[1] + c[2] * c[2];
    const double rij = sqrt(r2ij), rjk = sqrt(r2jk);
    double scp = (a[0] * c[0] + a[1] * c[1] + a[2] * c[2]) / (rij * rjk);
    scp = fmin(1.0, fmax(-1.0, scp));
    const double theta = acos(scp);
    const double db = theta - P[0];
    const double dv = wgt * P[1] * db;
    double f1 = sin(theta);
    f1 = fabs(f1) < 1.e-12 ? -1.e12 : -1.0 / f1;
    double di[3], dk[3];
    for (int q = 0; q < 3; ++q) {
      di[q] = f1 * (c[q] / (rij * rjk) - scp * a[q] / r2ij);
      dk[q] = f1 * (a[q] / (rij * rjk) - scp * c[q] / r2jk);
    }
    add_grad(d.f, i0, dv * di[0], dv * di[1], dv * di[2]);
    add_grad(d.f, k0, dv * dk[0], dv * dk[1], dv * dk[2]);
    add_grad(d.f, j0, -dv * (di[0] + dk[0]), -dv * (di[1] + dk[1]), -dv * (di[2] + dk[2]));
    if (en) state_restraint_energy(d, w, W, ipsi, 0.5 * P[1] * db * db);
  }
}

__global__ void __launch_bounds__(64) k_prestr(Dev d) { prestr_wave(d, blockIdx.x); }

// water polarisation restraint (watpol, md.f90:15122-15288), one block per
// (window, shell): the waters whose oxygen lies in the shell are collected in
// LDS with the angle theta between their dipole and the radial vector, each
// one's place in the order of the reference's first-minimum selection sort
// (theta ascending, ties by water index) gives its target angle theta0, energy
// and forces.  The block also advances the shell's theta averages.
//
// Bound by latency and by the one CU a shell has.  The members are ordered
// through buckets of theta: a count, a scan of the buckets' first places, and
// for each member a count of the smaller ones in its own bucket, usually none
// or one.  Counting the smaller ones among all members took n^2 LDS reads: 25 us
// alone for a 1693-water window with 1024 threads and most of the 41 us of a
// step's forces there (512 threads); a step of that window 65.9 -> 53.5 us, of a
// 1109-water one 43.6 -> 41.1, of 16 of the first 187 -> 181, of the 64-window
// ladder 445 -> 441.
__device__ __forceinline__ void water_dipole(const double* x, int i, const double cent[3], double rmu[3], double rcu[3],
                                             double* rm, double* rc) {
  for (int c = 0; c < 3; ++c) rmu[c] = x[3 * (i + 1) + c] + x[3 * (i + 2) + c] - 2. * x[3 * i + c];
  *rm = sqrt(rmu[0] * rmu[0] + rmu[1] * rmu[1] + rmu[2] * rmu[2]);
  for (int c = 0; c < 3; ++c) rmu[c] /= *rm;
  for (int c = 0; c < 3; ++c) rcu[c] = x[3 * i + c] - cent[c];
  *rc = sqrt(rcu[0] * rcu[0] + rcu[1] * rcu[1] + rcu[2] * rcu[2]);
  for (int c = 0; c < 3; ++c) rcu[c] /= *rc;
}
// cosine of the angle between the unit vectors, clipped to [-1, 1]
__device__ __forceinline__ double dipole_cos(const double rmu[3], const double rcu[3]) {
  const double scp = rmu[0] * rcu[0] + rmu[1] * rcu[1] + rmu[2] * rcu[2];
  return fmin(1.0, fmax(-1.0, scp));
}
// energy and forces of water atom group i (its oxygen) at place `rank` of the
// n members of its shell
__device__ __forceinline__ double watpol_force(const Dev& d, const WinDev& W, float cstb_f, float corr_f, int n, int i,
                                               int rank, double th) {
  const double pi = (double)(4.0f * atanf(1.0f));
  const double cstb = (double)cstb_f, tc = (double)corr_f;
  const int il = rank + 1;
  const float argf = 1.0f + (1.0f - 2.0f * (float)il) / (float)n;
  double th0 = acos((double)argf);
  th0 = th0 - 3. * sin(th0) * cstb / 2.;
  th0 = fmin(fmax(th0, 0.0), pi);
  const double dth = th - th0 + tc;
  const double dv = W.fkwpol * dth;
  double rmu[3], rcu[3], rm, rc;
  water_dipole(d.x, i, W.xwcent, rmu, rcu, &rm, &rc);
  const double scp = dipole_cos(rmu, rcu);
  double f0 = sin(acos(scp));
  if (fabs(f0) < 1.e-12) f0 = 1.e-12;
  f0 = dv * (-1.0 / f0);
  double f1[3], f2[3];
  for (int c = 0; c < 3; ++c) {
    f1[c] = (rcu[c] - rmu[c] * scp) / rm;
    f2[c] = (rmu[c] - rcu[c] * scp) / rc;
  }
  add_grad(d.f, i, f0 * (-2. * f1[0] + f2[0]), f0 * (-2. * f1[1] + f2[1]), f0 * (-2. * f1[2] + f2[2]));
  add_grad(d.f, i + 1, f0 * f1[0], f0 * f1[1], f0 * f1[2]);
  add_grad(d.f, i + 2, f0 * f1[0], f0 * f1[1], f0 * f1[2]);
  return 0.5 * W.fkwpol * dth * dth;
}

constexpr int kWpolSum = 256;        // threads of the theta sum (its order is part of the result)
constexpr int kWpolBuckets = 1024;   // of the ordering by theta
// (any monotone function of theta orders correctly)
__device__ __forceinline__ int wpol_bucket(double th) {
  return min(max((int)(th * (kWpolBuckets / 3.1415926535897932)), 0), kWpolBuckets - 1);
}
template <int kWpolBlock>            // threads per (window, shell) block
struct WpolLds {
  double th[kWpolLds];
  int iw[kWpolLds], start[kWpolBuckets], wsum[kWpolBlock / 64];
  int n;
  float corr;
  double red[kWpolSum / 64];
};
template <int kWpolBlock>
__device__ __forceinline__ void watpol_block(const Dev& d, int block, WpolLds<kWpolBlock>& L) {
  constexpr int kWpolHeld = kWpolLds / kWpolBlock;   // members per thread of a shell held in LDS
  const int w = block / kWpolMaxShell, is = block % kWpolMaxShell;
  if (w >= d.nwin) return;
  const WinState& st = d.ws[w];
  const WinDev& W = d.win[w];
  const int nsh = W.nshell;
  if (!st.active || !W.wpol || W.nwat == 0 || is >= nsh) return;
  const ShellDev* shells = d.shells + W.sh_off;
  ShellDev& sh = d.shells[W.sh_off + is];
  double *s_th = L.th, *s_red = L.red;
  int *s_iw = L.iw, *s_start = L.start;
  int& s_n = L.n;
  float& s_corr = L.corr;
  const int t = threadIdx.x;
  // theta_corr follows the shell's mean theta every 100 steps; only the
  // pot_energy calls of the run (MD steps and the final evaluation) advance
  // the shell averages, so extra evaluations (tuning, queries) leave them
  if (t == 0) {
    if (st.wpol_acc && st.istep != 0 && st.istep % 100 == 0) {
      sh.avtheta = sh.avtheta / 100.0f;
      sh.avn_insh = sh.avn_insh / 100.0f;
      sh.theta_corr = sh.theta_corr + sh.avtheta - acosf(sh.cstb);
      sh.avtheta = 0.0f;
      sh.avn_insh = 0.0f;
    }
    s_corr = sh.theta_corr;
    s_n = 0;
  }
  for (int b = t; b < kWpolBuckets; b += kWpolBlock) s_start[b] = 0;
  __syncthreads();
  // the shell's bounds: waters beyond the innermost radius (a single-precision
  // difference, as the bounds are real(4)) lie in the innermost shell whose
  // outer radius holds them, the rest in shell 0
  const double r_in = (double)(shells[nsh - 1].rout - shells[nsh - 1].dr);
  const double r_out = is > 0 ? (double)sh.rout : 1e300;
  const double r_next = is < nsh - 1 ? (double)shells[is + 1].rout : r_in;
  const int o0 = W.ao + W.nat_solute;
  // a window whose shells could outgrow LDS has a row of its waters' angles
  // per shell in memory (-1: not in the shell)
  double* row = W.nwat > kWpolLds ? d.wtheta + W.wp_off + (size_t)is * W.nwat : nullptr;
  for (int iw = t; iw < W.nwat; iw += kWpolBlock) {
    const int i = o0 + 3 * iw;
    if (row) row[iw] = -1.0;
    if (d.aflag[i] & 1) continue;
    double c[3];
    for (int k = 0; k < 3; ++k) c[k] = d.x[3 * i + k] - W.xwcent[k];
    const double rc = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
    if (!(rc > r_in && rc > r_next && rc <= r_out)) continue;
    double rmu[3], rcu[3], rm, rd;
    water_dipole(d.x, i, W.xwcent, rmu, rcu, &rm, &rd);
    const double th = acos(dipole_cos(rmu, rcu));
    if (row) row[iw] = th;
    const int k = atomicAdd(&s_n, 1);
    if (k < kWpolLds) { s_th[k] = th; s_iw[k] = iw; }
  }
  __syncthreads();
  const int n = s_n;
  const bool in_lds = n <= kWpolLds;
  double th[kWpolHeld];
  int iw[kWpolHeld], rank[kWpolHeld];
  if (in_lds) {
    // members per bucket, and each member's place among its bucket's (in any
    // order)
#pragma unroll
    for (int m = 0; m < kWpolHeld; ++m) {
      const int k = t + kWpolBlock * m;
      rank[m] = -1;
      if (k >= n) continue;
      th[m] = s_th[k];
      iw[m] = s_iw[k];
      rank[m] = atomicAdd(&s_start[wpol_bucket(th[m])], 1);
    }
    __syncthreads();
    // the buckets' first places
    constexpr int kPer = kWpolBuckets / kWpolBlock;
    int c[kPer], sum = 0;
    for (int q = 0; q < kPer; ++q) {
      c[q] = s_start[kPer * t + q];
      sum += c[q];
    }
    int incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o);
      if ((t & 63) >= o) incl += v;
    }
    if ((t & 63) == 63) L.wsum[t >> 6] = incl;
    __syncthreads();
    int first = incl - sum;
    for (int q = 0; q < (t >> 6); ++q) first += L.wsum[q];
    for (int q = 0; q < kPer; ++q) {
      s_start[kPer * t + q] = first;
      first += c[q];
    }
    __syncthreads();
    // the members by bucket
#pragma unroll
    for (int m = 0; m < kWpolHeld; ++m) {
      if (rank[m] < 0) continue;
      const int k = s_start[wpol_bucket(th[m])] + rank[m];
      s_th[k] = th[m];
      s_iw[k] = iw[m];
    }
    __syncthreads();
    // a member's rank: its bucket's first place and the smaller ones of its
    // bucket (at the same angle the lower water)
#pragma unroll
    for (int m = 0; m < kWpolHeld; ++m) {
      if (rank[m] < 0) continue;
      const int b = wpol_bucket(th[m]), j0 = s_start[b], j1 = b + 1 < kWpolBuckets ? s_start[b + 1] : n;
      int r = j0;
      for (int j = j0; j < j1; ++j) {
        const double tj = s_th[j];
        r += tj < th[m] || (tj == th[m] && s_iw[j] < iw[m]) ? 1 : 0;
      }
      rank[m] = r;
    }
    __syncthreads();
    // the members in order
#pragma unroll
    for (int m = 0; m < kWpolHeld; ++m) {
      if (rank[m] < 0) continue;
      s_th[rank[m]] = th[m];
      s_iw[rank[m]] = iw[m];
    }
    __syncthreads();
  }
  // the shell's theta sum in a fixed order: members in their order (or, from
  // memory, in water order), over kWpolSum threads, the waves, the wave sums
  if (t < kWpolSum) {
    double tsum = 0.0;
    if (in_lds) {
      for (int k = t; k < n; k += kWpolSum) tsum += s_th[k];
    } else {
      for (int k = t; k < W.nwat; k += kWpolSum) tsum += row[k] >= 0.0 ? row[k] : 0.0;
    }
    tsum = wave_sum(tsum);
    if ((t & 63) == 0) s_red[t >> 6] = tsum;
  }
  __syncthreads();
  if (t == 0) {
    if (n > 0 && st.wpol_acc) {
      const double avtdum = (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
      // real(4) + real(8) quotient, rounded once (md.f90:15285)
      sh.avtheta = (float)((double)sh.avtheta + avtdum / (double)(float)n);
      sh.avn_insh = sh.avn_insh + (float)n;
    }
    sh.n_insh = n;
  }
  // forces, every lane to the energy sum
  const int nloop = in_lds ? n : W.nwat;
  const bool en = st.energy_now;
  for (int k0 = 0; k0 < nloop; k0 += kWpolBlock) {
    const int k = k0 + t;
    double e = 0.0;
    bool on = k < nloop;
    if (on && in_lds) {
      e = watpol_force(d, W, sh.cstb, s_corr, n, o0 + 3 * s_iw[k], k, s_th[k]);
    } else if (on) {
      const double tk = row[k];
      on = tk >= 0.0;
      if (on) {
        int r = 0;
        for (int j = 0; j < W.nwat; ++j) {
          const double tj = row[j];
          r += tj >= 0.0 && (tj < tk || (tj == tk && j < k)) ? 1 : 0;
        }
        e = watpol_force(d, W, sh.cstb, s_corr, n, o0 + 3 * k, r, tk);
      }
    }
    wave_energy(d.ws, w, E_WPOL, e, on && en);
  }
}
__global__ void __launch_bounds__(1024) k_watpol(Dev d) {
  __shared__ WpolLds<1024> L;
  watpol_block<1024>(d, blockIdx.x, L);
}

// ------------------------------------------------ all forces at once --
// Engines whose step is too small to fill the GPU run every force kernel of a
// step as one launch, each block taking one kind of work (by block index, the
// longest kinds first): a step then takes as long as its slowest kind, where
// separate launches add up with the gaps between them.
// us a step, nine launches and one: one ligand-in-water window 75 and 53, one
// protein window 107 and 74, 11 small windows 97 and 68.  128 registers (the
// bonded terms spill 42) keep two blocks on a CU.
constexpr int kAllBlock = 512;       // 8 waves: two q items, 8 row clusters
// an engine of more blocks fills the GPU with the launches of a large engine
// (k_pairs), whose pair waves need fewer registers, so that more of them are in
// flight.  us a step, one launch and those: 11 small windows (550 blocks) 55 and
// 72, 4 protein windows (660) 82 and 89, 20 small windows (1000) 78 and 87, 8
// protein windows (1330) 120 and 115, 32 small windows (1600) 105 and 109, 16
// protein windows 209 and 181.  The results do not depend on it
constexpr int kAllMost = 1200;
struct AllPlan {
  int wpol, bonded, qp, qw, srow, wrow, qq, rst, terms;   // first block of each kind
  int total;
};
static AllPlan all_plan(const Dev& d, bool energy, bool terms) {
  AllPlan p;
  int n = 0;
  auto take = [&](int& first, long long work, int per_block) {
    first = n;
    n += (int)((work + per_block - 1) / per_block);
  };
  const int waves = kAllBlock / 64;
  take(p.wpol, d.nwat_total ? (long long)d.nwin * kWpolMaxShell : 0, 1);
  take(p.bonded, d.nbtile, 1);
  take(p.qp, d.nqp_work, waves / kQWaves);
  take(p.qw, d.nqw_work, waves / kQWaves);
  take(p.srow, d.rl[T_PP].nicl, waves);
  take(p.wrow, d.rl[T_WW].nicl, waves);
  take(p.qq, qq_waves(d, energy), waves);
  take(p.rst, d.nrst, waves);
  take(p.terms, terms ? d.ntot : 0, kAllBlock);
  p.total = n;
  return p;
}
template <bool W3, bool EK>
__global__ void __launch_bounds__(kAllBlock, 4) k_all(Dev d, AllPlan p) {
  __shared__ union {
    WpolLds<kAllBlock> wpol;
    struct { unsigned long long acc[3 * kBondSpan], e[E_NSLOT]; } bonded;
    long long q[kAllBlock / (64 * kQWaves)][9 * 64 * kQWaves];
  } L;
  const int b = blockIdx.x, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  constexpr int kWaves = kAllBlock / 64, kItems = kWaves / kQWaves;
  const int group = wv / kQWaves;
  if (b >= p.terms) return atom_terms<true>(d, (b - p.terms) * kAllBlock + (int)threadIdx.x);
  if (b >= p.rst) return prestr_wave(d, (b - p.rst) * kWaves + wv);
  if (b >= p.qq) return qq_wave<EK>(d, (b - p.qq) * kWaves + wv);
  if (b >= p.wrow) return wrow_wave<W3, EK, 3>(d, (b - p.wrow) * kWaves + wv);
  if (b >= p.srow) return srow_wave<W3, EK>(d, (b - p.srow) * kWaves + wv);
  if (b >= p.qw) return qw_group<W3, EK>(d, (b - p.qw) * kItems + group, L.q[group]);
  if (b >= p.qp) return qp_group<EK>(d, (b - p.qp) * kItems + group, L.q[group]);
  if (b >= p.bonded) return bonded_tile(d, b - p.bonded, L.bonded.acc, L.bonded.e);
  watpol_block<kAllBlock>(d, b, L.wpol);
}

// -------------------------------------------- forces of a large engine --
// A step of an engine that fills the GPU takes two launches, side by side: the
// pair forces with the per-atom terms, whose waves need few registers and
// issue most of the step's instructions, and the few latency-bound blocks of
// the water polarisation with the bonded terms.  The rows come first, which
// run longest, then the q items, then the short waves that fill the end.
// As nine launches on three streams the kernels queued behind each other on
// each stream and the last ones ran with the GPU half empty: 16 + 16 windows
// 264 us a step, now 233, 32 protein windows 393 and 378, the 64-window ladder
// 485 and 473.  The q items first: 244, 384, 475.  The bonded terms as a
// kernel of their own behind the polarisation: 245, 396, 479; on a third
// stream 258, 407, 496.
struct PairPlan {
  int srow, qw, qp, qq, terms;   // first block of each kind; the water rows come first
  int total;
};
constexpr int kPairBlock = 64 * kQWaves;   // a q item, 4 row clusters
static PairPlan pair_plan(const Dev& d, bool energy, bool terms) {
  PairPlan p;
  int n = 0;
  auto take = [&](int& first, long long work, int per_block) {
    first = n;
    n += (int)((work + per_block - 1) / per_block);
  };
  const int waves = kPairBlock / 64;
  int wrow;
  take(wrow, d.rl[T_WW].nicl, waves);
  take(p.srow, d.rl[T_PP].nicl, waves);
  take(p.qw, d.nqw_work, 1);
  take(p.qp, d.nqp_work, 1);
  take(p.qq, qq_waves(d, energy), waves);
  take(p.terms, terms ? d.ntot : 0, kPairBlock);
  p.total = n;
  return p;
}
// (windows with a 3-atom solvent have instances of the row and q kernels of
// their own, launched after this one)
template <bool EK>
__global__ void __launch_bounds__(kPairBlock, EK ? 4 : 6) k_pairs(Dev d, PairPlan p) {
  __shared__ long long s_q[9 * 64 * kQWaves];
  const int b = blockIdx.x, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  constexpr int kWaves = kPairBlock / 64;
  if (b >= p.terms) return atom_terms<true>(d, (b - p.terms) * kPairBlock + (int)threadIdx.x);
  if (b >= p.qq) return qq_wave<EK>(d, (b - p.qq) * kWaves + wv);
  if (b >= p.qp) return qp_group<EK>(d, b - p.qp, s_q);
  if (b >= p.qw) return qw_group<false, EK>(d, b - p.qw, s_q);
  if (b >= p.srow) return srow_wave<false, EK>(d, (b - p.srow) * kWaves + wv);
  wrow_wave<false, EK, 3>(d, b * kWaves + wv);
}
// polarisation blocks first: they take longest
__global__ void __launch_bounds__(256) k_other(Dev d, int nwp) {
  __shared__ union {
    WpolLds<256> wpol;
    struct { unsigned long long acc[3 * kBondSpan], e[E_NSLOT]; } bonded;
  } L;
  const int b = blockIdx.x;
  if (b >= nwp) return bonded_tile(d, b - nwp, L.bonded.acc, L.bonded.e);
  watpol_block<256>(d, b, L.wpol);
}

// the FP32 coordinates of atom i from its FP64 ones, into x32 and, for a
// water or solute atom, into its cluster slot (with the FP64 ones), for a q-atom
// into its q-cluster slot
__device__ __forceinline__ void store_copies(const Dev& d, int i, int ws, int qs, float q, double x, double y, double z) {
  const float4 n = make_float4((float)x, (float)y, (float)z, q);
  d.x32[i] = n;
  if (ws >= 0) {
    d.xw[ws] = n;
    d.xwd[ws] = make_double4(x, y, z, 0.0);
  }
  if (qs >= 0) d.xq[qs] = n;
}
__device__ __forceinline__ void store_x32(const Dev& d, int i) {
  store_copies(d, i, d.wslot[i], d.qmslot[i], d.x32[i].w, d.x[3 * i], d.x[3 * i + 1], d.x[3 * i + 2]);
}

// ------------------------------------------------------- integrator --
// The end of a step in one kernel, k_integrate: the leapfrog of every atom,
// the SHAKE sweeps of every constraint component, v = (x - xx)/dt and the
// kinetic energy.  Every atom's arithmetic is that of the reference's three
// loops in their order; only the kinetic-energy sum goes to fixed point.

// leapfrog (md.f90:4081-4111) of atom i with gradient gfix (fixed point):
// v = (v - d*winv*dt)*Tscale; xx = x; x += v*dt, into x[], xx[], v[]
__device__ __forceinline__ void leapfrog_vals(const Dev& d, double ts, double wi, double dt, int i,
                                              const long long gfix[3], double x[3], double xx[3], double v[3]) {
#pragma clang fp contract(off)
  for (int c = 0; c < 3; ++c) {
    const int k = 3 * i + c;
    const double g = (double)gfix[c] * (1.0 / kFScale);
    v[c] = (d.v[k] - g * wi * dt) * ts;
    xx[c] = d.x[k];
    x[c] = xx[c] + v[c] * dt;
  }
}

// gradient of atom i (entry r of the row buffers) for the integrator: the
// step's per-atom terms (LRF evaluation, fixed/shell and radial solvent
// restraints, stored by k_atom_terms<true>), the row kernels' and q kernels'
// sums, and the gradient the other kernels added up, which is cleared for the
// next step where there was any; the complete gradient takes the place of the
// per-atom terms
__device__ __forceinline__ void step_gradient(const Dev& d, int i, int r, long long g[3]) {
  long long f[3];
  for (int c = 0; c < 3; ++c) {
    f[c] = d.f[3 * i + c];
    g[c] = d.fterm[3 * i + c] + f[c];
    if (r >= 0) g[c] += d.grow[3 * (size_t)r + c] + d.gq[3 * (size_t)r + c];
  }
  for (int c = 0; c < 3; ++c) {
    d.fterm[3 * i + c] = g[c];
    if (f[c]) d.f[3 * i + c] = 0;
  }
}

// SHAKE (md.f90:14445-14566): one thread per connected component of a
// molecule's constraint graph; components share no atoms, so iterating them
// separately gives the reference's result for the whole molecule.
// Constraints are swept in order, Gauss-Seidel, until every one is within
// tol*d0^2 (at most 1000 sweeps).
// a unit whose coordinates are in LDS (sx new, sxx old, its atoms numbered
// as sc_loc numbers them), any size.  Units of at most kShakeHeld
// constraints (the waters' three) take theirs from a ShakeHeld loaded
// before (at the start of the integrator, so the loads overlap its first
// phase) and hold the old-coordinate differences in registers over the
// sweeps; larger ones load each constraint per sweep.  The sums are the same
// either way.
constexpr int kShakeHeld = 3;
struct ShakeHeld {
  int li[kShakeHeld], lj[kShakeHeld];
  double d2[kShakeHeld];
  float2 w[kShakeHeld];
};
__device__ __forceinline__ void shake_hold(const Dev& d, int c0, int nc, ShakeHeld& h) {
#pragma unroll
  for (int c = 0; c < kShakeHeld; ++c) {
    const bool on = c < nc;
    h.li[c] = on ? d.sc_loc[2 * (c0 + c)] : 0;
    h.lj[c] = on ? d.sc_loc[2 * (c0 + c) + 1] : 0;
    h.d2[c] = on ? d.sc_d2[c0 + c] : 0.0;
    h.w[c] = on ? d.sc_w[c0 + c] : make_float2(0.f, 0.f);
  }
}
template <bool HELD>
__device__ __forceinline__ void shake_lds(const Dev& d, WinState& st, int c0, int nc, double (*sx)[3],
                                          const double (*sxx)[3], const ShakeHeld& h) {
#pragma clang fp contract(off)
  const double tol = (double)0.0001f;
  unsigned long long ready = 0ull;  // up to 64 constraints per component
  const unsigned long long all = nc >= 64 ? ~0ull : ((1ull << nc) - 1ull);
  double hxx[HELD ? kShakeHeld : 1][3];
  if (HELD) {
#pragma unroll
    for (int c = 0; c < kShakeHeld; ++c)
      for (int k = 0; k < 3; ++k) hxx[c][k] = c < nc ? sxx[h.li[c]][k] - sxx[h.lj[c]][k] : 0.0;
  }
  // one constraint: the correction of the Gauss-Seidel sweep
  auto fix_pair = [&](int c, int li, int lj, double d2, const double xxij[3], float wvi, float wvj) {
#pragma clang fp contract(off)
    double xij[3];
    for (int k = 0; k < 3; ++k) xij[k] = sx[li][k] - sx[lj][k];
    const double xij2 = xij[0] * xij[0] + xij[1] * xij[1] + xij[2] * xij[2];
    const double diff = d2 - xij2;
    if (fabs(diff) < tol * d2) ready |= 1ull << c;
    const double scp = xij[0] * xxij[0] + xij[1] * xxij[1] + xij[2] * xxij[2];
    const float wsum = wvi + wvj;
    const double corr = diff / (2. * scp * (double)wsum);
    const double wi = (double)wvi, wj = (double)wvj;
    for (int k = 0; k < 3; ++k) {
      sx[li][k] = sx[li][k] + xxij[k] * corr * wi;
      sx[lj][k] = sx[lj][k] - xxij[k] * corr * wj;
    }
  };
  int nits = 0;
  while (true) {
    if constexpr (HELD) {
#pragma unroll
      for (int c = 0; c < kShakeHeld; ++c)
        if (c < nc && !(ready & (1ull << c))) fix_pair(c, h.li[c], h.lj[c], h.d2[c], hxx[c], h.w[c].x, h.w[c].y);
    } else {
      for (int c = 0; c < nc; ++c) {
        if (ready & (1ull << c)) continue;
        const int li = d.sc_loc[2 * (c0 + c)], lj = d.sc_loc[2 * (c0 + c) + 1];
        const float2 wv = d.sc_w[c0 + c];
        double xxij[3];
        for (int k = 0; k < 3; ++k) xxij[k] = sxx[li][k] - sxx[lj][k];
        fix_pair(c, li, lj, d.sc_d2[c0 + c], xxij, wv.x, wv.y);
      }
    }
    ++nits;
    if ((ready & all) == all) break;
    if (nits >= 1000) { st.shake_fail = 1; break; }
  }
}

// the same for a unit of three constraints among three atoms (every water),
// in registers: the same arithmetic in the same order (a difference taken the
// other way round only changes signs that cancel)
__device__ __forceinline__ bool shake_tri(const double d2[3], const float w[3], const double xx[3][3], double x[3][3]) {
#pragma clang fp contract(off)
  const double tol = (double)0.0001f;
  constexpr int ci[3] = {0, 0, 1}, cj[3] = {1, 2, 2};
  double o[3][3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    for (int k = 0; k < 3; ++k) o[c][k] = xx[ci[c]][k] - xx[cj[c]][k];
  unsigned ready = 0;
  for (int nits = 1;; ++nits) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (ready & (1u << c)) continue;
      const int i = ci[c], j = cj[c];
      double xij[3];
      for (int k = 0; k < 3; ++k) xij[k] = x[i][k] - x[j][k];
      const double xij2 = xij[0] * xij[0] + xij[1] * xij[1] + xij[2] * xij[2];
      const double diff = d2[c] - xij2;
      if (fabs(diff) < tol * d2[c]) ready |= 1u << c;
      const double scp = xij[0] * o[c][0] + xij[1] * o[c][1] + xij[2] * o[c][2];
      const float wsum = w[i] + w[j];
      const double corr = diff / (2. * scp * (double)wsum);
      const double wi = (double)w[i], wj = (double)w[j];
      for (int k = 0; k < 3; ++k) {
        x[i][k] = x[i][k] + o[c][k] * corr * wi;
        x[j][k] = x[j][k] - o[c][k] * corr * wj;
      }
    }
    if (ready == 7u) return true;
    if (nits >= 1000) return false;
  }
}

// kinetic energy of the step (md.f90:3813-3830): the lanes' fixed-point sums
// added to their window's accumulators, one wave sum and one atomic each when
// all valid lanes hold the same window.  Integer sums: the result does not
// depend on the order.  Every lane calls it.
__device__ __forceinline__ void wave_ekin(const Dev& d, int w, const long long ek[4], bool valid) {
  const unsigned long long vm = __ballot(valid);
  if (vm == 0ull) return;
  const int first = __ffsll((long long)vm) - 1;
  const int w0 = __builtin_amdgcn_readlane(valid ? w : -1, first);   // first is uniform over the wave
  const bool uniform = __ballot(valid && w != w0) == 0ull;
  for (int c = 0; c < 4; ++c) {
    if (uniform) {
      const long long s = wave_sum_i(valid ? ek[c] : 0ll);
      if ((int)(threadIdx.x & 63) == first && s != 0)
        atomicAdd((unsigned long long*)&d.ws[w0].ekin_fix[c], (unsigned long long)s);
    } else if (valid && ek[c] != 0) {
      atomicAdd((unsigned long long*)&d.ws[w].ekin_fix[c], (unsigned long long)ek[c]);
    }
  }
}

// (outside the integrator's contract(off): its sum is fused)
__device__ __forceinline__ double kinetic(double mass, const double v[3]) {
  return 0.5 * mass * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
}

// k_integrate: one block per run of whole integration units (Dev::ib), in
// three phases.  1: one atom per thread, its gradient and leapfrog, the new
// and old coordinates into LDS.  2: one unit per thread, the SHAKE sweeps,
// in registers for three constraints among three atoms, else on the unit's
// coordinates in LDS.  3: one atom per thread again: v = (x - xx)/dt when
// `post` (md.f90:4117-4120), the copies of x, the kinetic energy (solute all,
// solute free, solvent all, solvent free).
// For one window it is a chain of dependent loads and sweeps, for many it is
// bound by memory: what it needs of an atom stands in one record in the order
// of the entries, so that the coordinates and gradients are one load away, and
// nothing is loaded after the sweeps.  One ligand-in-water window 16 -> 11 us,
// the 64-window ladder 69 -> 52.
__global__ void __launch_bounds__(kIntBlock) k_integrate(Dev d, int post) {
#pragma clang fp contract(off)
  __shared__ double s_x[kIntBlock][3], s_xx[kIntBlock][3];
  __shared__ int s_on[kIntBlock];
  const int4 B = d.ib[blockIdx.x];   // first entry, atoms, first unit, units
  const int t = threadIdx.x;
  // the thread's SHAKE unit of the second phase and its constraints
  int tri = 0, c0 = 0, nc = 0;
  int4 U = make_int4(0, 0, 0, -1);   // window, first entry, atoms, SHAKE unit
  ShakeHeld h;
  double d2[3] = {0, 0, 0};
  float wt[3] = {0, 0, 0};
  if (t < B.w) {
    const float4 p = d.tri[B.z + t];
    tri = __float_as_int(p.w);
    wt[0] = p.x; wt[1] = p.y; wt[2] = p.z;
    for (int k = 0; k < 3; ++k) d2[k] = d.tri_d2[3 * (B.z + t) + k];
    U = d.iu[B.z + t];
    if (!tri && U.w >= 0) {
      c0 = d.su_start[U.w];
      nc = d.su_n[U.w];
    }
  }
  shake_hold(d, c0, nc, h);
  int4 A = make_int4(d.ntot, 0, -1, -1);   // atom, window, row entry, slot
  float4 P = make_float4(0.f, 0.f, 0.f, 0.f);
  double mass = 0.0;
  bool on = false;
  if (t < B.y) {
    A = d.ie_i[B.x + t];
    P = d.ie_f[B.x + t];
    mass = d.ie_m[B.x + t];
    on = d.ws[A.y].active;
  }
  const int i = A.x, fl = __float_as_int(P.w);
  const WinState& st = d.ws[A.y];
  const double dt = d.win[A.y].dt;
  double x[3], xx[3], v[3];
  if (on) {
    const double ts = fl & 1 ? st.tscale_solute : st.tscale_solvent;
    long long g[3];
    step_gradient(d, i, A.z, g);
    leapfrog_vals(d, ts, (double)P.y, dt, i, g, x, xx, v);
    for (int c = 0; c < 3; ++c) {
      s_x[t][c] = x[c];
      s_xx[t][c] = xx[c];
    }
  }
  s_on[t] = on;
  __syncthreads();
  if (tri) {
    const int l0 = tri & kTriFirst, l[3] = {l0 + (tri >> kTriA & 3), l0 + (tri >> kTriB & 3), l0 + (tri >> kTriC & 3)};
    if (s_on[l0]) {
      double xs[3][3], os[3][3];
#pragma unroll
      for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 3; ++c) {
          xs[a][c] = s_x[l[a]][c];
          os[a][c] = s_xx[l[a]][c];
        }
      if (!shake_tri(d2, wt, os, xs)) d.ws[U.x].shake_fail = 1;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 3; ++c) s_x[l[a]][c] = xs[a][c];
    }
  } else if (nc > 0 && s_on[U.y - B.x]) {
    WinState& su = d.ws[U.x];
    const int l0 = U.y - B.x;
    if (nc <= kShakeHeld) shake_lds<true>(d, su, c0, nc, &s_x[l0], &s_xx[l0], h);
    else shake_lds<false>(d, su, c0, nc, &s_x[l0], &s_xx[l0], h);
  }
  __syncthreads();
  long long ek[4] = {0, 0, 0, 0};
  if (on) {
    for (int c = 0; c < 3; ++c) {
      x[c] = s_x[t][c];
      d.x[3 * i + c] = x[c];
      if (post) v[c] = (x[c] - xx[c]) / dt;
      d.v[3 * i + c] = v[c];
    }
    store_copies(d, i, A.w, __float_as_int(P.z), P.x, x[0], x[1], x[2]);
    const long long e = fix(kinetic(mass, v), kEScale);
    const bool solute = fl & 1, freeat = !(fl & 2);
    ek[0] += solute ? e : 0ll;
    ek[1] += solute && freeat ? e : 0ll;
    ek[2] += solute ? 0ll : e;
    ek[3] += !solute && freeat ? e : 0ll;
  }
  wave_ekin(d, A.y, ek, on);
}

// FP32 coordinates (and their slot copies) from the FP64 ones, after a
// state upload
__global__ void k_refresh32(Dev d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < d.ntot) store_x32(d, i);
}

// temperature and Berendsen scaling factors (md.f90:3813-3914) outside the
// step (at the start of a run, after a state upload): kTempParts blocks per
// window sum strided atoms (solute, solute free, solvent, solvent free) and
// store the block's partials; k_temperature adds the partials in part order,
// so the sum does not depend on scheduling.  Inside the step k_integrate
// sums the kinetic energy instead.
__global__ void __launch_bounds__(256) k_ekin_part(Dev d) {
  const int w = blockIdx.x / kTempParts, part = blockIdx.x % kTempParts;
  if (w >= d.nwin) return;
  const WinDev& W = d.win[w];
  double acc[4] = {0, 0, 0, 0};  // solute, solute free, solvent, solvent free
  for (int li = part * blockDim.x + threadIdx.x; li < W.natom; li += kTempParts * blockDim.x) {
    const int i = W.ao + li;
    const double* v = &d.v[3 * i];
    const double ek = 0.5 * d.mass[i] * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    const bool solute = li < W.nat_solute;
    const bool freeat = !(d.aflag[i] & 1);
    acc[solute ? 0 : 2] += ek;
    if (freeat) acc[solute ? 1 : 3] += ek;
  }
  __shared__ double red[4][4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int k = 0; k < 4; ++k) {
    double s = wave_sum(acc[k]);
    if (lane == 0) red[wv][k] = s;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += red[q][threadIdx.x];
    d.t_part[((size_t)w * kTempParts + part) * 4 + threadIdx.x] = t;
  }
}

// temperatures and Berendsen factors (one wave per window) from the
// kinetic-energy partials of k_ekin_part, or with `advance` (the end of a
// step) from the fixed-point sums of k_integrate, which it clears for the
// next step; with `advance` also the ring records of the step, the step
// count, and the start of the next step (begin_step).  The lanes copy the
// energy accumulators into the step's ring slot, lane 0 does the rest.
// `variant`: what the step launched, bit 0 the list kernels, bit 1 the kernel
// instances with energy terms; a window that needed more is flagged.
__global__ void __launch_bounds__(64) k_temperature(Dev d, int advance, int variant) {
  const int w = blockIdx.x;
  if (w >= d.nwin) return;
  WinState& st = d.ws[w];
  const WinDev& W = d.win[w];
  if (!st.active && advance) return;   // uniform over the block
  if (advance && st.energy_now) {
    const int slot = (st.istep - st.ring_base) % d.ring_n;
    long long* er = &d.e_ring[((size_t)slot * d.nwin + w) * E_NSLOT];
    for (int k = threadIdx.x; k < E_NSLOT; k += blockDim.x) er[k] = st.E[k];
  }
  __syncthreads();   // every lane has read istep before lane 0 advances it
  if (threadIdx.x != 0) return;
  double t[4] = {0, 0, 0, 0};
  if (advance) {
    for (int k = 0; k < 4; ++k) {
      t[k] = (double)st.ekin_fix[k] * (1.0 / kEScale);
      st.ekin_fix[k] = 0;
    }
  } else {
    for (int p = 0; p < kTempParts; ++p)
      for (int k = 0; k < 4; ++k) t[k] += d.t_part[((size_t)w * kTempParts + p) * 4 + k];
  }
  {
    const double boltz = (double)0.001986f;
    const double tfree_e = t[1] + t[3];
    const double temp_e = t[0] + t[2];
    st.ekin = temp_e;
    st.temp = 2.0 * temp_e / boltz / (double)(float)W.ndegf;
    st.tfree = 2.0 * tfree_e / boltz / (double)(float)W.ndegfree;
    st.tfree_solute = W.ndegfree_solute ? 2.0 * t[1] / boltz / (double)(float)W.ndegfree_solute : 0.0;
    st.tfree_solvent = W.ndegfree_solvent ? 2.0 * t[3] / boltz / (double)(float)W.ndegfree_solvent : 0.0;
    if (W.separate_scaling) {
      if (st.tfree_solvent != 0) st.tscale_solvent = W.temp0 / st.tfree_solvent - 1.0;
      st.tscale_solvent = sqrt(1 + W.dt / W.tau_t * st.tscale_solvent);
      if (st.tfree_solute != 0) st.tscale_solute = W.temp0 / st.tfree_solute - 1.0;
      st.tscale_solute = sqrt(1 + W.dt / W.tau_t * st.tscale_solute);
    } else {
      if (st.tfree != 0) st.tscale_solvent = W.temp0 / st.tfree - 1.0;
      st.tscale_solvent = sqrt(1 + W.dt / W.tau_t * st.tscale_solvent);
      st.tscale_solute = st.tscale_solvent;
    }
    if (advance) {
      const int slot = (st.istep - st.ring_base) % d.ring_n;
      double* tr = &d.t_ring[((size_t)slot * d.nwin + w) * kTRing];
      tr[0] = st.temp; tr[1] = st.tfree; tr[2] = st.ekin;
      tr[3] = (double)st.istep + 4294967296.0 * (double)st.run_epoch;
      tr[4] = st.tfree_solute; tr[5] = st.tfree_solvent;
      if (st.list_now && !(variant & 1)) st.list_missed = 1;
      if (st.energy_now && !(variant & 2)) st.list_missed = 2;
      st.istep += 1;
      begin_step(st, W);
    }
  }
}

// ------------------------------------------------------ launchers --
static inline int blocks(long long n, int bs) { return (int)((n + bs - 1) / bs); }

void launch_begin(const Dev& d, hipStream_t s, int eval, int rebuild) {
  k_begin<<<blocks(d.nwin, 64), 64, 0, s>>>(d, eval, rebuild);
}
void launch_offdiag(const Dev& d, hipStream_t s) {
  if (d.noffd_all) k_offdiag<<<blocks(d.noffd_all, 64), 64, 0, s>>>(d);
}

void launch_lrf_build(const Dev& d, hipStream_t s) {
  if (!d.nlrfw) return;
  k_lrf_pack<<<blocks(std::max(d.ngrp_all, d.nls), 256), 256, 0, s>>>(d);
  if (d.nlrfw <= kLrfSplitMost) k_lrf_build<true><<<2 * d.nlrfw, 64, 0, s>>>(d);
  else k_lrf_build<false><<<d.nlrfw, 64, 0, s>>>(d);
  k_lrf_reduce<<<blocks((long long)kLrfSums * d.ngrp_all, 256), 256, 0, s>>>(d);
}

// list update: group centres and cluster spheres, then the neighbour rows
// and the LRF expansions (independent of each other)
static void launch_list_prep(const Dev& d, hipStream_t s, int ngrp, int nwc, int nsc) {
  if (d.any_qdyn) k_qin<<<blocks(d.ntot, 256), 256, 0, s>>>(d);
  k_centres<<<blocks(ngrp, 128), 128, 0, s>>>(d, ngrp);
  k_bounds<<<blocks(nwc + nsc, 128), 128, 0, s>>>(d, nwc, nsc);
}
static void launch_list_rows(const Dev& d, hipStream_t s) {
  const int nb = 2 * (blocks(d.rl[T_PP].nicl, 4) + blocks(d.rl[T_WW].nicl, 4));
  if (nb) k_build_rows<<<nb, 256, 0, s>>>(d);
}
void launch_lists(const Dev& d, hipStream_t s, int ngrp, int nwc, int nsc) {
  launch_list_prep(d, s, ngrp, nwc, nsc);
  launch_list_rows(d, s);
  launch_lrf_build(d, s);
}

// the q-atoms against water and solute; `energy`: the instances that also
// evaluate the energy terms of windows at an energy step.  launch_*3: the
// instances for windows with a 3-atom solvent
static void launch_qw3(const Dev& d, hipStream_t s, bool energy) {
  if (!d.nqw_work) return;
  if (energy) k_qw<true, true><<<d.nqw_work, 64 * kQWaves, 0, s>>>(d);
  else k_qw<true, false><<<d.nqw_work, 64 * kQWaves, 0, s>>>(d);
}
static void launch_qw(const Dev& d, hipStream_t s, bool energy) {
  if (!d.nqw_work) return;
  if (energy) k_qw<false, true><<<d.nqw_work, 64 * kQWaves, 0, s>>>(d);
  else k_qw<false, false><<<d.nqw_work, 64 * kQWaves, 0, s>>>(d);
  if (d.any_wat3) launch_qw3(d, s, energy);
}
static void launch_qp(const Dev& d, hipStream_t s, bool energy) {
  if (!d.nqp_work) return;
  if (energy) k_qp<true><<<d.nqp_work, 64 * kQWaves, 0, s>>>(d);
  else k_qp<false><<<d.nqp_work, 64 * kQWaves, 0, s>>>(d);
}
void launch_q(const Dev& d, hipStream_t s, bool energy) {
  launch_qw(d, s, energy);
  launch_qp(d, s, energy);
}

// water rows; part: k_wrow's PART
constexpr int kRowBlock = 256;   // 4 clusters
template <bool EK, int PART>
static void launch_wrow_k(const Dev& d, hipStream_t s) {
  const int nb = blocks((long long)d.rl[T_WW].nicl * 64, kRowBlock);
  if (d.rl[T_WW].nicl) k_wrow<false, EK, PART><<<nb, kRowBlock, 0, s>>>(d);
  if (d.rl[T_WW].nicl && d.any_wat3) k_wrow<true, EK, PART><<<nb, kRowBlock, 0, s>>>(d);
}
static void launch_wrow3(const Dev& d, hipStream_t s, bool energy) {
  const int nb = blocks((long long)d.rl[T_WW].nicl * 64, kRowBlock);
  if (!d.rl[T_WW].nicl) return;
  if (energy) k_wrow<true, true, 3><<<nb, kRowBlock, 0, s>>>(d);
  else k_wrow<true, false, 3><<<nb, kRowBlock, 0, s>>>(d);
}
void launch_ww(const Dev& d, hipStream_t s, bool energy) {
  if (energy) launch_wrow_k<true, 1>(d, s);
  else launch_wrow_k<false, 1>(d, s);
}
// solute rows
template <bool EK>
static void launch_srow_k(const Dev& d, hipStream_t s) {
  const int nb = blocks((long long)d.rl[T_PP].nicl * 64, kRowBlock);
  if (d.rl[T_PP].nicl) k_srow<false, EK><<<nb, kRowBlock, 0, s>>>(d);
  if (d.rl[T_PP].nicl && d.any_wat3) k_srow<true, EK><<<nb, kRowBlock, 0, s>>>(d);
}
static void launch_srow3(const Dev& d, hipStream_t s, bool energy) {
  const int nb = blocks((long long)d.rl[T_PP].nicl * 64, kRowBlock);
  if (!d.rl[T_PP].nicl) return;
  if (energy) k_srow<true, true><<<nb, kRowBlock, 0, s>>>(d);
  else k_srow<true, false><<<nb, kRowBlock, 0, s>>>(d);
}
static void launch_srow(const Dev& d, hipStream_t s, bool energy) {
  if (energy) launch_srow_k<true>(d, s);
  else launch_srow_k<false>(d, s);
}

void launch_nonbonded(const Dev& d, hipStream_t s, bool energy) {
  launch_wrow_k<false, 2>(d, s);   // added to what launch_ww stored
  launch_srow(d, s, energy);
  launch_q(d, s, energy);
  launch_qq(d, s, energy);
}
void launch_pair_forces(const Dev& d, hipStream_t s) {
  launch_wrow_k<false, 3>(d, s);
  launch_srow(d, s, false);
  launch_q(d, s, false);
  launch_qq(d, s, false);
}

// Shells beyond LDS are ordered by counting in memory, for which the blocks are
// wide (one window with a shell of more than 4096 of its 13056 waters: an
// evaluation 20 ms, with the 512 threads of k_all 33); else 256 threads order as fast as 1024 (a step of 8 protein windows 116
// and 116 us) and share a launch with the bonded terms
void launch_other_forces(const Dev& d, hipStream_t s) {
  const int nwp = d.nwat_total ? d.nwin * kWpolMaxShell : 0;
  if (d.wpol_wide) {
    if (nwp) k_watpol<<<nwp, 1024, 0, s>>>(d);
    if (d.nbtile) k_bonded<<<d.nbtile, 256, 0, s>>>(d);
  } else if (nwp + d.nbtile) {
    k_other<<<nwp + d.nbtile, 256, 0, s>>>(d, nwp);
  }
  if (d.nrst) k_prestr<<<d.nrst, 64, 0, s>>>(d);
}
// the per-atom terms of an evaluation, after all its other kernels: completes
// the gradient
static void launch_complete(const Dev& d, hipStream_t s) {
  if (d.ntot) k_atom_terms<false><<<blocks(d.ntot, 256), 256, 0, s>>>(d);
}

static void launch_all(const Dev& d, hipStream_t s, bool energy, bool terms) {
  const AllPlan p = all_plan(d, energy, terms);
  if (!p.total) return;
  if (d.any_wat3) {
    if (energy) k_all<true, true><<<p.total, kAllBlock, 0, s>>>(d, p);
    else k_all<true, false><<<p.total, kAllBlock, 0, s>>>(d, p);
  } else {
    if (energy) k_all<false, true><<<p.total, kAllBlock, 0, s>>>(d, p);
    else k_all<false, false><<<p.total, kAllBlock, 0, s>>>(d, p);
  }
}
bool small_engine(const Dev& d, bool mixed_solvent) {
  return !mixed_solvent && !d.wpol_wide && all_plan(d, true, true).total <= kAllMost;
}

// the lists and forces of a small engine: one launch for the forces, and on
// list steps the LRF expansions beside the rows and the forces
static hipError_t launch_small_forces(const Dev& d, hipStream_t s, hipStream_t s2, const hipEvent_t ev[2], bool lists,
                                      int ngrp, int nwc, int nsc, bool energy, bool eval) {
  if (!eval) launch_offdiag(d, s);
  if (lists) {
    launch_list_prep(d, s, ngrp, nwc, nsc);
    if (d.any_lrf) {
      hipError_t err = hipEventRecord(ev[0], s);
      if (err == hipSuccess) err = hipStreamWaitEvent(s2, ev[0], 0);
      if (err != hipSuccess) return err;
      launch_lrf_build(d, s2);
      if (!eval) launch_atom_terms(d, s2);
      err = hipEventRecord(ev[1], s2);
      if (err != hipSuccess) return err;
    }
    launch_list_rows(d, s);
    launch_all(d, s, energy, !eval && !d.any_lrf);
    if (d.any_lrf) {
      hipError_t err = hipStreamWaitEvent(s, ev[1], 0);
      if (err != hipSuccess) return err;
    }
  } else {
    launch_all(d, s, energy, !eval);
  }
  if (eval) launch_complete(d, s);
  return hipSuccess;
}

// the pair forces (terms: with the per-atom terms)
static void launch_pairs(const Dev& d, hipStream_t s, bool energy, bool terms) {
  const PairPlan p = pair_plan(d, energy, terms);
  if (p.total) {
    if (energy) k_pairs<true><<<p.total, kPairBlock, 0, s>>>(d, p);
    else k_pairs<false><<<p.total, kPairBlock, 0, s>>>(d, p);
  }
  if (d.any_wat3) {
    launch_qw3(d, s, energy);
    launch_wrow3(d, s, energy);
    launch_srow3(d, s, energy);
  }
}

// The lists and forces of an MD step, or of an evaluation (eval: the per-atom
// terms come last and complete the gradient), on two streams:
//   s:  on list steps the group centres and the rows; the pair forces; on list
//       steps the LRF expansions and then the per-atom terms;
//   s2: water polarisation, bonded terms and restraints.
// s then waits for s2.  The LRF build comes last because it fills every CU for
// more than a millisecond of FP64 work: beside the row builds and pair kernels
// it starves them (they wait for its long-running blocks), and cutting its
// occupancy so that they fit slows it more than it frees them.
// The kernels write the energies and the shared gradient only through integer
// atomic adds, and everything else to buffers of their own, which the
// integrator adds, so the result does not depend on how they overlap.
hipError_t launch_step_forces(const Dev& d, hipStream_t s, hipStream_t s2, const hipEvent_t ev[2], bool lists, int ngrp,
                              int nwc, int nsc, bool energy, bool eval) {
  if (d.small) return launch_small_forces(d, s, s2, ev, lists, ngrp, nwc, nsc, energy, eval);
  hipError_t err = hipEventRecord(ev[0], s);
  if (err == hipSuccess) err = hipStreamWaitEvent(s2, ev[0], 0);
  if (err != hipSuccess) return err;
  if (!eval) launch_offdiag(d, s2);
  launch_other_forces(d, s2);
  err = hipEventRecord(ev[1], s2);
  if (err != hipSuccess) return err;
  if (lists) {
    launch_list_prep(d, s, ngrp, nwc, nsc);
    launch_list_rows(d, s);
  }
  const bool lrf = lists && d.any_lrf;
  launch_pairs(d, s, energy, !eval && !lrf);
  if (lrf) {
    launch_lrf_build(d, s);
    if (!eval) launch_atom_terms(d, s);
  }
  err = hipStreamWaitEvent(s, ev[1], 0);
  if (err == hipSuccess && eval) launch_complete(d, s);
  return err;
}

void launch_atom_terms(const Dev& d, hipStream_t s) {
  if (d.ntot) k_atom_terms<true><<<blocks(d.ntot, 256), 256, 0, s>>>(d);
}

void launch_integrate(const Dev& d, hipStream_t s, int shake_any, int variant) {
  if (d.nib) k_integrate<<<d.nib, kIntBlock, 0, s>>>(d, shake_any ? 1 : 0);
  k_temperature<<<d.nwin, 64, 0, s>>>(d, 1, variant);
}

void launch_temperature(const Dev& d, hipStream_t s) {
  k_ekin_part<<<d.nwin * kTempParts, 256, 0, s>>>(d);
  k_temperature<<<d.nwin, 64, 0, s>>>(d, 0, 0);
}

void launch_refresh32(const Dev& d, hipStream_t s) { k_refresh32<<<blocks(d.ntot, 256), 256, 0, s>>>(d); }



}  // namespace qmi
