// Device-side layout of the batched engine.  Every window's atoms, groups,
// clusters and terms live in flat arrays with per-window offsets, so each
// kernel launch covers all windows at once.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace qmi {

constexpr int kMaxS = 4;            // states handled on the GPU (2 in FEP windows)
constexpr double kFScale = 4294967296.0;        // 2^32: forces, fixed point
constexpr double kEScale = 68719476736.0;       // 2^36: energies, fixed point
constexpr int kCl = 8;               // cluster size (8 x 8 tile = one wave64)

// energy slots per window (int64 fixed point), order used by the finaliser
enum ESlot {
  E_PP_EL, E_PP_VDW, E_PW_EL, E_PW_VDW, E_WW_EL, E_WW_VDW, E_LRF,
  E_P_BOND, E_P_ANG, E_P_TOR, E_P_IMP, E_W_BOND, E_W_ANG, E_W_TOR, E_W_IMP,
  E_FIX, E_SHELL, E_RAD, E_WPOL,
  E_PROT,             // state-independent part of restraint%protein (sequence, wall)
  E_NBASE,
  // per state s: E_Q0 + s*8 + {qbond, qangle, qtors, qimp, qq_el, qq_vdw, qp_el, qp_vdw},
  // E_QW0 + s*2 + {qw_el, qw_vdw} and E_QR0 + s (state restraints)
  E_Q0 = E_NBASE,
  E_QW0 = E_Q0 + 8 * kMaxS,
  E_QR0 = E_QW0 + 2 * kMaxS,
  E_NSLOT = E_QR0 + kMaxS
};

// restraint records of p_restrain (md.f90:12940-13274)
enum RstKind { R_SEQ_ATOMS = 0, R_SEQ_GEOM, R_SEQ_MASS, R_POS, R_DIST, R_ANGLE, R_WALL };

// A and B of a pair's V = A/r^12 - B/r^6 from the two atoms' LJ columns a, b:
// products under the geometric rule (nonbond_pp, md.f90:10432-10439); under
// the arithmetic rule R* = a_i + a_j and eps = b_i b_j (b being the square
// root of epsilon), A = eps R*^12, B = 2 eps R*^6 (nonbon2_pp,
// md.f90:8993-9000, 9056-9058)
template <typename T>
__host__ __device__ __forceinline__ void lj_ab(T ai, T bi, T aj, T bj, bool arith, T* A, T* B) {
  if (!arith) {
    *A = ai * aj;
    *B = bi * bj;
    return;
  }
  const T s = ai + aj, s2 = s * s, s6 = s2 * s2 * s2, e = bi * bj;
  *A = e * s6 * s6;
  *B = T(2) * e * s6;
}

struct WinDev {
  int ao, natom, nat_solute, nwat;
  int nq, S, qvdw, natyps;
  int q_off, t_off;                 // first global q-atom / first entry of the type tables
  int qs_off, qsc_off;              // first entry of the [q][state] and [q][type][state] tables
  int g_off, ngrp, ngrp_solute;     // charge groups
  int wc_off, nwc, sc_off, nsc, qc_off, nqc;
  int nqch;                         // chunks of kQItem q-atoms (2 per 4 q-clusters)
  long long qp14_off;               // first entry of the window in Dev::qp14
  int sh_off, nshell;               // water polarisation shells
  long long wp_off;                 // first entry of the window's shell rows in Dev::wtheta
  int nsteps, nbcycle, iene, iout;
  int use_lrf, wpol, separate_scaling, iac_ow;   // iac_ow: 0-based type of water O
  int ndegf, ndegfree, ndegf_solute, ndegfree_solute, ndegf_solvent, ndegfree_solvent;
  float el14, crg_ow, crg_hw, aO1, bO1;   // aO1, bO1: LJ columns of the water oxygen type
  int arith;                        // arithmetic LJ combination rule (topology vdW rule 2)
  // the Q-atom lists are rebuilt at list updates (q_atom cut-off within the
  // exclusion radius, nbqplist / nbqwlist md.f90:7875-7964, 8066-8118)
  int qlist_dynamic;
  double rcq2;
  float ww_a, ww_b;                 // A, B of the water O-O pair
  // 3-atom solvent (topology solvent type 1): LJ on all three atoms and the
  // charges of the first solvent molecule; crg_w is (crg_ow, crg_hw, crg_hw)
  // for SPC
  int wat3;
  int iac_w[3];                     // 0-based types of the solvent atoms
  float crg_w[3], aw[3], bw[3];     // charges and LJ columns of the solvent atoms
  float ww3_a[9], ww3_b[9];         // A, B of solvent atom pairs (p, q) at [3p + q]
  // the same in FP64, for the energy terms of energy steps
  double el14d, aO1d, bO1d, ww_ad, ww_bd;
  double awd[3], bwd[3], ww3_ad[9], ww3_bd[9];
  double dt, tau_t, temp0;
  double rcpp2, rcpw2, rcww2, rclrf2;
  double fk_pshell, fk_wsphere, fkwpol, dwmz, awmz, rwat;
  double xwcent[3], xpcent[3];
  double lambda[kMaxS];
};

struct WinState {
  int istep;          // current step (counts from 0 at the start of the run)
  int stop_at;        // the current qmi_run stops this window at this step
  int ring_base;      // step at the start of the current qmi_run: ring slot = (istep - ring_base) % ring_n
  int run_epoch;      // number of the current qmi_run, stored with each ring record
  int list_now, energy_now, active;
  int wpol_acc;       // this evaluation is a pot_energy call of the run: water-polarisation shell averages advance
  double tscale_solute, tscale_solvent;
  double temp, tfree, tfree_solute, tfree_solvent, temp_solute, temp_solvent, ekin;
  // kinetic energy of the step's atoms, fixed point (kEScale): solute all,
  // solute free, solvent all, solvent free; k_integrate adds, k_temperature
  // reads and clears
  long long ekin_fix[4];
  int shake_fail;
  int list_overflow;  // a neighbour row exceeded its capacity
  int list_missed;    // 1 (2): a step needing pair lists (energies) was launched without those kernels
  long long E[E_NSLOT];
};

struct ShellDev { float rout, dr, cstb, theta_corr, avtheta, avn_insh; int n_insh; int pad; };

// dynamic pair lists (i-centric): WW, W<-P, P<-W, P<-P
enum RowType { T_WW = 0, T_WP, T_PW, T_PP, T_NTYPES };

// temperature ring record per window and step: T_tot, T_free, Ekin, step tag,
// T_free solute, T_free solvent
constexpr int kTRing = 6;
constexpr int kTempParts = 8;      // blocks per window of the kinetic-energy sum
// the LRF build splits a window's source groups in this many parts, summed in
// part order; a constant, so the expansions do not depend on launch shapes
constexpr int kLrfParts = 8;
constexpr int kIntBlock = 256;     // atoms per block of the integrator
// bits of a three-constraint unit: its first entry within the block, the places
// of a, b and c among its atoms, and that it is one
constexpr int kTriFirst = 0xff, kTriA = 8, kTriB = 10, kTriC = 12, kTri = 1 << 14;
constexpr int kWpolMaxShell = 8;
constexpr int kWpolLds = 4096;     // waters of one polarisation shell held (and ordered) in LDS
constexpr int kBondTileTerms = 512; // bonded terms per tile
constexpr int kBondSpan = 1024;     // atoms of a tile's LDS gradient sums
constexpr int kQItem = 16;          // q-atoms of a chunk of the q kernels: half the members of 4 q-clusters

// Neighbour rows of the dynamic pair lists (WW, W<-P, P<-W, P<-P): row
// ic*8 + a belongs to member a of i-cluster ic and holds the j entries of
// that member: the index in xw of a water's oxygen, or a solute slot (P<-P
// entries carry the 1-4 flag in bit 30), in a fixed capacity `cap` per row, a
// multiple of the entries the row kernels take in a pass.
struct RowList {
  int* cnt;        // entries per row
  int* ent;        // [row * cap + k]
  int cap;
  int nicl;        // i-clusters; rows = 8 * nicl
};
constexpr int kRow14 = 1 << 30;

// index in Dev::xw of site k (O, H1, H2) of member m of water cluster c
__host__ __device__ __forceinline__ int xw_at(int c, int m, int k) { return 3 * kCl * c + kCl * k + m; }

struct Dev {
  int nwin, ntot;
  const WinDev* win;
  WinState* ws;
  // atoms
  double *x, *v, *xtop;
  float4* x32;          // x, y, z, scaled charge
  // x32 again in cluster-slot order, the order in which rows name their
  // entries: per water cluster its 8 members' O, H1 and H2 (xw_at), so that a
  // row's 8 lanes, which mostly hold the members of one cluster, read one
  // 128-byte line a load; then one per solute slot (cluster * 8 + member).
  // Zero for empty members.  wslot: per atom, its index, or -1 (q-atoms)
  float4* xw;
  const int* wslot;
  double4* xwd;         // the same in FP64 (x, y, z, unused), for the energy terms
  float4* sljp;         // avdw1, bvdw1, avdw3, bvdw3 of the solute slots
  const double4* sljd;  // the same in FP64
  // the q-atoms' x32 again, per q-cluster member slot (cluster * 8 + member;
  // zero for empty members); qmslot: per atom, its slot or -1
  float4* xq;
  const int* qmslot;
  long long* f;         // shared gradient, 3 per atom, fixed point 2^-32; zero between steps
  // the row kernels' and the q kernels' sums, 3 per entry: entry 3 * slot +
  // site for the waters' cluster slots (nwslot of them), then one per solute
  // slot; rslot: an atom's entry, or -1 (q-atoms)
  long long *grow, *gq;
  int nwslot;
  const int* rslot;
  long long* fterm;     // per-atom terms of the step (LRF evaluation, atom restraints), then the complete gradient
  const double* mass;
  const int* wid;       // window of atom
  const int* iac;       // 0-based window-local atom type
  const int* grp;       // charge group (global) of atom
  const uint8_t* aflag; // bit0 excl, bit1 shell, bit2 heavy, bit3 q-atom
  // Q-atom lists: whether a non-q atom is within the q_atom cut-off of the
  // Q centre (the switching atom of its group, or its water's oxygen) at
  // the last list update; always 1 where the lists are static
  uint8_t* qin;
  const int* qref;      // the atom whose distance decides qin, -1: never updated
  int any_qdyn;         // some window's Q lists are rebuilt at list updates
  // charge groups
  const int* g_sw;      // switch atom (global); water groups: O
  const int* g_first;   // into g_atoms
  const int* g_n;
  const int* g_atoms;   // global atoms
  const int* g_win;
  double* g_cent;       // 3 per group
  double* g_lrf;        // 20 per group: phi0, phi1(3), phi2(6: xx xy xz yy yz zz), phi3(10)
  int ngrp_all;         // groups of all windows
  int nlrfw;            // LRF build blocks: (window, first target group, count <= 64, source part)
  const int4* lrf_work;
  double* g_lrf_part;    // [part][group][20] sums over the kLrfParts source parts
  // LRF sources, packed at every build: switching atom of each group
  // (x, y, z, excluded) and the group's non-q atoms (x, y, z, charge)
  double4* ls_sw;
  double4* ls_xq;
  const int* ls_first; const int* ls_n; const int* ls_atom;
  int nls;
  // special partners of solute atoms (exclusions / 1-4), CSR
  const int* sp_start;  // per atom (ntot+1)
  const int* sp_j;
  const uint8_t* sp_t;  // 1 = excluded, 2 = 1-4
  const int2* sp_rng;   // per atom: smallest and largest partner in sp_j
  // clusters
  const int* wc_o;      // 8 per water cluster: O atom or -1
  const int* sc_a;      // 8 per solute cluster: atom or -1
  // per q-cluster member (8 per cluster): its global atom (or -1), and per
  // state (kMaxS per member) the water-side factors of k_qw: A and B of the
  // pair with the water oxygen, the charge products with O and with H, and
  // the soft-core term against the oxygen type
  const int* qc_atom;
  const float4* qcw_par;
  const float* qcw_sc;
  // 3-atom solvent: per member, state and hydrogen k = 1, 2 of the water:
  // A, B, charge product and soft-core term ([(m * kMaxS + s) * 2 + k - 1])
  const float4* qcw_h;
  int any_wat3;          // some window has a 3-atom solvent
  int small;             // a step's force kernels run as one launch
  int any_lrf;           // some window uses LRF
  // the same in FP64 for the energy terms: A, B, soft-core term, charge
  // product of member, state and water atom ([(m * kMaxS + s) * 3 + k])
  const double4* qcw_e;
  // static Q lists: whether the water (solute atom) of a cluster slot is in
  // them, the 1-4 pairs of a solute slot with the q-atoms of a chunk (bit
  // 4 member + cluster, [qp14_off + slot of the window * nqch + chunk]), and the
  // work items: window, first slot, slots (at most 64)
  const uint8_t* qw_on; const uint8_t* qp_on;
  const uint16_t* qp14;
  int nqw_work, nqp_work;
  const int4* qw_work; const int4* qp_work;
  const int* wc_win; const int* sc_win;
  double* wc_bs;        // bounding sphere per water cluster (x, y, z, r)
  double* sc_bs;        // bounding sphere of the switch atoms of the members
  // per cluster member, written at list steps: its switching atom's x, y, z
  // and w = 0 (listed), 1 (switching atom excluded) or -1 (no member)
  double4* wc_cm;
  double4* sc_cm;
  // q tables (per window, offset q_off)
  const int* q_atom;     // global atom
  const float* q_crg;    // [q*S + s]
  const float4* q_lj;    // [q*S + s]: qavdw1, qbvdw1, qavdw3, qbvdw3 (or topology params)
  const double* q_ljd;   // same in double, for the energy path
  const float* q_sc;     // [(q*natyps + t)*S + s]
  const double* q_scd;
  RowList rl[T_NTYPES];  // neighbour rows
  // bonded tiles, each of one window: (first entry of btile_terms, terms, first
  // atom, atoms spanned); btile_terms: term indices, grouped by kind within a tile
  int nbtile;
  const int4* btile;
  const int* btile_terms;
  // q-q pairs per atom for the forces: atom qqg_atom[k] has the records
  // qqg_start[k] .. qqg_start[k+1]-1 of two float4 each: charge product,
  // el_scale, A, B; soft-core term, partner atom, state (| 8: LJ code 3,
  // | 16: exponential repulsion), unused
  int nqqg;
  const int* qqg_atom;
  const int* qqg_start;
  const float4* qqg_ent;
  // q-q pairs (static)
  int nqq;
  const int4* qq_ij;     // iq (window-local), j (global), jq (1-based q or 0), ljcod
  const float* qq_es;    // el_scale
  const int* qq_st;      // state
  const int* qq_win;
  const float* qq_sc;    // soft-core term of the pair
  const double2* qq_ab;  // A, B of the pair in its state
  const float2* qq_q;    // charges (scaled, real(4)) of the pair's two atoms in its state
  // bonded terms
  int nbond, nang, ntor, nimp;
  const int2* b_ij; const double2* b_par; const int* b_win; const uint8_t* b_solv;
  const int4* a_ijk; const double4* a_par; const int* a_win; const uint8_t* a_solv;  // fk, ang0, ureyfk, ureyr0
  const int4* t_ijkl; const float4* t_par; const int* t_win; const uint8_t* t_solv;  // fk, rmult, deltor, paths
  const int4* i_ijkl; const float2* i_par; const int* i_win; const uint8_t* i_solv;
  const int* i_kind;     // 1 harmonic (improper), 2 periodic (improper2) per window
  const int* urey;       // per window: CHARMM Urey-Bradley on
  // q bonded (one entry per term and state)
  int nqb, nqa, nqt, nqi;
  const int2* qb_ij; const double4* qb_par; const int2* qb_ws;   // Dmz, amz, r0, fk; (window, state)
  const int4* qa_ijk; const double2* qa_par; const int2* qa_ws;
  const int4* qt_ijkl; const double4* qt_par; const int2* qt_ws; // fk, rmult, deltor
  const int4* qi_ijkl; const double2* qi_par; const int2* qi_ws; // fk, imp0
  // restraints: (kind, window, i, j) global atoms; (k, flag) with flag = ih
  // (sequence, wall) or ipsi (position, distance, angle); 8 parameters each
  int nrst;
  const int4* rs_kwij; const int2* rs_kf; const double* rs_par;
  // shake units (independent constraint components): their constraints
  const int* su_start; const int* su_n;
  const double* sc_d2;     // per constraint: d0^2
  const float2* sc_w;      // per constraint: inverse masses of i and j
  const uint8_t* sc_loc;   // per constraint: local atom numbers of i and j within the unit
  // integration units of k_integrate, each a SHAKE component or one
  // unconstrained atom: (window, first entry, number of atoms, SHAKE unit or
  // -1); a component's atoms are listed in the order its sc_loc numbers them.
  // Blocks of k_integrate: runs of whole units of at most kIntBlock atoms,
  // (first entry, atoms, first unit, units)
  int nib;
  const int4* iu; const int4* ib;
  // per entry, what the integrator needs of the atom: (atom, window, rslot,
  // wslot), (charge, inverse mass, qmslot, 1 solute | 2 excluded), mass
  const int4* ie_i; const float4* ie_f; const double* ie_m;
  // per unit: for three constraints among three atoms, the squared distances
  // and (inverse masses of a, b and c, kTri bits), the constraints being a-b,
  // a-c and b-c in their order; kTri 0 for other units
  const double* tri_d2; const float4* tri;
  // water shells
  ShellDev* shells;
  double* wtheta;        // windows of more than kWpolLds waters: theta per shell and water, at WinDev::wp_off
  int wpol_wide;         // some shell starts with more waters than LDS holds
  int nwat_total;
  // energy snapshots for output: [ring slot][window][E_NSLOT] + temperature
  long long* e_ring;
  double* t_ring;        // [slot][window][4]: temp, tfree, ekin, istep
  double* t_part;        // [window][kTempParts][4]: kinetic-energy partial sums
  int ring_n;
  // EVB off-diagonal functions of all windows: window, q-atoms k, l (global
  // atoms), A and mu; every MD step records Hij and r_kl at its start
  int noffd_all;
  const int* offd_win;
  const int2* offd_kl;
  const double2* offd_par;
  double* o_ring;        // [slot][noffd_all][2]: Hij, r_kl
};

}  // namespace qmi
