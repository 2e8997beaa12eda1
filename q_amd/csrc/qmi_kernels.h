// Launchers of the kernels in qmi_kernels.hip (all windows per launch).
#pragma once
#include <hip/hip_runtime.h>

#include "qmi_device.h"

namespace qmi {
// the start of a run's first step (eval 0) or of an evaluation (k_begin)
void launch_begin(const Dev& d, hipStream_t s, int eval, int rebuild);
// EVB off-diagonal elements at an MD step's starting coordinates
void launch_offdiag(const Dev& d, hipStream_t s);
void launch_lists(const Dev& d, hipStream_t s, int ngrp, int nwc, int nsc);
// the timing pass: the water-water rows alone, then all other pair kernels;
// `energy`: the instances that also evaluate the energy terms of windows at an
// energy step (false: forces only)
void launch_ww(const Dev& d, hipStream_t s, bool energy);
void launch_nonbonded(const Dev& d, hipStream_t s, bool energy);
// single families, for timing: the q kernels, the LRF build, the pair kernels
void launch_q(const Dev& d, hipStream_t s, bool energy);
void launch_lrf_build(const Dev& d, hipStream_t s);
void launch_pair_forces(const Dev& d, hipStream_t s);
// water polarisation, bonded terms and restraint records
void launch_other_forces(const Dev& d, hipStream_t s);
// the per-atom terms of an MD step into their own array (Dev::fterm)
void launch_atom_terms(const Dev& d, hipStream_t s);
// whether a step's force kernels run as one launch (Dev::small)
bool small_engine(const Dev& d, bool mixed_solvent);
// the lists and forces of an MD step or (eval) of an evaluation on two
// streams (see the definition)
hipError_t launch_step_forces(const Dev& d, hipStream_t s, hipStream_t s2, const hipEvent_t ev[2], bool lists, int ngrp,
                              int nwc, int nsc, bool energy, bool eval);
// the end of an MD step; the gradient is completed with the per-atom terms
// of launch_atom_terms, which must have run in the same step
// variant: bit 0 the step's list kernels were launched, bit 1 its energy terms
void launch_integrate(const Dev& d, hipStream_t s, int shake_any, int variant);
void launch_temperature(const Dev& d, hipStream_t s);
void launch_refresh32(const Dev& d, hipStream_t s);
}  // namespace qmi
