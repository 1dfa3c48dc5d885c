// pdmd_engine.h -- launch wrappers of the gfx950 DMD kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "pdmd_device.h"

namespace pdmd {

// LDS bytes of one system's workgroup of nw wavefronts with work areas (the
// calendar wavefront among them) for a calendar of nblk 16-entry blocks and
// work lists of maxw entries, before its leaves; at least one wavefront's
// list rebuild scratch.
size_t engine_lds_bytes(int nblk, int maxw, int nw);
// most event wavefronts per system in a launch of n systems of up to max_n beads
int engine_max_waves(int n, int max_n, int maxw, size_t lds_limit);
// work-list capacity of the event kernels for a list capacity
int engine_maxw(int cap);
// Opt the event-loop kernels in to lds_limit bytes of LDS per workgroup.
hipError_t engine_prepare(size_t lds_limit);
// Lists, pseudo-event seeds and events() for n systems of up to max_n beads,
// each step one launch over all of them.
hipError_t engine_setup(const SysDev* d_sys, const int* d_ids, int n, int max_n, hipStream_t s);
// A list update forced at the current time for n systems (origin shift,
// nbor + events), likewise.
hipError_t engine_rebuild(const SysDev* d_sys, const int* d_ids, int n, int max_n, hipStream_t s);
// Event loop: every listed system runs until its SysState::target.
// budget_ticks: wall_clock64 ticks after the launch's start after which
// each system stops between rounds (0 = run to the event targets), with
// launch_t0 a device word that takes the start (needed with a budget);
// waves: event wavefronts per system (1 to 8; seven run at most, three in a
// launch of more systems than compute units, fewer where lds_limit asks for
// it), each round runs up to that many conflict-free pair events side by side
constexpr int kStopAtOutput = 1;  // engine_run flag: stop after the next output pseudo-event
hipError_t engine_run(const SysDev* d_sys, const int* d_ids, const long long* d_inc, int n, int max_n, int maxw,
                      size_t lds_limit, hipStream_t s, long long budget_ticks = 0, int flags = 0, int waves = 1,
                      unsigned long long* launch_t0 = nullptr);
// Debug checks (checkover.f, check_nc_int.f) of system id's n beads: out[8]
// counters (zeroed by the caller, out[3] preset to all ones); alt replaces
// the resident state records when not null.
hipError_t engine_check(const SysDev* d_sys, int id, int n, const Rec* alt, unsigned long long* out, hipStream_t s);
// Observables of system id of n beads (energy.f, radgyr.f, end2end.f):
// outd[7] ered, tred, sumvel, ehh_ii, ehh_ij, rg_avg, e2e_avg; outi[3]
// hb_alpha, hb_ii, hb_ij.  cstart/clen: nch chains (addresses the device can
// read); nfirst: chains of the leading species block; boxl in Angstrom.
hipError_t engine_observables(const SysDev* d_sys, int id, int n, const int* cstart, const int* clen, int nch, int nfirst,
                              double boxl, double* outd, int* outi, hipStream_t s);
// State arrays of system id of n beads into out (StateLayout), those in
// `want` (kStateSv ...).
hipError_t engine_state(const SysDev* d_sys, int id, int n, int want, double* out, hipStream_t s);
// SysState::status, and all counters, of n systems.
hipError_t engine_status(const SysDev* d_sys, const int* d_ids, int n, int* out, hipStream_t s);
hipError_t engine_stats(const SysDev* d_sys, const int* ids, int n, SysStats* out, hipStream_t s);
// Test hook: collision times of (i, j) pairs (1-based) of system id.
hipError_t engine_predict(const SysDev* d_sys, int id, int n, const int* pi, const int* pj, double* tij, int* type,
                          hipStream_t s);

}  // namespace pdmd
