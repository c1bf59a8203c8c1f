// engine_internal.h — what other parts of the library (the MD step and the
// batch of systems) need from engine handles beyond the public C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <functional>
#include <vector>

#include "batch.h"
#include "bonded.h"
#include "common.h"
#include "forces.h"

struct dyn_engine;
struct dyn_energies;

namespace dyn {

// One evaluation pass over engines that share a stream: every kernel is one
// launch for all of them.  A single engine is a set of one.  The SPME chain
// (and the caller's side work, such as bonded forces) runs on a second
// stream of the same priority, forked after the preparation launch and
// joined before the finalize launch, so that it overlaps the list build,
// the pair kernel and the corrections.
struct EngineSet {
  std::vector<dyn_engine*> e;
  BatchRun R;          // main stream
  BatchRun side;       // second stream (side.stream null: everything on R)
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  Profiler* prof = nullptr;
};

// Enqueue one evaluation of every engine in the set (DYN_COMPUTE_* flags,
// the same for all).  Each engine decides on the device whether it rebuilds
// its pair list (DYN_COMPUTE_REBUILD, or a list never built, forces it).
// side, when given, are bonded terms to evaluate in the same pass (they read
// no nonbonded forces).
// Internal compute flag (beside the public DYN_COMPUTE_* bits): list builds
// the device decides on go to the staging list on the second stream, beside
// the pair kernel, and become current at the next evaluation; an evaluation
// whose current list has gone stale is void (status) and its call repeats.
constexpr uint32_t kComputeStagedBuild = 1u << 30;
// The caller's next launch sums the site forces from their parts and ends
// the evaluation's list bookkeeping (engine_force_parts); no finalize launch,
// and the engine's force array stays stale until a later evaluation
// finalizes.
constexpr uint32_t kComputeFusedFinalize = 1u << 29;
void engine_set_enqueue(EngineSet& S, uint32_t flags, const SideWork* side = nullptr);
// Wait for the set's work and check each engine's device status (throws the
// first engine's error; buffers that overflowed have been enlarged).
void engine_set_check(EngineSet& S);
// The set of this engine alone (its stream, argument packs and readings).
EngineSet engine_self_set(dyn_engine* eng);

Profiler* engine_profiler(dyn_engine* eng);
hipStream_t engine_stream(const dyn_engine* eng);
// The engine's device status word (non-zero after a failed evaluation).
const unsigned int* engine_status_device(const dyn_engine* eng);
// Whether the engine's evaluations may be recorded into a graph (no test
// hook pending, no profiling).
bool engine_graph_safe(const dyn_engine* eng);
// Whether the engine asks for every kernel on one stream (no second stream).
bool engine_single_stream(const dyn_engine* eng);
void engine_set_stream(dyn_engine* eng, hipStream_t s);  // null: its own stream again
int engine_device(const dyn_engine* eng);
void engine_sizes(const dyn_engine* eng, uint32_t* n_dyn, uint32_t* n_water);
void engine_box(const dyn_engine* eng, float box[3]);
int engine_mode(const dyn_engine* eng);  // DYN_MODE_*
const int64_t* engine_forces_device(const dyn_engine* eng);
// The parts of the last evaluation's forces, and whether the engine's force
// array is stale (the evaluation was enqueued with kComputeFusedFinalize).
ForceParts engine_force_parts(const dyn_engine* eng);
bool engine_forces_stale(const dyn_engine* eng);
// The engine's report (status, counters, energy sums) and its place in pinned
// host memory; a kernel of the caller's read stores it there (report_out, one
// workgroup), and after the wait engine_check_report looks at the status.
struct ReportView {
  const double* src;
  double* dst;
  uint64_t n;
};
__device__ __forceinline__ void report_out(const ReportView& V) {
  for (uint32_t k = threadIdx.x; k < (uint32_t)V.n; k += blockDim.x) V.dst[k] = V.src[k];
}
ReportView engine_report_view(const dyn_engine* eng);
void engine_check_report(dyn_engine* eng);
// dyn_engine_get_energies without a wait, after a check (engine_check_report,
// engine_set_check) that followed the last evaluation.
void engine_report_energies(dyn_engine* eng, dyn_energies* out);
// Pinned host memory of the engine, 24 bytes per site, for the caller's
// next read.
void* engine_host_stage(dyn_engine* eng);
// Device arrays to copy, in words of 8 bytes.
struct CopySegs {
  static constexpr uint32_t kMax = 8;
  const uint2* src[kMax];
  uint2* dst[kMax];
  uint64_t words_of[kMax];
  uint64_t n;
  void add(void* to, const void* from, size_t bytes) {
    src[n] = static_cast<const uint2*>(from);
    dst[n] = static_cast<uint2*>(to);
    words_of[n++] = bytes / 8;
  }
  size_t words() const {
    size_t m = 0;
    for (uint64_t k = 0; k < n; ++k) m = std::max(m, (size_t)words_of[k]);
    return m;
  }
};
// Keep / put back the last evaluation's forces, SPME forces and energies (a
// checkpoint adds the copies its caller makes on the engine's stream); a
// restore also invalidates the list.
void engine_checkpoint(dyn_engine* eng, CopySegs& seg);
void engine_restore(dyn_engine* eng);
}  // namespace dyn
