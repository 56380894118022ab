// Gate-stream planner and multi-gate sweeps (LDS/register tiles, fused blocks).
#pragma once

#include <complex>
#include <string>
#include <vector>

#include "gvs.h"
#include "sweep_types.h"

namespace q1t {

// A planned step of the gate stream.
struct PlanStep {
    bool sweep = false;
    std::vector<int> tile;          // sweep: global bit positions of the tile (ascending)
    std::vector<size_t> gates;      // indices into the queue, in application order
};

// Default tile geometry per precision (interpreter kernels), and with the
// kernels specialised to each sweep program.
TileGeom tile_geometry(Precision p);
TileGeom tile_geometry_specialised(Precision p);
// Is (M, R) one of the compiled tile shapes for this precision?
bool tile_shape_supported(Precision p, int M, int R);

// Is a gate applicable inside a tile (targets that must be local, if any)?
bool sweepable(const GateOp& op, std::vector<int>* local_targets);

// Plan: runs of gates whose non-diagonal targets fit M tile bits (the L low
// bits always included); a gate may run before earlier gates it commutes
// with.  With fuse_k > 0 the non-diagonal gates need all their bits in the
// tile.  `search`: refine each greedy tile (and, in the programs below, each
// phase's register bits) by local search (GpuVectorState::tile_search,
// phase_search).
// `pairs`: dense two-qubit gates without controls join the sweeps (unfused
// programs; batches and fused plans apply them on their own).
std::vector<PlanStep> plan_gates(const std::vector<PendingGate>& q, int n, const TileGeom& g, int fuse_k,
                                 bool search = true, bool pairs = false);

// Everything plan_gates reads of the queue and its settings: equal keys give
// equal plans (a flush repeating the previous flush's gate structure, with
// any angles, reuses its steps).
std::vector<uint64_t> plan_key(const std::vector<PendingGate>& q, int n, const TileGeom& g, int fuse_k, bool search);

// Register phases of one sweep (per-gate arithmetic).  `order`, if given,
// receives the queue indices of the sweep's gates in the order the kernel
// applies them (per phase: its register ops, then its write-back gates).
// `factors`: diagonal ops on bits outside the tile become one tile factor
// (a kind-2 phase; the specialised kernels apply it, the interpreter kernels
// do not take such programs).
void build_program(const std::vector<PendingGate>& q, const PlanStep& step, int M, int R,
                   std::vector<SwPhase>& phases, std::vector<SwOp>& ops, bool search = true,
                   std::vector<size_t>* order = nullptr, bool factors = false);

// The factor that reduce_program has taken out of a flush's gates so far, and
// the number of gates it comes from.
struct Reduction {
    std::complex<long double> factor{1, 0};
    int gates = 0;
};
// The same sweep in fewer operations per amplitude, for kernels bound by them:
// uncontrolled rotations, reflections (H) and RX gates without their larger
// entry, uncontrolled diagonal gates on a register bit as the phase of its ones,
// and the factors that depend only on thread and outer bits multiplied per
// thread and applied once per phase.  The common factor is applied at the end
// of the program if `last`, and before it could leave the precision's range.
// The structure does not depend on the gates' angles.
// Measured: specialised kernels, 20 layers, 30 qubits complex128 133.3 -> 115.9
// ms, 28 qubits complex64 21.3 -> 19.0 ms (the sweeps of many gates are bound by
// FP64 issue: 154 ops on 2^18 tiles 15 ms); interpreted, 12 layers of 24 qubits
// 1866 -> 1695 us complex128, 1033 -> 979 us complex64.  Errors against 64-bit
// arithmetic fall with the roundings: 28 qubits complex64 4.3e-6 -> 1.5e-6.
// Batches keep the gates' own forms.
void reduce_program(std::vector<SwPhase>& phases, std::vector<SwOp>& ops, Precision prec, Reduction& red, bool last);

// The LDS places of the register phases for amplitudes of elem_bytes.
void place_phases(std::vector<SwPhase>& phases, int M, int R, size_t elem_bytes);

// An op as the interpreting kernels take it; `seq`: whole-state programs.
template <typename R> InterpOpT<R> interp_op(const SwOp& o, bool seq);

// States too small for tiles (below M+2 qubits) run whole in LDS, one
// workgroup per column: runs of gates that a register phase takes are one
// step (its tile: all M bits, M >= 3 bits whatever the state), others run on
// their own kernels between them.  Gates that round keep their order
// (Blocker), so the amplitudes are those of the gates applied one by one.
std::vector<PlanStep> plan_whole(const std::vector<PendingGate>& q, int M);
// The program of one such step with nr register bits; op_begin / op_end count
// from the step's first op.
template <typename R>
void build_whole(const std::vector<PendingGate>& q, const PlanStep& step, int M, int nr, std::vector<WholePhase>& phases,
                 std::vector<InterpOpT<R>>& ops);

// The order in which the plain (per-gate) plan of the specialised kernels
// applies the queue's gates (identity gates, which never run, are left out;
// tile factors last in their sweep).
std::vector<size_t> plan_order(const std::vector<PendingGate>& q, int n, const TileGeom& g, bool search);

// Fused program of one sweep: dense blocks of at most K local qubits
// (composed in FP64, real-embedded, rounded to FP32 into `blocks`) and
// register phases for the rest.
void build_fused_program(const std::vector<PendingGate>& q, const PlanStep& step, int M, int R, int K,
                         std::vector<SwPhase>& phases, std::vector<SwOp>& ops, std::vector<float>& blocks,
                         int* nblocks, bool search = true, bool factors = false);

// Features of a sweep program for the learned cost model (20 floats):
//  0 register phases, 1 blocks of 3 qubits, 2 blocks of 4 qubits (a block of
//  k > 4 qubits counts as 4^(k-4) four-qubit blocks), 3-6 one-qubit ops by
//  body (general, real/RX/Y, swap, phase/diagonal), 7-9 ops with thread,
//  register and outer controls, 10 precision, 11 M, 12 R, 13 phases holding
//  a local bit >= 8 in registers, 14 tile bits at positions >= 20 (long HBM
//  strides), 15 gates, 16 widest block, 17 tile bits at positions >= 26,
//  18 ops folded into the tile factors, 19 kernel specialised to the
//  program (1) or the interpreter (0).
constexpr int kSweepFeatures = 20;
void sweep_features(const std::vector<SwPhase>& phases, const std::vector<SwOp>& ops, const PlanStep& step,
                    int precision, const TileGeom& g, bool specialised, float* out);

// Device buffer that grows on demand (synchronising `stream` first).
struct DeviceBuffer {
    void* ptr = nullptr;
    size_t cap = 0;
    void* get(size_t bytes, hipStream_t stream);
    ~DeviceBuffer();
};

// Pinned host buffer that grows on demand; the caller makes sure no copy
// from it is in flight when it grows or is rewritten.
struct PinnedBuffer {
    void* ptr = nullptr;
    size_t cap = 0;
    void* get(size_t bytes);
    ~PinnedBuffer();
};

// Flush the pending gates of many states together (all of one precision,
// tile geometry and fusion setting, sharing `stream`): states at least
// M+2 qubits wide are planned into sweeps and the r-th sweep of every state
// runs in one launch over all their tiles; smaller states run whole in LDS,
// one workgroup per column, all in one launch.
// The table goes up from `stage` (the call ends with the stream
// synchronised, so the next call may rewrite it).  `plan_s` and `pack_s`
// (optional) accumulate the host planning and table-building time.
void run_planned_batch(const std::vector<GpuVectorState*>& states, hipStream_t stream, DeviceBuffer& prog,
                       PinnedBuffer& stage, ItemQueue& iq, RunStats& agg, unsigned tile_chunk,
                       double* plan_s = nullptr, double* pack_s = nullptr);

// Sources of the kernels specialised to the sweeps of the plan a flush of
// `q` would run (plain programs; with fusion_k > 0 greedy fixed-width
// fusion), block offsets as in the flush's merged table; `factors`: diagonal
// ops on bits outside the tile folded into tile factors.  Host only.
std::vector<std::string> plan_jit_sources(const std::vector<PendingGate>& q, int n, Precision prec, int fusion_k,
                                          bool search, bool prefetch = false, bool factors = true);

// Apply the pending gates to columns [col_begin, col_end) of the state with
// the planned schedule: runs of gates whose qubits fit one tile are applied
// in one HBM sweep; `fusion_k` > 0 composes runs into dense blocks of at most
// that many qubits first (complex64 path).  `fresh`: the state is one column
// |0..0> that is not in memory (tiling only).
void run_planned(GpuVectorState& st, const std::vector<PendingGate>& queue, size_t col_begin, size_t col_end,
                 int fusion_k, bool tiling, bool fresh, RunStats& stats);

}  // namespace q1t
