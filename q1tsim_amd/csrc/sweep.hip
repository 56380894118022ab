// Gate-stream planner and multi-gate tile sweeps.
//
// A sweep streams the state once through LDS in tiles of 2^M amplitudes.
// The tile's M local bits are the L lowest index bits (so every tile is made
// of 2^L-element contiguous runs: coalesced HBM traffic) plus up to M-L other
// bits chosen by the planner.  Inside a tile every thread keeps 2^R
// amplitudes in registers; a "phase" fixes which R local bits live in
// registers, so one-qubit updates on those bits are pure register work and a
// phase change is one LDS exchange.  Controls and diagonal gates need no
// local bits: controls outside the tile are a per-tile predicate, a diagonal
// factor on an outer bit is a per-tile constant.
#include "sweep.h"

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>
#include <cmath>
#include <cstring>
#include <map>
#include <set>

#include "costmodel.h"
#include "jit.h"
#include "kernels.h"
#include "sweep_dev.h"

namespace q1t {

#define SW_HIP_OK(expr)                                                                            \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            throw Error(e_ == hipErrorOutOfMemory ? ERR_OUT_OF_MEMORY : ERR_HIP,                    \
                        std::string("HIP error in " #expr ": ") + hipGetErrorString(e_));          \
    } while (0)

template <typename V> __device__ __forceinline__ void warm_sweep(const SweepArgs& sa)
{
    warm_program(sa.phases, uint32_t(sa.nphases) * uint32_t(sizeof(SwPhase)));
    if (sa.nops) warm_program(sa.ops, sa.nops * uint32_t(sizeof(InterpOpT<typename RealOf<V>::type>)));
}

// UNSET: launches with SweepArgs::unset bits, in a kernel of their own (the
// load that takes them costs the sweeps without).
// complex64 with 16 amplitudes per thread is held to 4 waves per SIMD (24 qubits
// 979 us when it took 44 bytes of scratch to get there, at 3 waves 1092 us).
template <typename V, int M, int R, int SW, int BLK, bool UNSET>
__global__ void __launch_bounds__(1 << (M - R))
__attribute__((amdgpu_waves_per_eu(sizeof(V) == 8 && M == 12 ? (R == 3 || BLK == 0 ? 4 : 3) : 2)))
k_sweep(V* __restrict__ amp, uint64_t col_stride, SweepArgs sa)
{
    __shared__ V lds[1 << M];
    V* a = amp + uint64_t(blockIdx.y) * col_stride;
    warm_sweep<V>(sa);
    for (uint64_t tile = blockIdx.x; tile < sa.ntiles; tile += gridDim.x) sweep_tile<V, M, R, SW, BLK, BLK == 0 || BLK == 3, UNSET>(a, sa, tile, lds);
}

// Sweeps of many states in one launch: item i covers flattened tiles
// [first_tile[i], first_tile[i+1]) of one state, its columns one after the
// other (column c at amp + c * col_stride, 2^log_ntiles tiles each), with the
// state's program.
struct SweepItem {
    void* amp;
    uint64_t first_tile;
    uint64_t col_stride;
    uint32_t ncols, log_ntiles;
    SweepArgs sa;
};

// The complex64 12-bit tiles with 3 register bits and no fused blocks fit
// 64 VGPRs (8 waves per SIMD, 4 workgroups per CU by LDS) without spilling.
template <typename V, int M, int R, int SW, int BLK>
__global__ void __launch_bounds__(1 << (M - R))
__attribute__((amdgpu_waves_per_eu(BLK == 0 && sizeof(V) == 8 && M == 12 && R == 3 ? 8 : 2)))
k_sweep_batched(const SweepItem* __restrict__ items, int nitems, uint64_t total_tiles, uint32_t chunk)
{
    __shared__ V lds[1 << M];
    // grid-stride over runs of `chunk` consecutive tiles: a workgroup keeps
    // one item (and its program, in the scalar cache) for a whole run, while
    // neighbouring workgroups still read neighbouring tiles
    const uint64_t nchunks = (total_tiles + chunk - 1) / chunk;
    for (uint64_t j = blockIdx.x; j < nchunks; j += gridDim.x) {
        const uint64_t t0 = j * chunk;
        const uint64_t t1 = t0 + chunk < total_tiles ? t0 + chunk : total_tiles;
        int lo = 0, hi = nitems - 1;   // last item with first_tile <= t0
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (items[mid].first_tile <= t0) lo = mid;
            else hi = mid - 1;
        }
        warm_sweep<V>(items[lo].sa);
        for (uint64_t t = t0; t < t1; ++t) {
            while (lo + 1 < nitems && items[lo + 1].first_tile <= t) ++lo;
            const SweepItem& it = items[lo];
            const uint64_t lt = t - it.first_tile;
            V* a = static_cast<V*>(it.amp) + (lt >> it.log_ntiles) * it.col_stride;
            sweep_tile<V, M, R, SW, BLK, false, false>(a, it.sa, lt & ((uint64_t(1) << it.log_ntiles) - 1), lds);
        }
    }
}

// One batched complex64 sweep round on the kernel holding the round's
// widest block (blk as block_level).
template <int M, int R, int SW>
static void launch_batched_c64(int blk, unsigned gx, hipStream_t stream, const SweepItem* items, int nitems,
                               uint64_t total_tiles, uint32_t chunk)
{
    const dim3 grid(gx), block(1u << (M - R));
    if (blk == 2) hipLaunchKernelGGL((k_sweep_batched<float2, M, R, SW, 2>), grid, block, 0, stream, items, nitems, total_tiles, chunk);
    else if (blk == 1) hipLaunchKernelGGL((k_sweep_batched<float2, M, R, SW, 1>), grid, block, 0, stream, items, nitems, total_tiles, chunk);
    else hipLaunchKernelGGL((k_sweep_batched<float2, M, R, SW, 0>), grid, block, 0, stream, items, nitems, total_tiles, chunk);
}

template <typename V, int M, int R, int SW>
static int launch_sweep(GpuVectorState& st, const PlanStep& step, const SwPhase* dphases, int nphases,
                         const SwOp* dops, int nops, const float* dblocks, size_t cb, size_t ce, int blk,
                         uint64_t unset, double bytes, hipFunction_t jit = nullptr)
{
    const int n = int(st.nr_bits());
    SweepArgs sa{};
    sa.ntiles = uint64_t(1) << (n - M);
    sa.tset.cnt = M;
    for (int j = 0; j < M; ++j) {
        sa.tset.s[j] = step.tile[j];
        sa.tpos[j] = step.tile[j];
    }
    sa.phases = dphases;
    sa.ops = dops;
    sa.blocks = dblocks;
    sa.nphases = nphases;
    sa.nops = uint32_t(nops);
    sa.unset = unset;
    const uint64_t dim = uint64_t(1) << n;
    // far more workgroups than the chip holds (1024): they start as others
    // finish, and loads, stores and arithmetic of neighbours spread out in
    // time.  28 qubits complex64, 10 sweeps: 512 workgroups 27.4 ms, 2048 18.7,
    // 16384 17.1, one per tile 17.4; specialised kernels, 30 qubits complex128:
    // 2048 89.0 ms, 16384 85.2.
    // Sweeps that skip tiles too: one workgroup per tile costs them 0.9 ms at
    // 2^18 tiles.
    const unsigned gx = unsigned(std::min<uint64_t>(sa.ntiles, 16384));
    int first = -1;
    for (size_t c0 = cb; c0 < ce; c0 += 65535) {
        const unsigned ny = unsigned(std::min<size_t>(65535, ce - c0));
        const int ps = st.prof_begin();
        if (first < 0) first = ps;
        if (jit) {
            // the kernel specialised to this program: same grid, block and arguments
            V* amp = static_cast<V*>(st.col_ptr(c0));
            uint64_t stride = dim;
            void* args[] = {&amp, &stride, &sa};
            SW_HIP_OK(hipModuleLaunchKernel(jit, gx, ny, 1, 1u << (M - R), 1, 1, 0, st.stream(), args, nullptr));
            st.prof_end(ps, sizeof(V) == 16 ? "q1t_jit_sweep_c128" : "q1t_jit_sweep_c64",
                        bytes * ny);
            continue;
        }
        V* amp = static_cast<V*>(st.col_ptr(c0));
        auto k = unset ? k_sweep<V, M, R, SW, 0, true> : k_sweep<V, M, R, SW, 0, false>;
        if (blk == 3) k = unset ? k_sweep<V, M, R, SW, 3, true> : k_sweep<V, M, R, SW, 3, false>;
        if constexpr (sizeof(V) == 8) {
            if (blk == 2) k = unset ? k_sweep<V, M, R, SW, 2, true> : k_sweep<V, M, R, SW, 2, false>;
            else if (blk == 1) k = unset ? k_sweep<V, M, R, SW, 1, true> : k_sweep<V, M, R, SW, 1, false>;
        }
        hipLaunchKernelGGL(k, dim3(gx, ny), dim3(1 << (M - R)), 0, st.stream(), amp, dim, sa);
        SW_HIP_OK(hipGetLastError());
        st.prof_end(ps, sizeof(V) == 16 ? "k_sweep_c128" : "k_sweep_c64", bytes * ny);
    }
    return first;
}

// Bytes of a program's ops as its kernel reads them, and the ops written so.
static size_t op_bytes(Precision prec, bool jit)
{
    return jit ? sizeof(SwOp) : prec == PREC_C128 ? sizeof(InterpOpT<double>) : sizeof(InterpOpT<float>);
}
static void put_ops(char* to, const std::vector<SwOp>& ops, Precision prec, bool jit)
{
    if (jit) {
        std::memcpy(to, ops.data(), ops.size() * sizeof(SwOp));
        return;
    }
    for (size_t i = 0; i < ops.size(); ++i) {
        if (prec == PREC_C128) reinterpret_cast<InterpOpT<double>*>(to)[i] = interp_op<double>(ops[i], false);
        else reinterpret_cast<InterpOpT<float>*>(to)[i] = interp_op<float>(ops[i], false);
    }
}

// The widest fused dense block of a program, as the kernels' BLK: 0 none,
// 1 blocks of 3 and 4 qubits, 2 wider ones; 3 dense pairs, which no program with
// blocks has (kernels of their own too: the pairs' registers would spill in the
// complex64 kernel of the others).
static int block_level(const std::vector<SwPhase>& phases)
{
    int lv = 0;
    for (const SwPhase& ph : phases) {
        if (ph.kind == 1) lv = std::max(lv, ph.reg_mask > 4 ? 2 : 1);
        if (ph.kind == 4) lv = 3;
    }
    return lv;
}

// ------------------------------------------------- whole states in LDS

constexpr int whole_regs(int n) { return n <= 13 ? 3 : 4; }   // register bits: at most 1024 threads
static int whole_bits(int n) { return std::max(n, whole_regs(n)); }

// One column of up to 2^14 amplitudes per workgroup, in LDS from its load to
// its store: 2^R amplitudes per thread in registers, the program's register
// phases as in the tile sweeps, one LDS exchange and barrier per phase.  Bound
// by latency: a few waves per SIMD, each op a uniform branch; so the next op's
// record is loaded while the current one runs.  Waves past the column's
// threads leave at once (barriers count the waves that are left).
// Before, one launch per gate (single states: 3.2 us per gate at 12 qubits) or
// one barrier and a full LDS pass per gate (batches: 9 us per gate at 13
// qubits).  Measured: 12 qubits complex128, 350 gates 1110 -> 115 us; 112
// columns of 10 to 13 qubits complex64 in a batch 2850 -> 150 us per round.
template <typename V, int R>
__global__ void __launch_bounds__(1024) k_whole(const WholeItem* __restrict__ items, uint64_t col_stride,
                                                const WholePhase* __restrict__ phases,
                                                const InterpOpT<typename RealOf<V>::type>* __restrict__ ops)
{
    constexpr int NR = 1 << R;
    extern __shared__ unsigned char smem_whole[];
    V* s = reinterpret_cast<V*>(smem_whole);
    const WholeItem it = load_uniform(items, col_stride ? 0u : blockIdx.x);
    const int M = int(it.n) > R ? int(it.n) : R, sw = sweep_swizzle_bits(M);
    const uint32_t nth = 1u << (M - R), N = 1u << it.n, tid = threadIdx.x;
    const uint32_t nops = it.nphases ? load_uniform(phases, it.phases + it.nphases - 1).op_end : 0u;
    if (it.nphases) warm_program(phases + it.phases, it.nphases * uint32_t(sizeof(WholePhase)));
    if (nops) warm_program(ops + it.ops, nops * uint32_t(sizeof(InterpOpT<typename RealOf<V>::type>)));
    if (tid >= nth) return;
    V* a = static_cast<V*>(it.amp) + uint64_t(blockIdx.x) * col_stride;
    {
        V x[NR];
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const uint32_t l = tid + uint32_t(k) * nth;
            x[k] = mkc<V>(it.fresh && l == 0 ? 1 : 0, 0);
            if (l < N && !it.fresh) x[k] = a[l];
        }
#pragma unroll
        for (int k = 0; k < NR; ++k) s[swizzle_slot(sw, M, int(tid + uint32_t(k) * nth))] = x[k];
    }
    __syncthreads();
    for (uint32_t p = 0; p < it.nphases; ++p) {
        const WholePhase ph = load_uniform(phases, it.phases + p);
        uint32_t t = ph.wxor << 16;
#pragma unroll
        for (int b = 0; b < 10; ++b) t ^= (0u - ((tid >> b) & 1u)) & ph.col[b];
        const uint32_t tin = t & 0xffffu, tout = t >> 16;
        V v[NR];
#pragma unroll
        for (int k = 0; k < NR; ++k) v[k] = s[tin ^ (ph.slot[k] & 0xffffu)];
        const uint32_t o1 = it.ops + ph.op_end;
        uint32_t oi = it.ops + ph.op_begin;
        V lane = mkc<V>(1, 0);
        InterpOpT<typename RealOf<V>::type> nxt = load_uniform(ops, oi);   // the table ends with a spare record
        while (oi < o1) {
            const InterpOpT<typename RealOf<V>::type> op = nxt;
            ++oi;
            nxt = load_uniform(ops, oi);
            interp_op<V, NR, R, true, false>(op, v, tid, 0, lane);
        }
        if (ph.wmap == 0) {
#pragma unroll
            for (int k = 0; k < NR; ++k) s[tin ^ (ph.slot[k] & 0xffffu)] = v[k];
        } else {
            __syncthreads();   // other threads' slots are overwritten
#pragma unroll
            for (int k = 0; k < NR; ++k) s[tout ^ (ph.slot[k] >> 16)] = v[k];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const uint32_t l = tid + uint32_t(k) * nth;
        if (l < N) a[l] = s[swizzle_slot(sw, M, int(l))];
    }
}

// `ncols` columns of states of at most n_max qubits (the LDS and threads of
// the widest): an item each, or one item for columns at stride col_stride.
// Tables in device memory; the op table ends with a spare record.
template <typename V>
static void launch_whole(int n_max, const WholeItem* items, size_t ncols, uint64_t col_stride,
                         const WholePhase* phases, const InterpOpT<typename RealOf<V>::type>* ops, hipStream_t stream)
{
    const int R = whole_regs(n_max), M = whole_bits(n_max);
    const size_t lds = sizeof(V) << M;
    const dim3 grid{unsigned(ncols)}, block{unsigned(std::max(64, 1 << (M - R)))};
    auto go = [&](auto kernel) {
        if (lds > (size_t(64) << 10))
            SW_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, items, col_stride, phases, ops);
    };
    if (R == 3) go(&k_whole<V, 3>);
    else if constexpr (sizeof(V) == 8) go(&k_whole<V, 4>);
    else throw Error(ERR_INVALID_ARGUMENT, "No whole-state kernel for 2^14 complex128 amplitudes");
    SW_HIP_OK(hipGetLastError());
}

// The programs of a small state's whole-state steps, appended to `phases` and
// `ops` (records of one step: phases [ph0[s], ph0[s] + nph[s]), ops from op0[s]).
template <typename R> struct WholeTables {
    std::vector<WholePhase> phases;
    std::vector<InterpOpT<R>> ops;
    std::vector<uint32_t> ph0, nph, op0;
    void build(const std::vector<PendingGate>& q, const std::vector<PlanStep>& steps, int n)
    {
        ph0.assign(steps.size(), 0);
        nph.assign(steps.size(), 0);
        op0.assign(steps.size(), 0);
        for (size_t s = 0; s < steps.size(); ++s) {
            if (!steps[s].sweep) continue;
            std::vector<WholePhase> p;
            std::vector<InterpOpT<R>> o;
            build_whole<R>(q, steps[s], whole_bits(n), whole_regs(n), p, o);
            ph0[s] = uint32_t(phases.size());
            nph[s] = uint32_t(p.size());
            op0[s] = uint32_t(ops.size());
            phases.insert(phases.end(), p.begin(), p.end());
            ops.insert(ops.end(), o.begin(), o.end());
        }
    }
};

// One sweep's program: phases, ops and its own block table (block phases
// index it through op_begin until the table is merged into the flush's).
struct SweepProgram {
    std::vector<SwPhase> phases;
    std::vector<SwOp> ops;
    std::vector<float> blocks;
    int nblocks = 0;
};

// kind 0: per-gate register phases; 3 .. 6: dense blocks of that width
static SweepProgram build_candidate(const std::vector<PendingGate>& q, const PlanStep& step, const TileGeom& g,
                                    int kind, bool search, bool factors)
{
    SweepProgram p;
    if (kind == 0) build_program(q, step, g.M, g.R, p.phases, p.ops, search, nullptr, factors);
    else build_fused_program(q, step, g.M, g.R, kind, p.phases, p.ops, p.blocks, &p.nblocks, search, factors);
    return p;
}

// The reduced programs of a flush (sweeps with dense blocks stay as they are):
// the factor taken out of the gates goes back in with the last of them that
// has a register phase.
static void reduce_programs(std::vector<SweepProgram>& progs, Precision prec)
{
    auto reducible = [](const SweepProgram& p) {
        const int lv = block_level(p.phases);
        return lv == 0 || lv == 3;
    };
    size_t last = progs.size();
    for (size_t s = 0; s < progs.size(); ++s)
        if (reducible(progs[s]))
            for (const SwPhase& ph : progs[s].phases)
                if (ph.kind == 0) last = s;
    Reduction red;
    for (size_t s = 0; s < progs.size(); ++s)
        if (reducible(progs[s])) reduce_program(progs[s].phases, progs[s].ops, prec, red, s == last);
}

// Wall-time estimate of a gate applied on its own: one read and one write
// of the columns at the measured streaming rate.
static double single_gate_us(double state_bytes) { return 2.0 * state_bytes / 4.9e12 * 1e6; }

// Pick the steps and sweep programs of a flush.  Plain (complex128, or
// complex64 without fusion): per-gate register phases on the greedy tiles.
// Fused complex64: greedy fixed-width blocks (PLAN_GREEDY), or the cheaper of
// two tilings -- the per-gate tiling and the fusion tiling, each sweep of
// either with the cheapest of {register phases, 3-qubit blocks, 4-qubit
// blocks, blocks of the configured width when it is 5 or 6} -- as ranked by
// the learned cost model (PLAN_LEARNED), or a seeded random choice among the
// same candidates (PLAN_EXPLORE).
// A state's last plan (choose_plan): its steps and each sweep's program kind.
struct PlanCacheEntry {
    std::vector<PlanStep> steps;
    std::vector<int> kind;
};

static void choose_plan(GpuVectorState& st, const std::vector<PendingGate>& queue, const TileGeom& g, int fusion_k,
                        double state_bytes, double tiles, std::vector<PlanStep>& steps,
                        std::vector<SweepProgram>& progs)
{
    const int n = int(st.nr_bits());
    const int prec = int(st.precision());
    const bool fused = st.precision() == PREC_C64 && fusion_k > 0;
    const bool search = st.tile_search(fused ? fusion_k : 0, state_bytes);
    const bool phase_search = st.phase_search(state_bytes), keep = st.plan_cache();
    const bool factors = st.tile_factors();   // specialised kernels only
    auto build_all = [&](const std::vector<PlanStep>& ss, int kind) {
        std::vector<SweepProgram> out(ss.size());
        for (size_t s = 0; s < ss.size(); ++s)
            if (ss[s].sweep) out[s] = build_candidate(queue, ss[s], g, kind, phase_search, factors);
        return out;
    };
    // A flush with the previous flush's gate structure (a repeated circuit,
    // new angles allowed) takes that flush's steps and per-sweep program
    // kinds and builds only those programs: the tile searches (and the
    // learned planner's candidates) are most of the planning time.
    std::vector<uint64_t> key;
    auto cache_hit = [&](std::vector<int>& kind) {
        const std::shared_ptr<void>& cached = st.plan_cache_steps();
        if (!cached || key != st.plan_cache_key()) return false;
        const PlanCacheEntry& e = *static_cast<const PlanCacheEntry*>(cached.get());
        steps = e.steps;
        kind = e.kind;
        return true;
    };
    auto cache_store = [&](const std::vector<int>& kind) {
        st.plan_cache_key() = key;
        st.plan_cache_steps() = std::shared_ptr<void>(new PlanCacheEntry{steps, kind},
                                                      [](void* p) { delete static_cast<PlanCacheEntry*>(p); });
    };
    if (!fused) {
        if (keep) {
            key = plan_key(queue, n, g, 0, search);
            key.insert(key.begin(), 1);   // the per-gate planner
            std::vector<int> kind;
            if (!cache_hit(kind)) {
                steps = plan_gates(queue, n, g, 0, search, true);
                cache_store(std::vector<int>(steps.size(), 0));
            }
        } else {
            steps = plan_gates(queue, n, g, 0, search, true);
        }
        progs = build_all(steps, 0);
        return;
    }
    // blocks of 3 to 6 local qubits: block_mfma holds 3 and 4, block_mfma_wide 5 and 6
    const int Kg = std::min(6, std::max(3, fusion_k));
    CostModel* cm = st.cost_model();
    const int mode = st.plan_mode();
    if (mode == PLAN_GREEDY || (mode == PLAN_LEARNED && (!cm || !cm->trained()))) {
        if (keep) {
            key = plan_key(queue, n, g, Kg, search);
            key.insert(key.begin(), 3);   // greedy fusion
            std::vector<int> kind;
            if (!cache_hit(kind)) {
                steps = plan_gates(queue, n, g, Kg, search);
                cache_store(std::vector<int>(steps.size(), Kg));
            }
        } else {
            steps = plan_gates(queue, n, g, Kg, search);
        }
        progs = build_all(steps, Kg);
        return;
    }
    const bool cacheable = keep && mode == PLAN_LEARNED;
    if (cacheable) {
        // both tilings' inputs, the block width, the model, the kernels the
        // predictions are for and the bytes swept (single gates are costed
        // by them)
        key = plan_key(queue, n, g, 0, search);
        const std::vector<uint64_t> k2 = plan_key(queue, n, g, Kg, search);
        key.insert(key.end(), k2.begin(), k2.end());
        key.insert(key.begin(), {2, uint64_t(Kg), reinterpret_cast<uintptr_t>(cm), cm->version(),
                                 uint64_t(st.jit_enabled()), uint64_t(factors), uint64_t(prec),
                                 uint64_t(state_bytes)});
        std::vector<int> kind;
        if (cache_hit(kind)) {
            progs.assign(steps.size(), SweepProgram{});
            for (size_t s = 0; s < steps.size(); ++s)
                if (steps[s].sweep) progs[s] = build_candidate(queue, steps[s], g, kind[s], phase_search, factors);
            return;
        }
    }
    // candidates: tiling A (per-gate tiles) and tiling B (fusion tiles), each
    // sweep of either with one program per block width (0: register phases,
    // 3, 4 and, above 4, fusion_k; in tiling A gates whose controls lie
    // outside the tile stay register ops beside the blocks)
    // (host planning runs on parallel threads: both tilings, then every
    // candidate program; a flush's planning would otherwise rival its kernels
    // on states of a few GiB)
    std::vector<PlanStep> tl[2];
    {
        std::exception_ptr e0, e1;
        std::thread other([&] {
            try {
                tl[1] = plan_gates(queue, n, g, Kg, search);
            } catch (...) {
                e1 = std::current_exception();
            }
        });
        try {
            tl[0] = plan_gates(queue, n, g, 0, search);
        } catch (...) {
            e0 = std::current_exception();
        }
        other.join();
        if (e0) std::rethrow_exception(e0);
        if (e1) std::rethrow_exception(e1);
    }
    std::vector<int> kinds = {0, 3, 4};
    if (Kg > 4) kinds.push_back(Kg);
    const int nk = int(kinds.size());
    std::vector<std::vector<SweepProgram>> cand[2];
    std::vector<int> pick[2];
    std::vector<std::array<size_t, 3>> work;   // (tiling, sweep, candidate)
    for (int t = 0; t < 2; ++t) {
        cand[t].assign(tl[t].size(), std::vector<SweepProgram>(kinds.size()));
        pick[t].assign(tl[t].size(), 0);
        for (size_t s = 0; s < tl[t].size(); ++s)
            if (tl[t][s].sweep)
                for (int c = 0; c < nk; ++c) work.push_back({size_t(t), s, size_t(c)});
    }
    {
        std::atomic<size_t> next{0};
        std::exception_ptr err;
        std::mutex err_mu;
        auto run = [&] {
            try {
                for (size_t i = next++; i < work.size(); i = next++) {
                    const auto& w = work[i];
                    cand[w[0]][w[1]][w[2]] = build_candidate(queue, tl[w[0]][w[1]], g, kinds[w[2]], phase_search, factors);
                }
            } catch (...) {
                std::lock_guard<std::mutex> lk(err_mu);
                if (!err) err = std::current_exception();
            }
        };
        const size_t hw = std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
        const size_t nth = std::min(hw, std::max<size_t>(1, work.size() / 4));
        std::vector<std::thread> pool;
        for (size_t i = 1; i < nth; ++i) pool.emplace_back(run);
        run();
        for (auto& th : pool) th.join();
        if (err) std::rethrow_exception(err);
    }
    int use = 1;
    if (mode == PLAN_EXPLORE) {
        Xoshiro256& rng = st.plan_rng();
        use = int(rng.next() >> 63);
        for (int t = 0; t < 2; ++t)
            for (size_t s = 0; s < tl[t].size(); ++s) pick[t][s] = int(rng.next() % uint64_t(nk));
    } else {
        std::vector<float> feat;
        struct Who {
            int t;
            size_t s;
            int c;
        };
        std::vector<Who> who;
        float f[kSweepFeatures];
        for (int t = 0; t < 2; ++t)
            for (size_t s = 0; s < tl[t].size(); ++s)
                if (tl[t][s].sweep)
                    for (int c = 0; c < nk; ++c) {
                        sweep_features(cand[t][s][c].phases, cand[t][s][c].ops, tl[t][s], prec, g, st.jit_enabled(), f);
                        feat.insert(feat.end(), f, f + kSweepFeatures);
                        who.push_back(Who{t, s, c});
                    }
        std::vector<float> y(who.size());
        cm->predict(feat.data(), who.size(), y.data());
        const double us_per_unit = tiles / 1024.0;   // the model predicts log(us per 1024 tiles)
        std::vector<std::vector<double>> pred[2];
        for (int t = 0; t < 2; ++t) pred[t].assign(tl[t].size(), std::vector<double>(nk, 0.0));
        for (size_t i = 0; i < who.size(); ++i)
            pred[who[i].t][who[i].s][who[i].c] = std::exp(double(y[i])) * us_per_unit;
        // per sweep: blocks replace the register program only when predicted at
        // least 10 % cheaper (the fit's error is ~7 % in time, and a wrong pick
        // of blocks costs more than a missed one); a tiling costs the sum of
        // its chosen programs' predictions
        constexpr double kBlockMargin = 0.9;
        double cost[2] = {0.0, 0.0};
        for (int t = 0; t < 2; ++t)
            for (size_t s = 0; s < tl[t].size(); ++s) {
                if (!tl[t][s].sweep) {
                    cost[t] += single_gate_us(state_bytes) * double(tl[t][s].gates.size());
                    continue;
                }
                int c_best = 0;
                for (int c = 1; c < nk; ++c)
                    if (pred[t][s][c] < kBlockMargin * pred[t][s][c_best] ||
                        (c_best != 0 && pred[t][s][c] < pred[t][s][c_best]))
                        c_best = c;
                pick[t][s] = c_best;
                cost[t] += pred[t][s][c_best];
            }
        use = cost[0] < cost[1] ? 0 : 1;
    }
    steps = std::move(tl[use]);
    progs.resize(steps.size());
    std::vector<int> kind(steps.size(), 0);
    for (size_t s = 0; s < steps.size(); ++s)
        if (steps[s].sweep) {
            progs[s] = std::move(cand[use][s][pick[use][s]]);
            kind[s] = kinds[pick[use][s]];
        }
    if (cacheable) cache_store(kind);
}

std::vector<std::string> plan_jit_sources(const std::vector<PendingGate>& q, int n, Precision prec, int fusion_k,
                                          bool search, bool prefetch, bool factors)
{
    const TileGeom g = tile_geometry_specialised(prec);
    const int K = prec == PREC_C64 && fusion_k > 0 ? std::min(6, std::max(3, fusion_k)) : 0;
    const std::vector<PlanStep> steps = plan_gates(q, n, g, K, search, K == 0);
    std::vector<SweepProgram> progs(steps.size());
    for (size_t s = 0; s < steps.size(); ++s)
        if (steps[s].sweep) progs[s] = build_candidate(q, steps[s], g, K, search, factors);
    reduce_programs(progs, prec);
    std::vector<std::string> out;
    size_t nblk_floats = 0;
    for (size_t s = 0; s < steps.size(); ++s) {
        if (!steps[s].sweep) continue;
        SweepProgram& p = progs[s];
        for (SwPhase& ph : p.phases)
            if (ph.kind == 1) ph.op_begin += uint32_t(nblk_floats);
        nblk_floats += p.blocks.size();
        out.push_back(jit_sweep_source(p.phases, p.ops, prec == PREC_C64, g.M, g.R, sweep_swizzle_bits(g.M), prefetch));
    }
    return out;
}

// The single-gate kernels of a step in a launch signature (they hold their
// matrices by value); false if one cannot be captured.
static bool put_single_gates(const std::vector<PendingGate>& queue, const PlanStep& step, std::vector<uint64_t>& sig)
{
    auto put = [&](uint64_t x) { sig.push_back(x); };
    bool ok = true;
    for (size_t i : step.gates) {
        const GateOp& op = queue[i].op;
        // kernels of 4 and more targets upload their matrix and synchronise;
        // those of 3 run eagerly with them
        if (op.kind == OpKind::Dense && op.targets.size() >= 3) ok = false;
        put(uint64_t(op.kind));
        put(op.ctrl_mask);
        put(op.targets.size());
        for (int t : op.targets) put(uint64_t(t));
        put(op.m.size());
        for (const cdouble& c : op.m) {
            double re = c.real(), im = c.imag();
            uint64_t u;
            std::memcpy(&u, &re, 8);
            put(u);
            std::memcpy(&u, &im, 8);
            put(u);
        }
    }
    return ok;
}

// Uploads a flush's table (`host`: the state's pinned staging memory, which
// the flush's final synchronisation frees for the next one) and launches its
// kernels; with a launch signature, as a graph: replayed while the signature
// repeats, else captured anew.
static void run_table(GpuVectorState& st, const char* host, size_t total, std::vector<uint64_t>* sig,
                      const std::function<void(char*)>& launch_all, RunStats& stats)
{
    auto upload = [&](char* dst) {
        upload_table(dst, host, total, st.stream());
    };
    if (!sig) {
        char* dprog = total ? static_cast<char*>(st.scratch(GpuVectorState::SLOT_PROGRAM, total)) : nullptr;
        upload(dprog);
        launch_all(dprog);
        return;
    }
    if (GpuVectorState::FlushGraph* hit = st.find_graph(*sig)) {
        upload(static_cast<char*>(hit->table));
        SW_HIP_OK(hipGraphLaunch(hit->exec, st.stream()));
        const RunStats& d = hit->delta;
        stats.bytes += d.bytes;
        stats.launches += d.launches;
        stats.sweeps += d.sweeps;
        stats.gates += d.gates;
        stats.blocks += d.blocks;
        stats.phases += d.phases;
        stats.mfma_flops += d.mfma_flops;
        st.note_graph(false);
        return;
    }
    GpuVectorState::FlushGraph& fg = st.new_graph_slot(total);
    char* table = static_cast<char*>(fg.table);
    upload(table);
    const RunStats before = stats;
    SW_HIP_OK(hipStreamBeginCapture(st.stream(), hipStreamCaptureModeThreadLocal));
    try {
        launch_all(table);
    } catch (...) {
        hipGraph_t part = nullptr;
        (void)hipStreamEndCapture(st.stream(), &part);
        if (part) (void)hipGraphDestroy(part);
        throw;
    }
    hipGraph_t gr = nullptr;
    SW_HIP_OK(hipStreamEndCapture(st.stream(), &gr));
    hipGraphExec_t exec = nullptr;
    const hipError_t ie = hipGraphInstantiate(&exec, gr, nullptr, nullptr, 0);
    (void)hipGraphDestroy(gr);
    SW_HIP_OK(ie);
    fg.exec = exec;
    fg.sig = std::move(*sig);
    fg.delta = RunStats{};
    fg.delta.bytes = stats.bytes - before.bytes;
    fg.delta.launches = stats.launches - before.launches;
    fg.delta.sweeps = stats.sweeps - before.sweeps;
    fg.delta.gates = stats.gates - before.gates;
    fg.delta.blocks = stats.blocks - before.blocks;
    fg.delta.mfma_flops = stats.mfma_flops - before.mfma_flops;
    fg.delta.phases = stats.phases - before.phases;
    st.note_graph(true);
    SW_HIP_OK(hipGraphLaunch(exec, st.stream()));
}

// Gates up to which a run of a small state goes to the single-gate kernels (2.9 us
// a gate, with the rounding of k_whole): a launch of k_whole reads its program
// first and holds a column in one workgroup.  us per two-qubit unitary and run of
// gates, k_whole / single kernels: complex128, 8 qubits 1 gate 8.4 / 7.1, 2 gates
// 8.4 / 10.4; 12 qubits 1 10.3 / 7.3, 2 10.5 / 10.4, 3 11.2 / 13.4; 13 qubits 2 12.6 /
// 10.5, 3 13.4 / 13.3, 4 14.6 / 16.7; complex64, 12 qubits 1 9.9 / 7.2, 2 10.2 / 10.5;
// 13 qubits 2 10.5 / 10.3, 3 11.1 / 13.2; 512 columns of 12 qubits complex128 1 26.6 /
// 23.5, 2 26.9 / 33.4.  Where the run is the whole flush, one gate more saves the
// table's upload (8 qubits, 2 gates 17.5 / 14.6, 3 gates 18.2 / 17.2, 4 18.6 / 19.4).
static size_t lone_gates(int n, size_t ncols, size_t elem_bytes, bool whole_flush)
{
    const uint64_t amps = uint64_t(ncols) << n;
    const int few = amps > (uint64_t(1) << 20) ? 1 : std::max(1, n - (elem_bytes == 16 ? 10 : 11));
    return size_t(few) + (whole_flush && amps <= (uint64_t(1) << 17));
}

// A flush of a state that is too small for tiles: whole-state programs
// (k_whole), one launch for all columns, and single-gate kernels for the gates
// no register phase takes and for short runs of gates.
template <typename V>
static void run_whole(GpuVectorState& st, const std::vector<PendingGate>& queue, size_t col_begin, size_t col_end,
                      bool fresh, RunStats& stats)
{
    using R = typename RealOf<V>::type;
    const int n = int(st.nr_bits());
    const size_t ncols = col_end - col_begin;
    bool graph = st.graph_enabled();
    std::vector<PlanStep> steps = plan_whole(queue, whole_bits(n));
    // not for a graph, which replays programs with new angles but no single gates,
    // nor for the first gates of an unwritten state
    if (!graph) {
        const size_t few = lone_gates(n, ncols, sizeof(V), steps.size() == 1);
        for (size_t s = fresh ? 1 : 0; s < steps.size(); ++s)
            if (steps[s].gates.size() <= few) steps[s].sweep = false;
    }
    WholeTables<R> wt;
    wt.build(queue, steps, n);
    bool any = false;   // a step of k_whole
    for (const PlanStep& step : steps) any = any || step.sweep;
    wt.ops.push_back(InterpOpT<R>{});   // the spare record
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    const size_t ooff = up(wt.phases.size() * sizeof(WholePhase));
    const size_t ioff = up(ooff + wt.ops.size() * sizeof(InterpOpT<R>));
    const size_t total = any ? up(ioff + steps.size() * sizeof(WholeItem)) : 0;
    char* const host = any ? st.stage(total) : nullptr;
    if (any) {
        std::memcpy(host, wt.phases.data(), wt.phases.size() * sizeof(WholePhase));
        std::memcpy(host + ooff, wt.ops.data(), wt.ops.size() * sizeof(InterpOpT<R>));
        WholeItem* items = reinterpret_cast<WholeItem*>(host + ioff);   // one per step, of its first column
        for (size_t s = 0; s < steps.size(); ++s)
            items[s] = WholeItem{st.col_ptr(col_begin), uint32_t(n), wt.nph[s], wt.ph0[s], wt.op0[s], fresh && s == 0, 0};
    }
    if (fresh && (steps.empty() || !steps[0].sweep)) st.write_zero_state();
    const double S = double(uint64_t(1) << n) * sizeof(V) * double(ncols);
    auto launch_all = [&](char* d) {
        for (size_t s = 0; s < steps.size(); ++s) {
            if (!steps[s].sweep) {
                for (size_t i : steps[s].gates) st.apply_op(queue[i].op, col_begin, col_end, true);
                continue;
            }
            const int ps = st.prof_begin();
            launch_whole<V>(n, reinterpret_cast<const WholeItem*>(d + ioff) + s, ncols, uint64_t(1) << n,
                            reinterpret_cast<const WholePhase*>(d),
                            reinterpret_cast<const InterpOpT<R>*>(d + ooff), st.stream());
            st.prof_end(ps, sizeof(V) == 16 ? "k_whole_c128" : "k_whole_c64", 2.0 * S);
            stats.launches += 1;
            stats.sweeps += 1;
            stats.gates += steps[s].gates.size();
            stats.bytes += 2.0 * S;
            stats.phases += wt.nph[s];
        }
    };
    std::vector<uint64_t> sig;
    if (graph) {
        for (uint64_t x : {uint64_t(n), uint64_t(st.precision()), uint64_t(col_begin), uint64_t(col_end),
                           uint64_t(total), uint64_t(ooff), uint64_t(ioff),
                           uint64_t(reinterpret_cast<uintptr_t>(st.col_ptr(col_begin)))})
            sig.push_back(x);
        for (const PlanStep& step : steps) {
            sig.push_back(step.sweep ? 1 : 0);
            if (!step.sweep) graph = put_single_gates(queue, step, sig) && graph;
        }
    }
    run_table(st, host, total, graph ? &sig : nullptr, launch_all, stats);
}

void run_planned(GpuVectorState& st, const std::vector<PendingGate>& queue, size_t col_begin, size_t col_end,
                 int fusion_k, bool tiling, bool fresh, RunStats& stats)
{
    const int n = int(st.nr_bits());
    TileGeom g = st.geometry();
    if (!tiling) {
        for (const PendingGate& pg : queue) st.apply_op(pg.op, col_begin, col_end);
        return;
    }
    if (n < g.M + 2) {
        if (st.precision() == PREC_C128) run_whole<double2>(st, queue, col_begin, col_end, fresh, stats);
        else run_whole<float2>(st, queue, col_begin, col_end, fresh, stats);
        return;
    }
    const double S = double(uint64_t(1) << n) * double(st.elem_bytes()) * double(col_end - col_begin);
    const double tiles = double(col_end - col_begin) * double(uint64_t(1) << std::max(0, n - g.M));
    // complex64 interpreter with at most two tiles per CU: a sweep lasts as
    // long as one tile, so 8 amplitudes per thread and twice the waves win
    // over fewer phases.  12 layers, kernel time R=3 / R=4: 16 qubits 106 /
    // 119 us, 20 qubits 140 / 157, 21 qubits 188 / 199, 22 qubits 328 / 261.
    if (st.precision() == PREC_C64 && !st.geometry_set() && !st.jit_enabled() && fusion_k == 0 && tiles <= 512.0)
        g.R = 3;
    std::vector<PlanStep> steps;
    std::vector<SweepProgram> progs;
    choose_plan(st, queue, g, fusion_k, S, tiles, steps, progs);
    // recorded sweeps carry the features the planner predicts from: those of
    // the programs as it chose them
    std::vector<std::array<float, kSweepFeatures>> feat(st.recording() ? steps.size() : 0);
    for (size_t s = 0; s < feat.size(); ++s)
        if (steps[s].sweep)
            sweep_features(progs[s].phases, progs[s].ops, steps[s], int(st.precision()), g, st.jit_enabled(),
                           feat[s].data());
    reduce_programs(progs, st.precision());
    for (SweepProgram& p : progs) place_phases(p.phases, g.M, g.R, st.elem_bytes());

    // all sweep programs of this flush in one upload: [phases][ops] per sweep, then the block table
    std::vector<size_t> poff(steps.size()), ooff(steps.size()), boff_s(steps.size());
    size_t total = 0, nblk_floats = 0;
    int nblocks = 0;
    for (size_t s = 0; s < steps.size(); ++s) {
        if (!steps[s].sweep) continue;
        poff[s] = total;
        total += (progs[s].phases.size() * sizeof(SwPhase) + 255) / 256 * 256;
        ooff[s] = total;
        total += (progs[s].ops.size() * op_bytes(st.precision(), st.jit_enabled()) + 255) / 256 * 256;
        boff_s[s] = nblk_floats;
        nblk_floats += progs[s].blocks.size();
        nblocks += progs[s].nblocks;
    }
    const size_t boff = total;
    total += (nblk_floats * sizeof(float) + 15) / 16 * 16;
    char* const host = st.stage(total);
    for (size_t s = 0; s < steps.size(); ++s) {
        if (!steps[s].sweep) continue;
        // block phases address the merged table
        for (SwPhase& ph : progs[s].phases)
            if (ph.kind == 1) ph.op_begin += uint32_t(boff_s[s]);
        std::memcpy(host + poff[s], progs[s].phases.data(), progs[s].phases.size() * sizeof(SwPhase));
        put_ops(host + ooff[s], progs[s].ops, st.precision(), st.jit_enabled());
        if (!progs[s].blocks.empty())
            std::memcpy(host + boff + boff_s[s] * sizeof(float), progs[s].blocks.data(),
                        progs[s].blocks.size() * sizeof(float));
    }
    // A state still |0..0> (`fresh`, one column, none of it in memory): each
    // sweep's unset bits, and the bytes a column moves.  Gates between sweeps
    // and bits that no sweep reaches need the zeros in memory.
    std::vector<uint64_t> unset(steps.size(), 0);
    std::vector<double> col_bytes(steps.size(), 2.0 * std::ldexp(double(st.elem_bytes()), n));
    if (fresh) {
        const uint64_t all = (uint64_t(1) << n) - 1;
        uint64_t un = ~uint64_t(0);
        bool zeros = false;
        for (size_t s = 0; s < steps.size(); ++s) {
            if (!steps[s].sweep) {
                zeros = zeros || un != 0;
                un = 0;
                continue;
            }
            unset[s] = un & all ? un : 0;
            const double read = un == ~uint64_t(0) ? 0.0 : std::ldexp(1.0, __builtin_popcountll(~un & all));
            for (int b : steps[s].tile) un &= ~(uint64_t(1) << b);
            col_bytes[s] = (read + std::ldexp(1.0, __builtin_popcountll(~un & all))) * double(st.elem_bytes());
        }
        if (zeros || (un & all)) st.write_zero_state();
    }
    // kernels specialised to each sweep's program (compiled on first use)
    std::vector<hipFunction_t> jitfn(steps.size(), nullptr);
    if (st.jit_enabled()) {
        std::vector<std::string> src(steps.size());
        std::vector<std::string> all;
        for (size_t s = 0; s < steps.size(); ++s)
            if (steps[s].sweep) {
                src[s] = jit_sweep_source(progs[s].phases, progs[s].ops, st.precision() == PREC_C64, g.M, g.R,
                                          sweep_swizzle_bits(g.M), st.jit_prefetch(), unset[s] != 0);
                all.push_back(src[s]);
            }
        JitCache& jc = JitCache::get();
        jc.compile_all(all);
        for (size_t s = 0; s < steps.size(); ++s)
            if (steps[s].sweep) jitfn[s] = jc.function(src[s], false);
    }
    auto launch_all = [&](char* dprog) {
        const float* dblocks = reinterpret_cast<const float*>(dprog + boff);
        for (size_t s = 0; s < steps.size(); ++s) {
            const PlanStep& step = steps[s];
            if (!step.sweep) {
                for (size_t i : step.gates) st.apply_op(queue[i].op, col_begin, col_end);
                continue;
            }
            const SwPhase* dp = reinterpret_cast<const SwPhase*>(dprog + poff[s]);
            const SwOp* dop = reinterpret_cast<const SwOp*>(dprog + ooff[s]);
            const int np = int(progs[s].phases.size());
            const int blk = block_level(progs[s].phases);
            int slot;
            // the compiled tile shapes (M local bits, R register bits): see tile_shape_supported()
            const hipFunction_t jf = jitfn[s];
            if (!jf)
                for (const SwPhase& ph : progs[s].phases)
                    if (ph.kind == 2) throw Error(ERR_HIP, "A sweep program with tile factors needs its specialised kernel");
            const int shape = g.M * 16 + g.R;
            if (st.precision() == PREC_C128) {
                switch (shape) {
                case 12 * 16 + 3: slot = launch_sweep<double2, 12, 3, 4>(st, step, dp, np, dop, int(progs[s].ops.size()), dblocks, col_begin, col_end, blk, unset[s], col_bytes[s], jf); break;
                case 12 * 16 + 4: slot = launch_sweep<double2, 12, 4, 4>(st, step, dp, np, dop, int(progs[s].ops.size()), dblocks, col_begin, col_end, blk, unset[s], col_bytes[s], jf); break;
                default: throw Error(ERR_INVALID_ARGUMENT, "No sweep kernel for this complex128 tile shape");
                }
            } else {
                switch (shape) {
                case 13 * 16 + 4: slot = launch_sweep<float2, 13, 4, 5>(st, step, dp, np, dop, int(progs[s].ops.size()), dblocks, col_begin, col_end, blk, unset[s], col_bytes[s], jf); break;
                case 12 * 16 + 3: slot = launch_sweep<float2, 12, 3, 4>(st, step, dp, np, dop, int(progs[s].ops.size()), dblocks, col_begin, col_end, blk, unset[s], col_bytes[s], jf); break;
                case 12 * 16 + 4: slot = launch_sweep<float2, 12, 4, 4>(st, step, dp, np, dop, int(progs[s].ops.size()), dblocks, col_begin, col_end, blk, unset[s], col_bytes[s], jf); break;
                default: throw Error(ERR_INVALID_ARGUMENT, "No sweep kernel for this complex64 tile shape");
                }
            }
            if (st.recording() && col_end - col_begin <= 65535) st.add_sample(feat[s].data(), tiles, slot);
            stats.launches += 1;
            stats.sweeps += 1;
            stats.gates += step.gates.size();
            stats.bytes += col_bytes[s] * double(col_end - col_begin);
            stats.phases += progs[s].phases.size();
            for (const SwPhase& ph : progs[s].phases)
                if (ph.kind == 1)
                    stats.mfma_flops += std::ldexp(double(col_end - col_begin), n + int(ph.reg_mask) + 3);
        }
        stats.blocks += uint64_t(nblocks);
    };

    bool graph = st.graph_enabled();
    std::vector<uint64_t> sig;
    if (graph) {
        // the launch signature: everything a captured launch holds by value
        auto put = [&](uint64_t x) { sig.push_back(x); };
        put(reinterpret_cast<uintptr_t>(st.col_ptr(col_begin)));
        put(col_begin);
        put(col_end);
        put(uint64_t(n));
        put(uint64_t(st.precision()));
        put(uint64_t(g.M));
        put(uint64_t(g.R));
        put(total);
        put(boff);
        put(steps.size());
        for (size_t s = 0; s < steps.size() && graph; ++s) {
            put(steps[s].sweep ? 1 : 0);
            if (steps[s].sweep) {
                // a specialised kernel holds the program's structure in its code
                put(reinterpret_cast<uintptr_t>(jitfn[s]));
                for (int b : steps[s].tile) put(uint64_t(b));
                put(poff[s]);
                put(ooff[s]);
                put(progs[s].phases.size());
                put(uint64_t(block_level(progs[s].phases)));
                continue;
            }
            graph = put_single_gates(queue, steps[s], sig);
        }
    }
    run_table(st, host, total, graph ? &sig : nullptr, launch_all, stats);
}

// ------------------------------------------------------------- batches

void* DeviceBuffer::get(size_t bytes, hipStream_t stream)
{
    if (bytes > cap) {
        SW_HIP_OK(hipStreamSynchronize(stream));
        if (ptr) SW_HIP_OK(hipFree(ptr));
        ptr = nullptr;
        cap = 0;
        const size_t c = std::max<size_t>(bytes, size_t(1) << 20);
        SW_HIP_OK(hipMalloc(&ptr, c));
        cap = c;
    }
    return ptr;
}

DeviceBuffer::~DeviceBuffer()
{
    if (ptr) (void)hipFree(ptr);
}

void* PinnedBuffer::get(size_t bytes)
{
    if (bytes > cap) {
        if (ptr) SW_HIP_OK(hipHostFree(ptr));
        ptr = nullptr;
        cap = 0;
        const size_t c = std::max<size_t>(bytes, size_t(1) << 20) * 3 / 2;
        SW_HIP_OK(hipHostMalloc(&ptr, c, hipHostMallocDefault));
        cap = c;
    }
    return ptr;
}

PinnedBuffer::~PinnedBuffer()
{
    if (ptr) (void)hipHostFree(ptr);
}

void run_planned_batch(const std::vector<GpuVectorState*>& states, hipStream_t stream, DeviceBuffer& prog,
                       PinnedBuffer& stage, ItemQueue& iq, RunStats& agg, unsigned tile_chunk, double* plan_s,
                       double* pack_s)
{
    const auto t_plan = std::chrono::steady_clock::now();
    if (tile_chunk == 0) throw Error(ERR_INVALID_ARGUMENT, "tile chunk must be at least 1");
    std::vector<GpuVectorState*> live;
    for (GpuVectorState* s : states)
        if (!s->pending().empty()) {
            s->prepare_batched_flush(iq);
            live.push_back(s);
        }
    if (!iq.empty()) iq.launch(stream);   // compact columns written out before the sweeps
    if (live.empty()) return;
    const Precision prec = live[0]->precision();
    const TileGeom g = live[0]->geometry();
    const int K = (prec == PREC_C64 && live[0]->fusion() > 0) ? std::min(6, std::max(3, live[0]->fusion())) : 0;
    for (GpuVectorState* s : live)
        if (s->precision() != prec || s->geometry().M != g.M || s->geometry().R != g.R)
            throw Error(ERR_INVALID_ARGUMENT, "A batch needs one precision and tile shape");

    // 1. plans and programs (host): each state on its own, in parallel over
    // host threads; then merged into one upload
    struct Plan {
        std::vector<PlanStep> steps;
        std::vector<std::vector<SwPhase>> ph;
        std::vector<std::vector<SwOp>> ops;
        std::vector<float> blocks;
        WholeTables<double> wd;   // small states: the programs of their precision
        WholeTables<float> wf;
        std::vector<size_t> poff, ooff;
        std::vector<int> nph;
        std::vector<char> blk;    // per step: block_level of its program
        bool small = false;
        RunStats st;
        std::string error;
    };
    std::vector<Plan> plans(live.size());
    auto plan_one = [&](size_t i) {
        GpuVectorState& st = *live[i];
        const std::vector<PendingGate>& q = st.pending();
        Plan& p = plans[i];
        const int n = int(st.nr_bits());
        const double S = double(uint64_t(1) << n) * double(st.elem_bytes()) * double(st.nr_cols());
        if (n < g.M + 2) {
            p.small = true;
            p.steps = plan_whole(q, whole_bits(n));
            if (prec == PREC_C128) p.wd.build(q, p.steps, n);
            else p.wf.build(q, p.steps, n);
            const std::vector<uint32_t>& nph = prec == PREC_C128 ? p.wd.nph : p.wf.nph;
            for (size_t s = 0; s < p.steps.size(); ++s) {
                if (!p.steps[s].sweep) continue;
                p.st.sweeps += 1;
                p.st.launches += 1;
                p.st.gates += p.steps[s].gates.size();
                p.st.bytes += 2.0 * S;
                p.st.phases += nph[s];
            }
            return;
        }
        const bool search = live[i]->phase_search(S);
        // complex64: the greedy tiles, whose order of the gates' rounding a
        // seeded batch's outcomes depend on
        p.steps = plan_gates(q, n, g, K, prec == PREC_C128 ? live[i]->tile_search(0, S) : search);
        p.ph.resize(p.steps.size());
        p.ops.resize(p.steps.size());
        int nblocks = 0;
        for (size_t s = 0; s < p.steps.size(); ++s) {
            if (!p.steps[s].sweep) continue;
            if (K) build_fused_program(q, p.steps[s], g.M, g.R, K, p.ph[s], p.ops[s], p.blocks, &nblocks, search);
            else build_program(q, p.steps[s], g.M, g.R, p.ph[s], p.ops[s], search);
            place_phases(p.ph[s], g.M, g.R, st.elem_bytes());
            p.st.sweeps += 1;
            p.st.launches += 1;
            p.st.gates += p.steps[s].gates.size();
            p.st.bytes += 2.0 * S;
            p.st.phases += p.ph[s].size();
        }
        p.st.blocks = uint64_t(nblocks);
    };
    {
        const size_t hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
        const size_t nth = live.size() < 8 ? 1 : std::min(hw, live.size());
        std::atomic<size_t> next{0};
        auto work = [&]() {
            for (size_t i = next++; i < live.size(); i = next++) {
                try {
                    plan_one(i);
                } catch (const std::exception& e) {
                    plans[i].error = e.what();
                }
            }
        };
        std::vector<std::thread> pool;
        for (size_t t = 1; t < nth; ++t) pool.emplace_back(work);
        work();
        for (std::thread& t : pool) t.join();
        for (const Plan& p : plans)
            if (!p.error.empty()) throw Error(ERR_INVALID_ARGUMENT, "Batch planning failed: " + p.error);
    }
    if (plan_s) *plan_s += std::chrono::duration<double>(std::chrono::steady_clock::now() - t_plan).count();
    const auto t_pack = std::chrono::steady_clock::now();
    // 2. one table in pinned memory, uploaded in one copy: every state's
    // phases and ops, the block matrices, the small states' programs, and per
    // round one sweep item per state (all its columns) and one whole-state item
    // per small state's column.  Offsets first
    // (serial arithmetic), then the states fill their parts in parallel.
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    const size_t wop_bytes = prec == PREC_C128 ? sizeof(InterpOpT<double>) : sizeof(InterpOpT<float>);
    size_t off = 0, max_steps = 0, nblock_floats = 0, nwph = 0, nwops = 0;
    std::vector<size_t> bbase(live.size(), 0), wpbase(live.size(), 0), wobase(live.size(), 0);
    for (size_t i = 0; i < live.size(); ++i) {
        Plan& p = plans[i];
        max_steps = std::max(max_steps, p.steps.size());
        if (p.small) {
            wpbase[i] = nwph;
            wobase[i] = nwops;
            nwph += prec == PREC_C128 ? p.wd.phases.size() : p.wf.phases.size();
            nwops += prec == PREC_C128 ? p.wd.ops.size() : p.wf.ops.size();
            continue;
        }
        bbase[i] = nblock_floats;
        nblock_floats += p.blocks.size();
        p.poff.assign(p.steps.size(), 0);
        p.ooff.assign(p.steps.size(), 0);
        p.nph.assign(p.steps.size(), 0);
        p.blk.assign(p.steps.size(), 0);
        for (size_t s = 0; s < p.steps.size(); ++s) {
            if (!p.steps[s].sweep) continue;
            p.blk[s] = char(block_level(p.ph[s]));
            p.poff[s] = off;
            off = up(off + p.ph[s].size() * sizeof(SwPhase));
            p.ooff[s] = off;
            off = up(off + p.ops[s].size() * op_bytes(prec, false));
            p.nph[s] = int(p.ph[s].size());
        }
    }
    const size_t boff = off;
    off = up(off + nblock_floats * sizeof(float));
    const size_t wpoff = off;
    off = up(off + nwph * sizeof(WholePhase));
    const size_t wooff = off;
    off = up(off + (nwops + 1) * wop_bytes);   // and a spare record
    // whole-state items: round-major, within a round the widest states first;
    // the columns of state i in round r start at witem[r][i].  A round of up
    // to 256 items is one launch per register count (every item has a CU of
    // its own), a longer one a launch per width, so that narrow states do not
    // take the LDS of the widest.
    struct WholeGroup {
        size_t first, count;
        int n_max;
    };
    std::vector<std::vector<WholeGroup>> wgroups(max_steps);
    std::vector<std::vector<size_t>> witem(max_steps);
    size_t nwitems = 0;
    {
        std::vector<size_t> small;
        for (size_t i = 0; i < live.size(); ++i)
            if (plans[i].small) small.push_back(i);
        std::stable_sort(small.begin(), small.end(),
                         [&](size_t x, size_t y) { return live[x]->nr_bits() > live[y]->nr_bits(); });
        for (size_t r = 0; r < max_steps && !small.empty(); ++r) {
            witem[r].assign(live.size(), 0);
            size_t round = 0;
            for (size_t i : small)
                if (r < plans[i].steps.size() && plans[i].steps[r].sweep) round += live[i]->nr_cols();
            for (size_t i : small) {
                if (r >= plans[i].steps.size() || !plans[i].steps[r].sweep) continue;
                const int n = int(live[i]->nr_bits());
                std::vector<WholeGroup>& gr = wgroups[r];
                const bool same = !gr.empty() && whole_regs(gr.back().n_max) == whole_regs(n) &&
                                  (round <= 256 || gr.back().n_max == n || gr.back().n_max <= 10);
                if (!same) gr.push_back(WholeGroup{nwitems, 0, n});
                witem[r][i] = nwitems;
                nwitems += live[i]->nr_cols();
                gr.back().count += live[i]->nr_cols();
            }
        }
    }
    const size_t wioff = off;
    off = up(off + nwitems * sizeof(WholeItem));
    // sweep items: round-major; item (r, i) at item_at[r][i], tiles from
    // round_first[r][i]
    std::vector<std::pair<size_t, size_t>> round_items(max_steps);   // (first item, count)
    std::vector<uint64_t> round_tiles(max_steps, 0);
    std::vector<char> round_blk(max_steps, 0);
    std::vector<std::vector<uint64_t>> item_idx(max_steps), item_tile(max_steps);
    size_t wi = 0;
    for (size_t r = 0; r < max_steps; ++r) {
        round_items[r].first = wi;
        item_idx[r].assign(live.size(), SIZE_MAX);
        item_tile[r].assign(live.size(), 0);
        uint64_t tiles = 0;
        for (size_t i = 0; i < live.size(); ++i) {
            const Plan& p = plans[i];
            if (p.small || r >= p.steps.size() || !p.steps[r].sweep) continue;
            round_blk[r] = std::max(round_blk[r], p.blk[r]);
            item_idx[r][i] = wi++;
            item_tile[r][i] = tiles;
            tiles += uint64_t(live[i]->nr_cols()) << (live[i]->nr_bits() - size_t(g.M));
        }
        round_items[r].second = wi - round_items[r].first;
        round_tiles[r] = tiles;
    }
    const size_t items_off = off;
    const size_t total = up(items_off + wi * sizeof(SweepItem));
    char* dbase = static_cast<char*>(prog.get(total, stream));
    char* host = static_cast<char*>(stage.get(total));
    {
        std::atomic<size_t> next{0};
        auto fill = [&] {
            for (size_t i = next++; i < live.size(); i = next++) {
                Plan& p = plans[i];
                GpuVectorState& st = *live[i];
                if (p.small) {
                    auto copy = [&](const auto& wt) {
                        std::memcpy(host + wpoff + wpbase[i] * sizeof(WholePhase), wt.phases.data(),
                                    wt.phases.size() * sizeof(WholePhase));
                        std::memcpy(host + wooff + wobase[i] * wop_bytes, wt.ops.data(), wt.ops.size() * wop_bytes);
                        WholeItem* it = reinterpret_cast<WholeItem*>(host + wioff);
                        for (size_t s = 0; s < p.steps.size(); ++s) {
                            if (!p.steps[s].sweep) continue;
                            for (size_t c = 0; c < st.nr_cols(); ++c)
                                it[witem[s][i] + c] =
                                    WholeItem{st.col_ptr(c), uint32_t(st.nr_bits()), wt.nph[s],
                                              uint32_t(wpbase[i]) + wt.ph0[s], uint32_t(wobase[i]) + wt.op0[s], 0, 0};
                        }
                    };
                    if (prec == PREC_C128) copy(p.wd);
                    else copy(p.wf);
                    continue;
                }
                std::memcpy(reinterpret_cast<float*>(host + boff) + bbase[i], p.blocks.data(),
                            p.blocks.size() * sizeof(float));
                const int n = int(st.nr_bits());
                for (size_t s = 0; s < p.steps.size(); ++s) {
                    if (!p.steps[s].sweep) continue;
                    SwPhase* ph = reinterpret_cast<SwPhase*>(host + p.poff[s]);
                    for (size_t j = 0; j < p.ph[s].size(); ++j) {
                        ph[j] = p.ph[s][j];
                        if (ph[j].kind == 1) ph[j].op_begin += uint32_t(bbase[i]);
                    }
                    put_ops(host + p.ooff[s], p.ops[s], prec, false);
                    SweepItem it;
                    std::memset(&it, 0, sizeof(it));
                    it.amp = st.col_ptr(0);
                    it.col_stride = uint64_t(1) << n;
                    it.ncols = uint32_t(st.nr_cols());
                    it.log_ntiles = uint32_t(n - g.M);
                    it.first_tile = item_tile[s][i];
                    it.sa.ntiles = uint64_t(1) << (n - g.M);
                    it.sa.tset.cnt = g.M;
                    for (int j = 0; j < g.M; ++j) {
                        it.sa.tset.s[j] = p.steps[s].tile[j];
                        it.sa.tpos[j] = p.steps[s].tile[j];
                    }
                    it.sa.phases = reinterpret_cast<const SwPhase*>(dbase + p.poff[s]);
                    it.sa.ops = reinterpret_cast<const SwOp*>(dbase + p.ooff[s]);
                    it.sa.blocks = reinterpret_cast<const float*>(dbase + boff);
                    it.sa.nphases = p.nph[s];
                    it.sa.nops = uint32_t(p.ops[s].size());
                    std::memcpy(host + items_off + item_idx[s][i] * sizeof(SweepItem), &it, sizeof(it));
                }
            }
        };
        const size_t hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
        const size_t nth = live.size() < 64 ? 1 : std::min(hw, live.size() / 32);
        std::vector<std::thread> pool;
        for (size_t t = 1; t < nth; ++t) pool.emplace_back(fill);
        fill();
        for (std::thread& t : pool) t.join();
    }
    std::memset(host + wooff + nwops * wop_bytes, 0, wop_bytes);
    upload_table(dbase, host, total, stream);
    if (pack_s) *pack_s += std::chrono::duration<double>(std::chrono::steady_clock::now() - t_pack).count();

    // 3. rounds: single-gate steps of each state, then the whole-state
    // launches, then one batched sweep launch
    for (size_t r = 0; r < max_steps; ++r) {
        for (size_t i = 0; i < live.size(); ++i) {
            const Plan& p = plans[i];
            if (r >= p.steps.size() || p.steps[r].sweep) continue;
            for (size_t gi : p.steps[r].gates) live[i]->apply_op(live[i]->pending()[gi].op, 0, live[i]->nr_cols());
        }
        for (const WholeGroup& wg : wgroups[r]) {
            const WholeItem* wi = reinterpret_cast<const WholeItem*>(dbase + wioff) + wg.first;
            const WholePhase* wp = reinterpret_cast<const WholePhase*>(dbase + wpoff);
            if (prec == PREC_C128)
                launch_whole<double2>(wg.n_max, wi, wg.count, 0, wp,
                                      reinterpret_cast<const InterpOpT<double>*>(dbase + wooff), stream);
            else
                launch_whole<float2>(wg.n_max, wi, wg.count, 0, wp,
                                     reinterpret_cast<const InterpOpT<float>*>(dbase + wooff), stream);
            agg.launches += 1;
        }
        if (!round_items[r].second) continue;
        const SweepItem* ditems = reinterpret_cast<const SweepItem*>(dbase + items_off) + round_items[r].first;
        const int nit = int(round_items[r].second);
        // runs of tile_chunk tiles keep an item's program in the scalar cache,
        // but only once there are enough runs for every CU to hold several
        // workgroups: at most one run in 16384 of the round (256 circuits of 10
        // to 18 qubits complex64, ms per execute: runs of 16 31.0, 4 18.5, 1 17.9;
        // 1024 circuits of 10 to 20 qubits: 91, 88, 83)
        const unsigned chunk = unsigned(std::max<uint64_t>(1, std::min<uint64_t>(tile_chunk, round_tiles[r] / 16384)));
        const uint64_t nchunks = (round_tiles[r] + chunk - 1) / chunk;
        const unsigned gx = unsigned(std::min<uint64_t>(nchunks, 16384));
        if (prec == PREC_C128) {
            if (g.R == 3) hipLaunchKernelGGL((k_sweep_batched<double2, 12, 3, 4, 0>), dim3(gx), dim3(512), 0, stream, ditems, nit, round_tiles[r], chunk);
            else hipLaunchKernelGGL((k_sweep_batched<double2, 12, 4, 4, 0>), dim3(gx), dim3(256), 0, stream, ditems, nit, round_tiles[r], chunk);
        } else if (g.M == 13) {
            launch_batched_c64<13, 4, 5>(round_blk[r], gx, stream, ditems, nit, round_tiles[r], chunk);
        } else if (g.R == 3) {
            launch_batched_c64<12, 3, 4>(round_blk[r], gx, stream, ditems, nit, round_tiles[r], chunk);
        } else {
            launch_batched_c64<12, 4, 4>(round_blk[r], gx, stream, ditems, nit, round_tiles[r], chunk);
        }
        SW_HIP_OK(hipGetLastError());
        agg.launches += 1;
    }
    SW_HIP_OK(hipStreamSynchronize(stream));
    for (size_t i = 0; i < live.size(); ++i) {
        agg.sweeps += plans[i].st.sweeps;
        agg.gates += plans[i].st.gates;
        agg.bytes += plans[i].st.bytes;
        agg.phases += plans[i].st.phases;
        agg.blocks += plans[i].st.blocks;
        live[i]->finish_batched_flush(plans[i].st);
    }
}

}  // namespace q1t
