// Dense gates on 4..12 target qubits: Y = U X with U the 2^K x 2^K gate matrix
// and X the state seen as a 2^K x C matrix (rows: the target bits, columns:
// the other bits whose controls are set).  Bound by the matrix units from
// K = 6 on (2^(K+3) flop per amplitude against 16 / 32 bytes), by HBM below.
// The complex product is split into real ones with the column's real and
// imaginary parts as separate MFMA columns:
//   Yr = Ur Xr + Ui (-Xi),  Yi = Ur Xi + Ui Xr
// (v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64, accumulating in the state's
// precision).  Operand layouts of both: A[i][k] in lane i + 16k, B[k][j] in
// lane j + 16k.
#include "dense.h"

#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace q1t {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename V> struct Acc;
template <> struct Acc<float2> { using type = f32x4; };
template <> struct Acc<double2> { using type = f64x4; };

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f64x4 mfma(double a, double b, f64x4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// row of D held by element v of a lane's accumulator (its column: lane & 15)
template <typename V> __device__ __forceinline__ int acc_row(int lane, int v)
{
    return sizeof(V) == 8 ? 4 * (lane >> 4) + v : (lane >> 4) + 4 * v;
}

constexpr int kTileThreads = 512;   // k_dense_tile: 8 waves
constexpr int kRowThreads = 256;    // k_dense_rows: 4 waves

// log2 of the amplitudes a k_dense_tile workgroup holds: 64 KiB of LDS (two
// workgroups per CU), 128 KiB where 64 KiB would leave fewer than the 16
// columns of an MFMA.
constexpr int tile_log(size_t elem_bytes, int K)
{
    const int base = elem_bytes == 8 ? 13 : 12;
    return K + 4 > base ? K + 4 : base;
}
constexpr int tile_max_k(size_t elem_bytes) { return elem_bytes == 8 ? 10 : 9; }

// The index bits of a workgroup's amplitudes, ascending, and where each goes
// in the LDS tile (row-major, 2^log_cols columns: column bits first).
struct DenseMap {
    int nbits;
    int gpos[16];
    int lpos[16];     // 31 past nbits: a bit no tile index has
    uint64_t outer;   // the other free index bits: the block number's bits go there
    uint64_t cmask;
};

// The low bits of x at the set bits of mask, ascending.
__device__ __forceinline__ uint64_t spread(uint64_t x, uint64_t mask)
{
    uint64_t r = 0;
    for (; x; x >>= 1, mask &= mask - 1)
        if (x & 1) r |= mask & (~mask + 1);
    return r;
}

}  // namespace

// U in the order the kernels read it: for row tile t (16 rows) and 4 matrix
// columns s, lane l's entry is U[16 t + (l & 15)][4 s + (l >> 4)]; a lane's
// entries of consecutive s that make up 16 bytes are neighbours.
template <typename V>
__global__ void __launch_bounds__(kBlock) k_dense_pack(const V* __restrict__ raw, V* __restrict__ out, int K)
{
    constexpr int SP = 16 / int(sizeof(V));
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x, D = 1u << K;
    if (i >= D * D) return;
    const uint32_t e = i % SP, l = (i / SP) & 63, g = i / (SP * 64);
    const uint32_t gs = D / 4 / SP, t = g / gs, s = (g % gs) * SP + e;
    out[i] = raw[uint64_t(16 * t + (l & 15)) * D + 4 * s + (l >> 4)];
}

// One workgroup: all 2^K rows of 2^(LT-K) columns, staged in LDS, updated in
// place: coalesced reads and writes whatever the target bits, since the tile's
// columns are the lowest free index bits.  Each of the 8 waves owns RB row
// tiles x CB column tiles of 16 x 16 complex results in its accumulators,
// written back through LDS once every wave has read its operands.  The packed
// matrix is read from L2 (16-byte loads, one per row tile and 4 RB CB MFMAs of
// complex64).
// 21 qubits, K = 8, complex64: 1600 -> 48 us (with the matrix packing; the
// products alone take 27 us at the matrix peak); 25 qubits complex128: K = 5
// 1160 -> 251 us, K = 8 32.0 -> 1.05 ms.  Before, a thread per matrix row read
// it uncoalesced and the amplitudes from LDS one product at a time.
template <typename V, int K>
__global__ void __launch_bounds__(kTileThreads)
__attribute__((amdgpu_waves_per_eu((sizeof(V) << tile_log(sizeof(V), K)) > (64 << 10) ? 2 : 4)))
k_dense_tile(V* __restrict__ amp, uint64_t col_stride, DenseMap dm, uint64_t nblocks, const V* __restrict__ A)
{
    constexpr int LT = tile_log(sizeof(V), K), LC = LT - K, D = 1 << K, NC = 1 << LC, NK = D / 4;
    constexpr int W = kTileThreads / 64, TPW = (D / 16) * (NC / 16) / W;
    constexpr int CB = NC / 16 < TPW ? NC / 16 : TPW, RB = TPW / CB, RG = D / 16 / RB;
    static_assert(RB * CB == TPW && RG * (NC / 16 / CB) == W, "the waves cover the tile once");
    constexpr int PT = 1 << (LT - 9);   // amplitudes per thread
    constexpr int SP = 16 / int(sizeof(V));
    using R = typename RealOf<V>::type;
    using A4 = typename Acc<V>::type;
    extern __shared__ unsigned char smem_dense[];
    V* x = reinterpret_cast<V*>(smem_dense);
    V* a = amp + uint64_t(blockIdx.y) * col_stride;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rg = wave % RG, cg = wave / RG;
    uint64_t gt = 0;
    uint32_t lt = 0;
#pragma unroll
    for (int b = 0; b < 9; ++b)
        if ((tid >> b) & 1) {
            gt |= uint64_t(1) << dm.gpos[b];
            lt |= 1u << dm.lpos[b];
        }
    // uniform parts of the thread's amplitudes
    auto gpart = [&](int k) {
        uint64_t g = 0;
#pragma unroll
        for (int b = 0; b < LT - 9; ++b)
            if ((k >> b) & 1) g |= uint64_t(1) << dm.gpos[9 + b];
        return g;
    };
    auto lpart = [&](int k) {
        uint32_t l = 0;
#pragma unroll
        for (int b = 0; b < LT - 9; ++b)
            if ((k >> b) & 1) l |= 1u << dm.lpos[9 + b];
        return l;
    };
    for (uint64_t blk = blockIdx.x; blk < nblocks; blk += gridDim.x) {
        V* ab = a + (spread(blk, dm.outer) | dm.cmask) + gt;
        {
            V v[PT];
#pragma unroll
            for (int k = 0; k < PT; ++k) v[k] = ab[gpart(k)];
#pragma unroll
            for (int k = 0; k < PT; ++k) x[lt | lpart(k)] = v[k];
        }
        __syncthreads();
        A4 yr[RB][CB], yi[RB][CB];
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                yr[r][c] = A4{0, 0, 0, 0};
                yi[r][c] = A4{0, 0, 0, 0};
            }
        const V* xb = x + (lane >> 4) * NC + cg * CB * 16 + (lane & 15);
        const V* af = A + (uint64_t(rg) * RB * NK * 64 + uint64_t(lane) * SP);
        // steps in flight: 4, fewer where the accumulators leave no registers
        constexpr int UN = RB >= 4 ? 1 : NK / SP < 4 ? 2 : 4;
#pragma unroll UN
        for (int s = 0; s < NK; s += SP) {
            V u[RB][SP];
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int e = 0; e < SP; ++e) u[r][e] = af[(uint64_t(r) * NK + s) * 64 + e];
#pragma unroll
            for (int e = 0; e < SP; ++e) {
                V b[CB];
#pragma unroll
                for (int c = 0; c < CB; ++c) b[c] = xb[(4 * (s + e)) * NC + 16 * c];
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    const R bn = -b[c].y;
#pragma unroll
                    for (int r = 0; r < RB; ++r) {
                        yr[r][c] = mfma(u[r][e].x, b[c].x, yr[r][c]);
                        yi[r][c] = mfma(u[r][e].x, b[c].y, yi[r][c]);
                        yr[r][c] = mfma(u[r][e].y, bn, yr[r][c]);
                        yi[r][c] = mfma(u[r][e].y, b[c].x, yi[r][c]);
                    }
                }
            }
        }
        __syncthreads();   // every wave has read its operands
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    x[(16 * (rg * RB + r) + acc_row<V>(lane, v)) * NC + (cg * CB + c) * 16 + (lane & 15)] =
                        mkc<V>(yr[r][c][v], yi[r][c][v]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PT; ++k) ab[gpart(k)] = x[lt | lpart(k)];
        __syncthreads();   // the next block overwrites the tile
    }
}

// Few columns, or a matrix too tall for a 16-column tile: up to 8 columns per
// workgroup, their real parts in MFMA columns 0..7 and the imaginary ones in
// 8..15, so that 8 columns fill the unit, and 64 RTW rows (4 waves, RTW row
// tiles each); the rows of one block of columns are shared by gridDim.y
// workgroups.  X is staged in slices of up to 32 KiB.  Where one workgroup
// holds all rows and all of X in one slice, results go to the state in place;
// else to `out` (block by block, row-major), copied back by k_dense_back.
// Blocks are counted over all columns: block f is block f % nblocks of column
// f / nblocks.
// 21 qubits complex128: K = 10 8600 -> 550 us, K = 12 21300 -> 4250 us; 12
// qubits, K = 8: 51 -> 32 us.
constexpr size_t kSliceBytes = size_t(32) << 10;
template <typename V, int RTW>
__global__ void __launch_bounds__(kRowThreads) k_dense_rows(V* __restrict__ amp, V* __restrict__ out,
                                                            uint64_t col_stride, DenseMap dm, uint64_t nblocks,
                                                            uint64_t f0, uint64_t f1, int K, int LC, int LS,
                                                            const V* __restrict__ A)
{
    constexpr int SP = 16 / int(sizeof(V)), UN = RTW == 4 ? 1 : 2;
    using R = typename RealOf<V>::type;
    using A4 = typename Acc<V>::type;
    extern __shared__ unsigned char smem_dense[];
    V* x = reinterpret_cast<V*>(smem_dense);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int D = 1 << K, NK = D / 4, NC = 1 << LC, SL = 1 << LS;   // SL: rows per slice
    const int col = lane & 7;
    const bool imag = (lane & 8) != 0, used = col < NC;
    // index bits of tile element r * NC + c
    auto place = [&](uint32_t l) {
        uint64_t g = 0;
#pragma unroll
        for (int b = 0; b < 16; ++b)
            if ((l >> dm.lpos[b]) & 1) g |= uint64_t(1) << dm.gpos[b];
        return g;
    };
    const int rt0 = (int(blockIdx.y) * 4 + wave) * RTW;
    const bool active = rt0 < D / 16;
    for (uint64_t f = f0 + blockIdx.x; f < f1; f += gridDim.x) {
        const uint64_t c = f / nblocks;
        V* a = amp + c * col_stride + (spread(f - c * nblocks, dm.outer) | dm.cmask);
        A4 yu[RTW], yv[RTW];   // Ur [Xr | Xi] and Ui [-Xi | Xr]
#pragma unroll
        for (int t = 0; t < RTW; ++t) {
            yu[t] = A4{0, 0, 0, 0};
            yv[t] = A4{0, 0, 0, 0};
        }
        for (int r0 = 0; r0 < D; r0 += SL) {
            if (r0) __syncthreads();   // the last slice has been read
            for (uint32_t i = tid; i < uint32_t(SL) << LC; i += kRowThreads) x[i] = a[place((uint32_t(r0) << LC) + i)];
            __syncthreads();
            if (!active) continue;
            const V* af = A + (uint64_t(rt0) * NK + r0 / 4) * 64 + lane * SP;
#pragma unroll UN
            for (int s = 0; s < SL / 4; s += SP) {
                V u[RTW][SP];
#pragma unroll
                for (int t = 0; t < RTW; ++t)
#pragma unroll
                    for (int e = 0; e < SP; ++e) u[t][e] = af[(uint64_t(t) * NK + s) * 64 + e];
#pragma unroll
                for (int e = 0; e < SP; ++e) {
                    R bu = 0, bv = 0;
                    if (used) {
                        const V b = x[(4 * (s + e) + (lane >> 4)) * NC + col];
                        bu = imag ? b.y : b.x;
                        bv = imag ? b.x : -b.y;
                    }
#pragma unroll
                    for (int t = 0; t < RTW; ++t) {
                        yu[t] = mfma(u[t][e].x, bu, yu[t]);
                        yv[t] = mfma(u[t][e].y, bv, yv[t]);
                    }
                }
            }
        }
        if (active && used) {
#pragma unroll
            for (int t = 0; t < RTW; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t l = (uint32_t(16 * (rt0 + t) + acc_row<V>(lane, v)) << LC) + uint32_t(col);
                    V* dst = out ? out + ((f - f0) << (K + LC)) + l : a + place(l);
                    reinterpret_cast<R*>(dst)[imag ? 1 : 0] = yu[t][v] + yv[t][v];
                }
        }
        __syncthreads();   // the next block overwrites the slice
    }
}

// Blocks f0 .. f1 - 1 from `from` into the columns, in index order.
template <typename V>
__global__ void __launch_bounds__(kBlock) k_dense_back(V* __restrict__ amp, const V* __restrict__ from,
                                                       uint64_t col_stride, DenseMap dm, uint64_t nblocks, uint64_t f0,
                                                       uint64_t f1)
{
    const uint64_t nwork = (f1 - f0) << dm.nbits, step = uint64_t(gridDim.x) * kBlock;
    for (uint64_t j = uint64_t(blockIdx.x) * kBlock + threadIdx.x; j < nwork; j += step) {
        const uint64_t f = f0 + (j >> dm.nbits), c = f / nblocks;
        const uint32_t e = uint32_t(j) & ((1u << dm.nbits) - 1);
        uint64_t i = (spread(f - c * nblocks, dm.outer) | dm.cmask);
        uint32_t l = 0;
#pragma unroll
        for (int b = 0; b < 16; ++b)
            if ((e >> b) & 1) {
                i |= uint64_t(1) << dm.gpos[b];
                l |= 1u << dm.lpos[b];
            }
        amp[c * col_stride + i] = from[((f - f0) << dm.nbits) + l];
    }
}

// k_dense_tile where its blocks (times columns) occupy at least half of the
// 256 CUs, all of them for 128 KiB blocks (complex64, K = 8, us of k_dense_tile
// and k_dense_rows: 19 qubits, 64 blocks 43 and 42, 20 qubits 45 and 45, 21
// qubits 48 and 78; complex128, K = 9, 128 KiB: 20 qubits, 128 blocks 159 and
// 151, 21 qubits 171 and 285).  Up to K = 5 always: its products take
// microseconds however few the blocks are (18 qubits, K = 4: 9 and 14).  Else
// k_dense_rows, with as many rows per workgroup as leave two workgroups per CU
// and at most the matrix's row tiles per wave (1 and 2 at K = 4 and 5: those
// widths come here with the columns of states too small for k_dense_tile).
DensePlan plan_dense(const GateOp& op, int n, size_t ncols, size_t elem_bytes)
{
    DensePlan p;
    p.K = int(op.targets.size());
    const int free_bits = n - __builtin_popcountll(op.ctrl_mask) - p.K;
    p.matrix_bytes = (size_t(1) << (2 * p.K)) * elem_bytes;
    if (p.K <= tile_max_k(elem_bytes)) {
        const int lc = tile_log(elem_bytes, p.K) - p.K;
        const uint64_t fill = (elem_bytes << (p.K + lc)) > (size_t(64) << 10) ? 256 : 128;
        if (free_bits >= lc && ((uint64_t(1) << (free_bits - lc)) * ncols >= fill || p.K <= 5)) {
            p.tiles = true;
            p.log_cols = lc;
            p.nblocks = uint64_t(1) << (free_bits - lc);
            return p;
        }
    }
    p.log_cols = std::min(3, free_bits);
    p.nblocks = uint64_t(1) << (free_bits - p.log_cols);
    const uint64_t blocks = p.nblocks * ncols, tiles = (uint64_t(1) << p.K) / 16;
    p.rtw = blocks * tiles / 16 >= 512 ? 4 : blocks * tiles / 8 >= 512 ? 2 : 1;
    p.rtw = int(std::min<uint64_t>(uint64_t(p.rtw), tiles));
    p.splits = uint32_t(std::max<uint64_t>(1, tiles / (4 * p.rtw)));
    p.log_slice = p.K;
    while ((elem_bytes << (p.log_slice + p.log_cols)) > kSliceBytes) --p.log_slice;
    if (p.splits > 1 || p.log_slice < p.K) {
        // the copy: as many blocks at a time as 64 MiB hold (it stays in the
        // last-level cache), at least one
        const size_t block_bytes = elem_bytes << (p.K + p.log_cols);
        p.chunk = std::min<uint64_t>(blocks, std::max<uint64_t>(1, (size_t(64) << 20) / block_bytes));
        p.scratch_bytes = p.chunk * block_bytes;
    } else {
        p.chunk = blocks;
    }
    return p;
}

#define DN_OK(expr)                                                                                \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            throw Error(ERR_HIP, std::string("HIP error in " #expr ": ") + hipGetErrorString(e_)); \
    } while (0)

template <typename V, int K>
static void launch_tile(const DenseMap& dm, uint64_t nblocks, V* a, uint64_t col_stride, unsigned ncols, const V* A,
                        hipStream_t s)
{
    constexpr int lds = int(sizeof(V)) << tile_log(sizeof(V), K);
    DN_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_dense_tile<V, K>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    const dim3 grid(unsigned(std::min<uint64_t>(nblocks, 65536)), ncols);
    hipLaunchKernelGGL((k_dense_tile<V, K>), grid, dim3(kTileThreads), lds, s, a, col_stride, dm, nblocks, A);
    DN_OK(hipGetLastError());
}

template <typename V>
void launch_dense(const DensePlan& plan, const GateOp& op, int n, V* a, uint64_t col_stride, unsigned ncols,
                  const V* raw, V* packed, V* scratch, hipStream_t s)
{
    const int K = plan.K;
    // tile bits: the targets and the lowest other free bits as columns
    DenseMap dm{};
    for (int& l : dm.lpos) l = 31;
    uint64_t targets = 0, cols = 0;
    for (int t : op.targets) targets |= uint64_t(1) << t;
    const uint64_t taken = targets | op.ctrl_mask;
    for (int b = 0, left = plan.log_cols; left > 0; ++b)
        if (!((taken >> b) & 1)) {
            cols |= uint64_t(1) << b;
            --left;
        }
    int c = 0;
    for (int b = 0; b < n; ++b) {
        const uint64_t bit = uint64_t(1) << b;
        if (cols & bit) {
            dm.gpos[dm.nbits] = b;
            dm.lpos[dm.nbits++] = c++;
        } else if (targets & bit) {
            int q = 0;
            while (op.targets[size_t(q)] != b) ++q;
            dm.gpos[dm.nbits] = b;
            dm.lpos[dm.nbits++] = plan.log_cols + K - 1 - q;   // targets[0] is the row's MSB
        }
    }
    dm.outer = ((n >= 64 ? 0 : uint64_t(1) << n) - 1) & ~(taken | cols);
    dm.cmask = op.ctrl_mask;
    if (raw) {
        const uint32_t entries = 1u << (2 * K);
        hipLaunchKernelGGL(k_dense_pack<V>, dim3((entries + kBlock - 1) / kBlock), dim3(kBlock), 0, s, raw, packed, K);
        DN_OK(hipGetLastError());
    }
    if (plan.tiles) {
        switch (K) {
        case 4: launch_tile<V, 4>(dm, plan.nblocks, a, col_stride, ncols, packed, s); return;
        case 5: launch_tile<V, 5>(dm, plan.nblocks, a, col_stride, ncols, packed, s); return;
        case 6: launch_tile<V, 6>(dm, plan.nblocks, a, col_stride, ncols, packed, s); return;
        case 7: launch_tile<V, 7>(dm, plan.nblocks, a, col_stride, ncols, packed, s); return;
        case 8: launch_tile<V, 8>(dm, plan.nblocks, a, col_stride, ncols, packed, s); return;
        case 9: launch_tile<V, 9>(dm, plan.nblocks, a, col_stride, ncols, packed, s); return;
        default:
            if constexpr (sizeof(V) == 8) launch_tile<V, 10>(dm, plan.nblocks, a, col_stride, ncols, packed, s);
            return;
        }
    }
    const size_t lds = sizeof(V) << (plan.log_slice + plan.log_cols);
    const uint64_t blocks = plan.nblocks * ncols;
    // a wave takes rtw row tiles or none; all of them are taken once
    const uint32_t row_tiles = (1u << K) / 16, rtw = uint32_t(plan.rtw);
    if (row_tiles % rtw || 4 * rtw * plan.splits < row_tiles || 4 * rtw * (plan.splits - 1) >= row_tiles)
        throw Error(ERR_INVALID_ARGUMENT, "dense plan: the waves do not cover the matrix rows once");
    for (uint64_t f0 = 0; f0 < blocks; f0 += plan.chunk) {
        const uint64_t f1 = std::min(blocks, f0 + plan.chunk);
        const dim3 grid(unsigned(std::min<uint64_t>(f1 - f0, 65536)), plan.splits);
        auto rows = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(kRowThreads), lds, s, a, scratch, col_stride, dm, plan.nblocks, f0,
                               f1, K, plan.log_cols, plan.log_slice, packed);
        };
        if (plan.rtw == 4) rows(k_dense_rows<V, 4>);
        else if (plan.rtw == 2) rows(k_dense_rows<V, 2>);
        else rows(k_dense_rows<V, 1>);
        DN_OK(hipGetLastError());
        if (!scratch) continue;
        const uint64_t nwork = (f1 - f0) << (K + plan.log_cols);
        const unsigned gx = unsigned(std::min<uint64_t>((nwork + kBlock - 1) / kBlock, 65536));
        hipLaunchKernelGGL(k_dense_back<V>, dim3(gx), dim3(kBlock), 0, s, a, scratch, col_stride, dm, plan.nblocks, f0,
                           f1);
        DN_OK(hipGetLastError());
    }
}

// The order of k_dense_pack on the host, for matrices where a launch of its own
// would cost more (up to 2^6 rows: 4 us against 5 us for the launch).
template <typename V> void pack_dense(const cdouble* m, int K, V* out)
{
    constexpr uint32_t SP = 16 / sizeof(V);
    const uint32_t D = 1u << K;
    size_t o = 0;
    for (uint32_t t = 0; t < D / 16; ++t)
        for (uint32_t s = 0; s < D / 4; s += SP)
            for (uint32_t l = 0; l < 64; ++l)
                for (uint32_t e = 0; e < SP; ++e) {
                    const cdouble& c = m[size_t(16 * t + (l & 15)) * D + 4 * (s + e) + (l >> 4)];
                    out[o++] = mkc<V>(typename RealOf<V>::type(c.real()), typename RealOf<V>::type(c.imag()));
                }
}

template void pack_dense<double2>(const cdouble*, int, double2*);
template void pack_dense<float2>(const cdouble*, int, float2*);
template void launch_dense<double2>(const DensePlan&, const GateOp&, int, double2*, uint64_t, unsigned, const double2*,
                                    double2*, double2*, hipStream_t);
template void launch_dense<float2>(const DensePlan&, const GateOp&, int, float2*, uint64_t, unsigned, const float2*,
                                   float2*, float2*, hipStream_t);

}  // namespace q1t
