// Column work of many states in one launch per kind (ItemQueue).
#include "items.h"

#include <algorithm>
#include <cstring>
#include <mutex>

#include "gvs.h"
#include "kernels.h"

namespace q1t {

#define IQ_OK(expr)                                                                                \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            throw Error(e_ == hipErrorOutOfMemory ? ERR_OUT_OF_MEMORY : ERR_HIP,                    \
                        std::string("HIP error in " #expr ": ") + hipGetErrorString(e_));          \
    } while (0)

// work units of one column item per workgroup step
static constexpr uint64_t kChunk = uint64_t(kBlock) * 4;
// inputs of one tree workgroup step (kBlock outputs of the first level)
static constexpr uint64_t kTreeChunk = uint64_t(kBlock) * kTreeFanout;
static constexpr unsigned kMaxGrid = 8192;

// The item whose chunk range holds chunk c: the last with chunk0 <= c.
template <typename I>
__device__ __forceinline__ uint32_t find_item(const I* items, uint32_t n, uint64_t c)
{
    uint32_t lo = 0, hi = n - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (items[mid].chunk0 <= c) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Item of chunk c: a launch with one item has it in its arguments (items is
// null), so that nothing is uploaded.
template <typename I>
__device__ __forceinline__ I item_at(const I& one, const I* items, uint32_t n, uint64_t c)
{
    return items ? items[find_item(items, n, c)] : one;
}

__device__ __forceinline__ uint64_t insert_zero(uint64_t j, int p)
{
    const uint64_t bit = uint64_t(1) << p;
    return ((j >> p) << (p + 1)) | (j & (bit - 1));
}

// ------------------------------------------------------------- uploads

// Host table to device memory, read by a kernel over the bus.  The copy
// engine's hand-over to the compute queue takes about 40 us before the kernel
// that needs the table starts; this kernel's successor starts at once (17
// qubits complex64, 60 KB of sweep programs, time from the call that starts the
// upload to the first sweep: hipMemcpyAsync 75 us, and 65 us with a
// synchronisation before the sweep's launch; this kernel 43 us).
__global__ void __launch_bounds__(kBlock) k_upload(const uint4* __restrict__ from, uint4* __restrict__ to, uint32_t n)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) to[i] = from[i];
}

// Tables up to 1 MiB: above, the copy itself outweighs the hand-over.
static constexpr size_t kUploadKernelBytes = size_t(1) << 20;

void upload_table(void* dst, const void* pinned, size_t bytes, hipStream_t s)
{
    if (!bytes) return;
    if (bytes > kUploadKernelBytes) {
        IQ_OK(hipMemcpyAsync(dst, pinned, bytes, hipMemcpyHostToDevice, s));
        return;
    }
    void* from = nullptr;
    IQ_OK(hipHostGetDevicePointer(&from, const_cast<void*>(pinned), 0));
    const uint32_t n = uint32_t((bytes + 15) / 16);
    hipLaunchKernelGGL(k_upload, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, static_cast<const uint4*>(from),
                       static_cast<uint4*>(dst), n);
    IQ_OK(hipGetLastError());
}

// ------------------------------------------------------------ marginals

// One-qubit marginals: bound by HBM reads.  A column's work units (pairs of
// the qubit) are dealt to up to kMargBlocks workgroups in interleaved runs of
// marg_units(); each thread has 64 bytes in flight, 16 waves per CU.  A read
// of 8 GiB runs at 7.1 TB/s in this shape against 4.3 TB/s with 256 threads and
// 6.4 TB/s without the non-temporal hint (a plain read kernel on this part).
// Measured at 27 qubits complex128, Z on a high bit: 158 us (6.8 TB/s) against
// 479 us with 256 threads and one load in flight per thread; the average over
// all bits and bases went from 575 to 285 us, with complex64 Z at 28 qubits
// from 925 to 196 us.
static constexpr int kMargThreads = 1024;
static constexpr uint64_t marg_units(size_t elem_bytes) { return uint64_t(kMargThreads) * (64 / elem_bytes); }
// Columns from this size on are read with the non-temporal hint: they do not
// fit the 256 MiB last-level cache, so nothing of them is there at the next
// read.  Smaller ones may be.
static constexpr uint64_t kStreamBytes = uint64_t(512) << 20;

// Up to this many shares of all columns one launch does it all: the last share of
// a column adds them.  Its count takes an agent-scope release and acquire, which
// write back and invalidate an XCD's L2, so that many shares slow each other
// down: above, they are added by a launch of their own.  us per marginal (Z) in
// one launch / in two: 20 qubits complex128, 4 columns (512 shares) 30.4 / 23.9, 16
// columns 95 / 42; 22 qubits complex64, 8 columns 95 / 50; 4096 circuits of 10 to
// 22 qubits complex128 10050 / 2710.
static constexpr uint64_t kMargOneLaunch = kMargBlocks;
// Workgroups of the two launches' first: each takes consecutive shares and looks
// their item up once (the same circuits in complex64, us: a workgroup per share
// 1170, 4096 workgroups 920).
static constexpr uint64_t kMargGrid = 4096;
// Workgroups of a column: one per marg_units() work units, at most kMargBlocks
// (one per CU; the partial sums of a column then fit one workgroup).
static uint32_t marginal_blocks(bool c64, uint64_t nwork)
{
    return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(kMargBlocks, nwork / marg_units(c64 ? 8 : 16))));
}

template <bool NT, typename V> __device__ __forceinline__ V load_amp(const V* p)
{
    if constexpr (NT) {
        typedef typename RealOf<V>::type Rl2 __attribute__((ext_vector_type(2)));
        const Rl2 x = __builtin_nontemporal_load(reinterpret_cast<const Rl2*>(p));
        return mkc<V>(x.x, x.y);
    } else {
        return *p;
    }
}

// Outcome-0 weight of bit p over the work units of workgroup b of nb:
// |a0|^2 (Z), |a0 + a1|^2 / 2 (X) or |a0 - i a1|^2 / 2 (Y) per pair, in FP64
// with the fused multiply-adds spelled out.
template <typename V, bool NT>
__device__ __forceinline__ double marginal_acc(const V* a, uint64_t nwork, int p, int basis, uint32_t b, uint32_t nb)
{
    constexpr int U = 64 / int(sizeof(V));
    constexpr uint64_t units = marg_units(sizeof(V));
    const uint64_t bit = uint64_t(1) << p;
    double acc = 0.0;
    for (uint64_t base = uint64_t(b) * units; base < nwork; base += uint64_t(nb) * units) {
        V x0[U], x1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // nwork is a power of two: only columns below `units` have work
            // units past the end (zero weight)
            const uint64_t j = base + uint64_t(u) * kMargThreads + threadIdx.x;
            x0[u] = x1[u] = mkc<V>(0, 0);
            if (j < nwork) {
                const uint64_t i0 = insert_zero(j, p);
                x0[u] = load_amp<NT>(a + i0);
                if (basis != 0) x1[u] = load_amp<NT>(a + (i0 | bit));
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (basis == 0) {
                acc += weight(x0[u]);
                continue;
            }
            double re, im;
            if (basis == 1) {
                re = double(x0[u].x) + double(x1[u].x);
                im = double(x0[u].y) + double(x1[u].y);
            } else {   // a0 - i a1
                re = double(x0[u].x) + double(x1[u].y);
                im = double(x0[u].y) - double(x1[u].x);
            }
            acc = __fma_rn(0.5, __fma_rn(re, re, __dmul_rn(im, im)), acc);
        }
    }
    return acc;
}

template <int THREADS = kMargThreads> __device__ __forceinline__ double marg_block_total(double v)
{
    __shared__ double red[THREADS / 64];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int k = 0; k < THREADS / 64; ++k) s += red[k];
    __syncthreads();   // red is reused by the next call
    return s;
}

// Share b of nb of one column.
template <typename V>
__device__ __forceinline__ double marginal_share(const V* a, uint64_t nwork, int p, int basis, uint32_t b, uint32_t nb)
{
    const double acc = 2 * nwork * sizeof(V) >= kStreamBytes ? marginal_acc<V, true>(a, nwork, p, basis, b, nb)
                                                             : marginal_acc<V, false>(a, nwork, p, basis, b, nb);
    return marg_block_total(acc);
}

// Another share of a column of nb is in `partial`: the workgroup that brings the
// last one adds all of them (a fixed tree, so the result does not depend on which
// one that is) and writes the weight.  Partial sums and the count of finished
// shares go through agent-scope atomics: the XCDs' L2 caches are not coherent
// with each other.  The count is zero again when the column is done.
__device__ __forceinline__ void marginal_finish(uint32_t nb, const double* partial, uint32_t* done, double* w0)
{
    __shared__ uint32_t last;
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == nb - 1;
    __syncthreads();
    if (!last) return;
    double v = 0.0;
    if (threadIdx.x < nb) v = __hip_atomic_load(partial + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const double s = marg_block_total(v);
    if (threadIdx.x == 0) {
        *w0 = s;
        __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Chunk c: share c - chunk0 of its item; partial sums at partial[c].
template <typename V>
__global__ void __launch_bounds__(kMargThreads) k_marginal_items(MargItem one, const MargItem* __restrict__ items,
                                                                 uint32_t n, double* partial, uint32_t* done,
                                                                 double* w0)
{
    const uint64_t c = blockIdx.x;
    const uint32_t it = items ? find_item(items, n, c) : 0;
    const MargItem m = items ? items[it] : one;
    const double s = marginal_share<V>(static_cast<const V*>(m.amp), m.nwork, m.p, m.basis, uint32_t(c - m.chunk0),
                                       m.blocks);
    if (threadIdx.x == 0) {
        if (m.blocks == 1) w0[it] = s;
        else __hip_atomic_store(partial + c, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (m.blocks > 1) marginal_finish(m.blocks, partial + m.chunk0, done + it, w0 + it);
}

// The shares of many columns, `run` consecutive ones per workgroup; partial[c] is
// added up by k_marginal_sums.
template <typename V>
__global__ void __launch_bounds__(kMargThreads) k_marginal_shares(const MargItem* __restrict__ items, uint32_t n,
                                                                  uint64_t nchunks, uint32_t run,
                                                                  double* __restrict__ partial,
                                                                  double* __restrict__ w0)
{
    uint64_t c = uint64_t(blockIdx.x) * run;
    const uint64_t c1 = c + run < nchunks ? c + run : nchunks;
    for (uint32_t it = find_item(items, n, c); c < c1; ++it) {
        const MargItem m = items[it];
        const uint64_t end = m.chunk0 + m.blocks < c1 ? m.chunk0 + m.blocks : c1;
        for (; c < end; ++c) {
            const double s = marginal_share<V>(static_cast<const V*>(m.amp), m.nwork, m.p, m.basis,
                                               uint32_t(c - m.chunk0), m.blocks);
            if (threadIdx.x == 0) {
                if (m.blocks == 1) w0[it] = s;
                else partial[c] = s;
            }
        }
    }
}

// The weights of the columns of several shares, a workgroup per column: the sum of
// marginal_finish.  Without a table every column has nb shares, at stride
// kMargBlocks.
__global__ void __launch_bounds__(kMargBlocks) k_marginal_sums(const MargItem* __restrict__ items, uint32_t n,
                                                               uint32_t nb, const double* __restrict__ partial,
                                                               double* __restrict__ w0)
{
    for (uint32_t it = blockIdx.x; it < n; it += gridDim.x) {
        uint64_t at = uint64_t(it) * kMargBlocks;
        if (items) {
            at = items[it].chunk0;
            nb = items[it].blocks;
        }
        if (nb == 1) continue;
        const double s = marg_block_total<kMargBlocks>(threadIdx.x < nb ? partial[at + threadIdx.x] : 0.0);
        if (threadIdx.x == 0) w0[it] = s;
    }
}

// The shares of `gridDim.y` columns at stride col_stride (no item table: the
// allocation-free marginal); ONE: added here, else by k_marginal_sums.
template <typename V, bool ONE>
__global__ void __launch_bounds__(kMargThreads) k_marginal_cols(const V* __restrict__ amp, uint64_t col_stride,
                                                                uint64_t nwork, int p, int basis, double* partial,
                                                                uint32_t* done, double* w0)
{
    const uint32_t c = blockIdx.y, nb = gridDim.x;
    double* const part = partial + uint64_t(c) * kMargBlocks;
    const double s = marginal_share<V>(amp + uint64_t(c) * col_stride, nwork, p, basis, blockIdx.x, nb);
    if (threadIdx.x == 0) {
        if (nb == 1) w0[c] = s;
        else __hip_atomic_store(part + blockIdx.x, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if constexpr (ONE)
        if (nb > 1) marginal_finish(nb, part, done + c, w0 + c);
}

template <typename V>
static void marginal_cols(const V* amp, uint64_t col_stride, uint32_t ncols, uint64_t nwork, int p, int basis,
                          double* partial, uint32_t* done, double* w0, hipStream_t s)
{
    const uint32_t nb = marginal_blocks(sizeof(V) == 8, nwork);
    const bool one = nb == 1 || uint64_t(nb) * ncols <= kMargOneLaunch;
    auto k = one ? k_marginal_cols<V, true> : k_marginal_cols<V, false>;
    hipLaunchKernelGGL(k, dim3(nb, ncols), dim3(kMargThreads), 0, s, amp, col_stride, nwork, p, basis, partial, done,
                       w0);
    IQ_OK(hipGetLastError());
    if (one) return;
    hipLaunchKernelGGL(k_marginal_sums, dim3(ncols), dim3(kMargBlocks), 0, s, static_cast<const MargItem*>(nullptr),
                       ncols, nb, partial, w0);
    IQ_OK(hipGetLastError());
}

void launch_marginal_cols(bool c64, const void* amp, uint64_t col_stride, uint32_t ncols, uint64_t nwork, int p,
                          int basis, double* partial, uint32_t* done, double* w0, hipStream_t s)
{
    if (c64)
        marginal_cols(static_cast<const float2*>(amp), col_stride, ncols, nwork, p, basis, partial, done, w0, s);
    else
        marginal_cols(static_cast<const double2*>(amp), col_stride, ncols, nwork, p, basis, partial, done, w0, s);
}

// ------------------------------------------------------------- collapses

// Collapse of one pair (a0, a1) of bit p.  Z: dst0 keeps a0 s0, dst1 a1 s1.
// X/Y (the basis change back included): X, outcome 0: a0' = a1' =
// (a0 + a1) s0/2; outcome 1: a0' = -a1' = (a0 - a1) s1/2.  Y, outcome 0:
// u = a0 - i a1, a0' = u s0/2, a1' = i u s0/2; outcome 1: v = a0 + i a1,
// a0' = v s1/2, a1' = -i v s1/2.
template <typename V>
__device__ __forceinline__ void collapse_pair(const CollItem& m, uint64_t j)
{
    using Rl = typename RealOf<V>::type;
    const V* src = static_cast<const V*>(m.src);
    V* d0 = static_cast<V*>(m.dst0);
    V* d1 = static_cast<V*>(m.dst1);
    const uint64_t bit = uint64_t(1) << m.p;
    const uint64_t i0 = insert_zero(j, m.p), i1 = i0 | bit;
    const V x0 = src[i0], x1 = src[i1];
    const Rl s0 = Rl(m.s0), s1 = Rl(m.s1);
    if (m.basis == 0) {
        const V zero = mkc<V>(0, 0);
        if (d0) {
            d0[i0] = mkc<V>(x0.x * s0, x0.y * s0);
            d0[i1] = zero;
        }
        if (d1) {
            d1[i0] = zero;
            d1[i1] = mkc<V>(x1.x * s1, x1.y * s1);
        }
        return;
    }
    const Rl h0 = Rl(0.5) * s0, h1 = Rl(0.5) * s1;
    if (m.basis == 1) {
        const V u = mkc<V>((x0.x + x1.x) * h0, (x0.y + x1.y) * h0);
        const V v = mkc<V>((x0.x - x1.x) * h1, (x0.y - x1.y) * h1);
        if (d0) {
            d0[i0] = u;
            d0[i1] = u;
        }
        if (d1) {
            d1[i0] = v;
            d1[i1] = mkc<V>(-v.x, -v.y);
        }
    } else {
        const V u = mkc<V>((x0.x + x1.y) * h0, (x0.y - x1.x) * h0);   // (a0 - i a1) s0/2
        const V v = mkc<V>((x0.x - x1.y) * h1, (x0.y + x1.x) * h1);   // (a0 + i a1) s1/2
        if (d0) {
            d0[i0] = u;
            d0[i1] = mkc<V>(-u.y, u.x);   // i u
        }
        if (d1) {
            d1[i0] = v;
            d1[i1] = mkc<V>(v.y, -v.x);   // -i v
        }
    }
}

template <typename V>
__global__ void __launch_bounds__(kBlock) k_collapse_items(CollItem one, const CollItem* __restrict__ items,
                                                           uint32_t n, uint64_t nchunks)
{
    for (uint64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const CollItem m = item_at(one, items, n, c);
        const uint64_t j0 = (c - m.chunk0) * kChunk;
        const uint64_t j1 = j0 + kChunk < m.nwork ? j0 + kChunk : m.nwork;
        for (uint64_t j = j0 + threadIdx.x; j < j1; j += kBlock) collapse_pair<V>(m, j);
    }
}

// ------------------------------------------------------------ column gates

template <typename V> __device__ __forceinline__ V entry(const ColOp& o, int k)
{
    using Rl = typename RealOf<V>::type;
    return mkc<V>(Rl(o.m[2 * k]), Rl(o.m[2 * k + 1]));
}

template <typename V>
__device__ __forceinline__ void col_op_apply(V* a, const ColOp& o, const PosList& pl, uint64_t j)
{
    const uint64_t i = deposit(j, pl) | o.cmask;
    switch (o.kind) {
    case 0: {   // dense, one target
        const uint64_t i1 = i | (uint64_t(1) << o.t[0]);
        const V x = a[i], y = a[i1];
        a[i] = cadd(cmul(entry<V>(o, 0), x), cmul(entry<V>(o, 1), y));
        a[i1] = cadd(cmul(entry<V>(o, 2), x), cmul(entry<V>(o, 3), y));
        break;
    }
    case 1: {   // dense, two targets (t[0] the local MSB)
        const uint64_t b0 = uint64_t(1) << o.t[0], b1 = uint64_t(1) << o.t[1];
        const uint64_t ix[4] = {i, i | b1, i | b0, i | b0 | b1};
        V v[4];
#pragma unroll
        for (int l = 0; l < 4; ++l) v[l] = a[ix[l]];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            V acc = cmul(entry<V>(o, r * 4), v[0]);
#pragma unroll
            for (int c = 1; c < 4; ++c) acc = cmac(acc, entry<V>(o, r * 4 + c), v[c]);
            a[ix[r]] = acc;
        }
        break;
    }
    case 2: {   // diagonal on up to 3 targets
        int l = 0;
#pragma unroll
        for (int q = 0; q < 3; ++q)
            if (q < o.nt) l = (l << 1) | int((i >> o.t[q]) & 1);
        a[i] = cmul(entry<V>(o, l), a[i]);
        break;
    }
    case 3:   // phase where every bit of cmask is 1
        a[i] = cmul(entry<V>(o, 0), a[i]);
        break;
    default: {   // swap of the two targets
        const uint64_t ba = uint64_t(1) << o.t[0], bb = uint64_t(1) << o.t[1];
        const V x = a[i | bb], y = a[i | ba];
        a[i | bb] = y;
        a[i | ba] = x;
        break;
    }
    }
}

template <typename V>
__global__ void __launch_bounds__(kBlock) k_op_items(const OpItem* __restrict__ items, uint32_t n, uint64_t nchunks,
                                                     const ColOp* __restrict__ ops)
{
    for (uint64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const OpItem it = items[find_item(items, n, c)];
        const ColOp& o = ops[it.op];
        PosList pl;
        pl.cnt = o.npos;
#pragma unroll
        for (int k = 0; k < 16; ++k) pl.s[k] = o.pos[k];
        V* a = static_cast<V*>(it.amp);
        const uint64_t j0 = (c - it.chunk0) * kChunk;
        const uint64_t j1 = j0 + kChunk < it.nwork ? j0 + kChunk : it.nwork;
        for (uint64_t j = j0 + threadIdx.x; j < j1; j += kBlock) col_op_apply<V>(a, o, pl, j);
    }
}

// --------------------------------------------------------- basis columns

// Column of |k> (rot 0), H^n|k> (rot 1) or S^n H^n|k> (rot 2): amplitude j =
// (-1)^popcount(j&k) i^popcount(j) (the i factor for rot 2 only) times mag.
template <typename V>
__global__ void __launch_bounds__(kBlock) k_basis_items(BasisItem one, const BasisItem* __restrict__ items,
                                                        uint32_t n, uint64_t nchunks)
{
    using Rl = typename RealOf<V>::type;
    for (uint64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const BasisItem b = item_at(one, items, n, c);
        V* a = static_cast<V*>(b.amp);
        const Rl mag = Rl(b.mag);
        const uint64_t j0 = (c - b.chunk0) * kChunk;
        const uint64_t j1 = j0 + kChunk < b.dim ? j0 + kChunk : b.dim;
        for (uint64_t j = j0 + threadIdx.x; j < j1; j += kBlock) {
            V v;
            if (b.rot == 0) {
                v = mkc<V>(j == b.k ? Rl(1) : Rl(0), Rl(0));
            } else {
                const Rl s = (__popcll(j & b.k) & 1) ? -mag : mag;
                const int q = b.rot == 2 ? (__popcll(j) & 3) : 0;   // i^q
                v = q == 0 ? mkc<V>(s, 0) : q == 1 ? mkc<V>(0, s) : q == 2 ? mkc<V>(-s, 0) : mkc<V>(0, -s);
            }
            a[j] = v;
        }
    }
}

// ------------------------------------------------------------- sampling

__device__ __forceinline__ double leaf(double2 a) { return weight(a); }
__device__ __forceinline__ double leaf(float2 a) { return weight(a); }
__device__ __forceinline__ double leaf(double w) { return w; }

template <bool NT, typename V> __device__ __forceinline__ double load_leaf(const V* p) { return leaf(load_amp<NT>(p)); }
template <bool NT> __device__ __forceinline__ double load_leaf(const double* p) { return *p; }

// The weights of the kTreeChunk entries from `base` on, into LDS, 16 loads per
// thread in flight; entry e in a transposed, padded place, so that thread t
// reads entries 16t .. 16t+15 without bank conflicts.
template <typename T, bool NT>
__device__ __forceinline__ void load_leaves(const T* in, uint64_t size, uint64_t base, double* w)
{
    double v[kTreeFanout];
    if (base + kTreeChunk <= size) {
#pragma unroll
        for (int r = 0; r < kTreeFanout; ++r) v[r] = load_leaf<NT>(in + base + r * kBlock + threadIdx.x);
    } else {
#pragma unroll
        for (int r = 0; r < kTreeFanout; ++r) {
            const uint64_t k = base + r * kBlock + threadIdx.x;
            v[r] = k < size ? load_leaf<NT>(in + k) : 0.0;
        }
    }
#pragma unroll
    for (int r = 0; r < kTreeFanout; ++r) {
        const int e = r * kBlock + threadIdx.x;
        w[(e & (kTreeFanout - 1)) * (kBlock + 1) + (e >> 4)] = v[r];
    }
}

// Up to three levels of the sampling tree, a workgroup per 4096 inputs: bound
// by the read of the column at the first levels (the higher ones hold 1/16 of
// it and less) and by launches for small columns, so one launch makes three
// levels: 256 threads fold 16 entries each, 16 threads the 256 folds, one
// thread the 16 folds of those.  Sizes are powers of two above 16: every group
// that exists is full.  A column of 30 qubits complex128 takes 3.1 ms (5.5 TB/s),
// 3.7 ms with a level per launch and plain loads.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_tree_items(TreeItem one, const TreeItem* __restrict__ items, uint32_t n,
                                                       uint64_t nchunks)
{
    __shared__ double w[kTreeFanout * (kBlock + 1)];
    __shared__ double w2[kTreeFanout * (kTreeFanout + 1)];
    const uint32_t t = threadIdx.x;
    for (uint64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const TreeItem it = item_at(one, items, n, c);
        const T* in = static_cast<const T*>(it.in);
        const uint64_t base = (c - it.chunk0) * kTreeChunk;
        const uint64_t n1 = it.size / kTreeFanout, n2 = n1 / kTreeFanout;
        if (it.size * sizeof(T) >= kStreamBytes) load_leaves<T, true>(in, it.size, base, w);
        else load_leaves<T, false>(in, it.size, base, w);
        __syncthreads();
        double acc = 0.0;
        const uint64_t g = base / kTreeFanout + t;
        if (g < n1) {
            acc = w[t];
#pragma unroll
            for (int j = 1; j < kTreeFanout; ++j) acc += w[j * (kBlock + 1) + t];
            it.out[g] = acc;
        }
        if (it.levels > 1) {
            w2[(t & (kTreeFanout - 1)) * (kTreeFanout + 1) + (t >> 4)] = acc;
            __syncthreads();
            if (t < 64) {
                const uint64_t g2 = base / (kTreeFanout * kTreeFanout) + t;
                double a2 = 0.0;
                if (t < kTreeFanout && g2 < n2) {
                    a2 = w2[t];
#pragma unroll
                    for (int j = 1; j < kTreeFanout; ++j) a2 += w2[j * (kTreeFanout + 1) + t];
                    it.out[n1 + g2] = a2;
                }
                if (it.levels > 2) {
                    double a3 = __shfl(a2, 0, 64);
#pragma unroll
                    for (int j = 1; j < kTreeFanout; ++j) a3 += __shfl(a2, j, 64);
                    if (t == 0) it.out[n1 + n2 + base / kTreeChunk] = a3;
                }
            }
        }
        __syncthreads();
    }
}

// Entry k of a tree level of a column (level 0: its amplitudes).
template <typename V>
__device__ __forceinline__ double tree_at(const V* a, const double* lev, int l, uint64_t k)
{
    return l == 0 ? weight(a[k]) : lev[k];
}

// The last job whose key (run0 or col0) is at most x.
__device__ __forceinline__ SampleJob job_at(const SampleJob& one, const SampleJob* jobs, uint32_t njobs,
                                            uint64_t SampleJob::*key, uint64_t x)
{
    if (!jobs) return one;
    uint32_t lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (jobs[mid].*key <= x) lo = mid;
        else hi = mid - 1;
    }
    return jobs[lo];
}

// Inverse-CDF sampling of one run per thread by the canonical tree walk:
// t = u * T; within each group keep offset += S_j while offset + S_j <= t,
// descend into the first child where that fails, or the last positive one.
// The workgroups past the runs' write the total weight of each column (its
// top tree level summed in order), one thread per column of all jobs: the
// norm check of measure_all.
template <typename V>
__global__ void __launch_bounds__(kBlock) k_sample_items(SampleJob one, const SampleJob* __restrict__ jobs,
                                                         uint32_t njobs, const uint64_t* __restrict__ first,
                                                         const double* __restrict__ u01, uint64_t nruns,
                                                         uint64_t* __restrict__ out, uint64_t ncols,
                                                         double* __restrict__ tops)
{
    const uint64_t run_blocks = (nruns + kBlock - 1) / kBlock;
    const bool is_top = blockIdx.x >= run_blocks;
    const uint64_t r = (uint64_t(blockIdx.x) - (is_top ? run_blocks : 0)) * kBlock + threadIdx.x;
    if (r >= (is_top ? ncols : nruns)) return;
    const SampleJob jb = job_at(one, jobs, njobs, is_top ? &SampleJob::col0 : &SampleJob::run0, r);
    uint64_t col;
    if (is_top) {
        col = r - jb.col0;
    } else {
        const uint64_t rl = r - jb.run0;
        const uint64_t* fr = first + jb.first_off;
        int clo = 0, chi = jb.ncols - 1;
        while (clo < chi) {
            const int mid = (clo + chi + 1) >> 1;
            if (fr[mid] <= rl) clo = mid;
            else chi = mid - 1;
        }
        col = uint64_t(clo);
    }
    const V* a = static_cast<const V*>(jb.a0) + col * jb.col_stride;
    const int nb = jb.nbits, top = tree_top(nb);
    const double* lev = jb.tree + col * jb.per_col + tree_offset(nb, top);
    uint64_t gstart = 0, glen = uint64_t(1) << (nb - 4 * top), idx = 0;
    double total = tree_at(a, lev, top, 0);
    for (uint64_t k = 1; k < glen; ++k) total += tree_at(a, lev, top, k);
    if (is_top) {
        tops[r] = total;
        return;
    }
    const double t = u01[r] * total;
    double offset = 0.0;
    for (int l = top; l >= 0; --l) {
        double v[kTreeFanout];
        int last = 0;
#pragma unroll
        for (int j = 0; j < kTreeFanout; ++j) {
            v[j] = (uint64_t(j) < glen) ? tree_at(a, lev, l, gstart + j) : 0.0;
            if (v[j] > 0.0) last = j;
        }
        int chosen = last;
        for (int j = 0; j < last; ++j) {
            const double nx = offset + v[j];
            if (nx <= t) {
                offset = nx;
            } else {
                chosen = j;
                break;
            }
        }
        idx = gstart + uint64_t(chosen);
        gstart = idx * kTreeFanout;
        glen = kTreeFanout;
        if (l > 1) lev -= uint64_t(1) << (nb - 4 * (l - 1));
    }
    out[r] = idx;
}

// ------------------------------------------------------------- the queue

ItemQueue::ItemQueue(bool c64) : c64_(c64) {}

ItemQueue::~ItemQueue()
{
    if (last_stream_) (void)hipStreamSynchronize(last_stream_);
    if (dbuf_) (void)hipFree(dbuf_);
    if (hin_) (void)hipHostFree(hin_);
    if (hout_) (void)hipHostFree(hout_);
    if (stage_) (void)hipHostFree(stage_);
    if (in_done_) (void)hipEventDestroy(in_done_);
}

size_t ItemQueue::add_marginal(const MargItem& m)
{
    MargItem x = m;
    x.blocks = marginal_blocks(c64_, m.nwork);
    x.chunk0 = marg_chunks_;
    marg_chunks_ += x.blocks;
    marg_.push_back(x);
    return marg_.size() - 1;
}

void ItemQueue::add_collapse(const CollItem& c)
{
    if (!c.nwork) return;
    CollItem x = c;
    x.chunk0 = coll_chunks_;
    coll_chunks_ += (c.nwork + kChunk - 1) / kChunk;
    coll_.push_back(x);
}

uint32_t ItemQueue::add_op(const ColOp& op)
{
    ops_.push_back(op);
    return uint32_t(ops_.size() - 1);
}

void ItemQueue::add_op_item(void* amp, uint64_t nwork, uint32_t op)
{
    if (!nwork) return;
    OpItem it{amp, nwork, op_chunks_, op, 0};
    op_chunks_ += (nwork + kChunk - 1) / kChunk;
    opit_.push_back(it);
}

void ItemQueue::add_basis(const BasisItem& b)
{
    if (!b.dim) return;
    BasisItem x = b;
    x.chunk0 = basis_chunks_;
    basis_chunks_ += (b.dim + kChunk - 1) / kChunk;
    basis_.push_back(x);
}

size_t ItemQueue::add_sample(const SampleJob& job, const uint64_t* first, const double* u, size_t nruns)
{
    const int top = tree_top(job.nbits);
    if (job.ncols < 1 || job.nbits < 0 || top > 3 * kTreeSteps)
        throw Error(ERR_INVALID_ARGUMENT, "sampling job: inconsistent tree");
    for (int c = 0; c < job.ncols; ++c) {
        double* const tree = const_cast<double*>(job.tree) + uint64_t(c) * job.per_col;
        const char* a = static_cast<const char*>(job.a0) + uint64_t(c) * job.col_stride * (c64_ ? 8 : 16);
        for (int l = 0, k = 0; l < top; l += 3, ++k) {
            TreeItem it{};
            it.in = l == 0 ? static_cast<const void*>(a) : tree + tree_offset(job.nbits, l);
            it.out = tree + tree_offset(job.nbits, l + 1);
            it.size = uint64_t(1) << (job.nbits - 4 * l);
            it.levels = uint32_t(std::min(3, top - l));
            it.chunk0 = tree_chunks_[k];
            tree_chunks_[k] += (it.size + kTreeChunk - 1) / kTreeChunk;
            tree_[k].push_back(it);
        }
    }
    SampleJob j = job;
    j.first_off = first_.size();
    j.run0 = u_.size();
    j.col0 = cols_;
    cols_ += uint64_t(job.ncols);
    first_.insert(first_.end(), first, first + job.ncols + 1);
    u_.insert(u_.end(), u, u + nruns);
    jobs_.push_back(j);
    return jobs_.size() - 1;
}

void ItemQueue::release_after(void* p, size_t bytes, hipStream_t s)
{
    if (p) rel_.push_back(Release{p, bytes, s});
}

bool ItemQueue::empty() const
{
    bool lv = false;
    for (const auto& v : tree_) lv = lv || !v.empty();
    return marg_.empty() && coll_.empty() && opit_.empty() && basis_.empty() && jobs_.empty() && !lv &&
           rel_.empty();
}

static size_t up256(size_t x) { return (x + 255) / 256 * 256; }

void ItemQueue::launch(hipStream_t s)
{
    if (!marg_.empty() || !coll_.empty() || !opit_.empty() || !basis_.empty() || !jobs_.empty()) launch_items(s);
    clear_inputs();
}

void ItemQueue::clear_inputs()
{
    // the kernels that read the released blocks are enqueued: stream order
    // keeps later users of those blocks behind them
    for (const Release& r : rel_) DeviceCache::get().release(r.p, r.bytes, r.s);
    rel_.clear();
    marg_.clear();
    coll_.clear();
    ops_.clear();
    opit_.clear();
    basis_.clear();
    for (auto& v : tree_) v.clear();
    jobs_.clear();
    first_.clear();
    u_.clear();
    cols_ = 0;
    marg_chunks_ = coll_chunks_ = op_chunks_ = basis_chunks_ = 0;
    for (uint64_t& c : tree_chunks_) c = 0;
}

// What a launch moves besides the columns is small, and its cost is launches
// and copies: a kernel of one item has it in its arguments, and up to
// kHostBytes the kernels read the uniforms from pinned host memory and write
// the results there, where a copy would be a launch of its own at either end.
// A marginal of a 16-qubit state then is one launch, not three, and sampling it
// two, not seven: 16 marginals or peeks and one sampling of 4096 runs of 16
// complex64 qubits take 577 us, 845 us before; 21 marginals of 21 qubits 166 us
// less.
static constexpr size_t kHostBytes = size_t(1) << 20;

void ItemQueue::launch_items(hipStream_t s)
{
    // the device buffer: the count of finished workgroups of a single
    // marginal (zero between launches), inputs, partial sums, results
    size_t in = 256;
    auto take = [&](size_t bytes) {
        const size_t o = in;
        in = up256(in + bytes);
        return o;
    };
    auto many = [&](const auto& v) { return v.size() > 1 ? v.size() * sizeof(v[0]) : 0; };   // one: by argument
    const size_t o_marg = take(many(marg_));
    const size_t o_coll = take(many(coll_));
    const size_t o_ops = take(ops_.size() * sizeof(ColOp));
    const size_t o_opit = take(opit_.size() * sizeof(OpItem));
    const size_t o_basis = take(many(basis_));
    size_t o_tree[kTreeSteps];
    for (int k = 0; k < kTreeSteps; ++k) o_tree[k] = take(many(tree_[k]));
    const size_t o_jobs = take(many(jobs_));
    const size_t o_done = take(marg_.size() > 1 ? marg_.size() * sizeof(uint32_t) : 0);   // zeros
    const size_t u_bytes = up256(u_.size() * sizeof(double));
    const bool u_host = u_bytes <= kHostBytes;
    const size_t o_first = take(cols_ > jobs_.size() ? first_.size() * sizeof(uint64_t) : 0);   // not read for one column
    const size_t o_u = u_host ? in : take(u_bytes);
    const size_t up_bytes = in - 256;                                  // uploaded
    const size_t in_bytes = o_u + u_bytes - 256;                       // of hin_
    const size_t o_part = take(marg_chunks_ * sizeof(double));         // device only
    const size_t dev_bytes = in;
    size_t out = 0;
    const size_t p_w0 = out;
    out = up256(out + marg_.size() * sizeof(double));
    const size_t p_idx = out;
    out = up256(out + u_.size() * sizeof(uint64_t));
    const size_t p_top = out;
    out = up256(out + cols_ * sizeof(double));
    const size_t out_bytes = out;
    const bool out_host = out_bytes <= kHostBytes;

    // buffers: wait for the previous launch's reads before the host inputs
    // are rewritten; grow the device buffer after the stream has drained
    if (in_done_) IQ_OK(hipEventSynchronize(in_done_));
    else IQ_OK(hipEventCreateWithFlags(&in_done_, hipEventDisableTiming));
    if (dev_bytes + out_bytes > dcap_) {
        if (last_stream_) IQ_OK(hipStreamSynchronize(last_stream_));
        IQ_OK(hipStreamSynchronize(s));
        if (dbuf_) IQ_OK(hipFree(dbuf_));
        dbuf_ = nullptr;
        dcap_ = 0;
        const size_t cap = std::max<size_t>(dev_bytes + out_bytes, size_t(1) << 20) * 3 / 2;
        IQ_OK(hipMalloc(reinterpret_cast<void**>(&dbuf_), cap));
        IQ_OK(hipMemsetAsync(dbuf_, 0, 256, s));
        dcap_ = cap;
    }
    auto grow = [&](char*& host, char*& dev, size_t& have, size_t bytes) {
        if (bytes <= have) return;
        if (last_stream_) IQ_OK(hipStreamSynchronize(last_stream_));
        if (host) IQ_OK(hipHostFree(host));
        host = dev = nullptr;
        have = 0;
        const size_t cap = std::max<size_t>(bytes, size_t(1) << 20) * 3 / 2;
        IQ_OK(hipHostMalloc(reinterpret_cast<void**>(&host), cap, hipHostMallocDefault));
        IQ_OK(hipHostGetDevicePointer(reinterpret_cast<void**>(&dev), host, 0));
        have = cap;
    };
    grow(hin_, hin_dev_, hin_cap_, in_bytes);
    grow(hout_, hout_dev_, hout_cap_, out_bytes);
    last_stream_ = s;
    auto put = [&](size_t off, const void* src, size_t bytes) {
        if (bytes) std::memcpy(hin_ + off - 256, src, bytes);
    };
    put(o_marg, marg_.data(), many(marg_));
    put(o_coll, coll_.data(), many(coll_));
    put(o_ops, ops_.data(), ops_.size() * sizeof(ColOp));
    put(o_opit, opit_.data(), opit_.size() * sizeof(OpItem));
    put(o_basis, basis_.data(), many(basis_));
    for (int k = 0; k < kTreeSteps; ++k) put(o_tree[k], tree_[k].data(), many(tree_[k]));
    put(o_jobs, jobs_.data(), many(jobs_));
    if (marg_.size() > 1) std::memset(hin_ + o_done - 256, 0, marg_.size() * sizeof(uint32_t));
    if (cols_ > jobs_.size()) put(o_first, first_.data(), first_.size() * sizeof(uint64_t));
    put(o_u, u_.data(), u_.size() * sizeof(double));
    if (up_bytes) {
        upload_table(dbuf_ + 256, hin_, up_bytes, s);
        launches_ += 1;
    }
    // the next launch may rewrite hin_ once the upload has read it, or the
    // sampling kernel its uniforms
    const bool host_read = u_host && u_bytes;
    if (up_bytes && !host_read) IQ_OK(hipEventRecord(in_done_, s));
    char* d = dbuf_;
    char* dout = out_host ? hout_dev_ : dbuf_ + dev_bytes;
    auto table = [&](const auto& v, size_t off) {
        using I = typename std::decay<decltype(v[0])>::type;
        return v.size() > 1 ? reinterpret_cast<const I*>(d + off) : nullptr;
    };
    auto grid = [](uint64_t chunks, uint64_t cap) { return dim3(unsigned(std::min<uint64_t>(chunks, cap))); };
    auto run = [&](auto kernel, dim3 g, int threads, auto... args) {
        hipLaunchKernelGGL(kernel, g, dim3(unsigned(threads)), 0, s, args...);
        IQ_OK(hipGetLastError());
        launches_ += 1;
    };
    if (!basis_.empty())
        run(c64_ ? k_basis_items<float2> : k_basis_items<double2>, grid(basis_chunks_, kMaxGrid), kBlock, basis_[0],
            table(basis_, o_basis), uint32_t(basis_.size()), basis_chunks_);
    if (!coll_.empty())
        run(c64_ ? k_collapse_items<float2> : k_collapse_items<double2>, grid(coll_chunks_, kMaxGrid), kBlock, coll_[0],
            table(coll_, o_coll), uint32_t(coll_.size()), coll_chunks_);
    if (!opit_.empty())
        run(c64_ ? k_op_items<float2> : k_op_items<double2>, grid(op_chunks_, kMaxGrid), kBlock,
            reinterpret_cast<const OpItem*>(d + o_opit), uint32_t(opit_.size()), op_chunks_,
            reinterpret_cast<const ColOp*>(d + o_ops));
    if (!marg_.empty()) {
        const MargItem* const items = table(marg_, o_marg);   // null for one item, which has at most kMargBlocks shares
        const uint32_t ni = uint32_t(marg_.size());
        double* const part = reinterpret_cast<double*>(d + o_part);
        double* const w = reinterpret_cast<double*>(dout + p_w0);
        if (!items || marg_chunks_ <= kMargOneLaunch) {
            run(c64_ ? k_marginal_items<float2> : k_marginal_items<double2>, dim3(unsigned(marg_chunks_)), kMargThreads,
                marg_[0], items, ni, part, reinterpret_cast<uint32_t*>(items ? d + o_done : d), w);
        } else {
            const uint64_t share = (marg_chunks_ + kMargGrid - 1) / kMargGrid;
            run(c64_ ? k_marginal_shares<float2> : k_marginal_shares<double2>,
                dim3(unsigned((marg_chunks_ + share - 1) / share)), kMargThreads, items, ni, marg_chunks_,
                uint32_t(share), part, w);
            if (marg_chunks_ > ni)   // else every column is one share
                run(k_marginal_sums, grid(ni, kMaxGrid), int(kMargBlocks), items, ni, 0u, part, w);
        }
    }
    // trees: a workgroup per chunk, up to 2^20 of them
    for (int k = 0; k < kTreeSteps; ++k)
        if (!tree_[k].empty())
            run(k > 0 ? k_tree_items<double> : c64_ ? k_tree_items<float2> : k_tree_items<double2>,
                grid(tree_chunks_[k], uint64_t(1) << 20), kBlock, tree_[k][0], table(tree_[k], o_tree[k]),
                uint32_t(tree_[k].size()), tree_chunks_[k]);
    if (!jobs_.empty()) {
        const uint64_t nruns = u_.size();
        run(c64_ ? k_sample_items<float2> : k_sample_items<double2>,
            dim3(unsigned((nruns + kBlock - 1) / kBlock + (cols_ + kBlock - 1) / kBlock)), kBlock, jobs_[0],
            table(jobs_, o_jobs), uint32_t(jobs_.size()), reinterpret_cast<const uint64_t*>(d + o_first),
            reinterpret_cast<const double*>(u_host ? hin_dev_ + o_u - 256 : d + o_u), nruns,
            reinterpret_cast<uint64_t*>(dout + p_idx), cols_, reinterpret_cast<double*>(dout + p_top));
    }
    if (host_read) IQ_OK(hipEventRecord(in_done_, s));
    if (out_bytes && !out_host) {
        IQ_OK(hipMemcpyAsync(hout_, dout, out_bytes, hipMemcpyDeviceToHost, s));
        launches_ += 1;
    }
    out_w0_ = p_w0;
    out_idx_ = p_idx;
    out_top_ = p_top;
    res_run0_.clear();
    res_col0_.clear();
    for (const SampleJob& j : jobs_) {
        res_run0_.push_back(j.run0);
        res_col0_.push_back(j.col0);
    }
}

char* ItemQueue::stage(size_t bytes, hipStream_t s)
{
    if (stage_stream_) IQ_OK(hipStreamSynchronize(stage_stream_));
    stage_stream_ = nullptr;
    if (bytes > stage_cap_) {
        if (stage_) IQ_OK(hipHostFree(stage_));
        stage_ = nullptr;
        stage_cap_ = 0;
        const size_t cap = std::max<size_t>(bytes, size_t(1) << 18) * 3 / 2;
        IQ_OK(hipHostMalloc(reinterpret_cast<void**>(&stage_), cap, hipHostMallocDefault));
        stage_cap_ = cap;
    }
    stage_stream_ = s;
    return stage_;
}

double ItemQueue::w0(size_t item) const { return reinterpret_cast<const double*>(hout_ + out_w0_)[item]; }

const uint64_t* ItemQueue::indices(size_t job) const
{
    return reinterpret_cast<const uint64_t*>(hout_ + out_idx_) + res_run0_[job];
}

const double* ItemQueue::tops(size_t job) const
{
    return reinterpret_cast<const double*>(hout_ + out_top_) + res_col0_[job];
}

void ItemQueue::detach()
{
    if (last_stream_) (void)hipStreamSynchronize(last_stream_);
    last_stream_ = nullptr;
    if (stage_stream_) (void)hipStreamSynchronize(stage_stream_);
    stage_stream_ = nullptr;
    // the upload event belongs to the last owner's stream, which may be
    // destroyed and its handle reused: the next owner records a fresh one
    if (in_done_) (void)hipEventDestroy(in_done_);
    in_done_ = nullptr;
    clear_inputs();
}

namespace {
struct QueuePool {
    std::mutex mu;
    std::vector<std::unique_ptr<ItemQueue>> free[2];
};
QueuePool& queue_pool()
{
    static QueuePool* p = new QueuePool();   // never destroyed (the HIP runtime may be gone at exit)
    return *p;
}
}  // namespace

std::unique_ptr<ItemQueue> ItemQueuePool::take(bool c64)
{
    QueuePool& p = queue_pool();
    {
        std::lock_guard<std::mutex> lk(p.mu);
        auto& v = p.free[c64 ? 1 : 0];
        if (!v.empty()) {
            std::unique_ptr<ItemQueue> q = std::move(v.back());
            v.pop_back();
            return q;
        }
    }
    return std::make_unique<ItemQueue>(c64);
}

void ItemQueuePool::give(std::unique_ptr<ItemQueue> q)
{
    if (!q) return;
    q->detach();
    QueuePool& p = queue_pool();
    std::lock_guard<std::mutex> lk(p.mu);
    auto& v = p.free[q->c64() ? 1 : 0];
    if (v.size() < 64) v.push_back(std::move(q));
}

bool col_op_from(const GateOp& g, ColOp& o)
{
    std::memset(&o, 0, sizeof(o));
    std::vector<int> pos;
    for (int b = 0; b < 64; ++b)
        if ((g.ctrl_mask >> b) & 1) pos.push_back(b);
    o.cmask = g.ctrl_mask;
    const int nt = int(g.targets.size());
    auto put = [&](size_t k, const cdouble& c) {
        o.m[2 * k] = c.real();
        o.m[2 * k + 1] = c.imag();
    };
    switch (g.kind) {
    case OpKind::Dense:
        if (nt < 1 || nt > 2) return false;
        o.kind = nt == 1 ? 0 : 1;
        for (int q = 0; q < nt; ++q) {
            o.t[q] = g.targets[q];
            pos.push_back(g.targets[q]);
        }
        for (size_t k = 0; k < g.m.size(); ++k) put(k, g.m[k]);
        break;
    case OpKind::Diag:
        if (nt < 1 || nt > 3) return false;
        o.kind = 2;
        for (int q = 0; q < nt; ++q) o.t[q] = g.targets[q];
        for (size_t k = 0; k < g.m.size(); ++k) put(k, g.m[k]);
        break;
    case OpKind::PhaseOnes:
        o.kind = 3;
        put(0, g.m[0]);
        break;
    case OpKind::Swap2:
        o.kind = 4;
        o.t[0] = g.targets[0];
        o.t[1] = g.targets[1];
        pos.push_back(g.targets[0]);
        pos.push_back(g.targets[1]);
        break;
    default:
        return false;
    }
    if (pos.size() > 16) return false;
    std::sort(pos.begin(), pos.end());
    o.nt = nt;
    o.npos = int(pos.size());
    for (size_t k = 0; k < pos.size(); ++k) o.pos[k] = pos[k];
    return true;
}

}  // namespace q1t
