// Sweep program records (host and device): the in-tile ops and phases a
// tile sweep executes.  Plain C++ with fixed-width types only, so the
// sweep kernels specialised at run time can include it as text.
#pragma once

#ifndef __HIPCC_RTC__
#include <cstdint>
#else
// hipRTC: fixed-width types of its built-in runtime header
typedef __hip_internal::int32_t int32_t;
typedef __hip_internal::uint32_t uint32_t;
typedef __hip_internal::uint64_t uint64_t;
typedef __hip_internal::uint16_t uint16_t;
typedef __hip_internal::uint8_t uint8_t;
#endif

namespace q1t {

// One in-tile operation of a sweep program (read by every thread of a
// workgroup; uniform).
enum SwOpType : int32_t { SW_DENSE1 = 0, SW_PHASE = 1, SW_DIAG1 = 2, SW_BLOCK = 3, SW_APPLY = 4, SW_PAIR = 5 };

// Body of a SW_DENSE1 op, read off its 2x2 matrix (SwOp::aux).
// The _SEQ forms round as the general body does (its second product fused):
// whole-state programs use them, which give the bits of the gates applied one
// by one with the general body.
// The last six are reduced forms (reduce_program): the matrix without a factor
// that the flush applies once, rotations [[a, -b], [b, a]], reflections
// [[a, b], [b, -a]] and RX [[a, ib], [ib, a]] divided by their diagonal entry
// (_D, one coefficient m[0] = b / a) or their off-diagonal one (_O, m[0] = a / b):
// four fused multiply-adds per pair instead of eight operations.
enum SwDenseForm : uint32_t {
    SWF_GENERAL = 0, SWF_REAL = 1, SWF_SWAP = 2, SWF_RX = 3, SWF_Y = 4, SWF_REAL_SEQ = 5, SWF_RX_SEQ = 6,
    SWF_ROT_D = 7, SWF_ROT_O = 8, SWF_REFL_D = 9, SWF_REFL_O = 10, SWF_RX_D = 11, SWF_RX_O = 12
};
// Body of a SW_PHASE op (SwOp::aux): general, times i, times -i, times -1.
enum SwPhaseForm : uint32_t { SWP_GENERAL = 0, SWP_I = 1, SWP_MINUS_I = 2, SWP_NEG = 3 };

// Controls (and the ones-mask of a phase) are split by where their bits live
// during the op's phase: `cr` over register indices (uniform per register
// slot), `ct` over thread-index bits (one lane test per op), `co` over global
// bits outside the tile (uniform per tile).
struct SwOp {
    int32_t type;
    int32_t reg;       // SW_DENSE1: index of the target among the phase's register bits; SW_PHASE and
                       // SW_DIAG1 without register bits: 1 if the factor goes to the thread's product,
                       // which a SW_APPLY at the phase's end multiplies into its registers
    int32_t dreg;      // SW_DIAG1: register index of the target, or -1; reduced dense forms: 1 for the _O one
    int32_t dtid;      // SW_DIAG1: thread-index bit of the target, or -1
    int32_t dglobal;   // SW_DIAG1: global bit of the target when it is outside the tile, or -1
    uint32_t cr;       // control (or phase) mask over register indices
    uint32_t ct;       // control (or phase) mask over thread-index bits
    uint32_t aux;      // SW_DENSE1 / SW_PHASE: body form; SW_BLOCK: offset of the block matrix
    uint64_t co;       // control (or phase) mask over global bits outside the tile
    double m[8];       // SW_DENSE1: m00, m01, m10, m11 (re, im); SW_PHASE: m[0..1]; SW_DIAG1: d0, d1
    float mf[8];       // m rounded to FP32 once (the complex64 sweeps read these)
};

struct SwPhase {
    uint32_t op_begin, op_end;
    uint32_t reg_mask;   // local tile bits held in registers during this phase
    uint32_t kind;       // 0: register phase, 1: fused dense block on LDS,
                         // 2: tile factors -- ops [op_begin, op_end) are
                         // diagonal ops on bits outside the tile only; the
                         // tile is scaled by the product of their factors
                         // as it is stored (the program's last phase;
                         // programs of the specialised kernels only)
                         // 4: a dense gate on two local bits rpos[0] (the
                         // matrix's high bit) and rpos[1]; ops op_begin ..
                         // op_begin + 3 hold its rows in m
    uint8_t rpos[8];     // local positions of the register bits (ascending)
    uint8_t tbit[16];    // local positions of the thread bits (ascending)
    // register phases: an affine map over GF(2) of the local index, applied
    // when the phase writes the tile back to LDS -- amplitude l moves to
    // XOR over the set bits of l of their columns, XOR wxor.  wcol holds the
    // columns of the thread bits (tbit order), then of the register bits
    // (rpos order).  SWAP, X and singly controlled X on local bits are such
    // maps and cost no op of their own.
    uint32_t wmap;       // 0: identity (plain write-back)
    uint32_t wxor;
    uint16_t wcol[16];
    // register phases, for the interpreting kernels (place_phases): byte offsets
    // in LDS, swizzled.  A thread reads its element k at tin ^ slot_in[k] and
    // writes it back at tout ^ slot_out[k]; tin and tout are the low and high
    // halves of the XOR of col over the thread's set bits, wxor is in slot_out.
    uint32_t col[12];
    uint32_t slot_in[16], slot_out[16];
};

// LDS swizzle of local element l in a 2^M tile: XOR-fold of the bits above
// SW into the low SW bits (an involution, XOR-linear in l).
constexpr int swizzle_slot(int SW, int M, int l)
{
    int f = 0;
    for (int s = SW; s < M; s += SW) f ^= l >> s;
    return l ^ (f & ((1 << SW) - 1));
}

// Swizzle width of the sweep kernels for 2^M tiles (13 -> 5, else 4).
constexpr int sweep_swizzle_bits(int M) { return M == 13 ? 5 : 4; }

// ---- ops of the interpreting kernels (k_sweep, k_sweep_batched, k_whole)

// A SwOp in the state's precision: 80 bytes complex128, 48 complex64 (a
// program of 100 ops then stays in the 16 KiB scalar cache).  X, CX and Y have
// the body of their matrix, phases of any value the general product (0, 1 and
// +-i are exact factors).  `code`: bits 0-7 body (SwDenseForm or kInterp*),
// 8-15 register bit of the target, 16-23 thread bit or outer bit of a
// diagonal's target, 24 a factor that goes to the thread's product; `ctl`: controls over register indices (low half) and
// thread bits (high half); `co`: controls over bits outside the tile.
constexpr uint32_t kInterpPhase = 16, kInterpDiagReg = 17, kInterpDiagTid = 18, kInterpDiagOuter = 19,
                   kInterpApply = 20, kInterpLane = 1u << 24;
template <typename R> struct InterpOpT {
    uint32_t code;
    uint32_t ctl;
    uint64_t co;
    R m[8];
};

// ---- whole-state programs (k_whole): a state of up to 14 qubits in LDS

// A register phase: R register bits, thread bits the others.  The LDS slot of a
// thread's element k is tin ^ (slot[k] & 0xffff) when the phase reads the state
// and tout ^ (slot[k] >> 16) when it writes it back; tin and tout are the low
// and high halves of the XOR of col over the thread's set bits, tout also of
// wxor; all swizzled.
struct WholePhase {
    uint32_t op_begin, op_end;
    uint32_t wmap;       // 0: written back where it was read
    uint32_t wxor;
    uint32_t col[12];
    uint32_t slot[16];
};

struct WholeItem {
    void* amp;           // the column (the first of a launch with a column stride)
    uint32_t n;          // qubits
    uint32_t nphases;
    uint32_t phases, ops;   // first records in the tables
    uint32_t fresh, pad;    // 1: the column is |0..0> and not in memory yet
};

}  // namespace q1t
