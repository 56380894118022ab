// Dense gates on 4 to 12 target qubits as matrix products on the MFMA units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gates.h"

namespace q1t {

// How a dense gate on `op.targets` (4..12 of them) runs over `ncols` columns
// of 2^n amplitudes.
struct DensePlan {
    int K = 0;                // target qubits
    bool tiles = false;       // k_dense_tile (else k_dense_rows)
    int log_cols = 0;         // amplitude groups per block (log2)
    uint64_t nblocks = 0;     // blocks per column
    int rtw = 1;              // k_dense_rows: row tiles per wave
    int log_slice = 0;        // ... rows staged at a time (log2)
    uint32_t splits = 1;      // ... workgroups that share a block's rows
    uint64_t chunk = 0;       // ... blocks per launch
    size_t matrix_bytes = 0;  // device bytes of the packed matrix
    size_t scratch_bytes = 0; // device bytes of the results' copy (0: in place)
};
DensePlan plan_dense(const GateOp& op, int n, size_t ncols, size_t elem_bytes);

// The packed matrix of a gate on up to kHostPackK qubits, made on the host.
constexpr int kHostPackK = 6;
template <typename V> void pack_dense(const cdouble* m, int K, V* out);

// Launch the gate on columns a, a + col_stride, ... (2^n amplitudes each).
// Device memory: `packed` holds the packed matrix, or `raw` the gate's
// row-major matrix in the state's precision and `packed` gets
// plan.matrix_bytes; `scratch` has plan.scratch_bytes (null for none).
template <typename V>
void launch_dense(const DensePlan& plan, const GateOp& op, int n, V* a, uint64_t col_stride, unsigned ncols,
                  const V* raw, V* packed, V* scratch, hipStream_t s);

}  // namespace q1t
