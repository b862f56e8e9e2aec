// Decode of a whole column to memory, shared by the decode entry points.
// Internal to libfls.so.
#pragma once

#include "fls_columns.hpp"

namespace fls {

// Column c to d_out: rows 0..n_rows-1 in original order, or (rows = false)
// every vector's 1,024 stored positions.
int materialize(const ColDev& c, uint64_t n_rows, bool rows, uint32_t* d_out, hipStream_t s);

}  // namespace fls
