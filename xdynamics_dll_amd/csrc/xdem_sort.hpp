// xdem_sort.hpp -- stable sort of (cell hash, index) pairs and the cell table, on gfx950.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace xdem {

// Bytes of scratch the sort needs for n pairs (digit counts; the caller provides the
// key/value buffers).
size_t cell_sort_scratch_bytes(uint32_t n);

// Sorts n (hash, index) pairs in place by hash (the bits that ncell - 1 needs), stable: equal
// hashes keep their input order. Writes the sorted indices to sorted_index too, and to
// cstart/cend (ncell entries) the first and one-past-last position of every occupied cell,
// 0xffffffff and 0 for the others. buf: four arrays of n entries; every pointer is a device
// pointer; the work is queued on `stream`.
hipError_t cell_sort(uint32_t* hash, uint32_t* index, uint32_t* sorted_index, uint32_t* cstart, uint32_t* cend, uint32_t n,
                     uint32_t ncell, uint32_t* const buf[4], void* scratch, hipStream_t stream);

}  // namespace xdem
