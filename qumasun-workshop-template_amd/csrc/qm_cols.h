// Columns of a matrix made of up to kMaxColBlocks blocks, on the device.
#pragma once

#include "qm_internal.h"

namespace qm {

template <typename T>
using GlobalPtr = __attribute__((address_space(1))) T *;

// Column j of the chain without branches or indexed arrays (a branch per block,
// or pointers picked from an array in scratch, made each panel of the products
// wait for its addresses): the block's displacement is summed up from the
// steps between consecutive blocks.
template <typename T>
struct Cols {
    uint64_t base;                 // address of column 0
    int64_t step[kMaxColBlocks];   // bytes that block b starts off the continuation of block b - 1
    int first[kMaxColBlocks];      // its first column, INT32_MAX past the last block
    int64_t pitch;                 // bytes between columns of a block
    __device__ __forceinline__ Cols(const ColBlocks &c, int64_t ng) : base((uint64_t)c.ptr[0]), pitch(ng * sizeof(T)) {
        int f = 0;
#pragma unroll
        for (int b = 1; b < kMaxColBlocks; ++b) {
            f += c.ncols[b - 1];
            first[b] = b < c.nblk ? f : INT32_MAX;
            step[b] = (int64_t)((uint64_t)c.ptr[b] - (uint64_t)c.ptr[b - 1]) - c.ncols[b - 1] * pitch;
        }
    }
    __device__ __forceinline__ GlobalPtr<T> at(int j) const {
        uint64_t a = base + j * pitch;
#pragma unroll
        for (int b = 1; b < kMaxColBlocks; ++b) a += j >= first[b] ? step[b] : 0;
        return (GlobalPtr<T>)a;
    }
    // the first column after j that another block holds
    __device__ __forceinline__ int end(int j) const {
        int l = INT32_MAX;
#pragma unroll
        for (int b = kMaxColBlocks - 1; b > 0; --b) l = first[b] > j ? first[b] : l;
        return l;
    }
};

}  // namespace qm
