// Rows of a read's buckets (offset, count), one per map, read-major.
#pragma once

#include <cstdint>
#include <hip/hip_runtime.h>

// Two neighbouring buckets. A row of an odd number of maps starts on an 8-byte boundary, so a pair
// is promised no more than that (one 16-byte load either way: global loads need no
// alignment beyond a dword's).
typedef uint32_t BucketPair __attribute__((ext_vector_type(4), aligned(8)));

// Buckets u and u + 1 (u even) of a row of M maps as (offset, count, offset, count); 0 past its end.
__host__ __device__ inline uint4 bucketPair(const uint2* row, int u, int M){
    if(u + 1 < M){
        const BucketPair x = *reinterpret_cast<const BucketPair*>(row + u);
        return make_uint4(x.x, x.y, x.z, x.w);
    }
    if(u < M) return make_uint4(row[u].x, row[u].y, 0u, 0u);
    return make_uint4(0u, 0u, 0u, 0u);
}
