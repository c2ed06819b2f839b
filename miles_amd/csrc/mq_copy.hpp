// Byte copies: the workgroup that moves one chunk, in launches of its own (mq_core.hip) or behind the workgroups of another one.
#pragma once
#include <type_traits>

#include "mq_common.hpp"
#include "mq_group.hpp"

namespace mq {

// Grouped byte copies: a workgroup moves one 16 KiB chunk (four 16-byte units per lane) of one of the launch's runs.
// Runs whose pointers are 16-byte aligned use 16-byte accesses, the bytes behind the last whole unit a lane each; the others
// go byte by byte.  The runs of a sync are mostly records of a few bytes, where the launch is bound by its chain of memory
// round trips (descriptor, source): with the tail in one lane's loop, a byte after the other, 18 records of 8 bytes took
// 4.4 us, now 3.2.
constexpr int kCopyUnits = 4;
constexpr int kCopyChunk = kCopyUnits * 4096;
__device__ __forceinline__ void copy_chunk(const CopyJob& job, const int32_t local) {
    const int32_t row = local / job.chunks_per_row;
    const int64_t off0 = (int64_t)(local - row * job.chunks_per_row) * kCopyChunk, bytes = job.bytes;
    const uint8_t* __restrict__ src = (const uint8_t*)load_global_ptr(&job.src) + row * job.src_pitch;
    uint8_t* __restrict__ dst = (uint8_t*)load_global_ptr(&job.dst) + row * job.dst_pitch;
    const bool aligned = (((uintptr_t)src | (uintptr_t)dst) & 15) == 0;
    const int64_t stop = off0 + kCopyChunk < bytes ? off0 + kCopyChunk : bytes;
    if (aligned) {
        u32x4 v[kCopyUnits];
#pragma unroll
        for (int u = 0; u < kCopyUnits; u++) {
            const int64_t o = off0 + (u * 256 + threadIdx.x) * 16;
            if (o + 16 <= stop) v[u] = ld16(src + o);
        }
        const int64_t tail = stop & ~(int64_t)15;       // a chunk starts at a whole unit
        if (tail + threadIdx.x < stop) dst[tail + threadIdx.x] = src[tail + threadIdx.x];
#pragma unroll
        for (int u = 0; u < kCopyUnits; u++) {
            const int64_t o = off0 + (u * 256 + threadIdx.x) * 16;
            if (o + 16 <= stop) st16(dst + o, v[u]);
        }
    } else {
        for (int64_t b = off0 + threadIdx.x; b < stop; b += 256) dst[b] = src[b];
    }
}

// Copies that ride along: rows of workgroups beside those of the tensors of a launch, neither of which depends on the other.  A launch of
// their own cost 3.5 to 5 us, to move the few bytes of the shape records of a packed payload (48 INT4 matrices of [2048, 7168], 266 -> 262.5 us;
// 16 of [3072, 256] 20.5 -> 17.8, 29 of [1408, 256] 17.3 -> 15.3).
// Either the runs themselves in the kernel's arguments, or entries of the device table of a submitted list; each of at most
// kRiderChunks chunks.
constexpr int kRiderChunks = 4;
struct CopyRun {
    const uint8_t* src;
    uint8_t* dst;
    int64_t bytes;
};
struct NoRiders {};
struct Riders {
    int32_t row, rows;        // of the grid
    int32_t n, pad;
    CopyRun run[kMaxGroup];
};
struct RidersRef {
    int32_t row, rows;
    int32_t n, pad;
    const CopyTableEntry* entry;
};
// a chunk of one run; a unit at a time, so that the kernel of the tensors keeps its number of registers
__device__ __forceinline__ void ride_chunk(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, const int64_t bytes, const int32_t chunk) {
    const int64_t first = (int64_t)chunk * kCopyChunk, stop = first + kCopyChunk < bytes ? first + kCopyChunk : bytes;
    const bool aligned = (((uintptr_t)src | (uintptr_t)dst) & 15) == 0;
    const int64_t tail = aligned && first < stop ? stop & ~(int64_t)15 : first;       // a chunk starts at a whole unit
#pragma unroll 1
    for (int64_t o = first + threadIdx.x * 16; o < tail; o += 256 * 16) st16(dst + o, ld16(src + o));
#pragma unroll 1
    for (int64_t b = tail + threadIdx.x; b < stop; b += 256) dst[b] = src[b];
}
// whether this workgroup of 256 lanes was one of theirs
template <class R>
__device__ __forceinline__ bool ride_along(const R& r) {
    if constexpr (std::is_same<R, NoRiders>::value) return false;
    else {
        const uint32_t row = blockIdx.y - r.row;
        if (row >= (uint32_t)r.rows) return false;
        const uint32_t id = row * gridDim.x + blockIdx.x, i = id / kRiderChunks;
        const int32_t chunk = (int32_t)(id % kRiderChunks);
        if (i >= (uint32_t)r.n) return true;
        if constexpr (std::is_same<R, Riders>::value) {
            const CopyRun& run = r.run[i];
            ride_chunk(load_global_ptr(&run.src), load_global_ptr(&run.dst), run.bytes, chunk);
        } else {
            const CopyJob& job = r.entry[i].job;       // (one row)
            ride_chunk(load_global_ptr(&job.src), load_global_ptr(&job.dst), job.bytes, chunk);
        }
        return true;
    }
}
// the tensor of any other one
template <class R>
__device__ __forceinline__ uint32_t tensor_row(const R& r) {
    if constexpr (std::is_same<R, NoRiders>::value) return blockIdx.y;
    else return (int32_t)blockIdx.y < r.row ? blockIdx.y : blockIdx.y - r.rows;
}

// what a launcher is handed (n = 0: nobody rides): runs, or entries of a device table
struct RiderArgs {
    int n;
    const CopyRun* run;
    const CopyTableEntry* entry;
};
// Calls launch(rows of the grid, the riders as a kernel takes them) for `tensors` rows of `blocks` workgroups.  The riders come
// first, and are done long before the others; a long launch has them last, where its first workgroups are not held up (us, last /
// first: 87 tensors of 44 workgroups 16.6 / 15.3, 72 of 192 25.8 / 25.5, 48 of 3584 265.6 / 266.3).
constexpr int64_t kRidersLast = 32768;
template <class Launch>
inline void with_riders(const RiderArgs& args, int tensors, int64_t blocks, Launch launch) {
    const int32_t rows = (int32_t)(((int64_t)args.n * kRiderChunks + blocks - 1) / blocks);
    const int32_t row = blocks * tensors >= kRidersLast ? tensors : 0;
    if (args.n == 0) {
        launch((unsigned)tensors, NoRiders{});
    } else if (args.entry) {
        launch((unsigned)(rows + tensors), RidersRef{row, rows, args.n, 0, args.entry});
    } else {
        Riders r{row, rows, args.n, 0, {}};
        for (int i = 0; i < args.n; i++) r.run[i] = args.run[i];
        launch((unsigned)(rows + tensors), r);
    }
}

}  // namespace mq
