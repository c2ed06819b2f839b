// Library plumbing: version, thread-local error text, launch check, fill and copy kernels.
#include <stdio.h>
#include <string.h>

#include "mq_api_internal.hpp"
#include "mq_common.hpp"
#include "mq_copy.hpp"
#include "mq_group.hpp"

static thread_local char g_err[256] = "";
static thread_local uint32_t* g_amax_feedback = nullptr;
static thread_local uint32_t* g_amax_feedback_mirror = nullptr;
uint32_t* mq_amax_feedback() { return g_amax_feedback; }
uint32_t* mq_amax_feedback_mirror() { return g_amax_feedback_mirror; }
void mq_set_amax_feedback(uint32_t* device_counter, uint32_t* mirror) {
    g_amax_feedback = device_counter;
    g_amax_feedback_mirror = mirror;
}

int mq_fail(int code, const char* msg) {
    snprintf(g_err, sizeof(g_err), "%s", msg);
    return code;
}

int mq_check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        snprintf(g_err, sizeof(g_err), "%s: %s", what, hipGetErrorString(e));
        return MQ_ERR_HIP;
    }
    return MQ_OK;
}

extern "C" int mq_version(void) { return MQ_VERSION; }
extern "C" const char* mq_last_error(void) { return g_err; }

namespace mq {
__global__ void fill_u32_n_kernel(uint32_t* p, uint32_t v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}
__global__ __launch_bounds__(256) void copy_group_kernel(const CopyTable tab) {
    const JobRef r = find_job(tab, blockIdx.x);
    copy_chunk(tab.job[r.ji], blockIdx.x - r.start);
}
// descriptors in device memory, of runs of few chunks each: blockIdx.y the run, blockIdx.x the chunk (a launch of 64 records a
// time instead: 192 of them 14.6 us in three launches, 4.9 in this one; 114 of them 8.9 and 2.3)
__global__ __launch_bounds__(256) void copy_table_kernel(const CopyTableEntry* __restrict__ table) {
    const CopyJob& job = table[blockIdx.y].job;
    if ((int32_t)blockIdx.x < job.chunks) copy_chunk(job, blockIdx.x);
}
// one long aligned run: one 16-byte unit per lane, no table (the access pattern that streams fastest on MI355X)
__global__ __launch_bounds__(256) void copy_run_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                       int64_t bytes) {
    const int64_t o = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 16;
    if (o + 16 <= bytes) st16(dst + o, ld16(src + o));
    else for (int64_t b = o; b < bytes; b++) dst[b] = src[b];
}
}  // namespace mq

int mq_copy_launch_run(const void* src, void* dst, int64_t bytes, hipStream_t st) {
    const int64_t blocks = (bytes + 4095) / 4096;
    if (blocks > 0x7FFFFFF0) return mq_fail(MQ_ERR_ARG, "copy too large");
    hipLaunchKernelGGL(mq::copy_run_kernel, dim3((unsigned)blocks), dim3(256), 0, st, (const uint8_t*)src, (uint8_t*)dst, bytes);
    return mq_check_launch("copy");
}

// chunks of a run of `rows` rows (job.bytes and the pitches are set), or -1 if they are too many; fills the chunk fields
int64_t mq_copy_job_finish(mq::CopyJob& job, int64_t rows) {
    const int64_t per_row = (job.bytes + mq::kCopyChunk - 1) / mq::kCopyChunk;
    if (per_row > 0x7FFFFFF0 || rows * per_row > 0x7FFFFFF0) return -1;
    job.chunks_per_row = per_row > 0 ? (int32_t)per_row : 1;
    job.chunks = (int32_t)(rows * per_row);
    return rows * per_row;
}
// tab.job[0..n) finished by the caller
int mq_copy_launch_group(mq::CopyTable& tab, hipStream_t st) {
    int64_t run = 0;
    for (int i = 0; i < tab.n; i++) {
        run += tab.job[i].chunks;
        if (run > 0x7FFFFFF0) return mq_fail(MQ_ERR_ARG, "copy group too large");
        tab.end[i] = (int32_t)run;
    }
    mq::seal_table(tab);
    if (tab.total == 0) return MQ_OK;
    hipLaunchKernelGGL(mq::copy_group_kernel, dim3((unsigned)tab.total), dim3(256), 0, st, tab);
    return mq_check_launch("grouped copy");
}
// n finished descriptors in device memory; max_chunks: the most chunks one of them has
int mq_copy_launch_table(const mq::CopyTableEntry* device_jobs, int n, int64_t max_chunks, hipStream_t st) {
    if (n == 0 || max_chunks == 0) return MQ_OK;
    hipLaunchKernelGGL(mq::copy_table_kernel, dim3((unsigned)max_chunks, (unsigned)n), dim3(256), 0, st, device_jobs);
    return mq_check_launch("grouped copy");
}

extern "C" int mq_fill_u32(void* p, uint32_t value, int64_t n, void* stream) {
    if (!p || n < 0) return mq_fail(MQ_ERR_ARG, "bad argument");
    if (n == 0) return MQ_OK;
    int64_t blocks = (n + 255) / 256;
    if (blocks > mq_grid_cap()) blocks = mq_grid_cap();
    hipLaunchKernelGGL(mq::fill_u32_n_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (uint32_t*)p,
                       value, n);
    return mq_check_launch("fill");
}
