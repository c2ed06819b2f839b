// NVFP4 (e2m1 codes, one e4m3 scale per 1x16 block, one fp32 scale per tensor) for gfx950.
// Reference: miles/utils/nvfp4.py:19-114 (layout, global scale); block arithmetic as restated in
// miles/kernels/quant/nvfp4_qdq.py:716-743,859-889,1079-1081:
//   S_enc = min(e4m3_max*6 / amax, FLT_MAX), 1 if amax == 0 or the quotient is 0;  S_dec = 1 / S_enc
//   per block: bmax = max|x|; s8 = sat_e4m3(bmax == 0 ? 0 : bmax * (S_enc * f32(1/6)))
//              inv = min(1 / (f32(s8) * S_dec), FLT_MAX);  code = sat_e2m1(x * inv)
//   published global scale: 1 / min(e4m3_max*6/amax, FLT_MAX) with only the ==0 repair (nvfp4.py:19-39)
//
// Pass 1 (mq_nvfp4_amax): up to 256 workgroups per tensor stream its elements and each writes one partial maximum
// into the tensor's section of the amax record: plain stores, no atomics (thousands of agent-scope atomics
// on one address serialise at ~8 ns each on this multi-XCD part) and nothing to clear.
// Lists of tensors that fit the chip's registers a few at a time run in one pass instead (nvfp4_one_pass_kernel).
// Pass 2 (mq_nvfp4_quant): the partial maxima become the amax, S_enc/6 and 1/S_enc, and each tensor's global scale is
// published: in short passes by every workgroup while its loads are under way (a launch of its own for the fold took 4.2 us:
// four [1077, 64] tensors 12.8 -> 8.1 us for the two passes), in long ones by a launch in front (nv_published).  Two lanes own
// one 16-element block (16 bytes each), the block amax is one DPP step, and each lane emits four bytes of codes.  A gate/up
// pair writes two sections of one record.
#include <type_traits>

#include "mq_api_internal.hpp"
#include "mq_common.hpp"
#include "mq_group.hpp"

namespace mq {

constexpr int kNvThreads = 256;
#ifndef MQ_NV_UNROLL
#define MQ_NV_UNROLL 2
#endif
constexpr int kNvUnroll = MQ_NV_UNROLL;
constexpr float kSixth = 0.16666667163372040f;  // 0x3E2AAAAB

static_assert(kSectionWords == MQ_NVFP4_SECTION_WORDS && kRecordSections == MQ_NVFP4_SECTIONS, "record layout");
#ifndef MQ_AMAX_UNROLL
#define MQ_AMAX_UNROLL 4
#endif
constexpr int kAmaxUnroll = MQ_AMAX_UNROLL;             // 16-byte units per lane per loop trip

// grid (up to kSectionWords, tensors): workgroup b of a tensor strides over its 16 KiB chunks and writes word b of
// the section.  A launch whose largest tensor has fewer chunks takes that many workgroups, which write a zero into the
// words nobody owns (amax_section_store): fifty-nine tensors of 17 chunks 8.7 us with 256 workgroups each, 5.1 with 17.
// job.units counts whole 16-byte units; job.s carries the element count for the sub-unit tail.
// KEEP of a lane's four loads are left in the memory-side cache for the pass behind (kept_quarters).
// (descriptors of a device table are in the quantizer's form, whose tensors are whole units: no tail, and job.s is the
// block-scale pointer there)
// (16-bit inputs, bf16 or fp16: the maximum is taken on the absolute bit patterns and converted to the fp32 pattern once)
__device__ __forceinline__ void amax_section_store(uint32_t* __restrict__ section, int t, uint32_t m) {
    const uint32_t word = blockIdx.x + (uint32_t)t * gridDim.x;
    if (word < (uint32_t)kSectionWords) section[word] = t == 0 ? m : 0u;
}
template <class Table, int F16, int KEEP>
__global__ __launch_bounds__(256) void nvfp4_amax_bf16_kernel(const Table tab) {
    __shared__ uint32_t wave_amax[4];
    const FlatJob job = flat_job(tab);       // a copy in registers: a descriptor in device memory must not be re-read after the stores
    const uint16_t* __restrict__ w = (const uint16_t*)job.w;
    uint32_t* __restrict__ section = (uint32_t*)job.aux + job.section * kSectionWords;
    const int64_t n16 = job.units, numel = std::is_same<Table, FlatRef>::value ? n16 * 8 : (int64_t)(uintptr_t)job.s;
    const int t = threadIdx.x;
    uint32_t m2 = 0;
    for (int64_t base = (int64_t)blockIdx.x * (256 * kAmaxUnroll); base < n16; base += (int64_t)gridDim.x * 256 * kAmaxUnroll) {
        u32x4 v[kAmaxUnroll];
        // (a loop for each kind: loads that one loop chooses between lose the hint)
#pragma unroll
        for (int i = 0; i < KEEP; i++) {
            const int64_t unit = base + i * 256 + t;
            v[i] = unit < n16 ? ld16_keep(w + unit * 8) : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = KEEP; i < kAmaxUnroll; i++) {
            const int64_t unit = base + i * 256 + t;
            v[i] = unit < n16 ? ld16(w + unit * 8) : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < kAmaxUnroll; i++)
            m2 = max2_u16(m2, max2_u16(max2_u16(abs2(v[i].x), abs2(v[i].y)), max2_u16(abs2(v[i].z), abs2(v[i].w))));
    }
    uint32_t m = hmax_u16(m2);
    if (blockIdx.x == 0 && t == 0)
        for (int64_t i = n16 * 8; i < numel; i++) m = umax(m, (uint32_t)(w[i] & 0x7FFFu));
    m = wave_max(m);
    if ((t & 63) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    amax_section_store(section, t, f2u(elem_lo<F16>(umax(umax(wave_amax[0], wave_amax[1]), umax(wave_amax[2], wave_amax[3])))));
}

// fp32 input (units and the element count as above): 16-byte loads of four elements
template <class Table, int KEEP>
__global__ __launch_bounds__(256) void nvfp4_amax_f32_kernel(const Table tab) {
    __shared__ uint32_t wave_amax[4];
    const FlatJob job = flat_job(tab);
    const float* __restrict__ w = (const float*)job.w;
    const int64_t loads = job.units * 2, numel = std::is_same<Table, FlatRef>::value ? job.units * 8 : (int64_t)(uintptr_t)job.s;
    const int t = threadIdx.x;
    uint32_t m = 0;
    for (int64_t base = (int64_t)blockIdx.x * (256 * kAmaxUnroll); base < loads; base += (int64_t)gridDim.x * 256 * kAmaxUnroll) {
        u32x4 v[kAmaxUnroll];
#pragma unroll
        for (int i = 0; i < KEEP; i++) {
            const int64_t at = base + i * 256 + t;
            v[i] = at < loads ? ld16_keep(w + at * 4) : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = KEEP; i < kAmaxUnroll; i++) {
            const int64_t at = base + i * 256 + t;
            v[i] = at < loads ? ld16(w + at * 4) : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < kAmaxUnroll; i++)
            m = umax(m, umax(umax(v[i].x & 0x7FFFFFFFu, v[i].y & 0x7FFFFFFFu), umax(v[i].z & 0x7FFFFFFFu, v[i].w & 0x7FFFFFFFu)));
    }
    if (blockIdx.x == 0 && t == 0)
        for (int64_t i = loads * 4; i < numel; i++) m = umax(m, f2u(w[i]) & 0x7FFFFFFFu);
    m = wave_max(m);
    if ((t & 63) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    amax_section_store((uint32_t*)job.aux + job.section * kSectionWords, t,
                       umax(umax(wave_amax[0], wave_amax[1]), umax(wave_amax[2], wave_amax[3])));
}

__global__ __launch_bounds__(256) void nvfp4_amax_generic_kernel(const void* __restrict__ w, int dtype, int64_t numel,
                                                                 uint32_t* __restrict__ section) {
    __shared__ uint32_t wave_amax[4];
    const int t = threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    uint32_t m = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + t; i < numel; i += stride)
        m = umax(m, f2u(load_f32(w, i, dtype)) & 0x7FFFFFFFu);
    m = wave_max(m);
    if ((t & 63) == 0) wave_amax[t >> 6] = m;
    __syncthreads();
    if (t == 0) section[blockIdx.x] = umax(umax(wave_amax[0], wave_amax[1]), umax(wave_amax[2], wave_amax[3]));
}

struct NvScales {
    float enc_sixth;  // S_enc * (1/6)
    float s_dec;      // 1 / S_enc
    float enc;        // S_enc
};
__device__ __forceinline__ NvScales nv_scales(float amax, float numer) {
    float enc = __builtin_fminf(numer / amax, kFltMax);
    if (amax == 0.0f || enc == 0.0f) enc = 1.0f;
    NvScales r;
    r.enc_sixth = enc * kSixth;
    r.s_dec = 1.0f / enc;
    r.enc = enc;
    return r;
}
__device__ __forceinline__ float nv_published_scale(float amax, float numer) {
    float enc = numer / amax;
    if (enc > kFltMax) enc = kFltMax;  // NaN stays NaN
    if (enc == 0.0f) enc = 1.0f;
    return 1.0f / enc;
}

// words of a record behind its sections
constexpr int kRecEncSixth = kRecAmax + 1;                     // S_enc * (1/6)
constexpr int kRecSDec = kRecAmax + 2;                         // 1 / S_enc
constexpr int kRecEnc = kRecAmax + 3;                          // S_enc

// The tail of a record and the published scales, from the folded amax.
__device__ __forceinline__ void nv_record_tail(uint32_t* rec, float amax, const NvScales& gs) {
    rec[kRecAmax] = f2u(amax);
    rec[kRecEncSixth] = f2u(gs.enc_sixth);
    rec[kRecSDec] = f2u(gs.s_dec);
    rec[kRecEnc] = f2u(gs.enc);
}
// What a plain run (no carried-over amax) leaves behind, by one lane of every tensor's first workgroup: its own published
// scale, and for the last tensor of a record (job.section its place there, job.pad the number of tensors that share the
// record) the record's tail and state words.
__device__ __forceinline__ void nv_publish_plain(const FlatJob& job, float amax, const NvScales& gs, float numer, uint32_t* moved_counter) {
    if (job.aux2) *(float*)job.aux2 = nv_published_scale(amax, numer);
    if (job.section != job.pad - 1) return;
    uint32_t* rec = (uint32_t*)job.aux;
    amax_feedback(moved_counter, rec[kRecAmax] != f2u(amax), (uint32_t)job.pad);
    rec[kRecVolatile] = 0;
    rec[kRecMovedRuns] = 0;
    nv_record_tail(rec, amax, gs);
}
// an amax and its scales, as the quantizing code below asks for them once its loads are issued
struct NvAmaxScales {
    float amax;
    NvScales gs;
};
__device__ __forceinline__ float uniform_f(float v) { return u2f((uint32_t)__builtin_amdgcn_readfirstlane((int)f2u(v))); }
__device__ __forceinline__ NvAmaxScales nv_record_scales(const FlatJob& job) {
    const uint32_t* __restrict__ rec = (const uint32_t*)job.aux;
    return NvAmaxScales{u2f(rec[kRecAmax]), NvScales{u2f(rec[kRecEncSixth]), u2f(rec[kRecSDec]), u2f(rec[kRecEnc])}};
}
// The same from the partial maxima of an amax pass, folded by every workgroup of the pass behind it while its data is under
// way: a launch between the two passes that did it took 4.2 us, and the host's part of one (long passes: nv_published).  Only the first wavefront folds
// and divides (four words a lane and section), the others wait for its four values in LDS: Four Over Six is bound by vector
// instructions, and some sixty of them in every wavefront cost it a tenth (fifty [616, 1584] tensors 24.5 us with the scales
// read from a record, 30.0 folded by all four wavefronts, 27.3 by one).  Scalar registers hold the result, where values read
// from a record are.
__device__ __forceinline__ uint32_t nv_wave_fold(const uint32_t* __restrict__ words, int sections, int lane) {
    uint32_t m = 0;
    for (int k = 0; k < sections; k++) {
        const u32x4 v = *reinterpret_cast<const u32x4_at4*>(words + k * kSectionWords + lane * 4);
        m = umax(m, umax(umax(v.x, v.y), umax(v.z, v.w)));
    }
    return wave_max(m);
}
template <class AmaxBits>
__device__ __forceinline__ NvAmaxScales nv_shared_scales(const int t, float numer, AmaxBits first_wave_bits) {
    static_assert(kSectionWords == 4 * kWave, "a wavefront takes a section in one load");
    __shared__ float shared[4];
    if (t < kWave) {
        const float amax = u2f(first_wave_bits());
        const NvScales gs = nv_scales(amax, numer);
        shared[0] = amax;
        shared[1] = gs.enc_sixth;
        shared[2] = gs.s_dec;
        shared[3] = gs.enc;
    }
    __syncthreads();
    return NvAmaxScales{uniform_f(shared[0]), NvScales{uniform_f(shared[1]), uniform_f(shared[2]), uniform_f(shared[3])}};
}

// A partial maximum that the single pass of a carried run has collected: the amax pass of a plain run leaves its own in the
// same words, without the mark and below every word with it, so the sections need no clearing between the two.
constexpr uint32_t kCarriedMark = 0x80000000u;

// Fold kernel, one workgroup per tensor.
// MODE 0 (mq_nvfp4_fold, and single calls outside the packed kernels): fold the first job.section sections of the record
//   and publish the scales.  Tensors that share a record compute the same values and write them twice.
// MODE 2 (the job driver, after the single pass of a carried run): job.section is the tensor's place inside its record and
//   job.pad the number of tensors sharing it; they sit next to each other in the table.  Only the workgroup of the last one
//   works: it folds what the run left in all their sections (kCarriedMark), writes every one's global scale and clears the
//   sections for the next run.  It checks the amax and scales the record held before against the new ones: all four words
//   equal means the codes just written with the old values are final (kRecRedo = 0); otherwise the new values are stored
//   and kRecRedo = 1 asks for a second quantization.
//   A record whose amax moved on two syncs in a row is marked volatile (kRecVolatile): on the next carried sync the
//   single pass only collects its partial maxima (no codes are written with an amax that is likely stale again) and the
//   second pass quantizes it with the fresh amax -- the cost of the plain two-pass form, instead of two full
//   quantizations.  The mark is dropped as soon as the amax has held still for one sync (amax_record_after_carried_run).
template <int MODE, class Table>
__global__ __launch_bounds__(256) void nvfp4_fold_kernel(const Table tab, float numer, uint32_t* moved_counter, uint32_t* moved_mirror) {
    __shared__ uint32_t lds4[4];
    const int ji = blockIdx.x;
    const FlatJob& job = tab.job[ji];
    const int sections = MODE == 0 ? job.section : job.pad;
    if (MODE != 0) amax_feedback_folded(moved_counter, moved_mirror, gridDim.x);
    if (MODE != 0 && job.section != job.pad - 1) return;
    uint32_t* rec = (uint32_t*)job.aux;
    uint32_t m = 0;
    for (int i = threadIdx.x; i < sections * kSectionWords; i += 256) {
        const uint32_t word = rec[i];
        m = umax(m, MODE == 0 ? word : (word & kCarriedMark) != 0 ? word & ~kCarriedMark : 0u);
        if (MODE != 0) rec[i] = 0;
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float amax = u2f(umax(umax(lds4[0], lds4[1]), umax(lds4[2], lds4[3])));
        const NvScales gs = nv_scales(amax, numer);
        if (MODE == 2) {
            const bool moved = !(rec[kRecAmax] == f2u(amax) && rec[kRecEncSixth] == f2u(gs.enc_sixth) &&
                                 rec[kRecSDec] == f2u(gs.s_dec) && rec[kRecEnc] == f2u(gs.enc));
            amax_record_after_carried_run(rec, moved);
            amax_feedback(moved_counter, moved, (uint32_t)sections);
        }
        nv_record_tail(rec, amax, gs);
        const float published = nv_published_scale(amax, numer);
        if (MODE == 0) {
            if (job.aux2) *(float*)job.aux2 = published;
        } else {
            for (int k = 0; k < sections; k++)
                if (tab.job[ji - k].aux2) *(float*)tab.job[ji - k].aux2 = published;
        }
    }
}

// Publish kernel, one wavefront per tensor, grid (1, tensors): what every workgroup of a plain run's quantize pass does by
// itself where the pass is short (nv_shared_scales) is done once here, and the pass reads the record.
template <class Table>
__global__ __launch_bounds__(kWave) void nvfp4_publish_kernel(const Table tab, float numer, uint32_t* moved_counter, uint32_t* moved_mirror) {
    const FlatJob job = flat_job(tab);
    if (blockIdx.y == 0) amax_feedback_folded(moved_counter, moved_mirror, gridDim.y);
    const float amax = u2f(nv_wave_fold((const uint32_t*)job.aux, job.pad, (int)threadIdx.x));
    if (threadIdx.x != 0) return;
    ((uint32_t*)job.aux)[kRecRedo] = 0;
    nv_publish_plain(job, amax, nv_scales(amax, numer), numer, moved_counter);
}

// ---- Four Over Six block scaling (miles/kernels/quant/nvfp4_qdq.py:893-990) --------------------------------
// Every block is quantized twice: "map to 6" with scale6 = e4m3(min(RN(RN(bmax / 6) * S_enc), 448)) and "map to 4"
// with scale4 = e4m3(min(RN(that product * 1.5), 448)); the candidate with the strictly smaller reconstruction
// error wins, ties go to map-to-6.  The error is an fp32 sum over the 16 elements in element order:
//   default   | RN(RN(RN(value * f32(scale)) * amax) / (6 * e4m3_max)) - x |   (MQ_NVFP4_ERR_MSE: its square)
//   ERR_FP16  | f32(RN_f16(f16(value) * f16(scale))) - RN(x * S_enc) |
__device__ __forceinline__ void nv_decode8(uint32_t word, float q[8]) {
    const f32x2 a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 0), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 1);
    const f32x2 c = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 2), d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 3);
    q[0] = a.x; q[1] = a.y; q[2] = b.x; q[3] = b.y; q[4] = c.x; q[5] = c.y; q[6] = d.x; q[7] = d.y;
}
// x / d for d = 2688 or 1536 with y = RN(1/d): q0 = RN(x*y); r = x - q0*d (exact in an FMA); q = RN(q0 + r*y) is the
// correctly rounded quotient for every fp32 mantissa of x and both divisors (exhaustive CPU check, 2^23 mantissas
// each), provided no intermediate leaves the normal range, i.e. for |x| in 2^-91 .. 2^89 (and for zero, which comes
// out as +0 whatever its sign: no error term can see that).  The numerators here are RN(RN(value * f32(scale)) * amax)
// with value * f32(scale) either zero or in 2^-10 .. 2688, so one test of the tensor amax covers every element:
// nv_fast_division(amax) allows the sequence for the whole tensor, otherwise every quotient is the IEEE division.
// 0: IEEE divisions; 1: the sequence; 2: the sequence, and the amax has at most 12 significant bits (the amax of a bf16 or
// fp16 tensor has), so that value x f32(scale) x amax -- 2, 4 and 12 bits -- is exact in whatever order it is taken, and it is
// 2^-60 or more, so that a block maximum out of the range of div_by_shared (below 2^-91; S_enc is at most 2^72) has a scale of
// zero whatever its sixth comes to in the last place
__device__ __forceinline__ int nv_fast_division(float amax) {
    const uint32_t e = f2u(amax) & 0x7F800000u;
    if (!(e >= 0x17800000u /* 2^-80 */ && e <= 0x65800000u /* 2^76 */)) return 0;
    return (f2u(amax) & 0xFFFu) == 0 && e >= 0x21800000u /* 2^-60 */ ? 2 : 1;
}
template <int FASTDIV>
__device__ __forceinline__ float div_by_numer(float x, float d, float y) {
    if (!FASTDIV) return x / d;
    const float q0 = x * y;
    const float r = __builtin_fmaf(-q0, d, x);
    return __builtin_fmaf(r, y, q0);
}
// error terms of this lane's eight elements; EM bit 0: squared error, bit 1: fp16 candidate error
template <int EM, int FASTDIV>
__device__ __forceinline__ void nv_error_terms(const float f[8], uint32_t word, float s_f, float amax, float enc, float denom,
                                               float denom_inv, float term[8]) {
    float q[8];
    nv_decode8(word, q);
    // FASTDIV 2: every partial product of value x f32(scale) x amax is exact, one multiplication per element
    const float scale_amax = s_f * amax;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        float diff;
        if (EM & 2) {
            _Float16 h = (_Float16)q[j] * (_Float16)s_f;        // both factors exact in fp16; one fp16 rounding
            float hf = (float)h;
            asm volatile("" : "+v"(hf));                          // keep the fp16 product a value of its own
            diff = hf - f[j] * enc;
        } else {
            diff = div_by_numer<FASTDIV>(FASTDIV == 2 ? q[j] * scale_amax : (q[j] * s_f) * amax, denom, denom_inv) - f[j];
        }
        term[j] = (EM & 1) ? diff * diff : __builtin_fabsf(diff);
    }
}
// One lane works on one block.  With two lanes per block every block-level step (the two candidate scales, their
// reciprocals, the comparison) is done twice, and the error sum, which has to run through the sixteen terms in element
// order, takes sixteen additions in each lane of the pair.  The data is therefore regrouped first: a lane ends up with the
// thirty-two bytes of one whole block, and the kernels are bound by vector instructions, not by memory.
struct NvCandidate16 {
    uint32_t at;        // eight times the e4m3 byte of the scale: where the table has its entry
    uint32_t lo, hi;    // codes of elements 0..7 and 8..15
    float a;            // RN(f32(sc) * amax / denom): what one unit of the code grid is worth (tensors that take the estimate)
    __device__ __forceinline__ uint32_t sc() const { return at >> 3; }
};
// A candidate's block scale is one of 128 bytes, and what the quantizer needs of it -- the reciprocal
// min(1 / (f32(byte) * S_dec), FLT_MAX) and, for the error estimate, RN(f32(byte) * amax / denom) -- depends on the byte
// and the tensor only.  A workgroup therefore computes both for every byte once (128 lanes, one IEEE division each,
// while its loads are in flight) into LDS, and a candidate is one 8-byte LDS read instead of a decode, a multiplication,
// a range test, a refined reciprocal and a three-instruction division per block and candidate.
struct NvScaleEntry {
    float inv, a;
};
__device__ __forceinline__ void nv_fill_scale_table(NvScaleEntry* table, int t, float amax, float s_dec, bool estimate,
                                                    float denom, float denom_inv) {
    if (t < 128) {
        const float s_f = hw_e4m3x2_decode<false>((uint32_t)t).x;
        NvScaleEntry e;
        e.inv = __builtin_fminf(1.0f / (s_f * s_dec), kFltMax);
        // (only read where f32(byte) * amax is exact and the sequence gives its correctly rounded quotient)
        e.a = estimate ? div_by_numer<2>(s_f * amax, denom, denom_inv) : 0.0f;
        table[t] = e;
    }
}
__device__ __forceinline__ NvCandidate16 nv_candidate16(const float f[16], uint32_t at, const NvScaleEntry* table) {
    NvCandidate16 c;
    c.at = at;
    const NvScaleEntry e = *reinterpret_cast<const NvScaleEntry*>(reinterpret_cast<const char*>(table) + at);
    const float inv = e.inv;
    c.a = e.a;
    asm("" : "=v"(c.lo), "=v"(c.hi));      // (four conversions write all of each)
    c.lo = hw_e2m1x2<0>(f[0] * inv, f[1] * inv, c.lo);
    c.lo = hw_e2m1x2<1>(f[2] * inv, f[3] * inv, c.lo);
    c.lo = hw_e2m1x2<2>(f[4] * inv, f[5] * inv, c.lo);
    c.lo = hw_e2m1x2<3>(f[6] * inv, f[7] * inv, c.lo);
    c.hi = hw_e2m1x2<0>(f[8] * inv, f[9] * inv, c.hi);
    c.hi = hw_e2m1x2<1>(f[10] * inv, f[11] * inv, c.hi);
    c.hi = hw_e2m1x2<2>(f[12] * inv, f[13] * inv, c.hi);
    c.hi = hw_e2m1x2<3>(f[14] * inv, f[15] * inv, c.hi);
    return c;
}
template <int EM, int FASTDIV>
__device__ __forceinline__ float nv_block_error(const float f[16], const NvCandidate16& c, float amax, float enc, float denom,
                                                float denom_inv) {
    float term[8], error = 0.0f;
    const float s_f = hw_e4m3x2_decode<false>(c.sc()).x;
    nv_error_terms<EM, FASTDIV>(f, c.lo, s_f, amax, enc, denom, denom_inv, term);
#pragma unroll
    for (int j = 0; j < 8; j++) error = error + term[j];
    nv_error_terms<EM, FASTDIV>(f + 8, c.hi, s_f, amax, enc, denom, denom_inv, term);
#pragma unroll
    for (int j = 0; j < 8; j++) error = error + term[j];
    return error;
}
// A cheaper error sum that decides almost every block.  With a = RN(f32(scale) * amax / denom), the exact term's
// dequantized value RN(q * f32(scale) * amax / denom) IS q * a for the codes that are powers of two (0.5, 1, 2, 4: scaling
// by a power of two commutes with the rounding) and differs from q * a by at most 2^-23 of its size for 1.5, 3 and 6.
// The estimate sums |q * a - x|, each term rounded once (an FMA), in element order.  Every step is within a few units in
// the last place of the exact computation, so the estimated sum S' and the exact sum S of a candidate differ by at most
//   2^-20 (31.4 a + 2 bmax) + 30.3 * 2^-24 S'
// (per element: 2.01 * 2^-24 |deq| between the two dequantized values, 2^-24 (|deq| + |x|) for each of the two roundings
// of the difference, |deq| <= 6 a (1 + 2^-22), |x| <= bmax; for the sums: recursive summation of sixteen non-negative
// terms is within 15.1 * 2^-24 of their true sum, on both sides).  Whenever the two estimates are further apart than
// the two bounds together, the exact sums compare the same way.
//
// The squared error (SQUARED) has the same estimate with each difference d' = RN(q * a - x) squared.  Per element the
// exact difference d and d' are within E = 2^-24 (24.1 a + 2 bmax) of each other (the three contributions above), so
// the squares differ by at most E (2 |d'| + E) and, rounded, by 2^-23 d'^2 more; over the block, with
// sum |d'| <= 4 sqrt(sum d'^2), the estimated and the exact sum of a candidate differ by at most
//   8.1 E sqrt(S') + 16.1 E^2 + 32.5 * 2^-24 S'.
template <bool SQUARED>
__device__ __forceinline__ float nv_block_error_estimate(const float f[16], const NvCandidate16& c, float a) {
    float q[8], sum = 0.0f;
    nv_decode8(c.lo, q);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float d = __builtin_fmaf(q[j], a, -f[j]);
        sum = sum + (SQUARED ? d * d : __builtin_fabsf(d));
    }
    nv_decode8(c.hi, q);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float d = __builtin_fmaf(q[j], a, -f[8 + j]);
        sum = sum + (SQUARED ? d * d : __builtin_fabsf(d));
    }
    return sum;
}
struct NvCandidates16 {
    NvCandidate16 c4, c6;
};
// TRUSTED: bmax is a number not above amax, so that s6_hp is at most 448 (1 + 2^-22), which the conversion takes for 448
template <int FASTDIV, bool F32, bool TRUSTED>
__device__ __forceinline__ NvCandidates16 nv_candidates16(const float f[16], float bmax, const NvScales& gs, const NvScaleEntry* table) {
    float sixth;
    if (FASTDIV == 2) {
        sixth = div_by_shared(bmax, 6.0f, 0x1.555556p-3f);
    } else {
        const bool plain_bmax = shared_div_ok(bmax);
        // (an fp32 block's maximum has more bits than the shared-divisor sequence takes)
        sixth = !F32 && __builtin_amdgcn_ballot_w64(!plain_bmax) == 0 ? div_by_shared(bmax, 6.0f, 0x1.555556p-3f) : bmax / 6.0f;
    }
    const float s6_hp = sixth * gs.enc, s4_hp = s6_hp * 1.5f;
    uint32_t bytes;      // of both scales, which have no sign bit
    asm("" : "=v"(bytes));
    bytes = hw_e4m3x2<false>(__builtin_fminf(s4_hp, kFp8Max), TRUSTED ? s6_hp : __builtin_fminf(s6_hp, kFp8Max), bytes);
    return NvCandidates16{nv_candidate16(f, (bytes << 3) & 0x3F8u, table), nv_candidate16(f, (bytes >> 5) & 0x3F8u, table)};
}
// What the estimates say of two candidates (FASTDIV 2: f32(scale) * amax is exact and its quotient by denom comes correctly
// rounded from the sequence).
struct NvPick {
    bool decided, four;
};
template <int EM>
__device__ __forceinline__ NvPick nv_estimated_pick(const float f[16], float bmax, const NvCandidate16& c4, const NvCandidate16& c6) {
    const float a4 = c4.a, a6 = c6.a;
    const float g4 = nv_block_error_estimate<EM == 1>(f, c4, a4), g6 = nv_block_error_estimate<EM == 1>(f, c6, a6);
    float guard;
    if (EM == 0) {
        // twice the bound's first part and four times its second: rounding in this line cannot bring it below the bound
        guard = 0x1p-17f * (__builtin_fmaf(8.0f, a4 + a6, bmax) + (g4 + g6));
    } else {
        // twice the squared error's bound for both candidates, and more (the hardware square root is within one unit
        // in the last place; the small constant keeps a denormal sum from dropping out of it and is the floor below
        // which two sums are too small to call)
        const float e4 = 0x1p-24f * (25.0f * a4 + 2.0f * bmax), e6 = 0x1p-24f * (25.0f * a6 + 2.0f * bmax);
        guard = 17.0f * (e4 * __builtin_amdgcn_sqrtf(g4 + 0x1p-100f) + e6 * __builtin_amdgcn_sqrtf(g6 + 0x1p-100f)) +
                33.0f * (e4 * e4 + e6 * e6) + 0x1p-17f * (g4 + g6) + 0x1p-100f;
    }
    // (an all-zero block, or two candidates with one scale byte -- the block that holds the tensor's maximum, whose
    // scales both saturate: the candidates are the same, the tie goes to map-to-6, as g4 < g6 says; a NaN compares false)
    return NvPick{__builtin_fabsf(g4 - g6) > guard || bmax == 0.0f || c4.at == c6.at, g4 < g6};
}
template <int EM, int FASTDIV, bool F32 = false, bool TRUSTED = false>
__device__ __forceinline__ NvCandidate16 nv_four_over_six16(const float f[16], float bmax, float amax, const NvScales& gs,
                                                            float denom, float denom_inv, const NvScaleEntry* table) {
    const NvCandidates16 both = nv_candidates16<FASTDIV, F32, TRUSTED>(f, bmax, gs, table);
    const NvCandidate16 c4 = both.c4, c6 = both.c6;
    if constexpr ((EM == 0 || EM == 1) && FASTDIV == 2) {
        const NvPick pick = nv_estimated_pick<EM>(f, bmax, c4, c6);
        if (__builtin_amdgcn_ballot_w64(!pick.decided) == 0) return pick.four ? c4 : c6;
        // a wavefront with a block too close to call (a few blocks in 10 000, most of them exact ties) takes the exact sums below
    }
    const float e4 = nv_block_error<EM, FASTDIV>(f, c4, amax, gs.enc, denom, denom_inv);
    const float e6 = nv_block_error<EM, FASTDIV>(f, c6, amax, gs.enc, denom, denom_inv);
    return e4 < e6 ? c4 : c6;
}
// error mode of a flags word, as the EM template argument
static inline int nv_error_mode(int flags) { return ((flags & MQ_NVFP4_ERR_MSE) ? 1 : 0) | ((flags & MQ_NVFP4_ERR_FP16) ? 2 : 0); }

// The amax and scales that a fake quantization of job.w works with: the caller's fp32 scalar (job.aux2), or the maximum of
// the kSectionWords partial maxima an amax pass left in job.aux.
__device__ __forceinline__ NvAmaxScales nv_fake_scales(const FlatJob& job, const int t, float numer) {
    return nv_shared_scales(t, numer, [&] {
        return job.aux2 ? *(const uint32_t*)job.aux2 : nv_wave_fold((const uint32_t*)job.aux, 1, t);
    });
}
// eight values times a scale as a unit of 16-bit elements
template <int F16>
__device__ __forceinline__ u32x4 nv_scaled16(const float q[8], float scale) {
    uint32_t p[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float a = q[2 * i] * scale, b = q[2 * i + 1] * scale;
        if (F16) {
            asm volatile("" : "+v"(a), "+v"(b));     // keep the product apart from the conversion: a fused fma(.., +0) loses -0
            p[i] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)a) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)b) << 16);
        } else {
            p[i] = hw_bf16x2(a, b);
        }
    }
    return u32x4{p[0], p[1], p[2], p[3]};
}

// the largest magnitude of sixteen numbers (no NaN), three at a time
__device__ __forceinline__ float nv_numbers_max(const float f[16]) {
    float m = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(f[0]), __builtin_fabsf(f[1])), __builtin_fabsf(f[2]));
#pragma unroll
    for (int j = 3; j < 15; j += 2) m = __builtin_fmaxf(__builtin_fmaxf(m, __builtin_fabsf(f[j])), __builtin_fabsf(f[j + 1]));
    return __builtin_fmaxf(m, __builtin_fabsf(f[15]));
}
template <int F16>
__device__ __forceinline__ void nv_unpack16(const u32x4 lo, const u32x4 hi, float f[16]) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        f[2 * k] = elem_lo<F16>(lo[k]);
        f[2 * k + 1] = elem_hi<F16>(lo[k]);
        f[8 + 2 * k] = elem_lo<F16>(hi[k]);
        f[9 + 2 * k] = elem_hi<F16>(hi[k]);
    }
}

// Four Over Six over kNvThreads * 2 units starting at `base`: loaded as the standard quantizer loads them (lane t takes
// units t and kNvThreads + t, so a wavefront's loads are contiguous), then regrouped through LDS inside each wavefront so
// that the even lane of a pair holds the block made of units 2p, 2p + 1 and the odd lane the block kNvThreads + 2p, + 1.
// Returns the largest |element| of the lane's block (bf16 bits).  QDQ: job.q takes the dequantized values instead of the
// codes, the amax is that of the fake quantization below, and the values go back through LDS to the lanes that loaded them.
#ifndef MQ_NV_FOS_ROUNDS
#define MQ_NV_FOS_ROUNDS 2
#endif
// consecutive pieces of kNvThreads * 2 units one Four Over Six workgroup takes.  Measured on 96 DeepSeek-V3 expert
// matrices, steady state: 4.74 / 4.95 / 4.83 TB/s with one / two / three pieces (78 and 86 registers with two and three:
// six and five wavefronts per SIMD instead of seven).
constexpr int kFosRounds = MQ_NV_FOS_ROUNDS;
// units a workgroup of the quantizer covers (FOS as in nvfp4_quant_units)
constexpr int64_t nv_units_per_block(int fos) { return (int64_t)kNvThreads * kNvUnroll * (fos ? kFosRounds : 1); }
// `trusted`: the amax is the maximum of these very elements, so that a tensor whose amax is a number has no NaN in it.
template <int EM, int F16, bool QDQ, class Scales>
__device__ __forceinline__ uint32_t nvfp4_fos_units(const FlatJob& job, const int64_t base, const int t, const float denom,
                                                    const float inv_denom, const bool trusted, Scales scales) {
    static_assert(kNvUnroll == 2, "the regrouping pairs the two units of a lane");
    constexpr uint32_t kPiece = kNvThreads * 2;
    __shared__ u32x4 stage[kPiece];
    __shared__ NvScaleEntry scale_table[128];
    __shared__ float final_scale[QDQ ? 128 : 1];       // of the dequantized values, by the scale's byte
    const uint16_t* __restrict__ w = (const uint16_t*)job.w;
    uint32_t* __restrict__ q = (uint32_t*)job.q;
    uint8_t* __restrict__ s8 = (uint8_t*)job.s;
    uint16_t* __restrict__ y0 = (uint16_t*)job.q + base * 8;
    const int64_t left = job.units - base;
    const uint32_t rem_all = left < kPiece * kFosRounds ? (uint32_t)left : kPiece * kFosRounds;
    const uint16_t* __restrict__ w0 = w + base * 8;
    uint32_t* __restrict__ q0 = q + base;
    uint8_t* __restrict__ s80 = s8 + base / 2;
    // every load of every piece is issued before the first is waited for: this kernel is bound by its arithmetic, some
    // two hundred vector instructions per block, and a wavefront that computes on one piece while nothing of its own is
    // in flight leaves the memory system idle.  A lane past the end reads the workgroup's first unit again (always
    // there) and drops it.
    u32x4 in[kFosRounds][2];
#pragma unroll
    for (int r = 0; r < kFosRounds; r++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t off = r * kPiece + (uint32_t)t + i * kNvThreads;
            in[r][i] = ld16(w0 + (off < rem_all ? off : 0u) * 8u);
        }
    const NvAmaxScales known = scales();
    const NvScales gs = known.gs;
    const float amax = known.amax;
    const int fastdiv = nv_fast_division(amax);
    // the error's divisor 6 * e4m3_max is one of two constants and the same for the whole launch: its reciprocal is
    // picked on the scalar unit
    constexpr float kInv2688 = 1.0f / 2688.0f, kInv1536 = 1.0f / 1536.0f;
    const float denom_inv = denom == 2688.0f ? kInv2688 : denom == 1536.0f ? kInv1536 : 1.0f / denom;
    // (a workgroup that comes here again, in the striding second pass, writes the same values over the table: one tensor)
    nv_fill_scale_table(scale_table, t, amax, gs.s_dec, fastdiv == 2 && EM < 2, denom, denom_inv);
    if (QDQ && t < 128) final_scale[t] = (hw_e4m3x2_decode<false>((uint32_t)t).x * amax) * inv_denom;
    __syncthreads();
    uint32_t seen = 0;
#pragma unroll
    for (int r = 0; r < kFosRounds; r++) {
        if (r * kPiece >= rem_all) break;      // the same for the whole workgroup
        const uint32_t rem = rem_all - r * kPiece;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t off = (uint32_t)t + i * kNvThreads;
            stage[off] = in[r][i];      // (a unit past the end holds the workgroup's first unit: real data, nothing new to any maximum)
        }
        // A wavefront reads back only what its own lanes wrote, and the LDS serves one wavefront's accesses in the order
        // it issued them: no workgroup barrier, only the compiler is told not to move the reads above the writes.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint32_t first = ((t & 1) ? (uint32_t)kNvThreads : 0u) + ((uint32_t)t & ~1u);      // the block's first unit
        const u32x4 lo = stage[first], hi = stage[first + 1];
        // (and the next piece's writes stay below these reads)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        auto pattern_max = [&] {
            return hmax_u16(max2_u16(max2_u16(max2_u16(abs2(lo.x), abs2(lo.y)), max2_u16(abs2(lo.z), abs2(lo.w))),
                                     max2_u16(max2_u16(abs2(hi.x), abs2(hi.y)), max2_u16(abs2(hi.z), abs2(hi.w)))));
        };
        float f[16];
        nv_unpack16<F16>(lo, hi, f);
        NvCandidate16 c;
        if (trusted && fastdiv == 2) {
            c = nv_four_over_six16<EM, 2, false, true>(f, nv_numbers_max(f), amax, gs, denom, denom_inv, scale_table);
        } else {
            const uint32_t mb = pattern_max();
            seen = umax(seen, mb);
            const float bmax = elem_lo<F16>(mb);
            c = fastdiv == 2   ? nv_four_over_six16<EM, 2>(f, bmax, amax, gs, denom, denom_inv, scale_table)
                : fastdiv == 1 ? nv_four_over_six16<EM, 1>(f, bmax, amax, gs, denom, denom_inv, scale_table)
                               : nv_four_over_six16<EM, 0>(f, bmax, amax, gs, denom, denom_inv, scale_table);
        }
        if (QDQ) {
            const float scale = final_scale[c.sc()];
            float y[8];
            nv_decode8(c.lo, y);
            stage[first] = nv_scaled16<F16>(y, scale);
            nv_decode8(c.hi, y);
            stage[first + 1] = nv_scaled16<F16>(y, scale);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t off = (uint32_t)t + i * kNvThreads;
                const u32x4 o = stage[off];
                if (off < rem) st16(y0 + (r * kPiece + off) * 8u, o);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else if (first < rem) {      // the tensor is whole blocks: both units of a block are inside or outside
            st8(q0 + r * kPiece + first, u32x2{c.lo, c.hi});      // `first` is even and `base` a multiple of the piece
            s80[(r * kPiece + first) >> 1] = (uint8_t)c.sc();
        }
    }
    return seen;
}

// one 16-byte unit, half of a 1x16 block whose other half the neighbouring lane holds: the block's scale byte, the unit's
// codes and the block maximum (a 16-bit pattern)
struct NvUnitCodes {
    uint32_t sc, word, mb;
};
template <int F16>
__device__ __forceinline__ NvUnitCodes nvfp4_quant_unit(const u32x4 v, const NvScales& gs) {
    constexpr uint32_t kInfBits = F16 ? 0x7C00u : 0x7F80u;
    const uint32_t m2 = max2_u16(max2_u16(abs2(v.x), abs2(v.y)), max2_u16(abs2(v.z), abs2(v.w)));
    const uint32_t mb = group_max2(hmax_u16(m2));
    const float bmax = elem_lo<F16>(mb);
    const float s_hp = bmax == 0.0f ? 0.0f : bmax * gs.enc_sixth;
    const float f[8] = {elem_lo<F16>(v.x), elem_hi<F16>(v.x), elem_lo<F16>(v.y), elem_hi<F16>(v.y),
                        elem_lo<F16>(v.z), elem_hi<F16>(v.z), elem_lo<F16>(v.w), elem_hi<F16>(v.w)};
    uint32_t sc, word;
    if (mb < kInfBits && s_hp == s_hp) {
        sc = hw_e4m3x2<false>(__builtin_fminf(s_hp, kFp8Max), 0.0f, 0u) & 0xFFu;
        const float s_f = hw_e4m3x2_decode<false>(sc).x;
        // 1 / (block scale x global decode scale): the refined hardware reciprocal where it equals the division (every
        // divisor in 2^-91 .. 2^90, far below FLT_MAX), decided for the wavefront; an all-zero block has divisor 0
        const float d = s_f * gs.s_dec;
        float inv;
        if (__builtin_amdgcn_ballot_w64(!shared_div_ok(d)) == 0) inv = recip_shared(d);
        else inv = __builtin_fminf(1.0f / d, kFltMax);
        word = hw_e2m1x2<0>(f[0] * inv, f[1] * inv, 0u);
        word = hw_e2m1x2<1>(f[2] * inv, f[3] * inv, word);
        word = hw_e2m1x2<2>(f[4] * inv, f[5] * inv, word);
        word = hw_e2m1x2<3>(f[6] * inv, f[7] * inv, word);
    } else {
        sc = sw_e4m3fn_sat(s_hp);
        const float s_f = sw_e4m3fn_decode(sc);
        const float inv = __builtin_fminf(1.0f / (s_f * gs.s_dec), kFltMax);
        word = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) word |= sw_e2m1(f[j] * inv) << (4 * j);
    }
    return NvUnitCodes{sc, word, mb};
}

// kNvThreads * kNvUnroll units starting at `base` of one tensor; returns the largest |element| this lane saw (bf16 bits)
// FOS = 0: standard quantizer; FOS = 1 + error mode: Four Over Six, which returns nothing of use where `trusted` (nvfp4_fos_units)
template <int FOS, int F16, class Scales>
__device__ __forceinline__ uint32_t nvfp4_quant_units(const FlatJob& job, const int64_t base, const int t, const float denom, const bool trusted, Scales scales) {
    if (FOS) return nvfp4_fos_units<(FOS > 0 ? FOS - 1 : 0), F16, false>(job, base, t, denom, 0.0f, trusted, scales);
    const uint16_t* __restrict__ w = (const uint16_t*)job.w;
    uint32_t* __restrict__ q = (uint32_t*)job.q;
    uint8_t* __restrict__ s8 = (uint8_t*)job.s;
    const int64_t total_units = job.units;
    // everything a lane adds to the workgroup's (uniform) base addresses is a 32-bit offset
    const int64_t left = total_units - base;
    const uint32_t rem = left < kNvThreads * kNvUnroll ? (uint32_t)left : (uint32_t)(kNvThreads * kNvUnroll);
    const uint16_t* __restrict__ w0 = w + base * 8;
    uint32_t* __restrict__ q0 = q + base;
    uint8_t* __restrict__ s80 = s8 + base / 2;        // `base` is a multiple of the two lanes of a block
    u32x4 v[kNvUnroll];
#pragma unroll
    for (int i = 0; i < kNvUnroll; i++) {
        const uint32_t off = (uint32_t)t + i * kNvThreads;
        v[i] = off < rem ? ld16(w0 + off * 8u) : u32x4{0u, 0u, 0u, 0u};
    }
    const NvScales gs = scales().gs;
    uint32_t seen = 0;
#pragma unroll
    for (int i = 0; i < kNvUnroll; i++) {
        const uint32_t off = (uint32_t)t + i * kNvThreads;
        const NvUnitCodes c = nvfp4_quant_unit<F16>(v[i], gs);
        seen = umax(seen, c.mb);
        if (off < rem) {
            st4(q0 + off, c.word);
            if ((t & 1) == 0) s80[off >> 1] = (uint8_t)c.sc;
        }
    }
    return seen;
}

// the largest |element| (bf16 bits) this lane sees in kNvThreads * kNvUnroll units starting at `base`: what the single
// pass does for a record marked volatile
__device__ __forceinline__ uint32_t nvfp4_amax_units(const FlatJob& job, const int64_t base, const int t) {
    const uint16_t* __restrict__ w = (const uint16_t*)job.w;
    uint32_t m2 = 0;
#pragma unroll
    for (int i = 0; i < kNvUnroll; i++) {
        const int64_t unit = base + i * kNvThreads + t;
        const u32x4 v = unit < job.units ? ld16(w + unit * 8) : u32x4{0u, 0u, 0u, 0u};
        m2 = max2_u16(m2, max2_u16(max2_u16(abs2(v.x), abs2(v.y)), max2_u16(abs2(v.z), abs2(v.w))));
    }
    return hmax_u16(m2);
}

// Carried-over amax.  A weight tensor's amax rarely changes from one sync to the next (the largest element has to move
// to another bf16 value), and the amax record of a replayed job list still holds the last sync's amax and scales.
// PASS 1 quantizes with those in a single read of the tensor and collects this sync's partial maxima on the way (one
// atomic max per workgroup into the tensor's section, cleared by the previous fold); the fold kernel then compares, and
// PASS 2, a small grid striding over the blocks, quantizes again only the tensors whose amax did change.
// PASS 0 is the second pass of the plain two-pass form (amax kernel, then this): every workgroup folds the partial maxima,
// and the first one of each tensor publishes what comes of them, also for a tensor without elements.
// PASS 3 is the same behind nvfp4_publish_kernel.
// `own` (passes 0 and 3): the partial maxima are those of an amax pass over these very elements.  A caller of mq_nvfp4_quant
// may hand over a record that holds another amax, below some elements or without the NaN among them.
template <int FOS, int PASS, class Table, int F16>
__global__ __launch_bounds__(kNvThreads) void nvfp4_quant_bf16_kernel(const Table tab, float denom, const bool own, uint32_t* moved_counter, uint32_t* moved_mirror) {
    const FlatJob job = flat_job(tab);       // a copy in registers: a descriptor in device memory must not be re-read after the stores
    const int t = threadIdx.x;
    constexpr int64_t kPerBlock = nv_units_per_block(FOS);
    if (PASS == 2) {
        if (((const uint32_t*)job.aux)[kRecRedo] == 0) return;
        // an XCD takes a run of consecutive blocks in every trip of the grid, as the flat grids do (second pass 2 pct faster)
        const int64_t first = xcd_chunked_block(gridDim.x == kSectionWords ? kSectionWords / kXcds : tab.chunk);
        for (int64_t base = first * kPerBlock; base < job.units; base += (int64_t)gridDim.x * kPerBlock)
            nvfp4_quant_units<FOS, F16>(job, base, t, denom, true, [&] { return nv_record_scales(job); });
        return;
    }
    const int64_t base = flat_block(tab) * kPerBlock;
    if (PASS == 0) {
        if (base >= job.units && base > 0) return;
        if (base == 0 && blockIdx.y == 0) amax_feedback_folded(moved_counter, moved_mirror, gridDim.y);
        auto fold = [&] {
            const NvAmaxScales a = nv_shared_scales(t, denom, [&] { return nv_wave_fold((const uint32_t*)job.aux, job.pad, t); });
            if (base == 0 && t == 0) {
                ((uint32_t*)job.aux)[kRecRedo] = 0;
                nv_publish_plain(job, a.amax, a.gs, denom, moved_counter);
            }
            return a;
        };
        if (job.units == 0) fold();
        else nvfp4_quant_units<FOS, F16>(job, base, t, denom, own, fold);
        return;
    }
    if (base >= job.units) return;
    if (PASS == 3) {
        nvfp4_quant_units<FOS, F16>(job, base, t, denom, own, [&] { return nv_record_scales(job); });
        return;
    }
    uint32_t seen;
    if (PASS == 1 && ((const uint32_t*)job.aux)[kRecVolatile] != 0) {
        seen = 0;
        for (int64_t piece = base; piece < base + kPerBlock && piece < job.units; piece += kNvThreads * kNvUnroll)
            seen = umax(seen, nvfp4_amax_units(job, piece, t));
    } else seen = nvfp4_quant_units<FOS, F16>(job, base, t, denom, false, [&] { return nv_record_scales(job); });
    if (PASS == 1) {
        __shared__ uint32_t wave_seen[kNvThreads / 64];
        seen = wave_max(seen);
        if ((t & 63) == 0) wave_seen[t >> 6] = seen;
        __syncthreads();
        if (t == 0) {
            uint32_t m = 0;
#pragma unroll
            for (int k = 0; k < kNvThreads / 64; k++) m = umax(m, wave_seen[k]);
            atomicMax((uint32_t*)job.aux + job.section * kSectionWords + (blockIdx.x & (kSectionWords - 1)), kCarriedMark | f2u(elem_lo<F16>(m)));
        }
    }
}

// ---- one read of the tensor without an amax from before ----------------------------------------------------
// The two-pass form reads every element twice, and at 6.8 TB/s its amax pass is 43 % of its time.  Here a workgroup keeps its
// 64 KiB in registers (16 units per lane, 93 VGPRs, five workgroups per CU: 80 MB on the chip), publishes their maximum,
// waits for the tensor's other workgroups and quantizes what it holds.  While one tensor waits for its last loads, the
// workgroups of the next two are already loading.
//   exchange: a workgroup stores its maximum (with kOneFull, so that it is never zero) into a word of its own of the record's
//     sections, its slot; the record's first workgroup alone watches the slots and publishes the maximum of all of them in
//     kOneWords words, each a line of its own, one of which every other workgroup watches with one request at a time.
//     (With every workgroup watching all slots the polling itself filled the memory channels that hold them: 496 us
//     instead of 240 on 32 x [2048, 7168].)  No counters, so no atomic read-modify-writes.  What stays in the slots, however
//     the waits ended, is nothing to a carried run: it has no kCarriedMark and is below every word that has.
//   every wait ends: after kOnePolls looks the first workgroup of a record publishes that it has given up (kOneGaveUp) in place
//     of the maximum, and every workgroup that reads it leaves: that happens when workgroups of one record cannot all be on
//     the chip because something else occupies it; workgroups start in order of their ids, so otherwise the oldest
//     unfinished tensor always gets there.  A record that does not fit next to a busy neighbour so costs
//     one wait, not one for each batch of its workgroups that comes to the chip.  Medians beside a stream that is never idle, two
//     passes / this way: 32 x [2048, 7168] beside [8192, 8192] matrix products 1.8 / 1.0 ms (with what is left in a launch behind, which
//     starts when the neighbour makes room, 1.8), beside copies 0.38 / 0.38; lists of 24 to 56 MiB beside [8192, 8192] products 1.6 / 0.8 ms,
//     beside [4096, 4096] ones 0.20 / 0.10 to 0.17, beside copies 34 to 53 us / 35 to 45.
//   what is left: rows of workgroups behind those of the tensors (nv_one_rest), which start when all of these have, read every
//     record's word and quantize what its own workgroups did not.  (As a launch behind this one they cost 4.5 us.)
// 32 x [2048, 7168] (940 MB of bf16, all launches together): 313 us in two passes, 211 us this way (5.7 TB/s; 211.1 with slots that had
// to be cleared again, where [2048, 7168] took 13.0 us and now 12.3, 28 x [528, 3088] 28.3 and now 27.8; 214 with what
// is left in a launch behind, where 28 x [528, 3088] took 31.6 us, 48 x [1536, 2048] 73 and now 68).  Before, at 217: 226 with a
// block's scale computed in both lanes that hold it and its byte stored under a mask, 234 with the block maxima taken after the
// wait and a range test and a branch to the software forms in each unit.  24 units per lane at
// four workgroups per CU were 5 % slower, 8 units in 512 lanes 6 %, six workgroups per CU (20 registers spilled) 38 %; two
// units stored together, eight bytes a lane, 2 % slower here and 2 % faster on 18 x [1420, 1520].
// What bounds it: so many long-lived workgroups stream at 5.8 TB/s even if nobody waits for anybody (206 of the kernel's
// 209 us), where two units a lane stream at 6.9.  Two, four or six units a lane more, held in LDS, 222 to 234 us; four loads in flight
// at a time 225 to 236; a tensor's units dealt to its workgroups in turn 222; plain stores 220; starting the first
// workgroups of a CU one after the other, no difference.
// Four Over Six (the error modes that have an estimate): a lane holds eight whole blocks, regrouped through LDS before the wait;
// the last pair of units stays there, or 24 registers would go to scratch memory instead of five.  Blocks that were too close to
// call are taken up again behind the others, in a loop with the one copy of the exact sums, which reads them again.  32 x
// [2048, 7168]: 342 us in two passes, 298 this way, 48 x [1536, 2048] 111 and 95 (four workgroups per CU without the spills 319 and
// 103; regrouped by lane exchange after the wait 308 and 100; the next block's table lookups ahead of this block's sums 309 and
// 101); of weights N(0, 0.02^2), with all loads first, 318 and 273, 105 and 86.  Bound by the two hundred vector instructions of a block, which all workgroups of a tensor run at the same time: they
// overlap with the loads of the next two tensors, half as well as in the second of two passes.
constexpr int kOneThreads = 256, kOneUnits = 16, kOneWavesPerSimd = 5;
constexpr int64_t kOnePerBlock = kOneThreads * kOneUnits;
constexpr int kOneSlots = 2 * kSectionWords;         // the most workgroups of a tensor
constexpr int kOneRecordSlots = kRecordSections * kSectionWords;     // of the tensors of a record
constexpr uint32_t kOneFull = 0x8000u;               // marks a slot or word that holds a maximum
static_assert((kOneFull & kCarriedMark) == 0, "no slot passes for what a carried run has collected");
constexpr uint32_t kOneGaveUp = 0x10000u;            // in a word: the first workgroup has stopped waiting
constexpr int kOneWords = 7, kOneStride = 32, kRecOne = kRecAmax + 32;     // the published maximum, 128 bytes apart
static_assert(kRecOne + (kOneWords - 1) * kOneStride < MQ_NVFP4_RECORD_WORDS, "the published words lie inside the record");
constexpr int kOneLeaderSleep = 1, kOneSleep = 12;   // between two looks, in units of 64 cycles
// Looks of a first workgroup at each pair of slots: 0.04 ms where nothing else uses the memory (0.15 us a look), 0.16 ms beside a stream
// of copies (0.6); undisturbed, some 10 are enough.
constexpr int kOnePolls = 256;
// Looks of those that watch its word: 28 ms or 57 ms (0.43 or 0.87 us).  It has come to the chip before them and writes its word when its own
// looks are spent, so this ends a wait only where that workgroup itself is held up.
constexpr int kOnePatience = 1 << 16;

__device__ __forceinline__ void agent_store(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint32_t agent_load(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// slots of a record: the first one of the tensor in row `row`, and how many there are
struct NvOneSlots {
    uint32_t first, all;
};
__device__ __forceinline__ uint32_t nv_one_slots_of(const int64_t units) { return (uint32_t)((units + kOnePerBlock - 1) / kOnePerBlock); }
template <class Table>
__device__ __forceinline__ NvOneSlots nv_one_slots(const Table& tab, const FlatJob& job, const uint32_t row) {
    uint32_t first = 0;
    for (int k = job.section; k > 0; k--) first += nv_one_slots_of(tab.job[row - k].units);
    uint32_t all = first + nv_one_slots_of(job.units);
    for (int k = job.section + 1; k < job.pad; k++) all += nv_one_slots_of(tab.job[row + (k - job.section)].units);
    return NvOneSlots{first, all};
}
// one workgroup per tensor: no slot and no word written yet, and nothing in the sections of the record that a carried run would
// take for its own
template <class Table>
__global__ __launch_bounds__(256) void nvfp4_one_pass_clear_kernel(const Table tab) {
    const FlatJob job = flat_job_at(tab, blockIdx.x);
    uint32_t* rec = (uint32_t*)job.aux;
    const uint32_t slots = nv_one_slots(tab, job, blockIdx.x).all, sections = (uint32_t)(job.pad * kSectionWords);
    for (uint32_t word = job.section * kSectionWords + threadIdx.x; word < sections || word < slots; word += sections) rec[word] = 0;
    if (job.section == 0 && threadIdx.x < kOneWords) rec[kRecOne + threadIdx.x * kOneStride] = 0;
}

// a unit's maxima of its even and of its odd elements (16-bit patterns)
__device__ __forceinline__ uint32_t nv_unit_max(const u32x4 v) {
    return max2_u16(max2_u16(abs2(v.x), abs2(v.y)), max2_u16(abs2(v.z), abs2(v.w)));
}
// maximum of the block that a lane's unit and its neighbour's make up (16-bit pattern)
__device__ __forceinline__ uint32_t nv_block_max(const u32x4 v) { return group_max2(hmax_u16(nv_unit_max(v))); }
// The scale byte and the factor of a block with finite elements, for 1 / S_enc in 2^-82 .. 2^81: a block scale is 0 or in
// 2^-9 .. 448, so the divisor of every block with a scale is in the range of recip_shared.  For a divisor of zero that gives
// NaN, and the minimum with the largest factor is that factor, as for 1 / 0.
struct NvPlainScale {
    uint32_t sc;        // (only the low byte)
    float inv;
};
__device__ __forceinline__ NvPlainScale nv_plain_scale(const float bmax, const NvScales& gs) {
    uint32_t any;
    asm("" : "=v"(any));      // the bytes above are never read: nothing to clear before
    NvPlainScale s;
    s.sc = hw_e4m3x2<false>(__builtin_fminf(bmax * gs.enc_sixth, kFp8Max), 0.0f, any);
    s.inv = __builtin_fminf(recip_shared(hw_e4m3x2_decode<false>(s.sc).x * gs.s_dec), kFltMax);
    return s;
}
template <int F16>
__device__ __forceinline__ uint32_t nv_plain_codes(const u32x4 v, const float inv) {
    uint32_t word;
    asm("" : "=v"(word));      // the four conversions write all of it
    word = hw_e2m1x2<0>(elem_lo<F16>(v.x) * inv, elem_hi<F16>(v.x) * inv, word);
    word = hw_e2m1x2<1>(elem_lo<F16>(v.y) * inv, elem_hi<F16>(v.y) * inv, word);
    word = hw_e2m1x2<2>(elem_lo<F16>(v.z) * inv, elem_hi<F16>(v.z) * inv, word);
    return hw_e2m1x2<3>(elem_lo<F16>(v.w) * inv, elem_hi<F16>(v.w) * inv, word);
}
// the value that the even / the odd lane of each pair holds
template <int ODD>
__device__ __forceinline__ float pair_lane(const float v) {
    const int bits = (int)f2u(v);
    return u2f((uint32_t)__builtin_amdgcn_update_dpp(bits, bits, ODD ? 0xF5 /* 1, 1, 3, 3 */ : 0xA0 /* 0, 0, 2, 2 */, 0xF, 0xF, true));
}

// the maximum over the workgroup of what its lanes have (CALL: one number for each place that takes one, which has words of its own)
template <int CALL>
__device__ __forceinline__ uint32_t nv_one_max(uint32_t m, const int t) {
    __shared__ uint32_t part[kOneThreads / kWave];
    m = wave_max(m);
    if ((t & (kWave - 1)) == 0) part[t / kWave] = m;
    __syncthreads();
    m = 0;
#pragma unroll
    for (int k = 0; k < kOneThreads / kWave; k++) m = umax(m, part[k]);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
}
// What this lane sees of a record's slots, two at a time, as soon as they are all written; `late` if that took more than
// `polls` looks.
__device__ __forceinline__ uint32_t nv_one_collect(const uint32_t* rec, const uint32_t slots, const int t, const int polls, bool& late) {
    uint32_t m = 0;
    for (uint32_t slot = t; slot < slots; slot += 2 * kOneThreads) {
        const uint32_t* other = rec + (slot + kOneThreads < slots ? slot + kOneThreads : slot);
        uint32_t a = agent_load(rec + slot), b = agent_load(other);
        for (int n = 0; (a & b & kOneFull) == 0 && n < polls; n++) {
            __builtin_amdgcn_s_sleep(kOneLeaderSleep);
            a = agent_load(rec + slot);
            b = agent_load(other);
        }
        late |= (a & b & kOneFull) == 0;
        m = umax(m, umax(a & ~kOneFull, b & ~kOneFull));
    }
    return m;
}
// The record's published word for the whole workgroup, or 0 if its first workgroup has not come to write it in
// `patience` looks.
__device__ __forceinline__ uint32_t nv_one_watch(const uint32_t* word, const int t, const int patience) {
    __shared__ uint32_t seen;
    if (t < kWave) {
        uint32_t got = agent_load(word);
        for (int n = 0; got == 0 && n < patience; n++) {
            __builtin_amdgcn_s_sleep(kOneSleep);
            got = agent_load(word);
        }
        if (t == 0) seen = got;
    }
    __syncthreads();
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)seen);
}
// the same from the elements: for who has watched in vain
template <class Table>
__device__ __forceinline__ uint32_t nv_one_scan(const Table& tab, const uint32_t row, const int tensors_of_it, const int t) {
    uint32_t m2 = 0;
    for (int k = 0; k < tensors_of_it; k++) {
        const uint16_t* __restrict__ w = (const uint16_t*)load_global_ptr(&tab.job[row + k].w);
        const int64_t units = tab.job[row + k].units;
        for (int64_t u = t; u < units; u += kOneThreads) {
            const u32x4 v = ld16(w + u * 8);
            m2 = max2_u16(m2, max2_u16(max2_u16(abs2(v.x), abs2(v.y)), max2_u16(abs2(v.z), abs2(v.w))));
        }
    }
    return nv_one_max<2>(hmax_u16(m2), t);
}
// Tensors with an infinity or a NaN, or with a scale at the ends of the fp32 range, are left as well: the code behind
// has the software forms, which here, in sixteen copies, were 8 700 instructions in the way of the 2 000 that run.
template <int FOS, int F16>
__device__ __forceinline__ bool nv_one_leaves(const uint32_t m, const NvScales& gs) {
    if (FOS) return nv_fast_division(elem_lo<F16>(m)) != 2;
    const uint32_t dec = f2u(gs.s_dec);
    return m >= (F16 ? 0x7C00u : 0x7F80u) || !(dec >= 0x16800000u /* 2^-82 */ && dec <= 0x68000000u /* 2^81 */);
}

// Rows behind the tensors', `workers` workgroups to a tensor: they quantize the records that were left.  They come to the chip
// when every workgroup of the tensors has, most of which are done, and of a record that is done there is its word to read.
// Of a record whose first workgroup has given up every worker folds the slots.
template <int FOS, int F16, class Table>
__device__ __forceinline__ void nv_one_rest(const Table& tab, const FlatJob& job, const uint32_t row, const uint32_t worker,
                                            const uint32_t workers, const int patience, const int t, float numer, uint32_t* moved_counter) {
    uint32_t* rec = (uint32_t*)job.aux;
    const uint32_t got = nv_one_watch(rec + kRecOne + ((row + worker) % kOneWords) * kOneStride, t, patience);
    const bool gave_up = got == kOneGaveUp;
    uint32_t m = got & 0x7FFFu;
    bool late = got == 0;
    if (gave_up) m = nv_one_max<1>(nv_one_collect(rec, nv_one_slots(tab, job, row).all, t, patience, late), t);
    if (__syncthreads_or(late)) m = nv_one_scan(tab, row - job.section, job.pad, t);
    const float amax = elem_lo<F16>(m);
    const NvAmaxScales a{amax, nv_scales(amax, numer)};
    if ((got & kOneFull) != 0 && !nv_one_leaves<FOS, F16>(m, a.gs)) return;
    if ((got & kOneFull) == 0 && worker == 0 && t == 0) nv_publish_plain(job, a.amax, a.gs, numer, moved_counter);
    constexpr int64_t kPerBlock = nv_units_per_block(FOS);
    for (int64_t base = worker * kPerBlock; base < job.units; base += workers * kPerBlock)
        nvfp4_quant_units<FOS, F16>(job, base, t, numer, true, [&] { return a; });
}
// By a record's first workgroup, when it has nothing else to do: the record of a maximum that it has published, for all
// tensors that share it.
template <class Table>
__device__ __forceinline__ void nv_one_settle(const Table& tab, const FlatJob& job, const int t, float amax, const NvScales& gs, float numer,
                                              const bool left, uint32_t* moved_counter) {
    if (t != 0) return;
    ((uint32_t*)job.aux)[kRecRedo] = left;
    for (int k = 0; k < job.pad; k++) nv_publish_plain(flat_job_at(tab, blockIdx.y + k), amax, gs, numer, moved_counter);
}

// Of the units of two loads, the even lane of a pair takes the block of the first one and the odd lane that of the second.
__device__ __forceinline__ void nv_pair_blocks(u32x4* stage, u32x4& a, u32x4& b, const int t) {
    stage[t] = a;
    stage[kOneThreads + t] = b;
    // (as in nvfp4_fos_units: a wavefront reads back what its own lanes wrote)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t first = ((t & 1) ? (uint32_t)kOneThreads : 0u) + ((uint32_t)t & ~1u);
    a = stage[first];
    b = stage[first + 1];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// The blocks of a lane of the one-pass kernel with Four Over Six, the last one in `stage`, for an amax that nv_fast_division puts at
// 2; maxima: of the blocks, two to a register.
template <int EM, int F16>
__device__ __forceinline__ void nv_one_four_over_six(const FlatJob& job, const u32x4 (&v)[kOneUnits], const uint32_t (&maxima)[kOneUnits / 2], const u32x4* stage, const int64_t base, const uint32_t rem, const int t,
                                                     const float amax, const NvScales& gs, const float denom) {
    __shared__ NvScaleEntry scale_table[128];
    constexpr float kInv2688 = 1.0f / 2688.0f, kInv1536 = 1.0f / 1536.0f;
    const float denom_inv = denom == 2688.0f ? kInv2688 : denom == 1536.0f ? kInv1536 : 1.0f / denom;
    nv_fill_scale_table(scale_table, t, amax, gs.s_dec, true, denom, denom_inv);
    __syncthreads();
    const uint32_t odd = (uint32_t)t & 1u;
    uint32_t* __restrict__ q0 = (uint32_t*)job.q + base;
    uint8_t* __restrict__ s80 = (uint8_t*)job.s + base / 2;
    auto store = [&](const uint32_t load, const NvCandidate16& c) {
        const uint32_t first = ((uint32_t)t & ~1u) + (load + odd) * kOneThreads;      // the block's first unit
        if (first < rem) {
            st8(q0 + first, u32x2{c.lo, c.hi});
            s80[first >> 1] = (uint8_t)c.sc();
        }
    };
    uint32_t open = 0;      // blocks too close to call
#pragma unroll
    for (int i = 0; i < kOneUnits; i += 2) {
        float f[16];
        const uint32_t held = odd * kOneThreads + ((uint32_t)t & ~1u);
        if (i + 2 < kOneUnits) nv_unpack16<F16>(v[i], v[i + 1], f);
        else nv_unpack16<F16>(stage[held], stage[held + 1], f);
        const float bmax = i % 4 ? elem_hi<F16>(maxima[i / 4]) : elem_lo<F16>(maxima[i / 4]);
        const NvCandidates16 c = nv_candidates16<2, false, true>(f, bmax, gs, scale_table);
        const NvPick pick = nv_estimated_pick<EM>(f, bmax, c.c4, c.c6);
        store(i, pick.four ? c.c4 : c.c6);
        if (!pick.decided) open |= 1u << (i / 2);
        __builtin_amdgcn_sched_barrier(0);      // a block at a time: more do not fit the registers
    }
    if (__builtin_amdgcn_ballot_w64(open != 0) == 0) return;
#pragma unroll 1
    for (uint32_t i = 0; i < kOneUnits; i += 2) {
        if (__builtin_amdgcn_ballot_w64((open >> (i / 2)) & 1u) == 0) continue;
        // (the block is read again: with every unit kept, 28 registers went to scratch memory)
        const uint32_t first = ((uint32_t)t & ~1u) + (i + odd) * kOneThreads;
        const uint16_t* __restrict__ w = (const uint16_t*)job.w + (base + (first < rem ? first : 0)) * 8;
        float f[16];
        nv_unpack16<F16>(ld16(w), ld16(w + 8), f);
        const NvCandidates16 c = nv_candidates16<2, false, true>(f, nv_numbers_max(f), gs, scale_table);
        const float e4 = nv_block_error<EM, 2>(f, c.c4, amax, gs.enc, denom, denom_inv), e6 = nv_block_error<EM, 2>(f, c.c6, amax, gs.enc, denom, denom_inv);
        if ((open >> (i / 2)) & 1u) store(i, e4 < e6 ? c.c4 : c.c6);
    }
}

// job as for the quantize pass: section = place of the tensor inside its record, pad = tensors sharing it (neighbours)
// grid (workgroups of the largest tensor, tensors + rows behind)
template <int FOS, int F16, class Table>
__global__ __launch_bounds__(kOneThreads, kOneWavesPerSimd) void nvfp4_one_pass_kernel(const Table tab, float numer, int first_polls, int patience, uint32_t tensors,
                                                                                       uint32_t workers, uint32_t* moved_counter, uint32_t* moved_mirror) {
    const int t = threadIdx.x;
    const bool behind = blockIdx.y >= tensors;
    uint32_t row = blockIdx.y, worker = 0;
    if (behind) {
        const uint32_t id = (blockIdx.y - tensors) * gridDim.x + blockIdx.x;
        worker = id / tensors;
        row = id - worker * tensors;
    }
    // A descriptor of a device table is read before the branch: below one with stores the compiler takes its values to vector
    // registers, and with them sixteen addresses of each lane; three of the sixteen loads then waited for the others
    // (96 x [2048, 7168] 695 us, now 620; 200 x [768, 2048] 142 and now 132).
    constexpr bool kRef = std::is_same<Table, FlatRef>::value;
    FlatJob job;
    if (kRef || !behind) job = flat_job_at(tab, row);
    if (behind) {
        if (!kRef) job = flat_job_at(tab, row);
        if (worker < workers) nv_one_rest<FOS, F16>(tab, job, row, worker, workers, patience, t, numer, moved_counter);
        return;
    }
    const int64_t block = flat_block(tab), base = block * kOnePerBlock;
    if (base >= job.units) return;
    const int64_t left = job.units - base;
    const uint32_t rem = left < kOnePerBlock ? (uint32_t)left : (uint32_t)kOnePerBlock;
    const uint16_t* __restrict__ w0 = (const uint16_t*)job.w + base * 8;
    u32x4 v[kOneUnits];
    const bool whole = rem == kOnePerBlock;
    if (whole) {
#pragma unroll
        for (int i = 0; i < kOneUnits; i++) v[i] = ld16(w0 + i * kOneThreads * 8 + (uint32_t)t * 8u);
    } else {
#pragma unroll
        for (int i = 0; i < kOneUnits; i++) {
            const uint32_t off = (uint32_t)t + i * kOneThreads;
            v[i] = ld16(w0 + (off < rem ? off : (off & 1u)) * 8u);      // a lane past the end reads the first block again
        }
    }
    // Every load before the first use, else the last one waits for most of the others, and the slots meanwhile (us, 32 x [2048, 7168] with
    // Four Over Six 277 and 269, over a device table 96 of them 626 and 620; but standard blocks over kernel arguments 210 and 213).
    constexpr bool kEarly = FOS != 0 || kRef;
    const NvOneSlots early = kEarly ? nv_one_slots(tab, job, row) : NvOneSlots{};
    auto slots = [&] { return kEarly ? early : nv_one_slots(tab, job, row); };
    if constexpr (kEarly) __builtin_amdgcn_sched_barrier(0);
    // the block maxima, two to a register: what does not depend on the amax is done before the wait for it
    __shared__ u32x4 stage[FOS ? 2 * kOneThreads : 1];
    uint32_t maxima[kOneUnits / 2], m2 = 0;
#pragma unroll
    for (int i = 0; i < kOneUnits; i += 2) {
        if constexpr (FOS != 0) {
            nv_pair_blocks(stage, v[i], v[i + 1], t);
            const uint32_t bmax = hmax_u16(max2_u16(nv_unit_max(v[i]), nv_unit_max(v[i + 1])));
            maxima[i / 4] = i % 4 ? maxima[i / 4] | (bmax << 16) : bmax;
            m2 = max2_u16(m2, bmax);
            continue;
        }
        maxima[i / 2] = nv_block_max(v[i]) | (nv_block_max(v[i + 1]) << 16);
        if constexpr (std::is_same<Table, FlatRef>::value) asm("" : "+v"(maxima[i / 2]));      // (else its halves are kept as well, in scratch memory)
        m2 = max2_u16(m2, maxima[i / 2]);
    }
    uint32_t m = nv_one_max<0>(hmax_u16(m2), t);
    uint32_t* rec = (uint32_t*)job.aux;
    if (t == 0) agent_store(rec + slots().first + block, kOneFull | m);
    const bool first = block == 0 && job.section == 0;
    if (first) {
        // the record's first workgroup waits for every other one
        bool late = false;
        m = nv_one_max<1>(nv_one_collect(rec, slots().all, t, first_polls, late), t);
        const bool gave_up = __syncthreads_or(late);
        if (t < kOneWords) agent_store(rec + kRecOne + t * kOneStride, gave_up ? kOneGaveUp : kOneFull | m);
        if (blockIdx.y == 0) amax_feedback_folded(moved_counter, moved_mirror, tensors);
        if (gave_up) {
            if (t == 0) rec[kRecRedo] = 1;
            return;
        }
    } else {
        m = nv_one_watch(rec + kRecOne + (blockIdx.x % kOneWords) * kOneStride, t, patience);
        if (m == 0) m = kOneFull | nv_one_scan(tab, blockIdx.y - job.section, job.pad, t);
        if ((m & kOneFull) == 0) return;
        m &= 0x7FFFu;
    }
    const float amax = elem_lo<F16>(m);
    const NvScales scales = nv_scales(amax, numer), gs{uniform_f(scales.enc_sixth), uniform_f(scales.s_dec), uniform_f(scales.enc)};
    const bool leaves = nv_one_leaves<FOS, F16>(m, gs);
    if constexpr (FOS != 0) {
        if (!leaves) nv_one_four_over_six<FOS - 1, F16>(job, v, maxima, stage, base, rem, t, amax, gs, numer);
    } else if (!leaves) {
        // Both lanes of a pair hold the maxima of the same blocks: of two units the even lane takes the first one's scale and the
        // odd lane the second one's, so that a scale is computed once and every lane stores a byte.
        const uint32_t odd = (uint32_t)t & 1u;
        uint32_t* __restrict__ q0 = (uint32_t*)job.q + base;
        uint8_t* __restrict__ s80 = (uint8_t*)job.s + base / 2;
        auto quantize = [&](auto full) {
#pragma unroll
            for (int i = 0; i < kOneUnits; i += 2) {
                const uint32_t two = maxima[i / 2];
                const NvPlainScale s = nv_plain_scale(odd ? elem_hi<F16>(two) : elem_lo<F16>(two), gs);
                const uint32_t word0 = nv_plain_codes<F16>(v[i], pair_lane<0>(s.inv)), word1 = nv_plain_codes<F16>(v[i + 1], pair_lane<1>(s.inv));
                const uint32_t off = (uint32_t)t + i * kOneThreads;
                if (full || off < rem) st4(q0 + off, word0);
                if (full || off + kOneThreads < rem) st4(q0 + off + kOneThreads, word1);
                if (full || off + odd * kOneThreads < rem) s80[(off >> 1) + odd * (kOneThreads / 2)] = (uint8_t)s.sc;
                __builtin_amdgcn_sched_barrier(0);      // two units at a time: more do not fit the registers
            }
        };
        if (whole) quantize(std::true_type{});
        else quantize(std::false_type{});
    }
    if (first) nv_one_settle(tab, job, t, amax, gs, numer, leaves, moved_counter);
}

// fp32 input, the second pass of the two-pass form (the carried-over amax and the one-pass form are for 16-bit tensors).
// Standard blocks: four elements per 16-byte load, four lanes a block, two bytes of codes per lane; bound by HBM, 8.56
// bytes per element with the amax pass.  Four Over Six: a lane per block, 64 consecutive bytes each, and the exact error sums
// (the estimate wants an amax of twelve significant bits); bound by vector instructions.
// A stack of eight [2048, 4096] tensors: 92 us, Four Over Six 95 (769 and 762 in the element-wise kernels, a launch each).
constexpr int kNvF32Loads = 2;                     // 16-byte loads per lane, standard blocks
// 8-element units a workgroup covers
constexpr int64_t nv_f32_units_per_block(int fos) { return fos ? kNvThreads * 2 : kNvThreads * kNvF32Loads / 2; }
template <int FOS, int PASS, class Table>
__global__ __launch_bounds__(kNvThreads) void nvfp4_quant_f32_kernel(const Table tab, float denom, uint32_t* moved_counter, uint32_t* moved_mirror) {
    const FlatJob job = flat_job(tab);
    const uint32_t t = threadIdx.x;
    const int64_t first = flat_block(tab) * nv_f32_units_per_block(FOS);       // in 8-element units
    if (first >= job.units && (PASS == 3 || first > 0)) return;
    if (PASS == 0 && first == 0 && blockIdx.y == 0) amax_feedback_folded(moved_counter, moved_mirror, gridDim.y);
    auto fold = [&] {           // as in PASS 0 and PASS 3 of the 16-bit kernel
        if (PASS == 3) return nv_record_scales(job);
        const NvAmaxScales a = nv_shared_scales((int)t, denom, [&] { return nv_wave_fold((const uint32_t*)job.aux, job.pad, (int)t); });
        if (first == 0 && t == 0) {
            ((uint32_t*)job.aux)[kRecRedo] = 0;
            nv_publish_plain(job, a.amax, a.gs, denom, moved_counter);
        }
        return a;
    };
    if (job.units == 0) {
        fold();
        return;
    }
    const float* __restrict__ w0 = (const float*)job.w + first * 8;
    const int64_t left = (job.units - first) * 2;                              // 16-byte loads
    if constexpr (FOS != 0) {
        __shared__ NvScaleEntry scale_table[128];
        constexpr int EM = FOS - 1;
        const uint32_t rem = left < 4 * kNvThreads ? (uint32_t)left / 4 : (uint32_t)kNvThreads;      // blocks
        const uint32_t at = t < rem ? t : 0u;
        float f[16];
        uint32_t mb = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u32x4 v = ld16_keep(w0 + at * 16u + 4 * i);      // (each line is touched by four load instructions)
            mb = umax(mb, umax(umax(v.x & 0x7FFFFFFFu, v.y & 0x7FFFFFFFu), umax(v.z & 0x7FFFFFFFu, v.w & 0x7FFFFFFFu)));
            f[4 * i] = u2f(v.x); f[4 * i + 1] = u2f(v.y); f[4 * i + 2] = u2f(v.z); f[4 * i + 3] = u2f(v.w);
        }
        const NvAmaxScales known = fold();
        const NvScales gs = known.gs;
        const float amax = known.amax, denom_inv = 1.0f / denom;
        nv_fill_scale_table(scale_table, (int)t, amax, gs.s_dec, false, denom, denom_inv);
        __syncthreads();
        NvCandidate16 c = nv_fast_division(amax) != 0 ? nv_four_over_six16<EM, 1, true>(f, u2f(mb), amax, gs, denom, denom_inv, scale_table)
                                                      : nv_four_over_six16<EM, 0, true>(f, u2f(mb), amax, gs, denom, denom_inv, scale_table);
        // the hardware conversion hands a NaN's sign on; the code of a NaN is 7, as in the element-wise kernel
        if (__builtin_amdgcn_ballot_w64(mb > 0x7F800000u) != 0) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (f[j] != f[j]) c.lo &= ~(8u << (4 * j));
                if (f[8 + j] != f[8 + j]) c.hi &= ~(8u << (4 * j));
            }
        }
        if (t < rem) {
            ((uint32_t*)job.q + first)[2 * t] = c.lo;
            ((uint32_t*)job.q + first)[2 * t + 1] = c.hi;
            ((uint8_t*)job.s + first / 2)[t] = (uint8_t)c.sc();
        }
    } else {
        constexpr uint32_t kPerBlock = kNvThreads * kNvF32Loads;
        const uint32_t rem = left < kPerBlock ? (uint32_t)left : kPerBlock;
        uint16_t* __restrict__ q0 = (uint16_t*)job.q + first * 2;
        uint8_t* __restrict__ s80 = (uint8_t*)job.s + first / 2;
        u32x4 v[kNvF32Loads];
#pragma unroll
        for (int i = 0; i < kNvF32Loads; i++) {
            const uint32_t off = t + i * kNvThreads;
            v[i] = off < rem ? ld16(w0 + off * 4u) : u32x4{0u, 0u, 0u, 0u};
        }
        const NvScales gs = fold().gs;
#pragma unroll
        for (int i = 0; i < kNvF32Loads; i++) {
            const uint32_t off = t + i * kNvThreads;
            const uint32_t mb = group_max4(umax(umax(v[i].x & 0x7FFFFFFFu, v[i].y & 0x7FFFFFFFu), umax(v[i].z & 0x7FFFFFFFu, v[i].w & 0x7FFFFFFFu)));
            const float bmax = u2f(mb);
            const float s_hp = bmax == 0.0f ? 0.0f : bmax * gs.enc_sixth;
            const float f[4] = {u2f(v[i].x), u2f(v[i].y), u2f(v[i].z), u2f(v[i].w)};
            uint32_t sc, word = 0;
            if (mb < 0x7F800000u && s_hp == s_hp) {
                sc = hw_e4m3x2<false>(__builtin_fminf(s_hp, kFp8Max), 0.0f, 0u) & 0xFFu;
                const float d = hw_e4m3x2_decode<false>(sc).x * gs.s_dec;
                float inv;          // as in nvfp4_quant_unit
                if (__builtin_amdgcn_ballot_w64(!shared_div_ok(d)) == 0) inv = recip_shared(d);
                else inv = __builtin_fminf(1.0f / d, kFltMax);
                word = hw_e2m1x2<0>(f[0] * inv, f[1] * inv, word);
                word = hw_e2m1x2<1>(f[2] * inv, f[3] * inv, word);
            } else {
                sc = sw_e4m3fn_sat(s_hp);
                const float inv = __builtin_fminf(1.0f / (sw_e4m3fn_decode(sc) * gs.s_dec), kFltMax);
#pragma unroll
                for (int j = 0; j < 4; j++) word |= sw_e2m1(f[j] * inv) << (4 * j);
            }
            if (off < rem) {
                __builtin_nontemporal_store((uint16_t)word, q0 + off);
                if ((t & 3) == 0) s80[off >> 2] = (uint8_t)sc;
            }
        }
    }
}

// software candidate of the one-lane-per-block kernel: codes of sixteen values and their error
__device__ __forceinline__ float nv_candidate_sw(const float x[16], uint32_t sc, float amax, const NvScales& gs, float denom,
                                                 int flags, uint32_t codes[16]) {
    const float s_f = sw_e4m3fn_decode(sc);
    const float inv = __builtin_fminf(1.0f / (s_f * gs.s_dec), kFltMax);
    float error = 0.0f;
    for (int j = 0; j < 16; j++) {
        const uint32_t c = sw_e2m1(x[j] * inv);
        codes[j] = c;
        const float mag = (c & 7u) < 2u ? 0.5f * (float)(c & 7u) : u2f(0x3F000000u + ((c & 7u) << 22));
        const float cand = (c & 8u) ? -mag : mag;
        float diff;
        if (flags & MQ_NVFP4_ERR_FP16) {
            float hf = (float)((_Float16)cand * (_Float16)s_f);
            asm volatile("" : "+v"(hf));
            diff = hf - x[j] * gs.enc;
        } else {
            diff = ((cand * s_f) * amax) / denom - x[j];
        }
        error = error + ((flags & MQ_NVFP4_ERR_MSE) ? diff * diff : __builtin_fabsf(diff));
    }
    return error;
}

__global__ __launch_bounds__(256) void nvfp4_quant_generic_kernel(const void* __restrict__ w, int dtype,
                                                                  const uint32_t* __restrict__ amax_bits,
                                                                  uint8_t* __restrict__ q, uint8_t* __restrict__ s8,
                                                                  int64_t blocks16, int flags, float denom) {
    NvScales gs;
    gs.enc_sixth = u2f(amax_bits[kRecEncSixth]);
    gs.s_dec = u2f(amax_bits[kRecSDec]);
    gs.enc = u2f(amax_bits[kRecEnc]);
    const float amax = u2f(amax_bits[kRecAmax]);
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < blocks16; b += stride) {
        uint32_t m = 0;
        for (int j = 0; j < 16; j++) m = umax(m, f2u(load_f32(w, b * 16 + j, dtype)) & 0x7FFFFFFFu);
        const float bmax = u2f(m);
        if (flags & MQ_NVFP4_4OVER6) {
            float x[16];
            for (int j = 0; j < 16; j++) x[j] = load_f32(w, b * 16 + j, dtype);
            const float s6_hp = (bmax / 6.0f) * gs.enc, s4_hp = s6_hp * 1.5f;
            const uint32_t sc4 = sw_e4m3fn_sat(__builtin_fminf(s4_hp, kFp8Max)), sc6 = sw_e4m3fn_sat(__builtin_fminf(s6_hp, kFp8Max));
            uint32_t c4[16], c6[16];
            const float e4 = nv_candidate_sw(x, sc4, amax, gs, denom, flags, c4);
            const float e6 = nv_candidate_sw(x, sc6, amax, gs, denom, flags, c6);
            const bool pick4 = e4 < e6;
            s8[b] = (uint8_t)(pick4 ? sc4 : sc6);
            for (int j = 0; j < 16; j += 2)
                q[b * 8 + j / 2] = (uint8_t)(pick4 ? (c4[j] | (c4[j + 1] << 4)) : (c6[j] | (c6[j + 1] << 4)));
            continue;
        }
        const float s_hp = bmax == 0.0f ? 0.0f : bmax * gs.enc_sixth;
        const uint32_t sc = sw_e4m3fn_sat(s_hp);
        s8[b] = (uint8_t)sc;
        const float inv = __builtin_fminf(1.0f / (sw_e4m3fn_decode(sc) * gs.s_dec), kFltMax);
        for (int j = 0; j < 16; j += 2) {
            const uint32_t lo = sw_e2m1(load_f32(w, b * 16 + j, dtype) * inv);
            const uint32_t hi = sw_e2m1(load_f32(w, b * 16 + j + 1, dtype) * inv);
            q[b * 8 + j / 2] = (uint8_t)(lo | (hi << 4));
        }
    }
}

// ---- fused quantize + dequantize (training-forward fake quantization) -------------------------------
// Reference: miles/kernels/quant/nvfp4_qdq.py:877-890 (standard quantize), :993-1029 (dequantize), kernel :1067-1105.
// Given the tensor amax: codes and block scale exactly as the quantizer above, then
//   final = RN(RN(f32(s8) * amax) * f32(1 / (6 * e4m3_max)));  y = dtype(RN(e2m1_value * final))
// Nothing but x (and the amax, see nv_fake_scales) is read and nothing but y written.  job: w = x, q = y, units.
// Standard blocks: two lanes own one 1x16 block.  Four Over Six: nvfp4_fos_units.
// Both are bound by memory, the reads by the memory-side cache where the amax pass left its input there: sixteen [1536, 2048]
// weights in one launch 28.4 us (33 from HBM; one launch per weight 4.6 us each), four [4096, 7168] with Four Over Six 66 us
// (78 from HBM; 67 without the forms for an amax of the tensor's own; 120 with two lanes per block and the exact error sums throughout, where vector instructions were the bound).
template <int FOS, int F16>
__global__ __launch_bounds__(kNvThreads) void nvfp4_fake_kernel(const FlatTable tab, float numer, float inv_numer) {
    const FlatJob job = flat_job(tab);
    const int t = threadIdx.x;
    const int64_t base = flat_block(tab) * nv_units_per_block(FOS);
    if (base >= job.units) return;
    if constexpr (FOS != 0) {
        nvfp4_fos_units<FOS - 1, F16, true>(job, base, t, numer, inv_numer, job.aux2 == nullptr, [&] { return nv_fake_scales(job, t, numer); });
    } else {
        const int64_t left = job.units - base;
        const uint32_t rem = left < kNvThreads * kNvUnroll ? (uint32_t)left : (uint32_t)(kNvThreads * kNvUnroll);
        const uint16_t* __restrict__ x0 = (const uint16_t*)job.w + base * 8;
        uint16_t* __restrict__ y0 = (uint16_t*)job.q + base * 8;
        u32x4 v[kNvUnroll];
#pragma unroll
        for (int i = 0; i < kNvUnroll; i++) {
            const uint32_t off = (uint32_t)t + i * kNvThreads;
            v[i] = ld16(x0 + (off < rem ? off : 0u) * 8u);      // a lane past the end reads the first unit again
        }
        const NvAmaxScales known = nv_fake_scales(job, t, numer);
        const float amax = known.amax;
        const NvScales gs = known.gs;
#pragma unroll
        for (int i = 0; i < kNvUnroll; i++) {
            const uint32_t off = (uint32_t)t + i * kNvThreads;
            const float f[8] = {elem_lo<F16>(v[i].x), elem_hi<F16>(v[i].x), elem_lo<F16>(v[i].y), elem_hi<F16>(v[i].y),
                                elem_lo<F16>(v[i].z), elem_hi<F16>(v[i].z), elem_lo<F16>(v[i].w), elem_hi<F16>(v[i].w)};
            const uint32_t m2 = max2_u16(max2_u16(abs2(v[i].x), abs2(v[i].y)), max2_u16(abs2(v[i].z), abs2(v[i].w)));
            const uint32_t mb = group_max2(hmax_u16(m2));
            const float bmax = elem_lo<F16>(mb);
            const float s_hp = bmax == 0.0f ? 0.0f : bmax * gs.enc_sixth;
            float s_f, q[8];
            if (mb < (F16 ? 0x7C00u : 0x7F80u) && s_hp == s_hp) {
                const uint32_t sc = hw_e4m3x2<false>(__builtin_fminf(s_hp, kFp8Max), 0.0f, 0u) & 0xFFu;
                s_f = hw_e4m3x2_decode<false>(sc).x;
                const float d = s_f * gs.s_dec;
                float inv;          // as in nvfp4_quant_units
                if (__builtin_amdgcn_ballot_w64(!shared_div_ok(d)) == 0) inv = recip_shared(d);
                else inv = __builtin_fminf(1.0f / d, kFltMax);
                uint32_t word = hw_e2m1x2<0>(f[0] * inv, f[1] * inv, 0u);
                word = hw_e2m1x2<1>(f[2] * inv, f[3] * inv, word);
                word = hw_e2m1x2<2>(f[4] * inv, f[5] * inv, word);
                word = hw_e2m1x2<3>(f[6] * inv, f[7] * inv, word);
                nv_decode8(word, q);
            } else {
                const uint32_t sc = sw_e4m3fn_sat(s_hp);
                s_f = sw_e4m3fn_decode(sc);
                const float inv = __builtin_fminf(1.0f / (s_f * gs.s_dec), kFltMax);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t c = sw_e2m1(f[j] * inv);
                    const float mag = (c & 7u) < 2u ? 0.5f * (float)(c & 7u) : u2f(0x3F000000u + ((c & 7u) << 22));
                    q[j] = (c & 8u) ? -mag : mag;
                }
            }
            const u32x4 o = nv_scaled16<F16>(q, (s_f * amax) * inv_numer);
            if (off < rem) st16(y0 + off * 8u, o);
        }
    }
}

}  // namespace mq

using namespace mq;

bool mq_nvfp4_fast_ok(const void* w, int dtype, const void* q) {
    return dtype >= MQ_BF16 && dtype <= MQ_F32 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)q % 4) == 0;
}

// tab.job[i]: w, aux = amax record, section, units = numel / 8, s = (void*)numel; every tensor of the one dtype
static unsigned amax_blocks(int dtype, int64_t max_units) {
    const int64_t chunks = (max_units * (dtype == MQ_F32 ? 2 : 1) + 256 * kAmaxUnroll - 1) / (256 * kAmaxUnroll);
    return (unsigned)(chunks < 1 ? 1 : chunks < kSectionWords ? chunks : kSectionWords);
}
template <int KEEP, class Table>
static void launch_nvfp4_amax_kept(int dtype, const Table& tab, dim3 grid, hipStream_t st) {
    const dim3 blk(256);
    if (dtype == MQ_F32) hipLaunchKernelGGL((nvfp4_amax_f32_kernel<Table, KEEP>), grid, blk, 0, st, tab);
    else if (dtype == MQ_F16) hipLaunchKernelGGL((nvfp4_amax_bf16_kernel<Table, 1, KEEP>), grid, blk, 0, st, tab);
    else hipLaunchKernelGGL((nvfp4_amax_bf16_kernel<Table, 0, KEEP>), grid, blk, 0, st, tab);
}
// max_units: the largest tensor's units; all_units: of all n tensors
template <class Table>
static int launch_nvfp4_amax(int dtype, const Table& tab, int n, int64_t max_units, int64_t all_units, hipStream_t st) {
    const dim3 grid(amax_blocks(dtype, max_units), (unsigned)n);
    switch (kept_quarters(all_units * (dtype == MQ_F32 ? 32 : 16))) {
        case 4: launch_nvfp4_amax_kept<4>(dtype, tab, grid, st); break;
        case 2: launch_nvfp4_amax_kept<2>(dtype, tab, grid, st); break;
        default: launch_nvfp4_amax_kept<0>(dtype, tab, grid, st); break;
    }
    return mq_check_launch("nvfp4 amax");
}
int mq_nvfp4_amax_launch_group(int dtype, FlatTable& tab, hipStream_t st) {
    int64_t max_units = 0, all_units = 0;
    for (int i = 0; i < tab.n; i++) {
        max_units = tab.job[i].units > max_units ? tab.job[i].units : max_units;
        all_units += tab.job[i].units;
    }
    return launch_nvfp4_amax(dtype, tab, tab.n, max_units, all_units, st);
}
// the same over n descriptors of a device table (the quantizer's form: whole units, section = place inside the record);
// max_units: the largest tensor's units
int mq_nvfp4_amax_launch_table(int dtype, const FlatJob* device_jobs, int n, int64_t max_units, hipStream_t st) {
    if (n == 0) return MQ_OK;
    return launch_nvfp4_amax(dtype, FlatRef{device_jobs, 0, 0}, n, max_units, max_units * n, st);
}

template <int PASS, class Table, int F16>
static void launch_nvfp4_quant_dtype(const Table& tab, int flags, float numer, bool own, bool counted, dim3 grid, hipStream_t st) {
    const dim3 blk(kNvThreads);
    uint32_t *const moved = counted ? mq_amax_feedback() : nullptr, *const mirror = mq_amax_feedback_mirror();
    // Four Over Six keeps to launches of kernel-argument tables (its five error modes are not built in the other form)
    const int fos = (flags & MQ_NVFP4_4OVER6) ? 1 + nv_error_mode(flags) : 0;
    if constexpr (std::is_same<Table, FlatRef>::value) {
        hipLaunchKernelGGL((nvfp4_quant_bf16_kernel<0, PASS, Table, F16>), grid, blk, 0, st, tab, numer, own, moved, mirror);
    } else {
        switch (fos) {
            case 0: hipLaunchKernelGGL((nvfp4_quant_bf16_kernel<0, PASS, Table, F16>), grid, blk, 0, st, tab, numer, own, moved, mirror); break;
            case 1: hipLaunchKernelGGL((nvfp4_quant_bf16_kernel<1, PASS, Table, F16>), grid, blk, 0, st, tab, numer, own, moved, mirror); break;
            case 2: hipLaunchKernelGGL((nvfp4_quant_bf16_kernel<2, PASS, Table, F16>), grid, blk, 0, st, tab, numer, own, moved, mirror); break;
            case 3: hipLaunchKernelGGL((nvfp4_quant_bf16_kernel<3, PASS, Table, F16>), grid, blk, 0, st, tab, numer, own, moved, mirror); break;
            default: hipLaunchKernelGGL((nvfp4_quant_bf16_kernel<4, PASS, Table, F16>), grid, blk, 0, st, tab, numer, own, moved, mirror); break;
        }
    }
}
template <int PASS, class Table>
static void launch_nvfp4_quant_f32(const Table& tab, int flags, float numer, bool counted, dim3 grid, hipStream_t st) {
    const dim3 blk(kNvThreads);
    uint32_t *const moved = counted ? mq_amax_feedback() : nullptr, *const mirror = mq_amax_feedback_mirror();
    const int fos = (flags & MQ_NVFP4_4OVER6) ? 1 + nv_error_mode(flags) : 0;
    if constexpr (std::is_same<Table, FlatRef>::value) {
        hipLaunchKernelGGL((nvfp4_quant_f32_kernel<0, PASS, Table>), grid, blk, 0, st, tab, numer, moved, mirror);
    } else {
        switch (fos) {
            case 0: hipLaunchKernelGGL((nvfp4_quant_f32_kernel<0, PASS, Table>), grid, blk, 0, st, tab, numer, moved, mirror); break;
            case 1: hipLaunchKernelGGL((nvfp4_quant_f32_kernel<1, PASS, Table>), grid, blk, 0, st, tab, numer, moved, mirror); break;
            case 2: hipLaunchKernelGGL((nvfp4_quant_f32_kernel<2, PASS, Table>), grid, blk, 0, st, tab, numer, moved, mirror); break;
            case 3: hipLaunchKernelGGL((nvfp4_quant_f32_kernel<3, PASS, Table>), grid, blk, 0, st, tab, numer, moved, mirror); break;
            default: hipLaunchKernelGGL((nvfp4_quant_f32_kernel<4, PASS, Table>), grid, blk, 0, st, tab, numer, moved, mirror); break;
        }
    }
}
// own: see nvfp4_quant_bf16_kernel; counted: pass 0 adds to the counters of the call's feedback (in a carried run the fold does)
template <int PASS, class Table>
static void launch_nvfp4_quant(int dtype, const Table& tab, int flags, float numer, bool own, bool counted, dim3 grid, hipStream_t st) {
    // (fp32 has no instances of passes 1 and 2: nvfp4_quant_launch refuses mode 2 for it)
    if constexpr (PASS == 0 || PASS == 3) {
        if (dtype == MQ_F32) {
            launch_nvfp4_quant_f32<PASS>(tab, flags, numer, counted, grid, st);
            return;
        }
    }
    if (dtype == MQ_F16) launch_nvfp4_quant_dtype<PASS, Table, 1>(tab, flags, numer, own, counted, grid, st);
    else launch_nvfp4_quant_dtype<PASS, Table, 0>(tab, flags, numer, own, counted, grid, st);
}

// Whether a plain run's amax is folded by a launch between the two passes (nvfp4_publish_kernel), or by every workgroup of the
// second one.  The launch takes 1 to 2 us; what it saves grows with the pass and with the sections of a record.  `sections`:
// of all n tensors' records, `bytes`: of their elements.  Device time of both passes in us, folded in the pass / by the launch:
//   gate and up in pairs, bf16: 2 x [2048, 7168] (59 MB) 25.1 / 25.6, 4 of them 44.3 / 43.7, 16 of them 168 / 158, 64 of them
//     (1.9 GB) 646 / 615; fp32: 34 MB 16.6 / 17.3, 67 MB 26.8 / 27.0, 117 MB 42.1 / 41.2, 470 MB 156 / 148, 940 MB 314 / 293.
//     (A pair folds two sections, a quarter of the bytes that a workgroup quantizes.)
//   Four Over Six of 16-bit tensors, bound by vector instructions: 34 MB 19.8 / 20.3, 50 MB 25.6 / 26.0, 67 MB 31.5 / 31.4,
//     134 MB 55.4 / 53.6, 189 MB 75.6 / 72.6 (longer lists are read once, or by the carried form).
//   Four Over Six of fp32 tensors, as long as the second pass finds all of its input in the memory-side cache: 78 MB 34.1 / 34.8
//     (in pairs 35.8 / 35.3), 117 MB 46.3 / 46.2 (47.6 / 46.3), 235 MB 85.4 / 83.9 (86.8 / 84.0), 268 MB 112 / 111; but 403 MB
//     143.0 / 143.1, 470 MB 169 / 173 (170 / 173), 604 MB 207 / 211.
//   one section per record, standard scaling: fp32 67 MB 25.5 / 27.1, 470 MB 147 / 148, 2.1 GB 667 / 663; bf16 tensors too large
//     to be read once, [5120, 8192] 36.1 / 37.3, two [8192, 8192] 92.8 / 92.3, eight 355 / 359: folded in the pass.
constexpr int64_t kPublishMinBytes = 64ll << 20;
static bool nv_published(int dtype, bool four_over_six, int64_t sections, int64_t n, int64_t bytes) {
    if (bytes < kPublishMinBytes) return false;
    const bool paired = sections * 2 >= n * 3;       // half of the tensors at least
    if (!four_over_six) return paired;
    return dtype != MQ_F32 || (kept_quarters(bytes) == 4 && (paired || bytes >= 2 * kPublishMinBytes));
}
// quantize (carried run: and fold, and second pass) over a table whose grid is known: tab.chunk / tab.max_blocks are set
// (all_units: of all n tensors; sections: of their records)
template <class Table>
static int nvfp4_quant_launch(int dtype, const Table& tab, int n, int64_t all_units, int64_t sections, int e4m3_max, int flags, int mode, hipStream_t st) {
    if (mode == 2 && dtype == MQ_F32) return mq_fail(MQ_ERR_ARG, "a carried-over amax is for bf16 and fp16 tensors");
    const float numer = (float)e4m3_max * 6.0f;
    const dim3 folds((unsigned)n), blk(256);
    const dim3 grid((unsigned)tab.max_blocks, (unsigned)n);
    if (mode == 2) {
        if (tab.max_blocks > 0) launch_nvfp4_quant<1>(dtype, tab, flags, numer, false, false, grid, st);
        hipLaunchKernelGGL((nvfp4_fold_kernel<2, Table>), folds, blk, 0, st, tab, numer, mq_amax_feedback(), mq_amax_feedback_mirror());
        if (tab.max_blocks > 0) {
            const unsigned redo_blocks = tab.max_blocks < kSectionWords ? (unsigned)tab.max_blocks : (unsigned)kSectionWords;
            launch_nvfp4_quant<2>(dtype, tab, flags, numer, true, false, dim3(redo_blocks, (unsigned)n), st);
        }
        return mq_check_launch("nvfp4 quant (carried-over amax)");
    }
    if (nv_published(dtype, (flags & MQ_NVFP4_4OVER6) != 0, sections, n, all_units * (dtype == MQ_F32 ? 32 : 16))) {
        hipLaunchKernelGGL((nvfp4_publish_kernel<Table>), dim3(1, (unsigned)n), dim3(kWave), 0, st, tab, numer,
                           mode == 1 ? mq_amax_feedback() : nullptr, mq_amax_feedback_mirror());
        launch_nvfp4_quant<3>(dtype, tab, flags, numer, mode == 1, false, grid, st);
        return mq_check_launch("nvfp4 quant");
    }
    // (a list of empty tensors still has its scales published, by the first workgroup of each)
    launch_nvfp4_quant<0>(dtype, tab, flags, numer, mode == 1, mode == 1, dim3(grid.x > 0 ? grid.x : 1u, grid.y), st);
    return mq_check_launch("nvfp4 quant");
}

// tab.job[i]: w, q, s = block scales, aux = amax record, aux2 = fp32 global scale out (may be null), units = numel / 8.
// section = place of the tensor inside its record, pad = tensors sharing the record (adjacent entries).
// mode 0 (single calls, whose record is the caller's) and 1 (job driver), after the amax pass: quantize; mode 1 is counted in
//   the call's feedback.
// (fp32 tensors take modes 0 and 1.)
// mode 2 (job driver, carried-over amax): quantize with the record's old scales while collecting the new partial maxima,
//   fold and compare, quantize again where they differ.
int mq_nvfp4_quant_launch_group(int dtype, FlatTable& tab, int e4m3_max, int flags, int mode, hipStream_t st) {
    const int fos = flags & MQ_NVFP4_4OVER6;
    if (!flat_grid(tab, dtype == MQ_F32 ? nv_f32_units_per_block(fos) : nv_units_per_block(fos))) return mq_fail(MQ_ERR_ARG, "tensor too large");
    int64_t all_units = 0, sections = 0;
    for (int i = 0; i < tab.n; i++) {
        all_units += tab.job[i].units;
        sections += tab.job[i].pad;
    }
    return nvfp4_quant_launch(dtype, tab, tab.n, all_units, sections, e4m3_max, flags, mode, st);
}
// modes 1 and 2 over n descriptors of a device table (standard block scaling only); max_units: the largest tensor's units,
// sections: of all tensors' records
int mq_nvfp4_quant_launch_table(int dtype, const FlatJob* device_jobs, int n, int64_t max_units, int64_t sections, int e4m3_max,
                                int mode, hipStream_t st) {
    FlatRef ref{device_jobs, 0, 0};
    if (!flat_grid(ref, max_units, dtype == MQ_F32 ? nv_f32_units_per_block(0) : kNvThreads * kNvUnroll)) return mq_fail(MQ_ERR_ARG, "tensor too large");
    if (n == 0) return MQ_OK;
    return nvfp4_quant_launch(dtype, ref, n, max_units * n, sections, e4m3_max, 0, mode, st);
}

// Whether a chunk of NVFP4 jobs (packed kernels, no carried amax) takes the one-pass form.  `slots` is the
// largest number of workgroups that share a record, `bytes` the input of the whole chunk.  All workgroups of a record
// have to be on the chip together, and the records behind it should be loading meanwhile: half of what fits (640 workgroups,
// 40 MB, on 256 CUs).  A pair of [2048, 7168] weights, 896 workgroups, gained less (313 -> 265 us for 16 pairs) and is one
// busy neighbour away from waiting in vain, so it keeps two passes.  Short lists keep them as well: they find their second
// read in the memory-side cache, and the launch that clears the slots takes what is left of the gain (us, two passes / one, runs of
// one side differ by 0.1): 4 x [256, 1024] (2 MB) 6.4 / 8.9, 2 x [1024, 2048] 8.1 / 9.5, 4 of them (17 MB) 10.5 / 10.6, 1 x [2048, 4096] (17 MB)
// 11.3 / 10.7, 4 x [1537, 2064] (25 MB) 13.9 / 12.2, 1 x [2048, 7168] (29 MB) 16.2 / 13.0, 8 x [1024, 2048] (34 MB) 16.1 / 14.0, 2 x [2048, 7168]
// (59 MB) 23.8 / 18.3.  With Four Over Six the first two tensors' loads and the last one's arithmetic have nothing beside them,
// and what a list gains depends on its tensors and its values (blocks too close to call are looked at again): with slots that had to be
// cleared again, 33 x [528, 3088] (108 MB) 44 / 48, 45 x [740, 1952] (130 MB) 53.4 / 54.3, 24 x [1536, 2048]
// (151 MB) 59.5 / 57.3, 5 x [4096, 4096] (168 MB) 64.5 / 66.4, 6 x [2048, 7168] (176 MB) 68.6 / 67.4, 7 x [4096, 4096] (235 MB) 88.0 / 87.1, 38 x [1536,
// 2048] (239 MB) 90.8 / 80.4; weights N(0, 0.02^2) with the slots as they are 44.8 / 44.0, 52.3 / 49.7, 58.1 / 52.8, 62.3 / 63.3, 66.4 / 63.7, 85.3 / 81.0,
// 88.5 / 72.8.  From 200 MiB on it is ahead for all of them.
// A list of many small tensors (over a device table; 64 tensors of 24 MiB have 384 KiB each) has a grid row and a wait for each, and two
// passes have neither: us, two / one, 24 MiB in tensors of 64 KiB 13.8 / 34.1, of 256 KiB 13.3 / 15.9, of 320 KiB 13.3 / 14.7; 32 MiB of
// 320 KiB 16.1 / 17.7, of 384 KiB 15.7 / 15.4; 50 MiB of 264 KiB 23.7 / 25.0, of 330 KiB 23.1 / 21.9; 64 MiB of 192 KiB 27.6 / 33.0, of 320 KiB
// 27.5 / 26.3.  Lists of 64 MiB and more are read once whatever their tensors are, though two passes would be faster up to 192 KiB a
// tensor (400 MiB of 64 KiB 160 / 435, of 192 KiB 149 / 162, of 256 KiB 149 / 130).
constexpr int64_t kOneMinBytes = 24ll << 20, kOneFosMinBytes = 200ll << 20;
constexpr int64_t kOneAnyTensors = 64ll << 20;
static int64_t one_min_tensor(int64_t bytes) { return bytes >= kOneAnyTensors ? 0 : bytes >= (48ll << 20) ? 320 << 10 : 384 << 10; }
// n: tensors of the chunk
bool mq_nvfp4_one_pass_ok(int64_t max_units, int64_t slots, int64_t bytes, int64_t n, int flags) {
    int device = 0, cus = 0;
    const bool fos = (flags & MQ_NVFP4_4OVER6) != 0;
    if (fos && nv_error_mode(flags) > 1) return false;       // (an error in fp16 has no estimate)
    if (bytes < (fos ? kOneFosMinBytes : kOneMinBytes) || max_units > kOneSlots * kOnePerBlock || bytes < n * one_min_tensor(bytes)) return false;
    if (hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return slots <= kOneRecordSlots && slots * 2 <= (int64_t)cus * kOneWavesPerSimd;       // a workgroup is one wavefront per SIMD
}
int64_t mq_nvfp4_one_pass_slots(int64_t units) { return (units + kOnePerBlock - 1) / kOnePerBlock; }

// workgroups behind the tensors' own, for each of n tensors of at most max_units: 64 of a list of 32 tensors (the launch has
// 0.4 ns for one that finds nothing to do), and enough to fill half of the chip for one that is left.  A list of more than 128 has 16 for
// each, or one for eight pieces of a smaller tensor: with 16, or one for each piece, 6400 x 64 KiB took 473 us, now 435, 2133 x 192 KiB 184 and 160,
// 1066 x 384 KiB 112 and 103 (452, 177 and 122 before there were any); all tensors left, 1600 x 256 KiB 180 and 162, 204 x 640 KiB 48.2 and 49.3.
constexpr int kOneWorkers = 2048, kOneFewest = 16, kOnePieces = 8;
static uint32_t nv_one_workers(int n, int64_t max_units, int fos) {
    const int64_t blocks = (max_units + nv_units_per_block(fos) - 1) / nv_units_per_block(fos);
    const int64_t few = (blocks + kOnePieces - 1) / kOnePieces, fewest = few < kOneFewest ? few : kOneFewest;
    int64_t workers = kOneWorkers / n;
    workers = workers < fewest ? fewest : workers > kSectionWords ? kSectionWords : workers;
    return (uint32_t)(workers < blocks ? workers : blocks);
}
// descriptors as for mode 1
template <class Table, int FOS, int F16>
static int nvfp4_one_pass_launch_dtype(const Table& tab, int n, int64_t max_units, float numer, int first_polls, int patience, hipStream_t st) {
    const uint32_t workers = nv_one_workers(n, max_units, FOS), blocks = (uint32_t)tab.max_blocks;
    const dim3 grid(blocks, (unsigned)(n + ((int64_t)n * workers + blocks - 1) / blocks));
    hipLaunchKernelGGL((nvfp4_one_pass_clear_kernel<Table>), dim3((unsigned)n), dim3(256), 0, st, tab);
    hipLaunchKernelGGL((nvfp4_one_pass_kernel<FOS, F16, Table>), grid, dim3(kOneThreads), 0, st, tab, numer, first_polls, patience, (uint32_t)n, workers,
                       mq_amax_feedback(), mq_amax_feedback_mirror());
    return mq_check_launch("nvfp4 quant (one pass)");
}
template <class Table>
static int nvfp4_one_pass_launch(int dtype, const Table& tab, int n, int64_t max_units, int e4m3_max, int flags, int first_polls, int patience, hipStream_t st) {
    const float numer = (float)e4m3_max * 6.0f;
    if constexpr (std::is_same<Table, FlatTable>::value) {
        if (flags & MQ_NVFP4_4OVER6) {
            const bool squared = nv_error_mode(flags) == 1;
            if (dtype == MQ_F16) return squared ? nvfp4_one_pass_launch_dtype<Table, 2, 1>(tab, n, max_units, numer, first_polls, patience, st)
                                                : nvfp4_one_pass_launch_dtype<Table, 1, 1>(tab, n, max_units, numer, first_polls, patience, st);
            return squared ? nvfp4_one_pass_launch_dtype<Table, 2, 0>(tab, n, max_units, numer, first_polls, patience, st)
                           : nvfp4_one_pass_launch_dtype<Table, 1, 0>(tab, n, max_units, numer, first_polls, patience, st);
        }
    }
    return dtype == MQ_F16 ? nvfp4_one_pass_launch_dtype<Table, 0, 1>(tab, n, max_units, numer, first_polls, patience, st)
                           : nvfp4_one_pass_launch_dtype<Table, 0, 0>(tab, n, max_units, numer, first_polls, patience, st);
}
static int nv_one_polls(int flags) { return (flags & MQ_NVFP4_NO_WAIT) ? 0 : kOnePolls; }
// (with limits of its own for the waits: for the tests of how they end)
int mq_nvfp4_one_pass_launch_waits(int dtype, FlatTable& tab, int64_t max_units, int e4m3_max, int flags, int first_polls, int patience, hipStream_t st) {
    if (!flat_grid(tab, kOnePerBlock)) return mq_fail(MQ_ERR_ARG, "tensor too large");
    return nvfp4_one_pass_launch(dtype, tab, tab.n, max_units, e4m3_max, flags, first_polls, patience, st);
}
int mq_nvfp4_one_pass_launch_group(int dtype, FlatTable& tab, int64_t max_units, int e4m3_max, int flags, hipStream_t st) {
    return mq_nvfp4_one_pass_launch_waits(dtype, tab, max_units, e4m3_max, flags, nv_one_polls(flags), kOnePatience, st);
}
int mq_nvfp4_one_pass_launch_table(int dtype, const FlatJob* device_jobs, int n, int64_t max_units, int e4m3_max, int flags,
                                   hipStream_t st) {
    FlatRef ref{device_jobs, 0, 0};
    if (!flat_grid(ref, max_units, kOnePerBlock)) return mq_fail(MQ_ERR_ARG, "tensor too large");
    return nvfp4_one_pass_launch(dtype, ref, n, max_units, e4m3_max, flags, nv_one_polls(flags), kOnePatience, st);
}

extern "C" int mq_nvfp4_amax(const void* w, int dtype, int64_t numel, void* record, int section, void* stream) {
    if ((!w && numel != 0) || !record) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (dtype < MQ_BF16 || dtype > MQ_F32 || numel < 0) return mq_fail(MQ_ERR_ARG, "bad argument");
    if (section < 0 || section >= MQ_NVFP4_SECTIONS) return mq_fail(MQ_ERR_ARG, "bad amax record section");
    hipStream_t st = (hipStream_t)stream;
    if (((uintptr_t)w % 16) == 0) {
        FlatTable tab{};
        tab.n = 1;
        tab.job[0] = FlatJob{w, nullptr, (void*)(uintptr_t)numel, record, numel / 8, nullptr, section, 0};
        return mq_nvfp4_amax_launch_group(dtype, tab, st);
    }
    hipLaunchKernelGGL(nvfp4_amax_generic_kernel, dim3(kSectionWords), dim3(256), 0, st, w, dtype, numel,
                       (uint32_t*)record + section * kSectionWords);
    return mq_check_launch("nvfp4 amax");
}

extern "C" int mq_nvfp4_quant(const void* w, int dtype, const void* record, int n_sections, void* q, void* block_scale,
                              float* global_scale, int64_t M, int64_t K, int e4m3_max, int flags, void* stream) {
    if (((!w || !q || !block_scale) && M != 0 && K != 0) || !record) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (dtype < MQ_BF16 || dtype > MQ_F32 || M < 0 || K < 0) return mq_fail(MQ_ERR_ARG, "bad argument");
    if (n_sections < 1 || n_sections > MQ_NVFP4_SECTIONS) return mq_fail(MQ_ERR_ARG, "bad amax record section count");
    if (K % 16 != 0) return mq_fail(MQ_ERR_ARG, "Last dim must be divisible by 16 for NVFP4");
    if (e4m3_max != 448 && e4m3_max != 256) return mq_fail(MQ_ERR_ARG, "e4m3_max must be 448 or 256");
    if (flags & ~(MQ_NVFP4_4OVER6 | MQ_NVFP4_ERR_MSE | MQ_NVFP4_ERR_FP16)) return mq_fail(MQ_ERR_ARG, "unknown NVFP4 flag");
    hipStream_t st = (hipStream_t)stream;
    const float numer = (float)e4m3_max * 6.0f;
    const int64_t blocks16 = M * (K / 16);
    if (blocks16 == 0 || mq_nvfp4_fast_ok(w, dtype, q)) {
        FlatTable tab{};
        tab.n = 1;
        tab.job[0] = FlatJob{w, q, block_scale, const_cast<void*>(record), blocks16 * 2, global_scale, n_sections - 1, n_sections};
        return mq_nvfp4_quant_launch_group(blocks16 == 0 ? MQ_BF16 : dtype, tab, e4m3_max, flags, 0, st);
    }
    FlatTable fold{};
    fold.n = 1;
    fold.job[0] = FlatJob{w, q, block_scale, const_cast<void*>(record), 0, global_scale, n_sections, 0};
    hipLaunchKernelGGL((nvfp4_fold_kernel<0, FlatTable>), dim3(1), dim3(256), 0, st, fold, numer, (uint32_t*)nullptr, (uint32_t*)nullptr);
    int64_t nb = (blocks16 + 255) / 256;
    if (nb > mq_grid_cap()) nb = mq_grid_cap();
    hipLaunchKernelGGL(nvfp4_quant_generic_kernel, dim3((unsigned)nb), dim3(256), 0, st, w, dtype,
                       (const uint32_t*)record, (uint8_t*)q, (uint8_t*)block_scale, blocks16, flags, numer);
    return mq_check_launch("nvfp4 quant");
}

extern "C" int mq_nvfp4_fold(void* record, int n_sections, int e4m3_max, void* stream) {
    if (!record) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (n_sections < 1 || n_sections > MQ_NVFP4_SECTIONS) return mq_fail(MQ_ERR_ARG, "bad amax record section count");
    if (e4m3_max != 448 && e4m3_max != 256) return mq_fail(MQ_ERR_ARG, "e4m3_max must be 448 or 256");
    FlatTable tab{};
    tab.n = 1;
    tab.job[0] = FlatJob{nullptr, nullptr, nullptr, record, 0, nullptr, n_sections, 0};
    hipLaunchKernelGGL((nvfp4_fold_kernel<0, FlatTable>), dim3(1), dim3(256), 0, (hipStream_t)stream, tab, (float)e4m3_max * 6.0f, (uint32_t*)nullptr, (uint32_t*)nullptr);
    return mq_check_launch("nvfp4 fold");
}

template <int F16>
static void nvfp4_fake_launch_dtype(const FlatTable& tab, int fos, float numer, float inv_numer, hipStream_t st) {
    const dim3 grid((unsigned)tab.max_blocks, (unsigned)tab.n), blk(kNvThreads);
    switch (fos) {
        case 0: hipLaunchKernelGGL((nvfp4_fake_kernel<0, F16>), grid, blk, 0, st, tab, numer, inv_numer); break;
        case 1: hipLaunchKernelGGL((nvfp4_fake_kernel<1, F16>), grid, blk, 0, st, tab, numer, inv_numer); break;
        case 2: hipLaunchKernelGGL((nvfp4_fake_kernel<2, F16>), grid, blk, 0, st, tab, numer, inv_numer); break;
        case 3: hipLaunchKernelGGL((nvfp4_fake_kernel<3, F16>), grid, blk, 0, st, tab, numer, inv_numer); break;
        default: hipLaunchKernelGGL((nvfp4_fake_kernel<4, F16>), grid, blk, 0, st, tab, numer, inv_numer); break;
    }
}
// tab.job[i]: w = x, q = y, units, and the amax (see nv_fake_scales)
static int nvfp4_fake_launch(int dtype, FlatTable& tab, int e4m3_max, int flags, hipStream_t st) {
    if (!flat_grid(tab, nv_units_per_block(flags & MQ_NVFP4_4OVER6))) return mq_fail(MQ_ERR_ARG, "tensor too large");
    const float numer = (float)e4m3_max * 6.0f, inv_numer = (float)(1.0 / (double)(6 * e4m3_max));
    const int fos = (flags & MQ_NVFP4_4OVER6) ? 1 + nv_error_mode(flags) : 0;
    if (dtype == MQ_F16) nvfp4_fake_launch_dtype<1>(tab, fos, numer, inv_numer, st);
    else nvfp4_fake_launch_dtype<0>(tab, fos, numer, inv_numer, st);
    return mq_check_launch("nvfp4 fake quant");
}

extern "C" int mq_nvfp4_qdq(const void* x, int dtype, const float* amax, void* y, int64_t numel, int e4m3_max,
                            int flags, void* stream) {
    if (((!x || !y) && numel != 0) || !amax) return mq_fail(MQ_ERR_ARG, "null pointer");
    if ((dtype != MQ_BF16 && dtype != MQ_F16) || numel < 0) return mq_fail(MQ_ERR_ARG, "input must be bfloat16 or float16");
    if (numel % 16 != 0) return mq_fail(MQ_ERR_ARG, "element count must be a multiple of 16");
    if (e4m3_max != 448 && e4m3_max != 256) return mq_fail(MQ_ERR_ARG, "e4m3_max must be 448 or 256");
    if ((((uintptr_t)x | (uintptr_t)y) & 15) != 0) return mq_fail(MQ_ERR_ARG, "tensors must be 16-byte aligned");
    if (flags & ~(MQ_NVFP4_4OVER6 | MQ_NVFP4_ERR_MSE | MQ_NVFP4_ERR_FP16)) return mq_fail(MQ_ERR_ARG, "unknown NVFP4 flag");
    if (numel == 0) return MQ_OK;
    FlatTable tab{};
    tab.n = 1;
    tab.job[0] = FlatJob{x, y, nullptr, nullptr, numel / 8, const_cast<float*>(amax), 0, 0};
    return nvfp4_fake_launch(dtype, tab, e4m3_max, flags, (hipStream_t)stream);
}

extern "C" int mq_nvfp4_fake_quant(const mq_fake_quant_item* list, int64_t n, int dtype, void* partial_maxima, int e4m3_max,
                                   int flags, void* stream) {
    if (n < 0 || (n > 0 && (!list || !partial_maxima))) return mq_fail(MQ_ERR_ARG, "null pointer");
    if (dtype != MQ_BF16 && dtype != MQ_F16) return mq_fail(MQ_ERR_ARG, "input must be bfloat16 or float16");
    if (e4m3_max != 448 && e4m3_max != 256) return mq_fail(MQ_ERR_ARG, "e4m3_max must be 448 or 256");
    if (flags & ~(MQ_NVFP4_4OVER6 | MQ_NVFP4_ERR_MSE | MQ_NVFP4_ERR_FP16)) return mq_fail(MQ_ERR_ARG, "unknown NVFP4 flag");
    if (((uintptr_t)partial_maxima & 3) != 0) return mq_fail(MQ_ERR_ARG, "the partial maxima must be 4-byte aligned");
    for (int64_t i = 0; i < n; i++) {
        if (!list[i].x || !list[i].y || list[i].numel <= 0) return mq_fail(MQ_ERR_ARG, "empty tensor");
        if (list[i].numel % 16 != 0) return mq_fail(MQ_ERR_ARG, "element count must be a multiple of 16");
        if ((((uintptr_t)list[i].x | (uintptr_t)list[i].y) & 15) != 0) return mq_fail(MQ_ERR_ARG, "tensors must be 16-byte aligned");
    }
    hipStream_t st = (hipStream_t)stream;
    for (int64_t i = 0; i < n;) {
        FlatTable tab{};
        int64_t sum = 0, mx = 0;
        for (; i < n && tab.n < kMaxGroup; i++) {
            const int64_t e = list[i].numel, nmx = e > mx ? e : mx;
            if (tab.n > 0 && nmx * (tab.n + 1) * 4 > (sum + e) * 5) break;       // padding of the 2-D grid under 25 %
            sum += e;
            mx = nmx;
            // (the amax kernel takes the element count in `s`)
            tab.job[tab.n++] = FlatJob{list[i].x, list[i].y, (void*)(uintptr_t)e, (uint32_t*)partial_maxima + i * kSectionWords,
                                       e / 8, nullptr, 0, 0};
        }
        int rc = mq_nvfp4_amax_launch_group(dtype, tab, st);
        if (rc == MQ_OK) rc = nvfp4_fake_launch(dtype, tab, e4m3_max, flags, st);
        if (rc != MQ_OK) return rc;
    }
    return MQ_OK;
}
