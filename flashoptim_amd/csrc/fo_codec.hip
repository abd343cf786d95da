// Standalone group codec and ECC kernels for gfx950 with their C entry points: the companions of the fused step
// kernels (state initialisation, checkpoints, fp32 export/import of master weights).  They share the access shape
// of the step kernels (fo_device.h), and their output equals an IEEE evaluation of the reference formulas operation
// by operation.
//
// All of them only move memory at heart, so each reads its inputs once and writes its result in its final type; and
// a checkpoint holds hundreds of tensors, most of them short, so the conversions of a whole list share one launch
// (convert_kernel below).
//
// "ref:" cites /root/reference/flashoptim/optimizers.py.
#include "fo_device.h"
#include "fo_host.h"
#include "../../include/flashoptim_hip.h"
#ifdef FO_DIAG
#include "../../include/flashoptim_hip_diag.h"
#endif

namespace fo {

constexpr int kCodecThreads = 64;   // one wavefront per workgroup, like the step kernels

// Value of code byte b before the group scale: q / IN_MAX, then y / (2 - |y|) when the softsign companding is on
// (ref:2591-2597), each operation correctly rounded.  Evaluated by the compiler, one table per flag combination;
// a lookup replaces two IEEE divisions per element.
template <bool SIGNED, bool SOFTSIGN> struct CodeTable {
    float v[256];
    constexpr CodeTable() : v() {
        for (int b = 0; b < 256; ++b) {
            const int q = (SIGNED && b >= 128) ? b - 256 : b;
            const float t = (float)q / (SIGNED ? 127.0f : 255.0f);
            const float a = t < 0.0f ? -t : t;
            v[b] = SOFTSIGN ? t / (2.0f - a) : t;
        }
    }
};
__device__ const CodeTable<false, false> kCodeTableU = CodeTable<false, false>();
__device__ const CodeTable<false, true> kCodeTableUS = CodeTable<false, true>();
__device__ const CodeTable<true, false> kCodeTableS = CodeTable<true, false>();
__device__ const CodeTable<true, true> kCodeTableSS = CodeTable<true, true>();

// ------------------------------------------------------------------------------------------------
// one launch over a list of tensors
// ------------------------------------------------------------------------------------------------

// The list travels as the kernel's argument (3.3 KiB of the 4 KiB a launch may pass): no table is uploaded and no
// memory has to outlive the call.  A workgroup (one wavefront) finds its job with one vector load and a ballot: lane l
// reads where job l's workgroups start, the number of lanes that start at or before this workgroup names the job.
constexpr int kJobsPerLaunch = 64;
struct JobBatch {
    fo_convert_job job[kJobsPerLaunch];
    u32 first_block[kJobsPerLaunch];
    int32_t count, reserved;
};
static_assert(sizeof(JobBatch) <= 3584, "a batch must fit the kernel argument segment");

// Op: kEpl elements per lane and span, kSpans neighbouring spans of 64 * kEpl elements per workgroup; a Raw holds
// what a lane has loaded for one span; all loads of a workgroup are issued before the first span is finished.
// kSpans is each Op's best over five sets of 2^27 elements in turn (more than the caches hold), bf16 where the type is
// free (TB/s of the bytes in and out):
//     spans per workgroup         1      2      3      4      6      8
//     fp32 masters out          6.02   6.62   6.28   6.35   6.12   6.27
//     fp32 masters in           6.09   6.59   6.34   6.36   6.04   6.09
//     dequantise to bf16        4.80   6.48   6.12   6.32   5.96   6.13
//     dequantise to fp32        3.98   5.48   5.91   6.29   5.89   6.13
//     quantise, first moments   4.22   6.02   6.03   6.20   5.86   5.94
//     quantise, second moments  3.95   5.65   5.74   5.99   5.77   5.82
//     quantise fp32             4.53   5.78   6.03   6.46   6.32   6.12
//     int8 to bf16              5.25   6.48   6.14   6.17   6.04   6.15
//     bf16 to int8              5.77   6.58   6.42   6.35   6.20   6.17
// One span leaves what a workgroup costs to start (its place in the list, the table in LDS, the spread of its loads) over
// too few bytes, many spans widen the window of addresses in flight; odd counts start workgroups at odd KiB.  A cap on the
// resident workgroups gains nothing on top.
template <class Op> struct ConvertShape {
    static constexpr int64_t kSpan = 64 * Op::kEpl;
    static constexpr int64_t kBlock = kSpan * Op::kSpans;
};

template <class Op, int MODE>
__device__ __forceinline__ void convert_block(const fo_convert_job& job, int64_t base, float* lut) {
    typename Op::Raw raw[Op::kSpans];
    const int lane = (int)threadIdx.x * Op::kEpl;
#pragma unroll
    for (int i = 0; i < Op::kSpans; ++i) Op::template load<MODE>(job, Where{base + i * ConvertShape<Op>::kSpan, lane}, raw[i]);
    Op::prepare(job, lut);
#pragma unroll
    for (int i = 0; i < Op::kSpans; ++i) Op::template finish<MODE>(job, Where{base + i * ConvertShape<Op>::kSpan, lane}, raw[i], lut);
}

template <class Op> __global__ __launch_bounds__(kCodecThreads) void convert_kernel(JobBatch b) {
    __shared__ __align__(16) float lut[Op::kLutFloats];
    const u32 start = (int)threadIdx.x < b.count ? b.first_block[threadIdx.x] : 0xffffffffu;
    const int j = __builtin_popcountll(__builtin_amdgcn_ballot_w64(start <= blockIdx.x)) - 1;  // job 0 starts at 0
    const fo_convert_job job = b.job[j];
    const int64_t base = (int64_t)(blockIdx.x - b.first_block[j]) * ConvertShape<Op>::kBlock;
    // workgroup-uniform choice of the access mode
    if (!Op::aligned(job)) convert_block<Op, kGuarded>(job, base, lut);
    else if (base + ConvertShape<Op>::kBlock <= job.n) convert_block<Op, kVector>(job, base, lut);
    else convert_block<Op, kLane>(job, base, lut);
}

__device__ __forceinline__ bool aligned16(const void* a, const void* b) { return (((uintptr_t)a | (uintptr_t)b) & 15u) == 0; }

// x where it is a number, the quiet NaN 0x7fc00000 otherwise: in front of a conversion to bf16 the result then has the
// bits of torch's cast, which writes 0x7fc0 for every NaN (the conversion instruction keeps sign and payload; for fp16
// the cast does so too).
template <int DT> __device__ __forceinline__ float one_nan(float x) { return (DT == DT_BF16 && x != x) ? as_f32(0x7fc00000u) : x; }

// ref:2541-2607 _triton_dequantize_kernel, with the cast to the output type that follows it in a checkpoint (ref:167).
// Bound by memory: 1.06 bytes in and 4 (fp32) or 2 (bf16) out per element.  kSpans: the 1 KiB table that a workgroup
// copies to LDS serves 1024 elements; reading the table through the vector cache instead is slower by a third.  An AdamW
// checkpoint of 2.2e8 weights (bf16, 24-bit masters; this kernel and Int8WidenOp) takes 306 us, 6.5 TB/s, where fp32
// values, their casts and torch's int8 cast (1.3 TB/s) took 1453.
template <int ODT> struct DequantizeOp {
    static constexpr int kEpl = DTypeInfo<ODT>::epl, kSpans = ODT == DT_F32 ? 4 : 2, kLutFloats = 256;
    struct Raw { Pack<1, kEpl> codes; uint16_t scale; };
    __device__ __forceinline__ static bool aligned(const fo_convert_job& j) { return aligned16(j.src, j.dst); }
    template <int MODE> __device__ __forceinline__ static void load(const fo_convert_job& j, Where w, Raw& r) {
        load_lane<1, kEpl, MODE>(r.codes, j.src, w, j.n);
        r.scale = 0x3c00;                                                   // ref:2577-2582 masked scales read 1.0
        if (MODE == kVector || w.first() < j.n) r.scale = load_scale(static_cast<const uint16_t*>(j.src2), w);
    }
    __device__ __forceinline__ static void prepare(const fo_convert_job& j, float* lut) {
        const bool is_signed = j.flags & FO_CODEC_SIGNED, softsign = j.flags & FO_CODEC_SOFTSIGN;
        const float* table = is_signed ? (softsign ? kCodeTableSS.v : kCodeTableS.v) : (softsign ? kCodeTableUS.v : kCodeTableU.v);
        *reinterpret_cast<u32x4*>(lut + 4 * threadIdx.x) = *reinterpret_cast<const u32x4*>(table + 4 * threadIdx.x);
        __syncthreads();  // one wavefront: no hardware barrier is needed, the compiler drops it
    }
    template <int MODE> __device__ __forceinline__ static void finish(const fo_convert_job& j, Where w, Raw& r, const float* lut) {
        const float scale = f16_bits_to_f32(r.scale);
        float x[kEpl];
#pragma unroll
        for (int k = 0; k < kEpl; ++k) {
            x[k] = lut[byte_of<kEpl>(r.codes, k)] * scale;                  // ref:2591-2600
            if (j.flags & FO_CODEC_SQRT) x[k] = x[k] * x[k];                // ref:2603-2604
        }
        Pack<DTypeInfo<ODT>::bytes, kEpl> o;
#pragma unroll
        for (int k = 0; k < kEpl; k += 2) {
            float wa, wb;
            narrow_pair<ODT, kEpl>(o, k, one_nan<ODT>(x[k]), one_nan<ODT>(x[k + 1]), wa, wb);
        }
        store_lane<DTypeInfo<ODT>::bytes, kEpl, MODE>(o, j.dst, w, j.n);
    }
};

// One span of values as the verified flow sees it from a lane (fo_math.h: codec_verified).
template <int EPL> struct CodecLane {
    const float (&v)[EPL];
    float am;
    Pack<1, EPL>& out;
    float x[EPL], slack[EPL], least;
    __device__ __forceinline__ void convert(const float (&q)[EPL]) {
        if constexpr (EPL == 8) {
            const float lo[4] = {q[0], q[1], q[2], q[3]}, hi[4] = {q[4], q[5], q[6], q[7]};
            convert_pack8<kFloor, kFloor>(lo, hi, out.w[0], out.w[1]);
        } else {
            u32 c[EPL];
#pragma unroll
            for (int k = 0; k < EPL; ++k) c[k] = (u32)hw::floor_to_int(q[k]);
            pack_codes<1, EPL>(c, out);
        }
    }
    __device__ __forceinline__ void set_code(int k, u32 code) { fo::set_code<EPL>(out, k, code); }
};

// ref:2610-2676 _triton_quantize_kernel.  2 (4) bytes in and 1.06 out per element; two IEEE divisions (or one and an
// IEEE root) per element would make it a matter of vector instructions (2.4 TB/s on bf16), so the two kinds of state
// the optimizers hold go through the quick forms with verification, which give the same codes (fo_math.h).  Loading an
// AdamW checkpoint of 2.2e8 weights (bf16, 24-bit masters; this kernel and Int8NarrowOp) takes 301 us, 6.6 TB/s, where
// it took 912 with the IEEE form and torch's cast to int8 (1.3 TB/s).
template <int XDT> struct QuantizeOp {
    static constexpr int kEpl = DTypeInfo<XDT>::epl, kSpans = 4, kLutFloats = 4;
    struct Raw { Pack<DTypeInfo<XDT>::bytes, kEpl> x; };
    __device__ __forceinline__ static bool aligned(const fo_convert_job& j) { return aligned16(j.src, j.dst); }
    template <int MODE> __device__ __forceinline__ static void load(const fo_convert_job& j, Where w, Raw& r) {
        load_lane<DTypeInfo<XDT>::bytes, kEpl, MODE>(r.x, j.src, w, j.n);
    }
    __device__ __forceinline__ static void prepare(const fo_convert_job&, float*) {}
    template <int MODE> __device__ __forceinline__ static void finish(const fo_convert_job& j, Where w, Raw& r, const float*) {
        float v[kEpl];
        float am = 0.0f;
        Pack<1, kEpl> out;
#pragma unroll
        for (int k = 0; k < kEpl; ++k) v[k] = widen<XDT, kEpl>(r.x, k);
        if (j.flags == (FO_CODEC_SIGNED | FO_CODEC_SOFTSIGN)) {
#pragma unroll
            for (int k = 0; k < kEpl; ++k) am = fmaxf(am, fabsf(v[k]));
            am = fmaxf(group_max<kEpl>(am), 1e-12f);                            // ref:2657-2658
            CodecLane<kEpl> lane{v, am, out};
            HwWave<CodecLane<kEpl>> wave{lane};
            codec_verified<kEpl, false>(wave);
        } else if (j.flags == FO_CODEC_SQRT) {
            // the root is monotone, so the largest root is the root of the largest value; negative values are NaN after
            // the root and take no part in the maximum either way
#pragma unroll
            for (int k = 0; k < kEpl; ++k) am = fmaxf(am, v[k]);
            am = fmaxf(sqrt_rn(group_max<kEpl>(am)), 1e-12f);
            CodecLane<kEpl> lane{v, am, out};
            HwWave<CodecLane<kEpl>> wave{lane};
            codec_verified<kEpl, true>(wave);
        } else {
#pragma unroll
            for (int k = 0; k < kEpl; ++k) {
                if (j.flags & FO_CODEC_SQRT) v[k] = sqrt_rn(v[k]);              // ref:2650-2651
                am = fmaxf(am, fabsf(v[k]));
            }
            am = fmaxf(group_max<kEpl>(am), 1e-12f);
            const float out_max = (j.flags & FO_CODEC_SIGNED) ? 127.0f : 255.0f;
            u32 q[kEpl];
#pragma unroll
            for (int k = 0; k < kEpl; ++k) {
                const float nrm = div_rn(v[k], am);                             // ref:2661
                const float t = (j.flags & FO_CODEC_SOFTSIGN) ? div_rn(2.0f * nrm, 1.0f + fabsf(nrm)) : nrm;   // ref:2664-2667
                q[k] = (u32)(int)floorf(t * out_max + 0.5f);                    // ref:2670-2671
            }
            pack_codes<1, kEpl>(q, out);
        }
        store_lane<1, kEpl, MODE>(out, j.dst, w, j.n);
        if ((MODE == kVector || w.first() < j.n) && (threadIdx.x & (32 / kEpl - 1)) == 0)                      // ref:2675-2676
            store_scale(static_cast<uint16_t*>(j.dst2), w, f32_to_f16_bits(am));
    }
};

// int8 codes as values of a 2-byte type (exact): the form in which a checkpoint holds 1-byte correction codes
// (ref:900-927).  One byte in, two out.
template <int DT> struct Int8WidenOp {
    static constexpr int kEpl = 8, kSpans = 2, kLutFloats = 4;
    struct Raw { Pack<1, 8> codes; };
    __device__ __forceinline__ static bool aligned(const fo_convert_job& j) { return aligned16(j.src, j.dst); }
    template <int MODE> __device__ __forceinline__ static void load(const fo_convert_job& j, Where w, Raw& r) {
        load_lane<1, 8, MODE>(r.codes, j.src, w, j.n);
    }
    __device__ __forceinline__ static void prepare(const fo_convert_job&, float*) {}
    template <int MODE> __device__ __forceinline__ static void finish(const fo_convert_job& j, Where w, Raw& r, const float*) {
        Pack<2, 8> o;
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            float wa, wb;
            narrow_pair<DT, 8>(o, k, ecc_to_float<1, 8>(r.codes, k), ecc_to_float<1, 8>(r.codes, k + 1), wa, wb);
        }
        store_lane<2, 8, MODE>(o, j.dst, w, j.n);
    }
};

// The way back: values of a 2-byte type truncated to int8.
template <int DT> struct Int8NarrowOp {
    static constexpr int kEpl = 8, kSpans = 2, kLutFloats = 4;
    struct Raw { Pack<2, 8> x; };
    __device__ __forceinline__ static bool aligned(const fo_convert_job& j) { return aligned16(j.src, j.dst); }
    template <int MODE> __device__ __forceinline__ static void load(const fo_convert_job& j, Where w, Raw& r) {
        load_lane<2, 8, MODE>(r.x, j.src, w, j.n);
    }
    __device__ __forceinline__ static void prepare(const fo_convert_job&, float*) {}
    template <int MODE> __device__ __forceinline__ static void finish(const fo_convert_job& j, Where w, Raw& r, const float*) {
        u32 c[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) c[k] = (u32)(int)widen<DT, 8>(r.x, k);
        Pack<1, 8> out;
        pack_codes<1, 8>(c, out);
        store_lane<1, 8, MODE>(out, j.dst, w, j.n);
    }
};

// Import of fp32 master weights: the cast to the parameter's type and the correction codes of what it rounded off
// (ref:2806-2832 _compute_ecc_bits_kernel) in one pass, 4 bytes in and 3 or 4 out per element:
// 2.2e8 weights (bf16, 24-bit masters) take 230 us, 6.6 TB/s, where a cast, a copy and the split took 594.
template <int DT, int ECCB> struct EccNarrowOp {
    static constexpr int kEpl = 4, kSpans = 2, kLutFloats = 4;
    struct Raw { Pack<4, 4> x; };
    __device__ __forceinline__ static bool aligned(const fo_convert_job& j) { return aligned16(j.src, j.dst) && aligned16(j.dst2, nullptr); }
    template <int MODE> __device__ __forceinline__ static void load(const fo_convert_job& j, Where w, Raw& r) {
        load_lane<4, 4, MODE>(r.x, j.src, w, j.n);
    }
    __device__ __forceinline__ static void prepare(const fo_convert_job&, float*) {}
    template <int MODE> __device__ __forceinline__ static void finish(const fo_convert_job& j, Where w, Raw& r, const float*) {
        Pack<2, 4> narrow;
        u32 eb[4];
#pragma unroll
        for (int k = 0; k < 4; k += 2) {
            const float a = as_f32(r.x.w[k]), b = as_f32(r.x.w[k + 1]);
            float wa, wb;
            narrow_pair<DT, 4>(narrow, k, one_nan<DT>(a), one_nan<DT>(b), wa, wb);
            eb[k] = ecc_split_bits<DT, ECCB, true>(a, wa);
            eb[k + 1] = ecc_split_bits<DT, ECCB, true>(b, wb);
        }
        Pack<ECCB, 4> ecc;
        pack_codes<ECCB, 4>(eb, ecc);
        store_lane<2, 4, MODE>(narrow, j.dst, w, j.n);
        store_lane<ECCB, 4, MODE>(ecc, j.dst2, w, j.n);
    }
};

// ref:2779-2803 _reconstruct_fp32_kernel, the way out again: narrow value and correction code in (3 or 4 bytes), the fp32
// master out.  Bound by memory: 2.2e8 weights (bf16, 24-bit masters) take 232 us, 6.6 TB/s; the export of a model took
// 483 as long as it also cast every narrow weight and joined tensor by tensor.
template <int DT, int ECCB> struct EccJoinOp {
    static constexpr int kEpl = 4, kSpans = 2, kLutFloats = 4;
    struct Raw { Pack<2, 4> narrow; Pack<ECCB, 4> ecc; };
    __device__ __forceinline__ static bool aligned(const fo_convert_job& j) { return aligned16(j.src, j.dst) && aligned16(j.src2, nullptr); }
    template <int MODE> __device__ __forceinline__ static void load(const fo_convert_job& j, Where w, Raw& r) {
        load_lane<2, 4, MODE>(r.narrow, j.src, w, j.n);
        load_lane<ECCB, 4, MODE>(r.ecc, j.src2, w, j.n);
    }
    __device__ __forceinline__ static void prepare(const fo_convert_job&, float*) {}
    template <int MODE> __device__ __forceinline__ static void finish(const fo_convert_job& j, Where w, Raw& r, const float*) {
        Pack<4, 4> o;
#pragma unroll
        for (int k = 0; k < 4; ++k) o.w[k] = as_u32(ecc_join<DT, ECCB>(widen<DT, 4>(r.narrow, k), ecc_to_float<ECCB, 4>(r.ecc, k)));
        store_lane<4, 4, MODE>(o, j.dst, w, j.n);
    }
};

// ref:2806-2832 _compute_ecc_bits_kernel
template <int DT, int ECCB, bool FAST>
__device__ __forceinline__ void ecc_split_lane(const float* x, const void* narrow, void* ecc, int64_t first, int64_t n) {
    constexpr int EPL = 4;
    Pack<4, EPL> xraw;
    Pack<DTypeInfo<DT>::bytes, EPL> nraw;
    load_lane<4, EPL, FAST>(xraw, x, first, n);
    load_lane<DTypeInfo<DT>::bytes, EPL, FAST>(nraw, narrow, first, n);
    u32 eb[EPL];
#pragma unroll
    for (int k = 0; k < EPL; ++k) eb[k] = ecc_split_bits<DT, ECCB, true>(as_f32(xraw.w[k]), widen<DT, EPL>(nraw, k));
    Pack<ECCB, EPL> eout;
    pack_codes<ECCB, EPL>(eb, eout);
    store_lane<ECCB, EPL, FAST>(eout, ecc, first, n);
}

// Work loop shared by the kernels over one tensor, in the step kernels' geometry: a workgroup is one wavefront and takes one
// span of 64 x EPL elements (it only iterates for tensors beyond 2^31 - 1 spans); `first` is the lane's first element.
#define FO_SPAN_LOOP(N, EPL_, ALIGNED, CALL_FAST, CALL_SLOW)                                      \
    {                                                                                             \
        constexpr int64_t kSpan_ = 64 * (EPL_);                                                   \
        const int64_t n_spans_ = ((N) + kSpan_ - 1) / kSpan_;                                     \
        for (int64_t span_ = blockIdx.x; span_ < n_spans_; span_ += gridDim.x) {                  \
            const int64_t first = span_ * kSpan_ + (int64_t)threadIdx.x * (EPL_);                 \
            if ((ALIGNED) && (span_ + 1) * kSpan_ <= (N)) { CALL_FAST; } else { CALL_SLOW; }      \
        }                                                                                         \
    }

template <int DT, int ECCB>
__global__ __launch_bounds__(kCodecThreads) void ecc_split_kernel(const float* x, const void* narrow, void* ecc, int64_t n) {
    const bool aligned = ((((uintptr_t)narrow) | ((uintptr_t)ecc) | ((uintptr_t)x)) & 15u) == 0;
    FO_SPAN_LOOP(n, 4, aligned, (ecc_split_lane<DT, ECCB, true>(x, narrow, ecc, first, n)), (ecc_split_lane<DT, ECCB, false>(x, narrow, ecc, first, n)))
}

}  // namespace fo

namespace {
using namespace fo_host;

// A launch takes fewer than 2^32 work-items.
constexpr int64_t kMaxBlocks = UINT32_MAX / fo::kCodecThreads;

// One short-lived workgroup per span of 64 x EPL elements (one pass streams better than a persistent grid here).
unsigned grid_for(int64_t n, int epl) {
    const int64_t spans = (n + 64 * epl - 1) / (64 * epl);
    return (unsigned)(spans < kMaxBlocks ? spans : kMaxBlocks);
}

int32_t codec_flags(int is_signed, int do_sqrt, int softsign) {
    return (is_signed ? FO_CODEC_SIGNED : 0) | (do_sqrt ? FO_CODEC_SQRT : 0) | (softsign ? FO_CODEC_SOFTSIGN : 0);
}

// One launch's share of a job list: the jobs before `end` that have elements, and the workgroups they take together.
struct JobRange { int64_t end, blocks; };

// The jobs from `first` on that share a launch, at `per_block` elements to a workgroup; no job takes more than kMaxBlocks.
JobRange jobs_of_launch(const fo_convert_job* jobs, int64_t n_jobs, int64_t first, int64_t per_block) {
    JobRange r{first, 0};
    for (int count = 0; r.end < n_jobs; ++r.end) {
        const int64_t need = (jobs[r.end].n + per_block - 1) / per_block;
        if (need == 0) continue;
        if (count == fo::kJobsPerLaunch || r.blocks + need > kMaxBlocks) break;
        ++count;
        r.blocks += need;
    }
    return r;
}

// Enqueues the jobs, kJobsPerLaunch to a launch; the caller has checked their pointers.
template <class Op> int launch_jobs(const fo_convert_job* jobs, int64_t n_jobs, hipStream_t stream) {
    constexpr int64_t kBlock = fo::ConvertShape<Op>::kBlock;
    for (int64_t i = 0; i < n_jobs; ++i)
        if (jobs[i].n > kMaxBlocks * kBlock)
            return fail(FO_ERR_INVALID_ARGUMENT, "tensor too large for one launch (%lld elements, at most %lld)", (long long)jobs[i].n, (long long)(kMaxBlocks * kBlock));
    for (int64_t first = 0; first < n_jobs;) {
        const JobRange r = jobs_of_launch(jobs, n_jobs, first, kBlock);
        fo::JobBatch b;
        b.count = 0; b.reserved = 0;
        fo::u32 block = 0;
        for (; first < r.end; ++first) {
            if (jobs[first].n == 0) continue;
            b.job[b.count] = jobs[first];
            b.first_block[b.count++] = block;
            block += (fo::u32)((jobs[first].n + kBlock - 1) / kBlock);
        }
        if (r.blocks == 0) continue;
        hipLaunchKernelGGL(fo::convert_kernel<Op>, dim3((unsigned)r.blocks), dim3(fo::kCodecThreads), 0, stream, b);
        if (int rc = check_hip(hipGetLastError(), "conversion kernel launch")) return rc;
    }
    return 0;
}

// What every job list has to satisfy before a kernel sees its pointers: src, dst (and src2, dst2 where the kernel uses
// them) are there, each aligned to `*_align` bytes.  An align of 0 is an unused pointer.
int validate_jobs(const fo_convert_job* jobs, int64_t n_jobs, unsigned src_align, unsigned src2_align, unsigned dst_align, unsigned dst2_align) {
    if (n_jobs < 0) return fail(FO_ERR_INVALID_ARGUMENT, "negative job count");
    if (n_jobs > 0 && !jobs) return fail(FO_ERR_INVALID_ARGUMENT, "jobs must not be NULL");
    for (int64_t i = 0; i < n_jobs; ++i) {
        const fo_convert_job& j = jobs[i];
        if (j.n < 0) return fail(FO_ERR_INVALID_ARGUMENT, "n must be >= 0");
        if (j.n == 0) continue;
        const void* p[4] = {j.src, j.src2, j.dst, j.dst2};
        const unsigned align[4] = {src_align, src2_align, dst_align, dst2_align};
        for (int k = 0; k < 4; ++k) {
            if (!align[k]) continue;
            if (!p[k]) return fail(FO_ERR_INVALID_ARGUMENT, "job %lld: pointers must not be NULL", (long long)i);
            if ((uintptr_t)p[k] & (align[k] - 1)) return fail(FO_ERR_INVALID_ARGUMENT, "job %lld: pointer not aligned to its element size", (long long)i);
        }
    }
    if (n_jobs > 0 && compute_units() <= 0) return fail(FO_ERR_NO_DEVICE, "no HIP device");
    return 0;
}

}  // namespace

extern "C" {

int fo_quantize(const void* x, int x_dtype, void* codes, void* scales, int64_t n, int is_signed, int do_sqrt, int softsign,
                void* stream) {
    if (n < 0) return fail(FO_ERR_INVALID_ARGUMENT, "n must be >= 0");
    if (x_dtype < FO_F32 || x_dtype > FO_F16) return fail(FO_ERR_INVALID_ARGUMENT, "unknown dtype %d", x_dtype);
    if (n == 0) return 0;  // ref:2485
    if (!x || !codes || !scales) return fail(FO_ERR_INVALID_ARGUMENT, "x, codes and scales must not be NULL");
    if (((uintptr_t)x & (x_dtype == FO_F32 ? 3 : 1)) || ((uintptr_t)scales & 1)) return fail(FO_ERR_INVALID_ARGUMENT, "x or scales not aligned to their element size");
    const fo_convert_job job{x, nullptr, codes, scales, n, codec_flags(is_signed, do_sqrt, softsign), 0};
    return fo_quantize_many(&job, 1, x_dtype, stream);
}

int fo_quantize_many(const fo_convert_job* jobs, int64_t n_jobs, int x_dtype, void* stream) {
    if (x_dtype < FO_F32 || x_dtype > FO_F16) return fail(FO_ERR_INVALID_ARGUMENT, "unknown dtype %d", x_dtype);
    if (int rc = validate_jobs(jobs, n_jobs, x_dtype == FO_F32 ? 4 : 2, 0, 1, 2)) return rc;
    hipStream_t s = (hipStream_t)stream;
    switch (x_dtype) {
        case FO_F32: return launch_jobs<fo::QuantizeOp<fo::DT_F32>>(jobs, n_jobs, s);
        case FO_BF16: return launch_jobs<fo::QuantizeOp<fo::DT_BF16>>(jobs, n_jobs, s);
        default: return launch_jobs<fo::QuantizeOp<fo::DT_F16>>(jobs, n_jobs, s);
    }
}

int fo_dequantize(const void* codes, const void* scales, float* out, int64_t n, int is_signed, int do_sqrt, int softsign,
                  void* stream) {
    if (n < 0) return fail(FO_ERR_INVALID_ARGUMENT, "n must be >= 0");
    if (n == 0) return 0;  // ref:2533
    if (!codes || !scales || !out) return fail(FO_ERR_INVALID_ARGUMENT, "codes, scales and out must not be NULL");
    if (((uintptr_t)out & 3) || ((uintptr_t)scales & 1)) return fail(FO_ERR_INVALID_ARGUMENT, "out or scales not aligned to their element size");
    const fo_convert_job job{codes, scales, out, nullptr, n, codec_flags(is_signed, do_sqrt, softsign), 0};
    return fo_dequantize_many(&job, 1, FO_F32, stream);
}

int fo_dequantize_many(const fo_convert_job* jobs, int64_t n_jobs, int out_dtype, void* stream) {
    if (out_dtype != FO_F32 && out_dtype != FO_BF16) return fail(FO_ERR_INVALID_ARGUMENT, "output dtype must be fp32 or bf16 (got %d)", out_dtype);
    if (int rc = validate_jobs(jobs, n_jobs, 1, 2, out_dtype == FO_F32 ? 4 : 2, 0)) return rc;
    return out_dtype == FO_F32 ? launch_jobs<fo::DequantizeOp<fo::DT_F32>>(jobs, n_jobs, (hipStream_t)stream)
                               : launch_jobs<fo::DequantizeOp<fo::DT_BF16>>(jobs, n_jobs, (hipStream_t)stream);
}

int fo_int8_widen_many(const fo_convert_job* jobs, int64_t n_jobs, int dtype, void* stream) {
    if (dtype != FO_BF16 && dtype != FO_F16) return fail(FO_ERR_INVALID_ARGUMENT, "dtype must be bf16 or fp16 (got %d)", dtype);
    if (int rc = validate_jobs(jobs, n_jobs, 1, 0, 2, 0)) return rc;
    return dtype == FO_BF16 ? launch_jobs<fo::Int8WidenOp<fo::DT_BF16>>(jobs, n_jobs, (hipStream_t)stream)
                            : launch_jobs<fo::Int8WidenOp<fo::DT_F16>>(jobs, n_jobs, (hipStream_t)stream);
}

int fo_int8_narrow_many(const fo_convert_job* jobs, int64_t n_jobs, int dtype, void* stream) {
    if (dtype != FO_BF16 && dtype != FO_F16) return fail(FO_ERR_INVALID_ARGUMENT, "dtype must be bf16 or fp16 (got %d)", dtype);
    if (int rc = validate_jobs(jobs, n_jobs, 2, 0, 1, 0)) return rc;
    return dtype == FO_BF16 ? launch_jobs<fo::Int8NarrowOp<fo::DT_BF16>>(jobs, n_jobs, (hipStream_t)stream)
                            : launch_jobs<fo::Int8NarrowOp<fo::DT_F16>>(jobs, n_jobs, (hipStream_t)stream);
}

static int validate_ecc_args(const void* a, const void* b, const void* c, int narrow_dtype, int ecc_bytes, int64_t n) {
    if (n < 0) return fail(FO_ERR_INVALID_ARGUMENT, "n must be >= 0");
    if (narrow_dtype != FO_BF16 && narrow_dtype != FO_F16) return fail(FO_ERR_INVALID_ARGUMENT, "narrow dtype must be bf16 or fp16 (got %d)", narrow_dtype);  // ref:2858-2867, 2927-2930
    if (ecc_bytes != 1 && ecc_bytes != 2) return fail(FO_ERR_INVALID_ARGUMENT, "ecc_bytes must be 1 or 2 (got %d)", ecc_bytes);  // ref:2868-2869, 2944-2948
    if (n > 0 && (!a || !b || !c)) return fail(FO_ERR_INVALID_ARGUMENT, "NULL pointer");
    return 0;
}

#define FO_ECC_DISPATCH(KERNEL, ...)                                                                                     \
    if (narrow_dtype == FO_BF16 && ecc_bytes == 1) hipLaunchKernelGGL((fo::KERNEL<fo::DT_BF16, 1>), grid, block, 0, s, __VA_ARGS__); \
    else if (narrow_dtype == FO_BF16) hipLaunchKernelGGL((fo::KERNEL<fo::DT_BF16, 2>), grid, block, 0, s, __VA_ARGS__);  \
    else if (ecc_bytes == 1) hipLaunchKernelGGL((fo::KERNEL<fo::DT_F16, 1>), grid, block, 0, s, __VA_ARGS__);            \
    else hipLaunchKernelGGL((fo::KERNEL<fo::DT_F16, 2>), grid, block, 0, s, __VA_ARGS__);

#define FO_ECC_JOBS(OP)                                                                                                        \
    if (narrow_dtype == FO_BF16) {                                                                                             \
        return ecc_bytes == 1 ? launch_jobs<fo::OP<fo::DT_BF16, 1>>(jobs, n_jobs, (hipStream_t)stream)                         \
                              : launch_jobs<fo::OP<fo::DT_BF16, 2>>(jobs, n_jobs, (hipStream_t)stream);                        \
    }                                                                                                                          \
    return ecc_bytes == 1 ? launch_jobs<fo::OP<fo::DT_F16, 1>>(jobs, n_jobs, (hipStream_t)stream)                              \
                          : launch_jobs<fo::OP<fo::DT_F16, 2>>(jobs, n_jobs, (hipStream_t)stream);

int fo_ecc_join(const void* narrow, int narrow_dtype, const void* ecc, int ecc_bytes, float* out, int64_t n, void* stream) {
    if (int rc = validate_ecc_args(narrow, ecc, out, narrow_dtype, ecc_bytes, n)) return rc;
    if (n == 0) return 0;
    const fo_convert_job job{narrow, ecc, out, nullptr, n, 0, 0};
    return fo_ecc_join_many(&job, 1, narrow_dtype, ecc_bytes, stream);
}

int fo_ecc_join_many(const fo_convert_job* jobs, int64_t n_jobs, int narrow_dtype, int ecc_bytes, void* stream) {
    if (int rc = validate_ecc_args(nullptr, nullptr, nullptr, narrow_dtype, ecc_bytes, 0)) return rc;
    if (int rc = validate_jobs(jobs, n_jobs, 2, (unsigned)ecc_bytes, 4, 0)) return rc;
    FO_ECC_JOBS(EccJoinOp)
}

int fo_ecc_split(const float* x, const void* narrow, int narrow_dtype, void* ecc, int ecc_bytes, int64_t n, void* stream) {
    if (int rc = validate_ecc_args(x, narrow, ecc, narrow_dtype, ecc_bytes, n)) return rc;
    if (n == 0) return 0;
    if (((uintptr_t)narrow & 1) || ((uintptr_t)x & 3) || (ecc_bytes == 2 && ((uintptr_t)ecc & 1))) return fail(FO_ERR_INVALID_ARGUMENT, "pointer not aligned to its element size");
    if (compute_units() <= 0) return fail(FO_ERR_NO_DEVICE, "no HIP device");
    const dim3 grid(grid_for(n, 4)), block(fo::kCodecThreads);
    hipStream_t s = (hipStream_t)stream;
    FO_ECC_DISPATCH(ecc_split_kernel, x, narrow, ecc, n)
    return check_hip(hipGetLastError(), "ecc split kernel launch");
}

int fo_ecc_narrow_many(const fo_convert_job* jobs, int64_t n_jobs, int narrow_dtype, int ecc_bytes, void* stream) {
    if (int rc = validate_ecc_args(nullptr, nullptr, nullptr, narrow_dtype, ecc_bytes, 0)) return rc;
    if (int rc = validate_jobs(jobs, n_jobs, 4, 0, 2, (unsigned)ecc_bytes)) return rc;
    FO_ECC_JOBS(EccNarrowOp)
}

#ifdef FO_DIAG
int fo_conversion_launch(const fo_convert_job* jobs, int64_t n_jobs, int64_t first, int64_t elements_per_workgroup, int64_t* workgroups) {
    const JobRange r = jobs_of_launch(jobs, n_jobs, first, elements_per_workgroup);
    if (workgroups) *workgroups = r.blocks;
    return (int)(r.end - first);
}
#endif  // FO_DIAG

}  // extern "C"
