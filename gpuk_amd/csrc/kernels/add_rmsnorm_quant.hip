// residual-add -> RMSNorm -> (optional) FP8 e4m3fn quantisation, one workgroup per token row.
//
// This is the one-GPU share of the reference's all-reduce-fusion epilogue: the residual add at
// src/impl/all_reduce_fusion_impl.h:256-265 followed by epilogue<>() at :202-228 (rms_norm :159-181,
// reduce_abs_max :183-200, convert_to_fp8 :148-157), reached through the allreduce_rms host op
// (src/ops/all_reduce_fusion.cpp:363-396).  There is no all-reduce here.
//
// Numerics follow the reference's torch oracle (gpuk/__init__.py:147-164) op by op, *not* the
// reference kernel (which keeps fp32 until the fp8 cast):
//     res  = rT(x + r)                       rT = round-to-nearest-even into the 16-bit type
//     var  = sum(res^2) / H ; rstd = 1 / sqrt(var + eps)          (correctly rounded sqrt and divide)
//     n1   = rT(res * rstd) ; n2 = rT(gamma * n1)
//     scale = amax|n2| / fp8_max  (1 when the row is all zero, as the reference kernel: :217)
//     code = e4m3fn_rne(clamp(n2 / scale, +-fp8_max))             (fp32 IEEE quotient)
//
// Data movement per element: 2 B x + 2 B residual in, 2 B residual out, 1 B code (7 B); the row lives
// in registers between the three phases, so HBM sees each byte once.  Lane `t` of the workgroup owns
// 16-byte chunk `i*blockDim + t` of the row for i < NCHUNK (counted from the line boundary before the row where the row
// starts inside a line, see line_pad): every wave load/store instruction covers 1 KiB (loads) or 512 B (codes) of
// contiguous memory.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../../include/gpuk_amd.h"
#include "device_utils.h"
#include "host_utils.h"

namespace gpuk {

namespace {

constexpr int kMaxThreads = 1024;
constexpr int kMaxChunks = 8, kMaxChunksF32 = 4;  // chunks per lane the kernels of 16-bit and of fp32 rows have forms for

template <typename P>
__device__ __forceinline__ auto load_stream(P p) { return __builtin_nontemporal_load(p); }
template <typename P, typename V>
__device__ __forceinline__ void store_stream(P p, V v) { __builtin_nontemporal_store(v, p); }

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The scale reciprocal is usable by div_by_rcp when scale is comfortably normal.
__device__ __forceinline__ bool scale_in_fast_range(float s) {
    return s >= 0x1p-60f && s <= 0x1p60f;
}

// 1 / sqrt(sumsq / H + eps).  The mean as an exact IEEE quotient by multiply and two fused multiply-adds (exact on the guarded
// range, see div_by_rcp), then the short square root and reciprocal.  Every wave of a row walks this dependent chain before it
// can go on: one test behind it, and what any of the three is not made for takes the general operations.  A sum in the middle
// of the exponent range leaves the mean in [2^-91, 2^60) and, with an eps in [0, 2^60], the other two in theirs; sum_range is
// 0 for any other eps, so that no sum passes.
constexpr uint32_t kSumsFrom = 0x21800000u, kSumRange = 0x3c000000u;  // [2^-60, 2^60), see in_mid_range
__device__ __forceinline__ float row_rstd(float sumsq, float hidden_f, float rcp_hidden, float eps, uint32_t sum_range) {
    const float root = sqrt_rn_mid_range(div_by_rcp_finite(sumsq, hidden_f, rcp_hidden) + eps);
    const bool usual = __builtin_bit_cast(uint32_t, sumsq) - kSumsFrom < sum_range && !mantissa_all_ones(root);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!usual) == 0, 1)) return rcp_rn_mid_range(root);
    return 1.0f / sqrtf(sumsq / hidden_f + eps);
}

// scale = amax / fp8_max, 1 for an all-zero row; *fast: quotients by it take the short form.  rcp_fp8_max: see
// reciprocal_of_max.  One test decides for the common maxima, whose scales are then in the fast range and never have a
// significand of ones.
__device__ __forceinline__ float dynamic_scale(float amax, float fp8_max, float rcp_fp8_max, bool *fast) {
    const bool usual = __builtin_bit_cast(uint32_t, amax) - 0x26800000u < 0x37000000u && rcp_fp8_max > 0.f;  // amax in [2^-50, 2^60)
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!usual) == 0, 1)) {
        *fast = true;
        return div_by_rcp_finite(amax, fp8_max, rcp_fp8_max);
    }
    const float scale = amax == 0.f ? 1.f : amax / fp8_max;
    *fast = __builtin_amdgcn_ballot_w64(!(scale_in_fast_range(scale) && !mantissa_all_ones(scale) && rcp_fp8_max >= 0.f)) == 0;
    return scale;
}

// The parameters of the kernels of rows that stay in registers, ordered by when a wave needs them: the first fourteen dwords
// are handed to the wave in scalar registers at launch (-amdgpu-kernarg-preload-count), so that the loads of the row are
// issued without a round trip for the argument block.  They come as three vectors and a struct, not sixteen scalars: see
// launch_kernel (one row of 7168 elements, quantised, a call of the operator 5.36 / 4.79 us).
//   first:  x, residual_in, chunks_per_row, remap_end, lanes_and_shift, gate
//   second: gamma, residual_out
//   third:  norm_out
struct RowArgs {
    float *scale_io;
    float hidden_f, rcp_hidden, eps;
    uint32_t sum_range;  // see row_rstd
    float fp8_max, rcp_fp8_max;
};
static_assert(sizeof(u32x8) + sizeof(u32x4) + sizeof(u32x2) + sizeof(RowArgs) <= 112, "see launch_kernel");

// What a launch passes beside the workgroup size (lanes_and_shift, one argument register): lanes in bits 0-15, the row-run
// shift in bits 16-23, the mask of line_pad in bits 24-31.
__device__ __forceinline__ int lanes_of(uint32_t lanes_and_shift) { return (int)(lanes_and_shift & 0xffffu); }
__device__ __forceinline__ int shift_of(uint32_t lanes_and_shift) { return (int)((lanes_and_shift >> 16) & 0xffu); }
// Chunks by which a row's first one lies behind a line boundary.  The lanes of a row whose length is no multiple of a line
// start at the boundary, not at the row (the first `pad` of them idle), so that a wave's accesses cover whole lines but
// for the row's two ends: started at the row itself, every one of them splits its first and last line with the next wave,
// whose streamed access fetches or writes it again.  Multiples of 16 chunks, which are whole lines of codes as well, or of 8
// where the workgroup has no more lanes to spare: see line_mask.
// Lanes from the row's start / from the line: 16384 rows of 9000 elements 184.1 / 168.0 us, of 2568 55.1 / 50.3, of 7176 145.4 /
// 141.9; 8192 fp32 rows of 9000 181.5 / 165.2, of 2568 56.0 / 49.5; batches of a few hundred rows level.
// Rows of one chunk per lane that do not gate their stores stay at the row: small batches, which the arithmetic ahead of the
// first load costs more than it gains (one row of 1032 2.09 / 2.13 us, of 3208 2.44 / 2.48, one fp32 row of 2056 2.20 / 2.23; 40000
// rows of 264 19.4 / 19.4).  Behind a gate it costs nothing (1280 fp32 rows of 1032 without codes 5.30 / 5.15).  Half precision, where
// the two forms are level, keeps it throughout.
__device__ __forceinline__ int line_pad(uint32_t x_low, int64_t row_base, uint32_t lanes_and_shift) {
    return (int)(((x_low >> 4) + (uint32_t)row_base) & (lanes_and_shift >> 24));
}

// Two neighbouring elements of the normed row, rT(gamma * rT(res * rstd)), packed.
template <typename T>
__device__ __forceinline__ uint32_t normed_pair(uint32_t gamma, uint32_t res, float rstd) {
    using P = Pack16<T>;
    if constexpr (is_half<T>) return P::mul(gamma, P::scale_round(res, rstd));
    else return P::pack(P::lo(gamma) * P::round(P::lo(res) * rstd), P::hi(gamma) * P::round(P::hi(res) * rstd));
}

// The codes of one chunk by plain IEEE division, for scales so small or large (or not a number) that a reciprocal
// leaves the normal range.  Kept out of line: it is long (eight expanded divisions and clamps), it is almost never
// taken, and inlined it sat between the kernel's last two stretches of common-path code, which a wave then reached
// by a jump into instructions no prefetch had brought in.
typedef float f32x8 __attribute__((ext_vector_type(8)));
__device__ __attribute__((noinline)) u32x2 codes_by_division(f32x8 n, float scale, float fp8_max) {  // by value: in registers
    float q[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = clamp_sym(n[j] / scale, fp8_max);
    return u32x2{cvt4_e4m3fn(q[0], q[1], q[2], q[3]), cvt4_e4m3fn(q[4], q[5], q[6], q[7])};
}

// EXACT: lanes x NCHUNK equals the chunks of a row, so every lane owns NCHUNK live chunks and nothing is masked
// (true for every power-of-two row and for 7168 elements; it removes a sixth of the kernel's instructions, which is
// what a decode-sized batch waits for: with at most one row per compute unit the run time is the row's arithmetic).
// LANDED: the weights are asked for once the lane's row has landed, and the reduction hides them.  What bounds a row that has a
// compute unit to itself is that unit's path to the caches, 64 bytes a clock: asked for at once, the weights of its first waves
// go ahead of the rows of its last, and every wave waits for the last one's squares (one row of 16384 elements: the last wave's
// loads left 0.79 us after entry, a row's bytes take 0.47).  us, at once / landed, bf16: 40 rows of 7168 elements, dynamic scale,
// 3.59 / 3.54, 220 4.41 / 4.18, static 4.34 / 3.97, without codes 4.22 / 3.73; 90 of 14336 5.43 / 5.02, 5.27 / 4.77 and 4.79 / 4.29;
// fp16 40 of 12288 4.26 / 3.98, 4.10 / 3.84 and 3.70 / 3.44.  Which launches take it: see late_weights.
template <typename T, int NCHUNK, int QUANT, bool EXACT, bool GATED, bool LANDED>
__global__ void __launch_bounds__(kMaxThreads) __attribute__((amdgpu_waves_per_eu(GATED && NCHUNK <= 4 ? 8 : 4)))
add_rmsnorm_quant_rows(const u32x8 first, const u32x4 second, const u32x2 third, const RowArgs rest) {
    Global<const u32x4> *x = global_ptr<const u32x4>(first[0], first[1]), *residual_in = global_ptr<const u32x4>(first[2], first[3]);
    const int chunks_per_row = (int)first[4], remap_end = (int)first[5];
    const uint32_t lanes_and_shift = first[6], gate = first[7];  // (see lanes_of: the workgroup size need not be fetched from the dispatch packet)
    Global<const u32x4> *gamma = global_ptr<const u32x4>(second[0], second[1]);
    Global<u32x4> *residual_out = global_ptr<u32x4>(second[2], second[3]);
    Global<char> *norm_out = global_ptr<char>(third[0], third[1]);
    float *scale_io = rest.scale_io;
    const float hidden_f = rest.hidden_f, rcp_hidden = rest.rcp_hidden, eps = rest.eps, fp8_max = rest.fp8_max, rcp_fp8_max = rest.rcp_fp8_max;
    const int nthreads = lanes_of(lanes_and_shift), group_shift = shift_of(lanes_and_shift);
    using P = Pack16<T>;
    __shared__ float s_sum[kReduceSlots];
    __shared__ float s_max[kReduceSlots];
    GPUK_STAMPS_BEGIN();  // profiling build only
    // GATED (batches whose rows are all resident at once): no store before `gate` ticks of 10 ns after the wave's
    // entry, the time the launch's reads take; the chip then reads in the first part of the launch and writes in the
    // second instead of mixing the two, which the memory system charges for.  The residual is stored with the codes.
    // (A template parameter: as a run-time choice the branches around the early stores cost the large batches 1 %.)
    const uint64_t entry = GATED ? __builtin_amdgcn_s_memrealtime() : 0;

    const int tid = threadIdx.x;
    const int num_waves = nthreads >> 6;
    // Workgroup ids are handed to the 8 XCDs round-robin.  Below remap_end the rows are dealt out in runs of
    // 2^group_shift consecutive rows per XCD instead of one row each (which rows run concurrently stays the same;
    // which XCD's L2 and fabric port each row goes through changes).
    int row = blockIdx.x;
    if (row < remap_end) {
        const int xcd = row & 7, idx = row >> 3;
        row = ((((idx >> group_shift) << 3) | xcd) << group_shift) | (idx & ((1 << group_shift) - 1));
    }
    int64_t row_base = (int64_t)row * chunks_per_row;
    const int pad = EXACT || (NCHUNK == 1 && !GATED && !is_half<T>) ? 0 : line_pad(first[0], row_base, lanes_and_shift);
    row_base -= pad;  // where lane 0 stands: a lane's chunk c is chunk c - pad of the row

    // ---- phase 0: issue every load of the row before touching any of them.  The row is loaded whole before any of
    // it is stored, so residual_out may be the same buffer as residual_in or x.
    u32x4 xv[NCHUNK], rv[NCHUNK], gv[NCHUNK];
    bool live[NCHUNK];
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
        const int c = i * nthreads + tid;
        live[i] = EXACT || (uint32_t)(c - pad) < (uint32_t)chunks_per_row;
        if (live[i]) {
            xv[i] = load_stream(x + row_base + c);
            rv[i] = load_stream(residual_in + row_base + c);
        } else {
            xv[i] = u32x4{0, 0, 0, 0};
            rv[i] = u32x4{0, 0, 0, 0};
        }
    }
    auto load_weights = [&]() {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) gv[i] = live[i] ? (gamma - pad)[i * nthreads + tid] : u32x4{0, 0, 0, 0};
    };
    if constexpr (!LANDED) load_weights();
    // The arguments beyond the preloaded ones are fetched here, behind the row's loads and while those are in flight:
    // left to itself the compiler fetches them where they are first used, after the first barrier, and every wave of
    // the row then waits there for the scalar cache (0.1-0.15 us of a decode-sized call).
    asm volatile("" ::"s"(hidden_f), "s"(rcp_hidden), "s"(eps), "s"(rest.sum_range));
    if constexpr (QUANT != GPUK_QUANT_NONE) asm volatile("" ::"s"(fp8_max));
    if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) asm volatile("" ::"s"(rcp_fp8_max), "s"(scale_io));
    // ... and so is the static scale, which the kernel only reads (asked for here, needed in phase 3: fetched where it
    // is first used it put a round trip through the scalar cache between the last two phases)
    float static_scale = 0.f;
    if constexpr (QUANT == GPUK_QUANT_FP8_STATIC) static_scale = *(const __attribute__((address_space(4))) float *)scale_io;
    GPUK_STAMP(1);          // every load issued
    GPUK_STAMP_DRAINED(2);  // ... and landed

    // ---- phase 1: res = rT(x + r), stored once; sum of squares of the *rounded* residual.  Waves in this phase
    // are given issue priority over the arithmetic of phases 2-3 so that their residual stores leave early (+0.4 %).
    __builtin_amdgcn_s_setprio(1);
    if constexpr (LANDED) {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) asm volatile("" : "+v"(xv[i]), "+v"(rv[i]));
        load_weights();
        __builtin_amdgcn_sched_barrier(0);
    }
    // (A partial sum takes the squares of no more than two chunks: a row's sum in four chunks per lane is then as close to that in
    // 64 bits as in two, over 1536 rows of 8192 bfloat16 elements 3.9e-8 off in the mean square (4.4e-8 with two sums, two chunks 4.0e-8).)
    constexpr int kSums = NCHUNK >= 4 ? 4 : 2;
    float ss[kSums] = {};
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t w;
            if constexpr (is_half<T>) w = P::add(xv[i][j], rv[i][j]);
            else w = P::pack(P::lo(xv[i][j]) + P::lo(rv[i][j]), P::hi(xv[i][j]) + P::hi(rv[i][j]));
            xv[i][j] = w;  // xv now holds the residual
            float &sum = ss[(2 * i + (j & 1)) % kSums];
            sum = P::add_squares(w, sum);
        }
        if (!GATED && live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
    }
    if constexpr (GATED && NCHUNK == 4) {  // (the packed residual is what stays in registers, not the sums it was rounded from)
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(xv[i][j]));
    }
    if constexpr (QUANT == GPUK_QUANT_FP8_STATIC) asm volatile("" ::"s"(static_scale));  // (it has arrived by now)
    GPUK_STAMP(3);  // residual stored, the lane's squares summed
    // kUnpacked: the row and the weights are unpacked behind the wave's own part of the reduction, while it has the others to wait
    // for, and not in phase 2, where all waves of the row (two on most SIMDs of the only compute unit that a decode row has) issue
    // at once: one row of 16384 elements 4.11 / 4.02 us, 32 of 4096 2.89 / 2.85.  Without codes, whose only chain behind the
    // reduction is a store, it costs as much as it gains (256 rows of 4096 3.10 / 3.16), and four chunks per lane have no registers
    // for it.  Weights that were asked for late stay packed: a wave that unpacked them there would reach the barrier later (static
    // scale, 90 rows of 14336 4.85 / 4.77, 133 of 7168 3.64 / 3.62).
    constexpr bool kUnpacked = !is_half<T> && NCHUNK <= 2 && QUANT != GPUK_QUANT_NONE, kWeightsUnpacked = kUnpacked && !LANDED;
    float res[kUnpacked ? NCHUNK : 1][8], weight[kWeightsUnpacked ? NCHUNK : 1][8];
    SplitReciprocal rcp{};  // of the scale; `fast`: quotients take the short form
    bool fast = false;
    float lane_sum = ss[0] + ss[1];
    if constexpr (kSums == 4) lane_sum += ss[2] + ss[3];
    const float sumsq = block_allreduce<SumOp>(lane_sum, s_sum, num_waves, [&] {
        if constexpr (QUANT == GPUK_QUANT_FP8_STATIC) {
            fast = __builtin_amdgcn_ballot_w64(!(scale_in_fast_range(static_scale) && !mantissa_all_ones(static_scale))) == 0;
            rcp = split_reciprocal(static_scale);
            asm volatile("" : "+v"(rcp.hi), "+v"(rcp.lo));
        }
        if constexpr (kUnpacked) {
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    res[i][2 * j] = P::lo(xv[i][j]), res[i][2 * j + 1] = P::hi(xv[i][j]);
                    asm volatile("" : "+v"(res[i][2 * j]), "+v"(res[i][2 * j + 1]));
                    if constexpr (kWeightsUnpacked) {
                        weight[i][2 * j] = P::lo(gv[i][j]), weight[i][2 * j + 1] = P::hi(gv[i][j]);
                        asm volatile("" : "+v"(weight[i][2 * j]), "+v"(weight[i][2 * j + 1]));
                    }
                }
        }
    });
    // element e of the normed chunk i, rT(gamma * rT(res * rstd)), ahead of the last rounding
    const auto unrounded = [&](int i, int e, float rstd) {
        if constexpr (kWeightsUnpacked) return weight[i][e] * P::round(res[i][e] * rstd);
        else if constexpr (kUnpacked) return ((e & 1) ? P::hi(gv[i][e >> 1]) : P::lo(gv[i][e >> 1])) * P::round(res[i][e] * rstd);
        else return 0.f;
    };
    __builtin_amdgcn_s_setprio(0);
    GPUK_STAMP(4);  // sum of squares of the row known to every wave

    // ---- phase 2: n2 = rT(gamma * rT(res * rstd)); row amax for the dynamic scale.
    const float rstd = row_rstd(sumsq, hidden_f, rcp_hidden, eps, rest.sum_range);
    GPUK_STAMP(5);  // rstd
    if constexpr (QUANT == GPUK_QUANT_NONE) {
        auto *out = (Global<u32x4> *)norm_out + row_base;
        u32x4 normed[NCHUNK];
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                normed[i][j] = normed_pair<T>(gv[i][j], xv[i][j], rstd);
            }
            if (!GATED && live[i]) store_stream(out + i * nthreads + tid, normed[i]);
        }
        if constexpr (GATED) {
            // (the values to store are pinned down ahead of the wait: nothing ties the arithmetic to the clock, and the
            // compiler otherwise moves it behind the wait)
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i) asm volatile("" ::"v"(normed[i]));
            while (__builtin_amdgcn_s_memrealtime() < entry + gate) __builtin_amdgcn_s_sleep(1);
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i)
                if (live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i)
                if (live[i]) store_stream(out + i * nthreads + tid, normed[i]);
        }
        GPUK_STAMP(9);
        GPUK_STAMP_DRAINED(10);
        GPUK_STAMPS_WRITE(blockIdx.x * num_waves + (tid >> 6));
        return;
    } else {
        // the normed row stays in fp32 registers, every value already rounded to the 16-bit type.
        // (v_maximum3_f32 keeps a NaN, as the reference's amax does; tracked apart from v_max3_f32 it took a comparison per pair)
        // (kPacked, the gated four-chunk form: as 16-bit pairs instead, half the registers, so that eight waves fit a
        // SIMD with the residual kept for the gate as well; unpacked again in phase 3.  Half precision: always, its
        // arithmetic is packed and reads either half of a dword where bfloat16 needs an instruction to unpack it;
        // unpacked, the kernel took 410 vector instructions per wave at two chunks per lane and the four-chunk form
        // spilled: 4000 x 5120 ran in 34.3 us where bfloat16 takes 23.7; now 24.8, and 2000 x 7168 in 17.3
        // against 22.2)
        constexpr bool kPacked = (GATED && NCHUNK == 4) || is_half<T>;
        float nv[kPacked ? 1 : NCHUNK][8];
        uint32_t nw[kPacked ? NCHUNK : 1][4];
        float m0 = 0.f, m1 = 0.f;
        uint32_t half_max = 0;  // (half precision: both halves' largest magnitude, a NaN beating every number)
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float lo, hi;
                if constexpr (is_half<T>) {
                    nw[i][j] = normed_pair<T>(gv[i][j], xv[i][j], rstd);
                    if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) half_max = P::max_abs(half_max, nw[i][j]);
                    continue;
                } else if constexpr (kPacked) {
                    nw[i][j] = normed_pair<T>(gv[i][j], xv[i][j], rstd);
                    lo = P::lo(nw[i][j]);
                    hi = P::hi(nw[i][j]);
                } else {
                    if constexpr (kUnpacked) {
                        lo = P::round(unrounded(i, 2 * j, rstd));
                        hi = P::round(unrounded(i, 2 * j + 1, rstd));
                    } else {
                        lo = P::round(P::lo(gv[i][j]) * P::round(P::lo(xv[i][j]) * rstd));
                        hi = P::round(P::hi(gv[i][j]) * P::round(P::hi(xv[i][j]) * rstd));
                    }
                    nv[i][2 * j] = lo;
                    nv[i][2 * j + 1] = hi;
                }
                if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) {
                    if (j & 1) m1 = maximum3_abs(m1, lo, hi);
                    else m0 = maximum3_abs(m0, lo, hi);
                }
            }
        }
        float scale = static_scale;
        GPUK_STAMP(6);  // row normed, the lane's maximum known
        if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) {
            float amax = MaxOp::apply(m0, m1);
            if constexpr (is_half<T>) amax = MaxOp::apply(P::lo(half_max), P::hi(half_max));
            amax = block_allreduce<MaxOp>(amax, s_max, num_waves);
            GPUK_STAMP(7);  // row maximum known to every wave
            scale = dynamic_scale(amax, fp8_max, rcp_fp8_max, &fast);
            if (tid == 0) scale_io[row] = scale;
            rcp = split_reciprocal(scale);
        }

        // ---- phase 3: code = e4m3fn(clamp(n2 / scale)), 8 codes per chunk.  The quotient is the short one with the same
        // code (see SplitReciprocal; one row of 7168 elements, dynamic, 2.95 / 2.85 us with the correctly rounded quotient / this
        // one, 512 rows 5.85 / 5.74; with a static scale, whose reciprocal is taken while the wave waits at the first barrier,
        // 128 rows of 4096 3.24 / 3.13).  With the dynamic scale every value is finite and |n2 / scale| exceeds fp8_max by at
        // most one ULP, which the converter rounds to the same code: no clamp.  (Maxima where it does not, see
        // reciprocal_of_max, take the other path, which clamps.)  The static scale may meet anything: clamp; infinite and NaN
        // numerators come through the short quotient as through a division.
        constexpr bool kDynamic = QUANT == GPUK_QUANT_FP8_DYNAMIC;
        auto *out = (Global<u32x2> *)norm_out + row_base;
        if constexpr (kPacked && !is_half<T>) {  // (or the compiler keeps phase 2's unpacked copies alive instead)
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(nw[i][j]));
        }
        // (the scale is the same in every lane; deciding by ballot tells the compiler so, and the common path is
        // laid out as straight-line code with the other one out of the way)
        if (__builtin_expect(fast, 1)) {
            GPUK_STAMP(8);  // scale and its reciprocal
            u32x2 codes[NCHUNK];
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i) {
                float q[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if constexpr (is_half<T>) {  // (the numerator read in place)
                        const uint32_t w = nw[i][j >> 1];
                        q[j] = (j & 1) ? P::fma_hi(w, rcp.hi, P::mul_hi(w, rcp.lo)) : P::fma_lo(w, rcp.hi, P::mul_lo(w, rcp.lo));
                        continue;
                    }
                    float n;
                    if constexpr (kPacked) n = (j & 1) ? P::hi(nw[i][j >> 1]) : P::lo(nw[i][j >> 1]);
                    else n = nv[i][j];
                    q[j] = __builtin_fmaf(n, rcp.hi, n * rcp.lo);
                }
                if constexpr (!kDynamic) clamp8_sym(q, fp8_max);
                codes[i] = u32x2{cvt4_e4m3fn(q[0], q[1], q[2], q[3]), cvt4_e4m3fn(q[4], q[5], q[6], q[7])};
                if (!GATED && live[i]) store_stream(out + i * nthreads + tid, codes[i]);
            }
            if constexpr (GATED) {
#pragma unroll
                for (int i = 0; i < NCHUNK; ++i) asm volatile("" ::"v"(codes[i]));  // computed ahead of the wait, as above
                while (__builtin_amdgcn_s_memrealtime() < entry + gate) __builtin_amdgcn_s_sleep(1);
#pragma unroll
                for (int i = 0; i < NCHUNK; ++i)
                    if (live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
#pragma unroll
                for (int i = 0; i < NCHUNK; ++i)
                    if (live[i]) store_stream(out + i * nthreads + tid, codes[i]);
            }
        } else {
            if constexpr (GATED) {  // (no wait on this path: it is taken by rows whose scale is degenerate)
#pragma unroll
                for (int i = 0; i < NCHUNK; ++i)
                    if (live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
            }
            // (unrolled like the common path: a runtime index into the register arrays would move them to scratch)
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i) {
                f32x8 n;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if constexpr (kPacked) n[j] = (j & 1) ? P::hi(nw[i][j >> 1]) : P::lo(nw[i][j >> 1]);
                    else n[j] = nv[i][j];
                }
                const u32x2 codes = codes_by_division(n, scale, fp8_max);
                if (live[i]) store_stream(out + i * nthreads + tid, codes);
            }
        }
        GPUK_STAMP(9);           // codes stored (issued)
        GPUK_STAMP_DRAINED(10);  // every store of the wave acknowledged
        GPUK_STAMPS_WRITE(blockIdx.x * num_waves + (tid >> 6));
    }
}

// Calibration: the memory traffic of add_rmsnorm_quant_rows without its arithmetic.  Same launch shape, lane-to-chunk
// mapping, row-to-workgroup mapping, streaming loads and stores and the same two workgroup barriers; the "residual"
// is x ^ r and the "codes" fold it to half its size.  What this kernel reaches is the ceiling of the access pattern.
template <int NCHUNK>
__global__ void __launch_bounds__(kMaxThreads)
add_rmsnorm_quant_traffic_only(const u32x4 *x, const u32x4 *residual_in, int chunks_per_row, int remap_end,
                               uint32_t lanes_and_shift, uint32_t gate, u32x4 *residual_out, u32x2 *codes,
                               float *__restrict__ scale_out) {
    const int nthreads = lanes_of(lanes_and_shift), group_shift = shift_of(lanes_and_shift);
    const uint64_t entry = __builtin_amdgcn_s_memrealtime();  // the kernel's store gate, see there
    const int tid = threadIdx.x;  // arguments in the order of add_rmsnorm_quant_rows: the same ones arrive in registers
    int row = blockIdx.x;
    if (row < remap_end) {
        const int xcd = row & 7, idx = row >> 3;
        row = ((((idx >> group_shift) << 3) | xcd) << group_shift) | (idx & ((1 << group_shift) - 1));
    }
    int64_t row_base = (int64_t)row * chunks_per_row;
    const int pad = line_pad((uint32_t)(uintptr_t)x, row_base, lanes_and_shift);
    row_base -= pad;
    u32x4 xv[NCHUNK], rv[NCHUNK];
    bool live[NCHUNK];
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
        const int c = i * nthreads + tid;
        live[i] = (uint32_t)(c - pad) < (uint32_t)chunks_per_row;
        xv[i] = live[i] ? load_stream(x + row_base + c) : u32x4{0, 0, 0, 0};
        rv[i] = live[i] ? load_stream(residual_in + row_base + c) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
        xv[i] ^= rv[i];
        if (!gate && live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
    }
    __syncthreads();
    __syncthreads();
    if (gate) {
        while (__builtin_amdgcn_s_memrealtime() < entry + gate) __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i)
            if (live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
    }
    if (tid == 0) scale_out[row] = 1.0f;
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
        const u32x2 folded = {xv[i][0] + xv[i][1], xv[i][2] + xv[i][3]};
        if (live[i]) store_stream(codes + row_base + i * nthreads + tid, folded);
    }
}

// Rows too long to keep in registers (more than 8 chunks per lane at 1024 lanes, i.e. hidden > 65536):
// three sweeps over the row, re-reading what this same lane wrote to residual_out (L2-resident).
template <typename T, int QUANT>
__global__ void __launch_bounds__(kMaxThreads)
add_rmsnorm_quant_long_rows(const u32x4 *x, const u32x4 *residual_in,  // either may be residual_out: no __restrict__
                            const u32x4 *__restrict__ gamma, u32x4 *residual_out, void *norm_out,
                            float *__restrict__ scale_io, int chunks_per_row, float hidden_f, float eps,
                            float fp8_max) {
    using P = Pack16<T>;
    __shared__ float s_sum[kReduceSlots];
    __shared__ float s_max[kReduceSlots];
    const int tid = threadIdx.x;
    const int num_waves = blockDim.x >> 6;
    const int64_t row_base = (int64_t)blockIdx.x * chunks_per_row;

    float ss = 0.f;
    for (int c = tid; c < chunks_per_row; c += blockDim.x) {
        u32x4 xv = x[row_base + c], rv = residual_in[row_base + c];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t w = P::pack(P::lo(xv[j]) + P::lo(rv[j]), P::hi(xv[j]) + P::hi(rv[j]));
            xv[j] = w;
            ss = __builtin_fmaf(P::lo(w), P::lo(w), ss);
            ss = __builtin_fmaf(P::hi(w), P::hi(w), ss);
        }
        residual_out[row_base + c] = xv;
    }
    const float sumsq = block_allreduce<SumOp>(ss, s_sum, num_waves);
    const float rstd = 1.0f / sqrtf(sumsq / hidden_f + eps);

    auto normed = [&](int c) {
        u32x4 v = residual_out[row_base + c];  // written by this lane above
        const u32x4 g = gamma[c];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t n1 = P::pack(P::lo(v[j]) * rstd, P::hi(v[j]) * rstd);
            v[j] = P::pack(P::lo(g[j]) * P::lo(n1), P::hi(g[j]) * P::hi(n1));
        }
        return v;
    };

    if constexpr (QUANT == GPUK_QUANT_NONE) {
        u32x4 *out = reinterpret_cast<u32x4 *>(norm_out) + row_base;
        for (int c = tid; c < chunks_per_row; c += blockDim.x) out[c] = normed(c);
    } else {
        float scale;
        if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) {
            float amax = 0.f;
            for (int c = tid; c < chunks_per_row; c += blockDim.x) {
                const u32x4 v = normed(c);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    amax = MaxOp::apply(amax, __builtin_fabsf(P::lo(v[j])));  // keeps a NaN, like the reference's amax
                    amax = MaxOp::apply(amax, __builtin_fabsf(P::hi(v[j])));
                }
            }
            amax = block_allreduce<MaxOp>(amax, s_max, num_waves);
            scale = amax == 0.f ? 1.f : amax / fp8_max;
            if (tid == 0) scale_io[blockIdx.x] = scale;
        } else {
            scale = scale_io[0];
        }
        u32x2 *out = reinterpret_cast<u32x2 *>(norm_out) + row_base;
        for (int c = tid; c < chunks_per_row; c += blockDim.x) {
            const u32x4 v = normed(c);
            float q[8];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                q[2 * j] = clamp_sym(P::lo(v[j]) / scale, fp8_max);
                q[2 * j + 1] = clamp_sym(P::hi(v[j]) / scale, fp8_max);
            }
            out[c] = u32x2{cvt4_e4m3fn(q[0], q[1], q[2], q[3]), cvt4_e4m3fn(q[4], q[5], q[6], q[7])};
        }
    }
}

// fp32 rows that stay in registers (up to 4 x 1024 chunks of 4 elements): the arrangement of add_rmsnorm_quant_rows -- same
// arguments, lane-to-chunk mapping, store gate and short exact quotients -- around plain fp32 arithmetic, where every
// rounding to the activation type is the identity:
//   res = x + r;  rstd = 1/sqrt(mean(res^2) + eps);  n = gamma * (res * rstd);  scale = max|n| / fp8_max;
//   code = e4m3fn(clamp(n / scale))
// 13 bytes per element with codes, 16 without: bound by HBM.  The first version fetched gamma behind the first reduction,
// divided with the full expansion, stored codes 4 bytes per lane and had no store gate.  Per call, that version / this
// one, dynamic scale: 8192 x 4096 72.0 / 68.0 us (6.05 / 6.41 TB/s), 3000 x 7168 52.6 / 47.4, 2048 x 4096 22.3 / 18.3, 1024 x
// 7168 21.9 / 16.8, 512 x 4096 7.7 / 7.0, 256 x 7168 7.3 / 6.15, one row of 7168 4.5 / 4.1; 8192 x 4096 without codes 87.4 / 85.5.
//
// When the weights are asked for.  A row of them is half as many bytes as the row's own loads, and a compute unit that holds
// few rows waits for its own: asked for at once, the weights of its first waves go ahead of the rows of its last.  So batches
// of up to one round that do not gate their stores ask once the lane's row has landed, behind which the reduction hides them,
// and rows of 28 KB and more, which keep a compute unit's memory path busy by themselves, once rstd is known.  Larger batches
// have other rows to wait for and ask at once.  us, at once / landed / rstd known: 98 rows of 3320 elements without codes 3.43
// / 3.21 / 3.35, 32 of 5120 with 3.78 / 3.58 / 3.61, one of 2056 2.52 / 2.48 / 2.56, but 32 of 7168 4.60 / 4.16 / 4.01, of
// 12288 5.95 / 5.89 / 5.62, 98 of 8192 without codes 5.00 / 5.39 / 4.54, of 16384 with 8.49 / 8.22 / 7.94; 4000 of 7168 without
// 77.7 / 79.2 / 78.8; 32 of 1024, on two waves, 2.49 / 2.51 / 2.56.  At once as well: two chunks per lane on four waves and
// less, one row per compute unit (127 rows of 1504 without codes 2.51 / 2.65, with codes level), and without codes, whose short
// chain leaves the weights' latency open, up to 32 rows of more than 6144 elements (one of 8296 3.15 / - / 3.35, of 16384 3.73
// / - / 3.97, 30 of 7760 2.90 / - / 3.08) and rows of two chunks per lane that do not fill their lanes, on six waves and less
// or up to 128 of them on nine (one of 2968 1.90 / 2.01, 29 of 2424 2.31 / 2.44, 314 of 1456 2.70 / 2.82; filled rows 1-5 % the
// other way).
// (98 of 16384 without codes remain behind the sweep of each lane's chunks one by one that this kernel replaced: 8.3 us, it
// 7.8.)  Gated rows of one chunk per lane and eight waves or more without codes, the shortest computation, ask once landed as
// well: 400 of 2568 elements 5.1 / 4.6 us, 290 of 3840 5.5 / 4.9, but 1280 of 1032, on five waves, 5.2 / 5.4.
enum class F32Form { STREAM, GATED, LANDED, GATED_LANDED, LAST };
template <int NCHUNK, int QUANT, bool EXACT, F32Form FORM>
__global__ void __launch_bounds__(kMaxThreads) __attribute__((amdgpu_waves_per_eu(FORM == F32Form::GATED || FORM == F32Form::GATED_LANDED ? 8 : 4)))
add_rmsnorm_quant_f32_rows(const u32x8 first, const u32x4 second, const u32x2 third, const RowArgs rest) {
    Global<const f32x4> *x = global_ptr<const f32x4>(first[0], first[1]), *residual_in = global_ptr<const f32x4>(first[2], first[3]);
    const int chunks_per_row = (int)first[4], remap_end = (int)first[5];
    const uint32_t lanes_and_shift = first[6], gate = first[7];
    Global<const f32x4> *gamma = global_ptr<const f32x4>(second[0], second[1]);
    Global<f32x4> *residual_out = global_ptr<f32x4>(second[2], second[3]);
    Global<char> *norm_out = global_ptr<char>(third[0], third[1]);
    float *scale_io = rest.scale_io;
    const float hidden_f = rest.hidden_f, rcp_hidden = rest.rcp_hidden, eps = rest.eps, fp8_max = rest.fp8_max, rcp_fp8_max = rest.rcp_fp8_max;
    constexpr bool GATED = FORM == F32Form::GATED || FORM == F32Form::GATED_LANDED;
    constexpr bool LANDED = FORM == F32Form::LANDED || FORM == F32Form::GATED_LANDED;
    const int nthreads = lanes_of(lanes_and_shift), group_shift = shift_of(lanes_and_shift);
    __shared__ float s_sum[kReduceSlots];
    __shared__ float s_max[kReduceSlots];
    const uint64_t entry = GATED ? __builtin_amdgcn_s_memrealtime() : 0;
    const int tid = threadIdx.x;
    const int num_waves = nthreads >> 6;
    int row = blockIdx.x;
    if (row < remap_end) {
        const int xcd = row & 7, idx = row >> 3;
        row = ((((idx >> group_shift) << 3) | xcd) << group_shift) | (idx & ((1 << group_shift) - 1));
    }
    int64_t row_base = (int64_t)row * chunks_per_row;
    const int pad = EXACT || (NCHUNK == 1 && !GATED) ? 0 : line_pad(first[0], row_base, lanes_and_shift);  // (even: lanes stay paired)
    row_base -= pad;

    // every load of the row ahead of the first use of any (and of the first store: residual_out may be an input)
    f32x4 xv[NCHUNK], rv[NCHUNK], gv[NCHUNK];
    bool live[NCHUNK];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
        const int c = i * nthreads + tid;
        live[i] = EXACT || (uint32_t)(c - pad) < (uint32_t)chunks_per_row;
        xv[i] = live[i] ? load_stream(x + row_base + c) : zero;
        rv[i] = live[i] ? load_stream(residual_in + row_base + c) : zero;
    }
    auto load_weights = [&]() {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) gv[i] = live[i] ? (gamma - pad)[i * nthreads + tid] : zero;
    };
    if constexpr (FORM != F32Form::LAST && !LANDED) load_weights();
    asm volatile("" ::"s"(hidden_f), "s"(rcp_hidden), "s"(eps), "s"(rest.sum_range));
    if constexpr (QUANT != GPUK_QUANT_NONE) asm volatile("" ::"s"(fp8_max));
    if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) asm volatile("" ::"s"(rcp_fp8_max), "s"(scale_io));
    float static_scale = 0.f;
    if constexpr (QUANT == GPUK_QUANT_FP8_STATIC) static_scale = *(const __attribute__((address_space(4))) float *)scale_io;

    __builtin_amdgcn_s_setprio(1);
    if constexpr (LANDED) {
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) asm volatile("" : "+v"(xv[i]), "+v"(rv[i]));
        load_weights();
        __builtin_amdgcn_sched_barrier(0);
    }
    float ss0 = 0.f, ss1 = 0.f;
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float v = xv[i][j] + rv[i][j];
            xv[i][j] = v;  // xv now holds the residual
            if (j & 1) ss1 = __builtin_fmaf(v, v, ss1);
            else ss0 = __builtin_fmaf(v, v, ss0);
        }
        if (!GATED && live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
    }
    if constexpr (QUANT == GPUK_QUANT_FP8_STATIC) asm volatile("" ::"s"(static_scale));
    const float sumsq = block_allreduce<SumOp>(ss0 + ss1, s_sum, num_waves);
    __builtin_amdgcn_s_setprio(0);
    const float rstd = row_rstd(sumsq, hidden_f, rcp_hidden, eps, rest.sum_range);
    if constexpr (FORM == F32Form::LAST) load_weights();

    f32x4 nv[NCHUNK];
    float m0 = 0.f, m1 = 0.f;
#pragma unroll
    for (int i = 0; i < NCHUNK; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) nv[i][j] = gv[i][j] * (xv[i][j] * rstd);
        if constexpr (QUANT != GPUK_QUANT_NONE) {
            m0 = maximum3_abs(m0, nv[i][0], nv[i][1]);
            m1 = maximum3_abs(m1, nv[i][2], nv[i][3]);
        }
    }
    const float lane_max = MaxOp::apply(m0, m1);
    uint32_t codes[NCHUNK];
    if constexpr (QUANT != GPUK_QUANT_NONE) {
        float scale = static_scale;
        bool fast;
        if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) {
            const float amax = block_allreduce<MaxOp>(lane_max, s_max, num_waves);
            scale = dynamic_scale(amax, fp8_max, rcp_fp8_max, &fast);
            if (tid == 0) scale_io[row] = scale;
        } else {  // (a static scale may meet quotients that overflow)
            fast = __builtin_amdgcn_ballot_w64(!(scale_in_fast_range(scale) && lane_max <= 0x1p60f)) == 0;
        }
        // Quotients below the smallest code's half come out 0 with their sign whatever the correction step loses to
        // underflow; the others are the correctly rounded ones.  With the dynamic scale no clamp, as in
        // add_rmsnorm_quant_rows.
        if (__builtin_expect(fast, 1)) {
            float rcp;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(mantissa_all_ones(scale)) == 0, 1)) rcp = rcp_rn_mid_range(scale);
            else rcp = 1.0f / scale;
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i) {
                float q[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) q[j] = div_by_rcp_finite(nv[i][j], scale, rcp);
                    else q[j] = clamp_sym(div_by_rcp(nv[i][j], scale, rcp), fp8_max);
                }
                codes[i] = cvt4_e4m3fn(q[0], q[1], q[2], q[3]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NCHUNK; ++i) {
                float q[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) q[j] = clamp_sym(nv[i][j] / scale, fp8_max);
                codes[i] = cvt4_e4m3fn(q[0], q[1], q[2], q[3]);
            }
        }
    }
    if constexpr (GATED) {  // (what is stored is pinned down ahead of the wait, as in add_rmsnorm_quant_rows)
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i) {
            if constexpr (QUANT == GPUK_QUANT_NONE) asm volatile("" ::"v"(nv[i]));
            else asm volatile("" ::"v"(codes[i]));
        }
        while (__builtin_amdgcn_s_memrealtime() < entry + gate) __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i)
            if (live[i]) store_stream(residual_out + row_base + i * nthreads + tid, xv[i]);
    }
    if constexpr (QUANT == GPUK_QUANT_NONE) {
        auto *out = (Global<f32x4> *)norm_out + row_base;
#pragma unroll
        for (int i = 0; i < NCHUNK; ++i)
            if (live[i]) store_stream(out + i * nthreads + tid, nv[i]);
    } else if constexpr (NCHUNK == 1) {
        if (live[0]) store_stream((Global<uint32_t> *)norm_out + row_base + tid, codes[0]);
    } else {
        // 8 codes per lane and store: of two chunks, even lanes store the first one's codes of themselves and their odd
        // neighbour, odd lanes the second one's (a row is an even number of chunks: neighbours are live together)
        auto *out = (Global<uint32_t> *)norm_out + row_base;
        const bool odd = tid & 1;
#pragma unroll
        for (int i = 0; i < NCHUNK; i += 2) {
            const uint32_t give = odd ? codes[i] : codes[i + 1], keep = odd ? codes[i + 1] : codes[i];
            const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, DPP_QUAD_XOR1, 0xf, 0xf, true);
            if (odd ? live[i + 1] : live[i])
                store_stream((Global<u32x2> *)(out + (odd ? i + 1 : i) * nthreads + (tid & ~1)), odd ? u32x2{got, keep} : u32x2{keep, got});
        }
    }
}

// fp64 activations and longer fp32 rows: the reference dispatches both types through the same template
// (AT_DISPATCH_FLOATING_TYPES_AND2, src/ops/all_reduce_fusion.cpp:375-378).  4 elements per chunk; a lane keeps its
// CPL chunks of the summed row in registers (fp64 rows of up to 4 x 1024 chunks), or, with CPL = 0, sweeps a longer row
// three times, reading back what it stored to residual_out.  Rounding to the activation type is the identity here, so
// the oracle's sequence is plain arithmetic in that type around an fp32 variance:
//   res = x + r;  rstd = 1/sqrt(mean(float(res)^2) + eps) in fp32;  n = gamma * (res * F(rstd));
//   scale = max|float(n)| / fp8_max in fp32;  code = e4m3fn(float(clamp(n / F(scale))))
// (for F = double torch promotes tensor * fp32-tensor products to double and casts double -> float -> fp8).
template <typename F>
using wide4 = F __attribute__((ext_vector_type(4)));

template <typename F, int QUANT, int CPL>
__global__ void __launch_bounds__(kMaxThreads)
add_rmsnorm_quant_wide_rows(const wide4<F> *x, const wide4<F> *residual_in,  // either may be residual_out
                            const wide4<F> *__restrict__ gamma, wide4<F> *residual_out, void *norm_out,
                            float *__restrict__ scale_io, int chunks_per_row, float hidden_f, float eps, float fp8_max) {
    __shared__ float s_sum[kReduceSlots];
    __shared__ float s_max[kReduceSlots];
    const int tid = threadIdx.x;
    const int num_waves = blockDim.x >> 6;
    const int64_t row_base = (int64_t)blockIdx.x * chunks_per_row;
    constexpr int KEPT = CPL ? CPL : 1;
    // (no streaming accesses: measured 12 % slower for fp64)
    wide4<F> kept[KEPT];  // CPL > 0: chunk tid + i * blockDim.x of the summed row (and later of the normed row)

    // f(i, c) for every chunk c of the row this lane owns; i is its place in kept[]
    auto for_chunks = [&](auto f) {
        if constexpr (CPL > 0) {
#pragma unroll
            for (int i = 0; i < CPL; ++i) {
                const int c = tid + i * (int)blockDim.x;
                if (c < chunks_per_row) f(i, c);
            }
        } else {
            for (int c = tid; c < chunks_per_row; c += blockDim.x) f(0, c);
        }
    };

    float ss = 0.f;
    for_chunks([&](int i, int c) {
        const wide4<F> res = x[row_base + c] + residual_in[row_base + c];
        residual_out[row_base + c] = res;  // CPL = 0: read back below
        kept[i] = res;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float r = (float)res[j];
            ss = __builtin_fmaf(r, r, ss);
        }
    });
    const float sumsq = block_allreduce<SumOp>(ss, s_sum, num_waves);
    const F rstd = (F)(1.0f / sqrtf(sumsq / hidden_f + eps));

    // the normed chunk; with CPL = 0 the summed chunk is read back (this lane wrote it above)
    auto normed = [&](int i, int c) {
        const wide4<F> v = CPL > 0 ? kept[i] : residual_out[row_base + c];
        return gamma[c] * (v * rstd);
    };

    if constexpr (QUANT == GPUK_QUANT_NONE) {
        wide4<F> *out = reinterpret_cast<wide4<F> *>(norm_out) + row_base;
        for_chunks([&](int i, int c) { out[c] = normed(i, c); });
    } else {
        float scale;
        if constexpr (QUANT == GPUK_QUANT_FP8_DYNAMIC) {
            float amax = 0.f;
            for_chunks([&](int i, int c) {
                const wide4<F> v = normed(i, c);
                if constexpr (CPL > 0) kept[i] = v;
#pragma unroll
                for (int j = 0; j < 4; ++j) amax = MaxOp::apply(amax, __builtin_fabsf((float)v[j]));
            });
            amax = block_allreduce<MaxOp>(amax, s_max, num_waves);
            scale = amax == 0.f ? 1.f : amax / fp8_max;
            if (tid == 0) scale_io[blockIdx.x] = scale;
        } else {
            scale = scale_io[0];
        }
        const F wide_scale = (F)scale;
        uint32_t *out = reinterpret_cast<uint32_t *>(norm_out) + row_base;
        for_chunks([&](int i, int c) {
            wide4<F> n;
            if constexpr (CPL > 0 && QUANT == GPUK_QUANT_FP8_DYNAMIC) n = kept[i];
            else n = normed(i, c);
            const wide4<F> q = n / wide_scale;
            // clamping after the cast to fp32 equals the oracle's clamp before it: the bounds are fp32 numbers
            out[c] = cvt4_e4m3fn(clamp_sym((float)q[0], fp8_max), clamp_sym((float)q[1], fp8_max),
                                 clamp_sym((float)q[2], fp8_max), clamp_sym((float)q[3], fp8_max));
        });
    }
}

int g_force_nchunk = 0;   // 0 = heuristic; set through gpuk_set_tuning for sweeps
int g_force_threads = 0;  // 0 = heuristic
int g_row_group_shift = -1;  // -1 = heuristic, else log2 of the run of consecutive rows an XCD takes (0 = one row)
int g_gate = -1;             // store gate in ticks of 10 ns: -1 = built-in rule, 0 = none, > 0 = that many
int g_pieces = 0;            // launches per call: 0 = built-in rule, 1 = always one, 2 = two wherever each half fits one round
constexpr int kComputeUnits = 256;  // MI355X

// Rows resident at once, chip-wide, with `threads` lanes per row and `nchunk` chunks per lane: 2048 lanes per compute
// unit, eight waves per SIMD, which the gated instantiations of up to four chunks per lane are compiled for
// (amdgpu_waves_per_eu: at most 64 registers); with eight chunks per lane, up to 128 registers, half of that.
// Measured exception: of workgroups of 5 or 10 waves a compute unit takes 25 or 20 waves' worth, not 30 (1408 rows of
// 5120 elements, 5.5 per compute unit, run no faster gated than ungated, 1280 run 22 % faster; likewise 640 and 512
// rows of 10240), where 3, 6, 7, 9, 11-16 waves fill it as counted (30, 30, 28, 27, ... waves).
int64_t resident_rows(int threads, int nchunk) {
    const int waves = threads / 64;
    int waves_per_cu = nchunk >= 8 ? 16 : 32;
    if (waves == 5 || waves == 10) waves_per_cu = std::min(waves_per_cu, waves == 5 ? 25 : 20);
    return (int64_t)kComputeUnits * (waves_per_cu / waves);
}

enum class RowType { BF16, FP16, F32 };
template <typename T> constexpr RowType row_type = is_half<T> ? RowType::FP16 : RowType::BF16;

// The store gate of a launch: for batches whose workgroups are all resident at once (2048 lanes per compute unit) the time
// their reads take at 7 TB/s, the rate of a read-only kernel on this part, plus a twentieth; 0 (stores as soon as they are
// ready) for larger batches, whose later workgroups read while earlier ones write whatever a wave does.  Measured per call at
// 7168 elements: 6.35 against 7.2 us at 512 rows, 7.6 against 9.5 at 768, 9.0 against 11.7 at 1024 (gate 1.0-1.1 times the read
// time; 10.2 with 0.9, 9.6 with 1.2), nothing gained and 0.1 us lost below a quarter of a round; at 4096 elements 6.2 against
// 7.7 us at 1024 rows, 10.2 against 12.4 at 2048; 20-45 % slower where the batch does not fit one round.
// A compute unit reads no faster than its share of that rate by much, so a layer of rows (one per compute unit) that has just
// begun takes nearly the time of a full one where rows are wide and a compute unit holds few: the gate is at least 0.93 of the
// time of whole layers for 16-bit rows of four chunks per lane, else 0.86 with codes and 0.82 without (those store more, the
// rows' own gate / this one, us: bf16, four chunks, 522 rows of 16384 14.7 / 12.0, 614 15.1 / 12.9, 775 18.4 / 16.2, 780 of
// 10240 12.3 / 10.8, 1030 of 12288 17.6 / 15.8, 1044 of 8192 11.3 / 10.8; two chunks, fp16 559 of 8192 7.45 / 6.8, 377 of 16384
// 8.9 / 8.3, 300 of 8192 without codes 5.5 / 5.0; fp32 387 of 7168 8.1 / 7.4, 340 of 8192 8.9 / 7.6, 368 of 13184 14.5 / 12.1,
// without codes 318 of 5120 6.4 / 5.7; narrow rows and nearly full layers level.  More than that share holds back nearly full
// ones: fp32 without codes 592 of 4096 7.1 / 7.3 with 0.9, 7.5 with 0.94).  Only behind a full layer: in the first one a
// compute unit has one row or none, and the row's own share of the time is all there is to wait for (bf16 without codes, 32768
// elements, 128 rows 7.95 / 8.39, 160 8.71 / 8.99, 200 10.1 / 10.3; level up to 16384 elements and at 65536).
// short_rows: rows of two chunks per lane whose computation ends well ahead of the reads of a half-filled round (half
// precision, static scale).  From two fifths of a round to eleven twentieths they wait 1.16 times the read time: 460 rows of
// 8192 elements 6.28 / 5.72 us, 576 of 6144 6.55 / 6.05, 576 of 5120 5.46 / 5.3, level or slower below and above (1228 of 4096
// 6.6 / 6.8).
// 16-bit rows of one chunk per lane spread their stores by themselves, each wave as its row is done, and wait from three eighths
// of a round only (gated / not, us: 2800 of 512 elements 3.71 / 3.45, static 3.33 / 3.32, 400 of 2560 3.63 / 3.36, without codes
// 3.15 / 2.97, 128 of 5632 3.73 / 3.37, 130 of 7680 4.23 / 3.61; beyond, 580 of 2560 without codes 3.55 / 3.63, half precision 3.54
// / 3.93), ten waves a row not in the first layer (bfloat16, 200 of 5120 3.73 / 3.55, 256 3.97 / 3.75; 12 to 15 waves level to 6 %
// behind there).  The shortest of them, half precision without codes on one wave, from a quarter as the others (2800 of 512
// elements 3.25 / 3.47).
uint32_t store_gate(int64_t tokens, int64_t row_bytes, int threads, int nchunk, RowType type, int quant) {
    if (g_gate >= 0) return (uint32_t)g_gate;
    const int64_t resident = resident_rows(threads, nchunk);
    if (tokens > resident || 4 * tokens < resident) return 0;
    const bool quick = type == RowType::FP16 && quant == GPUK_QUANT_NONE && threads == 64;
    const bool early = 8 * tokens < 3 * resident || (threads <= 640 && tokens <= kComputeUnits);
    if (nchunk == 1 && type != RowType::F32 && early && !quick) return 0;
    // (four chunks per lane: the shape pick_shape takes to hold in one round what two chunks per lane cannot)
    const bool short_rows = type == RowType::FP16 && quant == GPUK_QUANT_FP8_STATIC;
    const bool half_filled = short_rows && nchunk == 2 && 5 * tokens >= 2 * resident && 20 * tokens <= 11 * resident;
    const double rows = (half_filled ? 1.16 : nchunk >= 4 ? 1.08 : 1.05) * (double)tokens;
    const double share = nchunk == 4 && type != RowType::F32 ? 0.93 : quant != GPUK_QUANT_NONE ? 0.86 : 0.82;
    const double layers = tokens > kComputeUnits ? share * (double)((tokens + kComputeUnits - 1) / kComputeUnits * kComputeUnits) : 0.0;
    const double ticks = 2 * std::max(rows, layers) * (double)row_bytes / 70000.0;  // 70,000 bytes per tick of 10 ns
    return (uint32_t)std::min(ticks, 5000.0);
}

// Whether a launch of the 16-bit kernel asks for the weights once the row has landed (LANDED, see add_rmsnorm_quant_rows): at most
// a round of rows, whose waves wait for their own loads and not for other rows', and more of them than short rows have.  us, at
// once / landed: without a gate, from five waves on, 30 rows of 8192 elements, static, 3.58 / 3.36, 4 of 14336 in half precision 3.62 / 3.29,
// 128 of 16384 5.7 / 5.45 (but not up to 4 rows of two chunks in bfloat16 without codes, one of 15576 3.35 / 3.46, 88 such calls
// 1.02; with codes or one chunk 0.98); four waves and fewer level to 3 % behind, but for
// 3 and 4 waves of two chunks behind the first layer (361 of 4096 static 3.9 / 3.7, 480 without codes 4.65 / 3.84).  Gated rows
// have the launch's reads to wait for: nine waves and more of one chunk 0.97, of two chunks in the first layer (131 of 12288
// 4.87 / 4.61, static 141 4.87 / 4.58, without codes 173 of 14688 5.35 / 5.02) and not behind it (338 of 12288 6.69 / 6.86);
// without codes, which have the time to be early, three waves and more up to three eighths of a round (379 of 7168 5.44 / 4.75, 597
// of 4096 4.86 / 4.50, but 537 of 7168 6.27 / 6.36).  Four chunks have the loads of a whole row in flight per lane and hide the weights'
// behind them unless the row has most of the lanes: with codes 1.04 of the time at 9 and 10 waves, level at 11 and 12, 0.96 from 13 on (700
// calls; 57 rows of 32512 elements in bfloat16, static, 9.0 / 8.3, but 40 of 18040 in half precision 5.5 / 5.9), without codes 1.11 and
// 1.06, and from 13 on 1.02 up to 32 rows (one of 17984 3.7 / 4.2) and 0.97 beyond (118 of 27112 8.2 / 7.5), in half precision; not in
// bfloat16 (14 rows of 32768 5.12 / 5.50), gated 1.00 to 1.19.  More than a round: 1.00 to 1.03 (8192 x 8192 75.6 / 76.7).
constexpr bool late_in_four_chunks(RowType type, int quant) { return type == RowType::FP16 || quant != GPUK_QUANT_NONE; }
bool late_weights(int64_t tokens, int threads, int nchunk, RowType type, int quant, bool gated) {
    const int64_t resident = resident_rows(threads, nchunk);
    if (tokens > resident || nchunk > 4) return false;
    if (type == RowType::BF16 && quant == GPUK_QUANT_NONE && nchunk == 2 && tokens <= 4) return false;
    const bool wide = threads >= 576;
    if (nchunk == 4) return !gated && threads >= 832 && late_in_four_chunks(type, quant) && (quant != GPUK_QUANT_NONE || tokens > 32);
    if (!gated) return threads >= 320 || (nchunk == 2 && threads >= 192 && 4 * tokens > 5 * kComputeUnits);
    if (nchunk == 1) return wide;
    return (wide && tokens <= kComputeUnits) || (quant == GPUK_QUANT_NONE && threads >= 192 && 8 * tokens <= 3 * resident);
}

// Lanes per row and chunks per lane.  Two chunks per lane on as many lanes as that needs (up to 1024) stream best or tie
// for 1024 .. 16384 16-bit elements (1-6 % over one or four chunks per lane; 7168 elements, per call: 3.3 us against 3.5
// with one chunk at one row, 5.0 against 5.6 at 256 rows), but for the small batches named below; longer rows double the chunks per lane.  Where rounding up to
// whole waves idles more lanes that way (an odd number of 64 chunks, or a little more than an even one), one chunk per lane
// serves what the chip holds in one round (1032 elements: 2.2 against 2.45 us at one row, 5.65 against 6.2 at 2048), but
// larger batches want the loads of two in flight: 12000 rows of 2560 / 3584 / 5632 / 7680 elements 37.0 / 49.6 / 76.6 /
// 102.8 us against 39.4 / 53.5 / 86.0 / 111.7, of 3208 45.7 against 47.1; fp32 rows of 2568 66.3 against 70.9.  Rows that one
// wave holds with one chunk per lane keep it, a second chunk would be dead in every lane (one / two chunks: 9000 rows of 256
// elements 5.4 / 6.7 us, 100000 rows 34.8 / 44.6, 20000 of 512 13.5 / 14.3; above 50000 rows of exactly 512 the two-chunk form is
// 4 % ahead in bfloat16, 150000 rows 90.4 / 86.8, level in half precision).
// codes: whether the rows are quantised.
void pick_shape(int64_t tokens, int chunks_per_row, RowType type, bool codes, int *threads, int *nchunk) {
    const int most_chunks = type == RowType::F32 ? kMaxChunksF32 : kMaxChunks;  // (a forced eight becomes four there)
    auto fits = [&](int n) { return (int64_t)n * kMaxThreads >= chunks_per_row; };
    int n;
    if (g_force_nchunk) {
        n = std::min(g_force_nchunk, most_chunks);
    } else {
        // one chunk per lane only where two would leave more lanes idle after rounding up to whole waves
        const int lanes1 = round_up(chunks_per_row, 64), lanes2 = round_up((chunks_per_row + 1) / 2, 64);
        n = (2 * lanes2 > lanes1 && lanes1 <= kMaxThreads) ? 1 : 2;
        while (n < most_chunks && chunks_per_row > kMaxThreads * n) n *= 2;
        if (n == 2 && !g_force_threads) {
            // A compute unit that has a row or two is bound by the instructions of its busiest SIMD, chunks per lane times the
            // waves there: lanes for 5 or 6 waves of two chunks put four chunks on one SIMD, 10 to 12 waves of one chunk three
            // (us, two / one: 12 rows of 6000 elements 3.44 / 3.20, 64 of 6144 3.45 / 3.10, without codes 3.21 / 2.82, 128 of
            // 5120 3.63 / 3.35, half precision 3.42 / 3.38; fp32 32 of 3072 3.11 / 2.89, 192 3.48 / 3.32).  As the first layer
            // fills, the waves share the units' load paths and only the 5 of bfloat16 still gain (256 of 5120 3.96 / 3.75,
            // without codes level, half precision 3.42 / 3.72, 256 of 5640 4.11 / 4.27); with a second row per unit they gain
            // again, up to the whole layer (320 of 5640 5.50 / 5.12, 270 of 5120 without codes 4.18 / 3.80, 416 of 6144 static 4.66 /
            // 4.24, 443 in half precision 5.01 / 4.84, 485 without codes 5.13 / 4.83, 505 of 5120 level).
            // 2 waves of two chunks and 4 of one are one wave a SIMD at most, of half the length: 4 rows of 2048 elements 2.48 /
            // 2.34, 300 3.39 / 2.81, 712 3.81 / 3.66, static 990 3.99 / 3.77, dynamic 1241 5.19 / 5.13; without codes 640 3.21 / 2.95 and,
            // gated as two chunks are from 1024 on, 932 4.23 / 3.76, but 768 3.25 / 3.43 and 1231 4.26 / 4.34 (fp32 gains less, 2-4 %, and
            // only for a few rows).
            // Where each of more than half of the units has one row, 3 or 4 full waves of four chunks wait for fewer of each
            // other (us, two / four: 160 rows of 6144 3.91 / 3.73, 256 4.29 / 4.02, without codes 4.00 / 3.60; 200 of 8192 4.49 /
            // 4.31, 256 without codes 4.52 / 4.09; 128 rows of 8192 and 7168 elements level, which idle lanes).
            const int lanes4 = round_up((chunks_per_row + 3) / 4, 64);
            const bool f32 = type == RowType::F32, f16 = type == RowType::FP16;
            if (!f32 && 2 * tokens > kComputeUnits && tokens <= kComputeUnits && (lanes4 == 192 || lanes4 == 256) &&
                15 * lanes4 < 4 * chunks_per_row) {
                n = 4;
            } else if (lanes2 == 128) {
                const bool gated_none = 4 * tokens > 13 * kComputeUnits && tokens <= 4 * kComputeUnits;
                if (!f32 && (2 * tokens <= 5 * kComputeUnits || (codes ? tokens <= 5 * kComputeUnits : gated_none))) n = 1;
            } else if (lanes2 == 320 || lanes2 == 384) {
                const bool few = 4 * tokens <= 3 * kComputeUnits;
                const bool first_layer = tokens <= kComputeUnits && lanes2 == 320 && !f16;
                const bool second_layer = tokens > kComputeUnits && tokens <= 2 * kComputeUnits;
                if (few || (!f32 && (first_layer || second_layer))) n = 1;
            }
        }
        // A batch that two chunks per lane cannot hold in one round but four can (half the lanes per row, so up to
        // 2048 rows of 7168 or 8192 elements instead of 1024) takes four: one round, with the store gate, against two
        // rounds of mixed reads and writes.  7168 elements: 10.8 against 12.8 us at 1100 rows, 10.9 against 14.3 at
        // 1280, 13.0 against 16.2 at 1536, 14.3 against 17.5 at 1700; 8192 elements: 12.4 against 15.5 us at 1280 rows,
        // 16.3 against 18.7 at 1700.  (That form keeps the normed row as 16-bit pairs between its last two phases:
        // with it in fp32 the kernel took 70 registers, seven waves per SIMD, 1792 rows.)
        // Not where four would idle a third of the lanes (3000 rows of 2312 elements: 12.4 us against 11.7 with two).
        if (n <= 2 && lanes2 < lanes1 && !g_force_threads && tokens > resident_rows(n == 1 ? lanes1 : lanes2, n)) {
            const int t4 = round_up((chunks_per_row + 3) / 4, 64);
            const int64_t round1 = resident_rows(lanes1, 1), round2 = resident_rows(lanes2, 2);
            // Rows that two chunks per lane leave a third of their lanes idle for (129 to 170 chunks, on three waves or on
            // two): one chunk between the round of the latter and three of the former (us, one chunk / two: 1160 elements 9.7 /
            // 10.2 at 4480 rows, 10.4 / 11.2 at 5120, 14.1 / 14.6 at 7680, 18.1 / 18.1 at 10240; 1288 10.1 / 10.9, 11.0 / 11.9,
            // 15.1 / 15.5, 19.2 / 19.5; 1032 9.5 / 9.7, 10.1 / 10.6, 13.9 / 13.8, 17.2 / 17.1; not fp32 rows, without codes
            // 4146 of 624 8.99 / 8.54, 6676 of 552 12.2 / 11.7, with codes level), and in bfloat16, whose arithmetic is
            // unpacked, where two idle two fifths also up to an eighth more than a round (2611 rows of 1032 6.36 / 6.81, 2816
            // 6.7 / 7.0, but 3072 7.5 / 7.2; half precision 6.35 / 5.97 at 2611).
            const bool thin = n == 1 && 3 * chunks_per_row < 4 * lanes2;
            const bool one = thin && (tokens > round2 ? type != RowType::F32 && tokens <= 3 * round1
                                                      : type == RowType::BF16 && 5 * chunks_per_row < 6 * lanes2 && 8 * tokens <= 9 * round1);
            n = one ? 1 : tokens > round2 && tokens <= resident_rows(t4, 4) && 8 * t4 <= 3 * chunks_per_row ? 4 : 2;
        }
    }
    while (n < most_chunks && !fits(n)) n *= 2;
    if (!fits(n)) {
        *nchunk = 0;
        *threads = kMaxThreads;
        return;
    }
    int t = round_up((chunks_per_row + n - 1) / n, 64);
    if (g_force_threads && (int64_t)g_force_threads * n >= chunks_per_row) t = g_force_threads;
    *nchunk = n;
    *threads = t;
}

// Rows of the first of two launches: a whole number of rows per compute unit (half of what the batch needs, rounded down),
// so that neither piece pays for a partly filled last row of workgroups twice.
int64_t half_of(int64_t tokens) { return (tokens + kComputeUnits - 1) / kComputeUnits / 2 * kComputeUnits; }

// Launches per call.  A batch of more than one round of workgroups and at most two runs as two launches of half the rows, each
// a round of its own with the store gate: a read phase and a write phase twice over instead of two rounds that mix the
// directions.  Only where each piece does fit a round in the shape it is given, rows start on line boundaries, and that shape
// idles few lanes: from 1.1 rounds on one in eight, or one in five of a single wave with four chunks per lane; from 1.25 rounds
// on one in five; from 1.5 on one in four of a single wave (fp32 rows of one wave: one in eight, always).  One launch / two,
// us:
// bf16 4600 rows of 4096 elements 23.6 / 22.7, 8000 rows 38.5 / 38.0, 2300 of 8192 24.4 / 23.2, 4600 of 3072 19.2 / 17.8; 3200
// of 5120 (a sixth idle) 22.1 / 23.3 but 4608 30.4 / 28.9; 9830 of 1664 (a fifth, one wave of four chunks) 22.2 / 21.5-22.0,
// 11900 25.9 / 24.5; 9830 of 832 (a fifth, of two chunks) 12.4 / 13.2, 14700 17.0 / 15.8; 14700 of 768 (a quarter, one wave)
// 16.1 / 15.3, 5500 of 3072 (a quarter, two waves) 22.3 / 24.3, 11900 of 640 (three eighths) 11.7 / 12.6; fp32 14700 of 416
// 15.3 / 15.8.  Pieces beyond a round: 5700 of 2688 21.0 / 24.6.  One chunk per lane (rows of at most 64 chunks): 11500 of 512
// 8.6 / 9.6, fp32 of 256 7.9 / 9.5.  Rows that end inside lines: 2500 of 9000 30.1 / 31.8.  Wide fp32 rows, four waves and
// more, of which a compute unit holds few, pay for a layer of workgroups (one per compute unit) that a piece does not fill: two
// launches where the rows fill 94 % of the two pieces' layers (92 on five waves, 96 on six), without codes 90 % (88 on five).
// Two / one by that share, codes: five waves 1.04 at 88 %, 1.00 at 92, 0.96 at 96; six 1.06 / 1.02 / 1.00, seven 1.04 / 1.01 /
// 0.98, eight 1.02 / 1.01 / 0.97; four 1.03 at 90, 1.00 at 94; without codes five to seven 1.00 at 88, 0.98 at 90, 0.95 at 96
// (1518 of 5120 with codes, 99 %, 20.1 / 17.8, but 1331 of 7168, 87 %, 24.5 / 27.0).  codes: for fp32, whether the rows are
// quantised.
int launches_for(int64_t tokens, int chunks_per_row, RowType type, bool codes) {
    if (g_pieces == 1 || g_force_nchunk || g_force_threads || chunks_per_row > 2 * kMaxThreads) return 1;
    const int64_t round = resident_rows(round_up((chunks_per_row + 3) / 4, 64), 4);
    if (tokens <= round || tokens > 2 * round) return 1;
    if (g_pieces == 2) return 2;
    const int64_t piece = tokens - half_of(tokens);  // (the larger one)
    int threads, nchunk;
    pick_shape(piece, chunks_per_row, type, codes, &threads, &nchunk);
    if (nchunk == 1 || piece > resident_rows(threads, nchunk) || chunks_per_row % 8 != 0) return 1;
    const int places = threads * nchunk;
    const bool one_wave = threads == 64, eighth = 8 * chunks_per_row >= 7 * places, fifth = 5 * chunks_per_row >= 4 * places;
    if (type == RowType::F32) {
        const int64_t layers = (tokens - piece + kComputeUnits - 1) / kComputeUnits + (piece + kComputeUnits - 1) / kComputeUnits;
        const int percent = !codes ? (threads == 320 ? 88 : 90) : threads == 320 ? 92 : threads == 384 ? 96 : 94;
        if ((!eighth && one_wave) || (threads >= 256 && 100 * tokens < percent * layers * kComputeUnits)) return 1;
    }
    if (eighth || (fifth && one_wave && nchunk == 4)) return 10 * tokens >= 11 * round ? 2 : 1;
    if (fifth) return 4 * tokens > 5 * round ? 2 : 1;
    return one_wave && 4 * chunks_per_row >= 3 * places && 2 * tokens >= 3 * round ? 2 : 1;
}

// log2 of the run of consecutive rows an XCD takes.  Runs of 64 rows: +1.1 % for 16 KiB rows (8192 rows), of 16-bit
// elements (75.5 -> 74.9 us) as of fp32 (68.8 -> 68.0, 16384 rows 138.0 -> 136.4, 1500 rows 14.1 -> 13.9); neutral or 1-10 %
// slower for every other row size tried (2, 3, 4, 8, 10, 14, 20, 28, 32 KiB) and for fewer rows, hence the narrow rule.
int row_group_shift(int64_t tokens, int64_t row_bytes) {
    return g_row_group_shift >= 0 ? g_row_group_shift : row_bytes == 16384 && tokens >= 1024 ? 6 : 0;
}

// The mask of line_pad: 15 where the lanes beyond the row's last chunk allow for it, else 7, else none.
uint32_t line_mask(int threads, int nchunk, int chunks) {
    const int idle = threads * nchunk - chunks;
    return idle >= 15 ? 15u : idle >= 7 ? 7u : 0u;
}

// What the kernels take for rcp_fp8_max: RN(1 / fp8_max) for the two maxima whose quotient was checked (448 and 240), 0 for
// others, and -1 where fp8_max and the next float round to different codes (400: 384 and 416), so that quotients by the
// dynamic scale, which may exceed fp8_max by that one ULP, have to be clamped.  Those calls take the kernels' dividing
// path, which clamps (8192 x 8192 at 400: 78.4 us, 76.0 at 448; 1024 x 7168, ungated on that path: 12.5 against 8.9; one row 3.6
// against 2.8): a clamp in the common path would add 55 to 440 instructions to every kernel for a handful of maxima.
float reciprocal_of_max(float fp8_max) {
    auto code = [](float v) {  // rounded to three bits of fraction, or to the spacing of the subnormal codes
        const float step = std::ldexp(1.0f, std::max(std::ilogb(v) - 3, -9));
        return std::nearbyint(v / step) * step;
    };
    if (fp8_max == 448.0f || fp8_max == 240.0f) return 1.0f / fp8_max;
    return code(fp8_max) == code(std::nextafter(fp8_max, INFINITY)) ? 0.0f : -1.0f;
}

// Rows of the first launch.
int64_t first_piece(int64_t tokens, int chunks_per_row, RowType type, bool codes = true) {
    if (launches_for(tokens, chunks_per_row, type, codes) == 1) return tokens;
    return half_of(tokens);
}

template <typename T, int QUANT>
int launch_rows(const void *x, const void *residual_in, const void *gamma, void *residual_out, void *norm_out,
                float *scale, int64_t tokens, int64_t hidden, float eps, float fp8_max, hipStream_t stream);

template <typename T, int QUANT>
int launch(const void *x, const void *residual_in, const void *gamma, void *residual_out, void *norm_out,
           float *scale, int64_t tokens, int64_t hidden, float eps, float fp8_max, hipStream_t stream) {
    const int64_t piece = first_piece(tokens, (int)(hidden / 8), row_type<T>);
    for (int64_t first = 0; first < tokens; first = first ? tokens : piece) {
        const int64_t in_bytes = first * hidden * 2, out_bytes = first * hidden * (QUANT == GPUK_QUANT_NONE ? 2 : 1);
        const int rc = launch_rows<T, QUANT>(static_cast<const char *>(x) + in_bytes, static_cast<const char *>(residual_in) + in_bytes,
                                             gamma, static_cast<char *>(residual_out) + in_bytes, static_cast<char *>(norm_out) + out_bytes,
                                             QUANT == GPUK_QUANT_FP8_DYNAMIC ? scale + first : scale, first ? tokens - first : piece,
                                             hidden, eps, fp8_max, stream);
        if (rc != GPUK_OK) return rc;
    }
    return GPUK_OK;
}

// What is passed to the kernels of rows that stay in registers, see RowArgs.  shape: lanes_and_shift.
struct RowParameters {
    u32x8 first;
    u32x4 second;
    u32x2 third;
    RowArgs rest;
};
RowParameters row_parameters(const void *x, const void *residual_in, const void *gamma, const void *residual_out, const void *norm_out,
                             float *scale, int64_t tokens, int chunks, uint32_t shape, uint32_t gate, int64_t hidden, float eps, float fp8_max) {
    const int group_shift = (int)((shape >> 16) & 0xffu);
    const uint32_t remap_end = group_shift > 0 ? (uint32_t)((tokens >> (3 + group_shift)) << (3 + group_shift)) : 0u;
    const float hf = (float)hidden;
    return {u32x8{low_half(x), high_half(x), low_half(residual_in), high_half(residual_in), (uint32_t)chunks, remap_end, shape, gate},
            u32x4{low_half(gamma), high_half(gamma), low_half(residual_out), high_half(residual_out)},
            u32x2{low_half(norm_out), high_half(norm_out)},
            RowArgs{scale, hf, 1.0f / hf, eps, eps >= 0.f && eps <= 0x1p60f ? kSumRange : 0u, fp8_max, reciprocal_of_max(fp8_max)}};
}

template <typename T, int QUANT>
int launch_rows(const void *x, const void *residual_in, const void *gamma, void *residual_out, void *norm_out,
                float *scale, int64_t tokens, int64_t hidden, float eps, float fp8_max, hipStream_t stream) {
    const int chunks = (int)(hidden / 8);
    int threads, nchunk;
    pick_shape(tokens, chunks, row_type<T>, QUANT != GPUK_QUANT_NONE, &threads, &nchunk);
    const dim3 grid((unsigned)tokens);
    if (nchunk == 0) {
        add_rmsnorm_quant_long_rows<T, QUANT><<<grid, kMaxThreads, 0, stream>>>(
            static_cast<const u32x4 *>(x), static_cast<const u32x4 *>(residual_in), static_cast<const u32x4 *>(gamma),
            static_cast<u32x4 *>(residual_out), norm_out, scale, chunks, (float)hidden, eps, fp8_max);
        return hip_status(hipGetLastError());
    }
    const uint32_t gate = store_gate(tokens, hidden * 2, threads, nchunk, row_type<T>, QUANT);
    const uint32_t shape = (uint32_t)threads | ((uint32_t)row_group_shift(tokens, hidden * 2) << 16) | (line_mask(threads, nchunk, chunks) << 24);
    const bool exact = (int64_t)threads * nchunk == chunks;
    const RowParameters p = row_parameters(x, residual_in, gamma, residual_out, norm_out, scale, tokens, chunks, shape, gate, hidden, eps, fp8_max);
    const bool late = late_weights(tokens, threads, nchunk, row_type<T>, QUANT, gate != 0);
#define GPUK_LAUNCH_NQ_AS(N, EXACT, GATED, LANDED)                                                                      \
    return launch_kernel(add_rmsnorm_quant_rows<T, N, QUANT, EXACT, GATED, LANDED>, grid, (uint32_t)threads, 0, stream, p.first, p.second, p.third, p.rest)
#define GPUK_LAUNCH_NQ_EXACT(N, EXACT)                                                                                 \
    do {                                                                                                               \
        if constexpr (N <= 2)                                                                                          \
            if (gate && late) GPUK_LAUNCH_NQ_AS(N, EXACT, true, true);                                                 \
        if (gate) GPUK_LAUNCH_NQ_AS(N, EXACT, true, false);                                                            \
        if constexpr (N <= 2 || (N == 4 && late_in_four_chunks(row_type<T>, QUANT)))                                  \
            if (late) GPUK_LAUNCH_NQ_AS(N, EXACT, false, true);                                                        \
        GPUK_LAUNCH_NQ_AS(N, EXACT, false, false);                                                                     \
    } while (0)
#define GPUK_LAUNCH_NQ(N)                                                                                              \
    do {                                                                                                               \
        if (exact) GPUK_LAUNCH_NQ_EXACT(N, true);                                                                      \
        else GPUK_LAUNCH_NQ_EXACT(N, false);                                                                           \
    } while (0)
    switch (nchunk) {
        case 1: GPUK_LAUNCH_NQ(1); break;
        case 2: GPUK_LAUNCH_NQ(2); break;
        case 4: GPUK_LAUNCH_NQ(4); break;
        case 8: GPUK_LAUNCH_NQ(8); break;
        default: return GPUK_ERR_INTERNAL;
    }
#undef GPUK_LAUNCH_NQ
#undef GPUK_LAUNCH_NQ_EXACT
#undef GPUK_LAUNCH_NQ_AS
}

// Lanes and kept chunks per lane of the fp64 kernel; 0 chunks kept = rows beyond 4096 chunks, swept (fp32 rows come here
// for that only).  One chunk (32 bytes) per lane up to 1024 lanes (6 % ahead of two).
void pick_wide_shape(int chunks, int *threads, int *cpl) {
    int n = 1;
    while (n < 4 && chunks > n * kMaxThreads) n *= 2;
    if (chunks > n * kMaxThreads) {
        *cpl = 0;
        *threads = kMaxThreads;
        return;
    }
    *cpl = n;
    *threads = round_up((chunks + n - 1) / n, 64);
}

// Bytes of both inputs from which on fp32 batches gate their stores: with less to read per compute unit than a 16-bit kernel of
// as many lanes has, a small batch has no reason to hold them.  Where the two cross depends on how long a row's own chain is:
// few waves and no codes early, many waves and two chunks per lane late.  Gated / ungated, batches of a quarter of a round to
// one: one wave of one chunk per lane with codes 0.994 at 4 MB, 0.97 at 6; without 0.98 / 0.92 below eleven twentieths of a
// round, above 1.02 at 6, 0.99 at 8; more waves of one chunk without codes 1.04 / 1.03 / 0.97 / 0.90 at 4 / 5 / 6 / 7, with
// 1.03 / 1.02 / 1.01 / 0.98; two chunks with codes 1.02 / 1.00 / 0.97 at 7 / 8 / 9, without 0.95 at 7 (0.99 on nine waves); of
// twelve waves 1.04 / 1.01 / 1.00 at 8 / 9 / 10, 1.01 / 0.97 at 8 / 9 without, four chunks 1.01 / 1.00 / 0.99.
int64_t f32_gate_from_bytes(int64_t tokens, int threads, int nchunk, bool codes) {
    const bool one_wave = threads == 64;
    if (nchunk == 4 || (nchunk == 2 && threads >= 768)) return codes || nchunk == 4 ? 9'200'000 : 8'800'000;
    if (nchunk == 2) return one_wave ? (codes ? 6'500'000 : 5'000'000) : codes ? 8'000'000 : threads < 576 ? 6'500'000 : 7'200'000;
    if (one_wave) return !codes && 20 * tokens > 11 * resident_rows(threads, nchunk) ? 7'500'000 : 4'000'000;
    return codes ? 7'000'000 : 6'000'000;
}

uint32_t f32_store_gate(int64_t tokens, int64_t hidden, int threads, int nchunk, int quant) {
    const bool gated = g_gate >= 0 || tokens * hidden * 8 >= f32_gate_from_bytes(tokens, threads, nchunk, quant != GPUK_QUANT_NONE);
    return gated ? store_gate(tokens, hidden * 4, threads, nchunk, RowType::F32, quant) : 0;
}

template <int QUANT>
int launch_f32_rows(const void *x, const void *residual_in, const void *gamma, void *residual_out, void *norm_out,
                    float *scale, int64_t tokens, int64_t hidden, float eps, float fp8_max, hipStream_t stream) {
    const int chunks = (int)(hidden / 4);
    int threads, nchunk;
    pick_shape(tokens, chunks, RowType::F32, QUANT != GPUK_QUANT_NONE, &threads, &nchunk);
    const bool exact = (int64_t)threads * nchunk == chunks;
    const uint32_t gate = f32_store_gate(tokens, hidden, threads, nchunk, QUANT);
    // Weights at once: more than a round, or waves that wait little for each other (see add_rmsnorm_quant_f32_rows).
    const bool few_waves = threads < 192 || (nchunk == 2 && threads <= 256 && tokens <= kComputeUnits);
    const bool short_chain = QUANT == GPUK_QUANT_NONE && ((hidden > 6144 && tokens <= 32) ||
                                                          (!exact && nchunk == 2 && (threads < 448 || (threads <= 576 && tokens <= 128))));
    const bool at_once = tokens > resident_rows(threads, nchunk) || few_waves || short_chain;
    const uint32_t shape = (uint32_t)threads | ((uint32_t)row_group_shift(tokens, hidden * 4) << 16) | ((line_mask(threads, nchunk, chunks) & ~1u) << 24);
    const RowParameters p = row_parameters(x, residual_in, gamma, residual_out, norm_out, scale, tokens, chunks, shape, gate, hidden, eps, fp8_max);
#define GPUK_LAUNCH_F32_AS(N, EXACT, FORM)                                                                              \
    return launch_kernel(add_rmsnorm_quant_f32_rows<N, QUANT, EXACT, F32Form::FORM>, dim3((unsigned)tokens), (uint32_t)threads, 0, stream, \
                         p.first, p.second, p.third, p.rest)
#define GPUK_LAUNCH_F32_EXACT(N, EXACT)                                                                                \
    do {                                                                                                               \
        if (gate) {                                                                                                    \
            if constexpr (N == 1 && QUANT == GPUK_QUANT_NONE) {                                                        \
                if (threads >= 512) GPUK_LAUNCH_F32_AS(N, EXACT, GATED_LANDED);                                        \
                else GPUK_LAUNCH_F32_AS(N, EXACT, GATED);                                                              \
            } else {                                                                                                   \
                GPUK_LAUNCH_F32_AS(N, EXACT, GATED);                                                                   \
            }                                                                                                          \
        }                                                                                                              \
        else if (at_once) GPUK_LAUNCH_F32_AS(N, EXACT, STREAM);                                                        \
        else if constexpr (N == 1) GPUK_LAUNCH_F32_AS(N, EXACT, LANDED);                                               \
        else if constexpr (N == 4) GPUK_LAUNCH_F32_AS(N, EXACT, LAST);                                                 \
        else if (hidden < 7168) GPUK_LAUNCH_F32_AS(N, EXACT, LANDED);                                                  \
        else GPUK_LAUNCH_F32_AS(N, EXACT, LAST);                                                                       \
    } while (0)
#define GPUK_LAUNCH_F32(N)                                                                                             \
    do {                                                                                                               \
        if (exact) GPUK_LAUNCH_F32_EXACT(N, true);                                                                     \
        else GPUK_LAUNCH_F32_EXACT(N, false);                                                                          \
    } while (0)
    switch (nchunk) {
        case 1: GPUK_LAUNCH_F32(1); break;
        case 2: GPUK_LAUNCH_F32(2); break;
        case 4: GPUK_LAUNCH_F32(4); break;
        default: return GPUK_ERR_INTERNAL;
    }
#undef GPUK_LAUNCH_F32
#undef GPUK_LAUNCH_F32_EXACT
#undef GPUK_LAUNCH_F32_AS
}

template <typename F, int QUANT>
int launch_wide(const void *x, const void *residual_in, const void *gamma, void *residual_out, void *norm_out,
                float *scale, int64_t tokens, int64_t hidden, float eps, float fp8_max, hipStream_t stream) {
    const int chunks = (int)(hidden / 4);
    if constexpr (sizeof(F) == 4) {
        if (chunks <= kMaxChunksF32 * kMaxThreads) {  // in pieces as for 16-bit rows, see launches_for
            const int64_t piece = first_piece(tokens, chunks, RowType::F32, QUANT != GPUK_QUANT_NONE);
            for (int64_t first = 0; first < tokens; first = first ? tokens : piece) {
                const int64_t in_bytes = first * hidden * 4, out_bytes = first * hidden * (QUANT == GPUK_QUANT_NONE ? 4 : 1);
                const int rc = launch_f32_rows<QUANT>(static_cast<const char *>(x) + in_bytes, static_cast<const char *>(residual_in) + in_bytes,
                                                      gamma, static_cast<char *>(residual_out) + in_bytes, static_cast<char *>(norm_out) + out_bytes,
                                                      QUANT == GPUK_QUANT_FP8_DYNAMIC ? scale + first : scale, first ? tokens - first : piece,
                                                      hidden, eps, fp8_max, stream);
                if (rc != GPUK_OK) return rc;
            }
            return GPUK_OK;
        }
    }
    int threads, cpl;
    pick_wide_shape(chunks, &threads, &cpl);
#define GPUK_LAUNCH_WIDE(CPL)                                                                                          \
    add_rmsnorm_quant_wide_rows<F, QUANT, CPL><<<dim3((unsigned)tokens), threads, 0, stream>>>(                        \
        static_cast<const wide4<F> *>(x), static_cast<const wide4<F> *>(residual_in),                                  \
        static_cast<const wide4<F> *>(gamma), static_cast<wide4<F> *>(residual_out), norm_out, scale, chunks,          \
        (float)hidden, eps, fp8_max)
    if constexpr (sizeof(F) == 4) {
        GPUK_LAUNCH_WIDE(0);
    } else {
        switch (cpl) {
            case 1: GPUK_LAUNCH_WIDE(1); break;
            case 2: GPUK_LAUNCH_WIDE(2); break;
            case 4: GPUK_LAUNCH_WIDE(4); break;
            default: GPUK_LAUNCH_WIDE(0); break;
        }
    }
#undef GPUK_LAUNCH_WIDE
    return hip_status(hipGetLastError());
}

template <typename F>
int launch_quant_wide(int quant_mode, const void *x, const void *residual_in, const void *gamma, void *residual_out,
                      void *norm_out, float *scale, int64_t tokens, int64_t hidden, float eps, float fp8_max,
                      hipStream_t stream) {
    switch (quant_mode) {
        case GPUK_QUANT_NONE:
            return launch_wide<F, GPUK_QUANT_NONE>(x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, stream);
        case GPUK_QUANT_FP8_DYNAMIC:
            return launch_wide<F, GPUK_QUANT_FP8_DYNAMIC>(x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, stream);
        case GPUK_QUANT_FP8_STATIC:
            return launch_wide<F, GPUK_QUANT_FP8_STATIC>(x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, stream);
        default:
            return GPUK_ERR_UNSUPPORTED;
    }
}

template <typename T>
int launch_quant(int quant_mode, const void *x, const void *residual_in, const void *gamma, void *residual_out,
                 void *norm_out, float *scale, int64_t tokens, int64_t hidden, float eps, float fp8_max,
                 hipStream_t stream) {
    switch (quant_mode) {
        case GPUK_QUANT_NONE:
            return launch<T, GPUK_QUANT_NONE>(x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, stream);
        case GPUK_QUANT_FP8_DYNAMIC:
            return launch<T, GPUK_QUANT_FP8_DYNAMIC>(x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, stream);
        case GPUK_QUANT_FP8_STATIC:
            return launch<T, GPUK_QUANT_FP8_STATIC>(x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, stream);
        default:
            return GPUK_ERR_UNSUPPORTED;
    }
}

}  // namespace

void set_norm_quant_tuning(int key, int value) {
    if (key == 0) g_force_nchunk = value;
    if (key == 1) g_force_threads = value;
    if (key == 5) g_row_group_shift = value;
    if (key == 6) g_gate = value;
    if (key == 7) g_pieces = value;
}

}  // namespace gpuk

// profiling build: where the kernels of this file write their phase stamps
GPUK_STAMPS_SETTER(gpuk_stamps_set_norm_quant)

extern "C" int gpuk_add_rmsnorm_quant_traffic_only(const void *x, const void *residual_in, void *residual_out,
                                                   void *codes, float *scale, int64_t tokens, int64_t hidden,
                                                   void *stream) {
    using namespace gpuk;
    if (tokens <= 0 || hidden <= 0 || hidden % 8 != 0 || tokens > 0x7fffffffLL) return GPUK_ERR_INVALID_ARG;
    if (!x || !residual_in || !residual_out || !codes || !scale) return GPUK_ERR_INVALID_ARG;
    if (!aligned16(x) || !aligned16(residual_in) || !aligned16(residual_out) || !aligned8(codes)) return GPUK_ERR_MISALIGNED;
    const int chunks = (int)(hidden / 8);
    if (const int64_t piece = first_piece(tokens, chunks, RowType::BF16); piece < tokens) {  // two launches where the op takes two
        const int rc = gpuk_add_rmsnorm_quant_traffic_only(x, residual_in, residual_out, codes, scale, piece, hidden, stream);
        if (rc != GPUK_OK) return rc;
        const int64_t wide = piece * hidden * 2, narrow = piece * hidden;
        return gpuk_add_rmsnorm_quant_traffic_only(static_cast<const char *>(x) + wide, static_cast<const char *>(residual_in) + wide,
                                                   static_cast<char *>(residual_out) + wide, static_cast<char *>(codes) + narrow,
                                                   scale + piece, tokens - piece, hidden, stream);
    }
    int threads, nchunk;
    pick_shape(tokens, chunks, RowType::BF16, true, &threads, &nchunk);
    if (nchunk == 0) return GPUK_ERR_UNSUPPORTED;  // rows that do not stay in registers
    const int group_shift = row_group_shift(tokens, hidden * 2);
    const int remap_end = group_shift > 0 ? (int)((tokens >> (3 + group_shift)) << (3 + group_shift)) : 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto xs = static_cast<const u32x4 *>(x), rs = static_cast<const u32x4 *>(residual_in);
    auto ro = static_cast<u32x4 *>(residual_out);
    auto co = static_cast<u32x2 *>(codes);
    const dim3 grid((unsigned)tokens);
    const uint32_t gate = store_gate(tokens, hidden * 2, threads, nchunk, RowType::BF16, GPUK_QUANT_FP8_DYNAMIC);
    // (one chunk per lane without a gate: the operator's rows start at lane 0)
    const uint32_t mask = nchunk == 1 && gate == 0 ? 0u : line_mask(threads, nchunk, chunks);
    const uint32_t shape = (uint32_t)threads | ((uint32_t)group_shift << 16) | (mask << 24);
    switch (nchunk) {
        case 1: add_rmsnorm_quant_traffic_only<1><<<grid, threads, 0, s>>>(xs, rs, chunks, remap_end, shape, gate, ro, co, scale); break;
        case 2: add_rmsnorm_quant_traffic_only<2><<<grid, threads, 0, s>>>(xs, rs, chunks, remap_end, shape, gate, ro, co, scale); break;
        case 4: add_rmsnorm_quant_traffic_only<4><<<grid, threads, 0, s>>>(xs, rs, chunks, remap_end, shape, gate, ro, co, scale); break;
        default: add_rmsnorm_quant_traffic_only<8><<<grid, threads, 0, s>>>(xs, rs, chunks, remap_end, shape, gate, ro, co, scale); break;
    }
    return hip_status(hipGetLastError());
}

extern "C" int gpuk_add_rmsnorm_quant_launch_shape_of(int64_t tokens, int64_t hidden, int dtype, int quant_mode, int *lanes_per_row,
                                                      int *chunks_per_lane) {
    using namespace gpuk;
    if (tokens <= 0 || hidden <= 0 || !lanes_per_row || !chunks_per_lane) return GPUK_ERR_INVALID_ARG;
    if (dtype != GPUK_DTYPE_BF16 && dtype != GPUK_DTYPE_FP16 && dtype != GPUK_DTYPE_F32 && dtype != GPUK_DTYPE_F64) return GPUK_ERR_UNSUPPORTED;
    if (quant_mode != GPUK_QUANT_NONE && quant_mode != GPUK_QUANT_FP8_DYNAMIC && quant_mode != GPUK_QUANT_FP8_STATIC) return GPUK_ERR_UNSUPPORTED;
    const bool wide = dtype == GPUK_DTYPE_F32 || dtype == GPUK_DTYPE_F64, codes = quant_mode != GPUK_QUANT_NONE;
    if (hidden % 8 != 0) return GPUK_ERR_UNSUPPORTED;  // the rule of gpuk_add_rmsnorm_quant, for every dtype
    if (dtype == GPUK_DTYPE_F32 && hidden / 4 <= kMaxChunksF32 * kMaxThreads) {
        const int chunks = (int)(hidden / 4);
        pick_shape(first_piece(tokens, chunks, RowType::F32, codes), chunks, RowType::F32, codes, lanes_per_row, chunks_per_lane);
        return GPUK_OK;
    }
    if (wide) {  // longer fp32 rows and fp64: 4-element chunks, 0 = rows swept three times
        pick_wide_shape((int)(hidden / 4), lanes_per_row, chunks_per_lane);
        return GPUK_OK;
    }
    const RowType type = dtype == GPUK_DTYPE_FP16 ? RowType::FP16 : RowType::BF16;
    pick_shape(first_piece(tokens, (int)(hidden / 8), type), (int)(hidden / 8), type, codes, lanes_per_row, chunks_per_lane);
    return GPUK_OK;
}

extern "C" int gpuk_add_rmsnorm_quant_launch_shape(int64_t tokens, int64_t hidden, int dtype, int *lanes_per_row, int *chunks_per_lane) {
    return gpuk_add_rmsnorm_quant_launch_shape_of(tokens, hidden, dtype, GPUK_QUANT_FP8_DYNAMIC, lanes_per_row, chunks_per_lane);
}

extern "C" int gpuk_add_rmsnorm_quant_store_gate(int64_t tokens, int64_t hidden, int dtype, int quant_mode, int *ticks) {
    using namespace gpuk;
    if (tokens <= 0 || hidden <= 0 || !ticks) return GPUK_ERR_INVALID_ARG;
    if (hidden % 8 != 0) return GPUK_ERR_UNSUPPORTED;
    if (quant_mode != GPUK_QUANT_NONE && quant_mode != GPUK_QUANT_FP8_DYNAMIC && quant_mode != GPUK_QUANT_FP8_STATIC) return GPUK_ERR_UNSUPPORTED;
    int threads, nchunk;
    *ticks = 0;
    if (dtype == GPUK_DTYPE_F64) return GPUK_OK;  // (no gate in the kernels of fp64 and of swept rows)
    if (dtype == GPUK_DTYPE_F32) {
        const int chunks = (int)(hidden / 4);
        if (chunks > kMaxChunksF32 * kMaxThreads) return GPUK_OK;
        tokens = first_piece(tokens, chunks, RowType::F32, quant_mode != GPUK_QUANT_NONE);
        pick_shape(tokens, chunks, RowType::F32, quant_mode != GPUK_QUANT_NONE, &threads, &nchunk);
        *ticks = (int)f32_store_gate(tokens, hidden, threads, nchunk, quant_mode);
        return GPUK_OK;
    }
    if (dtype != GPUK_DTYPE_BF16 && dtype != GPUK_DTYPE_FP16) return GPUK_ERR_UNSUPPORTED;
    const RowType type = dtype == GPUK_DTYPE_FP16 ? RowType::FP16 : RowType::BF16;
    tokens = first_piece(tokens, (int)(hidden / 8), type);
    pick_shape(tokens, (int)(hidden / 8), type, quant_mode != GPUK_QUANT_NONE, &threads, &nchunk);
    if (nchunk) *ticks = (int)store_gate(tokens, hidden * 2, threads, nchunk, type, quant_mode);
    return GPUK_OK;
}

extern "C" int gpuk_add_rmsnorm_quant(const void *x, const void *residual_in, const void *gamma, void *residual_out,
                                      void *norm_out, float *scale, int64_t tokens, int64_t hidden, float eps,
                                      int dtype, int quant_mode, float fp8_max, void *stream) {
    using namespace gpuk;
    if (tokens < 0 || hidden <= 0) return GPUK_ERR_INVALID_ARG;
    if (hidden % 8 != 0) return GPUK_ERR_UNSUPPORTED;           // rows are moved in 16-byte chunks
    if (tokens > 0x7fffffffLL || hidden / 8 > 0x7fffffffLL) return GPUK_ERR_UNSUPPORTED;
    if (!(fp8_max > 0.f) && quant_mode != GPUK_QUANT_NONE) return GPUK_ERR_INVALID_ARG;
    if (quant_mode == GPUK_QUANT_FP8_E4M3FNUZ) return GPUK_ERR_UNSUPPORTED;  // gfx950 encodes OCP e4m3fn only
    if (tokens == 0) return GPUK_OK;
    if (!x || !residual_in || !gamma || !residual_out || !norm_out) return GPUK_ERR_INVALID_ARG;
    if (quant_mode != GPUK_QUANT_NONE && !scale) return GPUK_ERR_INVALID_ARG;
    if (!aligned16(x) || !aligned16(residual_in) || !aligned16(gamma) || !aligned16(residual_out)) return GPUK_ERR_MISALIGNED;
    if (!(quant_mode == GPUK_QUANT_NONE ? aligned16(norm_out) : aligned8(norm_out))) return GPUK_ERR_MISALIGNED;
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (dtype) {
        case GPUK_DTYPE_BF16:
            return launch_quant<BF16>(quant_mode, x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, s);
        case GPUK_DTYPE_FP16:
            return launch_quant<FP16>(quant_mode, x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, s);
        case GPUK_DTYPE_F32:
            return launch_quant_wide<float>(quant_mode, x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, s);
        case GPUK_DTYPE_F64:
            return launch_quant_wide<double>(quant_mode, x, residual_in, gamma, residual_out, norm_out, scale, tokens, hidden, eps, fp8_max, s);
        default:
            return GPUK_ERR_UNSUPPORTED;
    }
}
