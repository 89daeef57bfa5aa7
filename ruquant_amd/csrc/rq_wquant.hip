// Weight-side quantizer and the dequantizers of the four block types, on the GPU: what ggml calls from_float_ref and
// to_float for W4A4 / W4A4H / A4 / A4H (reference patch lines 2507-2580, 2681-2710, 2738-2773).
//
// A converter quantizes whole tensors; the reference does it a row at a time on the host. The one quantity whose order of
// operations matters is the double-precision error sum of the scale search, and of it only which of the thirteen clip ratios
// has the smallest is kept. So the sums are taken in fp32 first, over all lanes and in any order, with a bound on what that
// can change; where the smallest two are further apart than the bound allows, the reference's sums are too, and the search is
// over. Where they are not (a row in a hundred of gaussian weights), the same again in double precision, and only where that cannot
// tell either (ties, infinities, NaNs, scales out of range) do lanes add up the reference's sums in its element order. A tensor that
// lies on an int4 grid (one that was dequantized) has a ratio without any error: settled at once.
//   * search kernels: a workgroup per row, or sixteen lanes per weight group of 256 or 64;
//   * encode kernel: a workgroup per row turns the chosen scale(s) into codes, row sum / multiplier headers and
//     blocks;
//   * dequantize kernel: a workgroup per row decodes blocks into the padded LDS row and, for the rotated types, runs
//     the Sylvester butterflies and the transposed Paley stage before the row leaves for memory.
// The forward rotation of W4A4H weights is the activation kernel's rotate-only mode.
#include "rq_hadamard.h"

#include <math.h>
#include <string.h>

#pragma clang fp contract(off)

namespace rq {

hipError_t launch_rotate_quant(const RotQuantArgs &a, hipStream_t stream);

namespace {

using namespace had;

__device__ __forceinline__ float absmax3_raw(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

constexpr int kRatios = 13;          // clip ratios 1.0, 0.975, ... 0.7 (reference lines 2514-2524)
constexpr int kSearchThreads = 64;   // four segments of sixteen lanes: single wavefronts spread evenly over the SIMDs

struct SearchArgs {
    const float *x;    // rows of K floats, ld apart
    int64_t ld;
    int64_t segments;  // rows * per_row
    int per_row;       // segments per row
    int n;             // floats per segment
    float *scale;      // [segments]
};

// What the fp32 sums may be off by, relative to the exact sum of the reference's squares. The quotient t = x * (1 / s) differs
// from x / s by less than 8e-6 (|x / s| is at most 10), so a code differs from the reference's only where x / s is that near
// to a half-way point; its error then is (0.5 +- 9e-6) s either way, and the square off by 7.2e-5 of itself. The errors
// themselves and their squares are rounded as the reference's or once (6e-8), and a sum goes through at most 148 additions: 128
// elements of a thread, four steps over its row of sixteen lanes, sixteen such rows: 8.9e-6. Together below 8.2e-5; the reference's
// own rounding (32768 additions in double precision, 4e-12) is nothing to that. Two sums can have their order changed only if they
// are within (1 + 8.2e-5) / (1 - 8.2e-5) of each other.
constexpr float kApart = 1.0f + 1.7e-4f;
// ... and squares below the normal numbers lose at most half of the smallest denormal each, 32768 of them 2.3e-41, in either sum. (A
// sum of zero, of a row that lies on the grid of one of the ratios, is told from the others by this alone.)
constexpr float kUnderflow = 1e-40f;
// The double-precision sums of the second look have the reference's terms and at most 400 roundings, the reference's own sums at
// most 32768: 3.7e-12 and 4.5e-14. (No square of a difference of floats underflows there: a sum is zero where every term is.)
constexpr double kApart64 = 1.0 + 1e-11;

__device__ __forceinline__ float ratio_scale(float amax, int r) { return amax * (1.0f - 0.025f * (float) r) / 7.0f; }
// what stands in place of a scale that these sums leave open, for rq_wsearch_open_kernel
constexpr float kOpen = -1.0f;
__device__ __forceinline__ bool reciprocal_holds(float rs) { return rs < 1e37f && rs > 2e-38f; }

// the sums of the squared errors of one element under all ratios (rs: reciprocals of the scales)
__device__ __forceinline__ void add_errors(float x, const float (&sc)[kRatios], const float (&rs)[kRatios], float (&acc)[kRatios]) {
#pragma unroll
    for (int r = 0; r < kRatios; ++r) {
        float q = rintf(x * rs[r]);
        if (r > 2) q = __builtin_amdgcn_fmed3f(q, -8.0f, 7.0f);   // (|x / s| is at most 7 / 0.95 before that)
        const float e = q * sc[r] - x;
        acc[r] = __builtin_fmaf(e, e, acc[r]);
    }
}

// v plus the value of lane `ctrl` of the same row of sixteen
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// the sum over a row of sixteen lanes, in all of them
__device__ __forceinline__ float row_sum(float v) {
    v = dpp_add<0xB1>(v);    // quad_perm [1, 0, 3, 2]
    v = dpp_add<0x4E>(v);    // quad_perm [2, 3, 0, 1]
    v = dpp_add<0x141>(v);   // row_half_mirror
    return dpp_add<0x140>(v);   // row_mirror
}

// a sum above this is larger than the smallest one in the reference's sums too
__device__ __forceinline__ float bound_of(float least) { return __builtin_fmaf(least, kApart, kUnderflow); }
// whether the smallest of the sums is the smallest in the reference's sums too (not with a NaN or an infinity among them)
__device__ __forceinline__ bool settled(const float (&sum)[kRatios], float &least) {
    float second = INFINITY, all = sum[0];
    least = sum[0];
#pragma unroll
    for (int r = 1; r < kRatios; ++r) {
        second = __builtin_amdgcn_fmed3f(least, second, sum[r]);
        least = fminf(least, sum[r]);
        all += sum[r];
    }
    return second > bound_of(least) && all < INFINITY;
}

// Weight groups of 256 (V = 4) or 64 (V = 1): sixteen lanes per group, V blocks of 64 elements in their registers.
// What bounds it: vector instructions, six per element and ratio. Search and encoding of 4096 x 17408, groups of 64, with a lane per
// ratio and the sums in order from the start 402 us, this way 306 (search 250); groups of 256 299 and 217 (134). 6144 x 5120 on a
// grid, groups of 64: in order 329 us, this way 129 (430 while a sum of zero was left to the search in order); of 256 298, 91 (423).
template <int V>
__global__ void __launch_bounds__(kSearchThreads, 4) rq_wsearch_groups_kernel(const SearchArgs a) {
    const int tid = threadIdx.x, r = tid & 15;
    int64_t seg = (int64_t) blockIdx.x * (kSearchThreads / 16) + (tid >> 4);
    const bool live = seg < a.segments;
    if (!live) seg = a.segments - 1;   // idle lanes follow a live segment
    const int64_t row = seg / a.per_row;
    const float *x = a.x + row * a.ld + (seg - row * a.per_row) * (int64_t) a.n;
    float4 v[V];
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = reinterpret_cast<const float4 *>(x)[16 * k + r];
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < V; ++k) amax = fmaxf(fmaxf(fmaxf(fmaxf(amax, fabsf(v[k].x)), fabsf(v[k].y)), fabsf(v[k].z)), fabsf(v[k].w));
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 16));

    const bool tries = amax > 0.0f && r < kRatios;
    const float s = tries ? ratio_scale(amax, r) : 1.0f;
    // lane r's scale to all lanes of the group (row_newbcast)
    const float inv = 1.0f / s;
    float sc[kRatios], rs[kRatios], sum[kRatios];
#define RQ_FROM_LANE(R)                                                                                                      \
    sc[R] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x150 + R, 0xF, 0xF, false)); \
    rs[R] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, inv), 0x150 + R, 0xF, 0xF, false));
    RQ_FROM_LANE(0) RQ_FROM_LANE(1) RQ_FROM_LANE(2) RQ_FROM_LANE(3) RQ_FROM_LANE(4) RQ_FROM_LANE(5) RQ_FROM_LANE(6)
    RQ_FROM_LANE(7) RQ_FROM_LANE(8) RQ_FROM_LANE(9) RQ_FROM_LANE(10) RQ_FROM_LANE(11) RQ_FROM_LANE(12)
#undef RQ_FROM_LANE
#pragma unroll
    for (int i = 0; i < kRatios; ++i) sum[i] = 0.0f;
    float4 w = v[0];
#pragma unroll 1
    for (int k = 0; k < V; ++k) {
        // (read again: kept, the registers of the four blocks let the compiler mix their sums, and spill)
        const float4 next = reinterpret_cast<const float4 *>(x)[16 * (k + 1 < V ? k + 1 : k) + r];
        add_errors(w.x, sc, rs, sum);
        add_errors(w.y, sc, rs, sum);
        add_errors(w.z, sc, rs, sum);
        add_errors(w.w, sc, rs, sum);
        w = next;
    }
#pragma unroll
    for (int i = 0; i < kRatios; ++i) sum[i] = row_sum(sum[i]);
    float least;
    // (the largest and the smallest reciprocal)
    bool sure = settled(sum, least) && reciprocal_holds(rs[0]) && reciprocal_holds(rs[kRatios - 1]);
    float scale = 0.0f;
#pragma unroll
    for (int i = 0; i < kRatios; ++i) scale = sum[i] == least ? sc[i] : scale;
    if (!(amax > 0.0f)) {   // (a group of zeros or of NaNs)
        scale = 0.0f;
        sure = true;
    }
    // Two ratios without an error, or one and squares that underflow (a group with one value, negative, beside zeros is on the grid
    // of the first ratio and of the sixth): the first whose errors are all zero, as the reference's sum then is, and of no ratio
    // before it. (No quotient at a half-way point has an error of zero, so its code is the reference's.)
    if (!sure && least == 0.0f && reciprocal_holds(rs[0]) && reciprocal_holds(rs[kRatios - 1])) {
#pragma unroll 1
        for (int i = 0; i < kRatios && !sure; ++i) {   // (the same for all lanes of the group)
            const float si = __shfl(s, i, 16), ri = __shfl(inv, i, 16);
            float worst = 0.0f;
#pragma unroll 1
            for (int k = 0; k < V; ++k) {
                const float4 y = reinterpret_cast<const float4 *>(x)[16 * k + r];
                const float ys[4] = { y.x, y.y, y.z, y.w };
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    worst = fmaxf(worst, fabsf(__builtin_amdgcn_fmed3f(rintf(ys[j] * ri), -8.0f, 7.0f) * si - ys[j]));
                }
            }
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) worst = fmaxf(worst, __shfl_xor(worst, off, 16));
            if (worst == 0.0f) {
                scale = si;
                sure = true;
            }
        }
    }
    if (live && r == 0) a.scale[seg] = sure ? scale : kOpen;
}

// Few groups go to the search in order at once: its one launch is as long as the two that spare it. Search and encoding of K = 256 /
// 1024 / 5120 gaussian inputs in us, in order -> this way: groups of 256 (at K = 256 whole rows), 3.2 Mi floats 31.4 -> 32.7 / 24.4 ->
// 25.6 / 23.8 -> 25.4, 4.6 Mi 41.2 -> 42.1 / 29.3 -> 30.5 / 28.7 -> 30.0, 6 Mi 50.0 -> 49.2 / 34.8 -> 35.3 / 34.1 -> 33.5; of 64, 2.6 Mi
// 26.9 -> 27.5 / 21.1 -> 21.5 / 20.9 -> 21.7, 3.2 Mi 31.5 -> 31.3 / 24.6 -> 24.5 / 23.9 -> 24.0, 4.6 Mi 42.8 -> 42.1 / 34.2 -> 33.0 / 32.4 ->
// 31.3. (Tensors on a grid are faster this way from the first row on: in order their quotients lie at half-way points, and lanes divide.)
constexpr int64_t few_floats(int n) { return n == 64 ? 7 << 19 : 5 << 20; }

// Rows: a workgroup each, which reads its row twice (the second time out of the caches).
// What bounds it: vector instructions, six per element and ratio (four of them of two cycles, beside a second wavefront).
// Search and encoding, 5120 inputs, with four rows per wavefront, a lane per ratio and the sums in order from the start: 2048 rows
// 137 us, 4096 173, 6144 187; this way 39, 63, 85 (search of 4096: 45). 17408 inputs, 1800 rows 441 and 97. 6144 x 5120 on a grid:
// in order 441, this way 86 (495 while a sum of zero was left open).
constexpr int kRowThreads = 256;
__global__ void __launch_bounds__(kRowThreads) rq_wsearch_rows_kernel(const SearchArgs a) {
    __shared__ float s_sum[kRowThreads / 16][kRatios];   // per row of sixteen lanes
    __shared__ float s_sc[kRatios], s_rs[kRatios], s_all[kRatios];
    __shared__ float s_max[kRowThreads / 64];
    __shared__ double s_err[kRowThreads / 64];
    const int tid = threadIdx.x, wave = tid >> 6;
    const float *x = a.x + (int64_t) blockIdx.x * a.ld;
    const float4 *xv = reinterpret_cast<const float4 *>(x);
    const int nv = a.n >> 2;   // (a multiple of 64: whole wavefronts have an element or none)
    float amax = 0.0f;
    constexpr int kBatch = 5;
    for (int i0 = tid; i0 < nv; i0 += kBatch * kRowThreads) {
        float4 v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int i = i0 + k * kRowThreads;
            v[k] = xv[i < nv ? i : i0];
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) amax = fmaxf(fmaxf(fmaxf(fmaxf(amax, fabsf(v[k].x)), fabsf(v[k].y)), fabsf(v[k].z)), fabsf(v[k].w));
    }
    amax = wave_max(amax);
    if ((tid & 63) == 0) s_max[wave] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    if (!(amax > 0.0f)) {   // (a row of zeros or of NaNs)
        if (tid == 0) a.scale[blockIdx.x] = 0.0f;
        return;
    }
    if (tid < kRatios) {
        const float s = ratio_scale(amax, tid);
        s_sc[tid] = s;
        s_rs[tid] = 1.0f / s;
    }
    __syncthreads();
    // (the same in all threads: scalar registers)
    float sc[kRatios], rs[kRatios], sum[kRatios];
#pragma unroll
    for (int r = 0; r < kRatios; ++r) {
        sc[r] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, s_sc[r])));
        rs[r] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, s_rs[r])));
        sum[r] = 0.0f;
    }
    float4 v = xv[tid < nv ? tid : 0];
    for (int i = tid; i < nv; i += kRowThreads) {
        const float4 next = xv[i + kRowThreads < nv ? i + kRowThreads : i];
        add_errors(v.x, sc, rs, sum);
        add_errors(v.y, sc, rs, sum);
        add_errors(v.z, sc, rs, sum);
        add_errors(v.w, sc, rs, sum);
        v = next;
    }
#pragma unroll
    for (int r = 0; r < kRatios; ++r) {
        const float t = row_sum(sum[r]);
        if ((tid & 15) == 0) s_sum[tid >> 4][r] = t;
    }
    __syncthreads();
    if (tid < kRatios) {
        float t = 0.0f;
#pragma unroll
        for (int k = 0; k < kRowThreads / 16; ++k) t += s_sum[k][tid];
        s_all[tid] = t;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRatios; ++r) sum[r] = s_all[r];
    float least;
    const bool normal = reciprocal_holds(rs[0]) && reciprocal_holds(rs[kRatios - 1]);
    if (settled(sum, least) && normal) {
        float scale = 0.0f;
#pragma unroll
        for (int r = 0; r < kRatios; ++r) scale = sum[r] == least ? sc[r] : scale;
        if (tid == 0) a.scale[blockIdx.x] = scale;
        return;
    }

    // The second look, at the ratios that the first could not tell from the smallest: the reference's terms, added up in
    // double precision by all threads.
    bool finite = normal;
#pragma unroll
    for (int r = 0; r < kRatios; ++r) finite = finite && sum[r] < INFINITY;
    if (finite) {
        double err64[2] = { INFINITY, INFINITY };   // the smallest and the second smallest
        int arg = 0;
        for (int r = 0; r < kRatios; ++r) {
            if (s_all[r] > bound_of(least)) continue;   // (uniform)
            const float s = s_sc[r], inv = s_rs[r];
            double err = 0.0;
            for (int i = tid; i < nv; i += kRowThreads) {
                const float4 w = xv[i];
                const float xs[4] = { w.x, w.y, w.z, w.w };
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float t = xs[j] * inv;
                    float q = rintf(t);
                    if (!(fabsf(t - q) < 0.49999f)) q = rintf(xs[j] / s);
                    const double e = (double) (fminf(fmaxf(q, -8.0f), 7.0f) * s - xs[j]);
                    err = __builtin_fma(e, e, err);
                }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) err += __shfl_xor(err, off, 64);
            __syncthreads();
            if ((tid & 63) == 0) s_err[wave] = err;
            __syncthreads();
            err = (s_err[0] + s_err[1]) + (s_err[2] + s_err[3]);
            if (err < err64[0]) {
                err64[1] = err64[0];
                err64[0] = err;
                arg = r;
            } else if (err < err64[1]) {
                err64[1] = err;
            }
        }
        if (err64[1] > err64[0] * kApart64 || err64[0] == 0.0) {   // (of ratios without any error the first)
            if (tid == 0) a.scale[blockIdx.x] = s_sc[arg];
            return;
        }
    }
    if (tid == 0) a.scale[blockIdx.x] = kOpen;
}

// The reference's search: sixteen lanes per segment, thirteen of them try one ratio each over the whole segment in element order, and
// a scan in ratio order keeps the first smallest error. (Lanes that are not live follow a live segment, so that the shuffles stay
// uniform.)
// ONE: segments of 64 (a scale per 64 inputs), one block each: nothing to fetch ahead and no eight loads to batch. (With the
// general form's, which fetch the one block again: 4096 x 17408, search and encoding, 450 us against 402.)
template <bool ONE>
__device__ __forceinline__ void search_in_order(const SearchArgs &a, int64_t seg, bool live, float4 (&s_x)[ONE ? 1 : 2][kSearchThreads]) {
    const int tid = threadIdx.x, r = tid & 15;
    const int64_t row = seg / a.per_row;
    const float *x = a.x + row * a.ld + (seg - row * a.per_row) * (int64_t) a.n;
    const int n = a.n;

    // Elements come by the sixteen lanes of a segment together, a block of 64 to a load (n is a multiple of 64). Eight loads at
    // once here: one after the other, this pass alone would be n / 64 trips to memory.
    constexpr int kBatch = ONE ? 1 : 8;
    const float4 *xv = reinterpret_cast<const float4 *>(x) + r;
    const int nv = ONE ? 1 : n >> 6;
    auto block = [&](int k) { return xv[16 * (k < nv ? k : nv - 1)]; };   // (past the end: the last again)
    float amax = 0.0f;
    for (int i0 = 0; i0 < nv; i0 += kBatch) {
        float4 v[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) v[j] = block(i0 + j);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            amax = fmaxf(fmaxf(fmaxf(fmaxf(amax, fabsf(v[j].x)), fabsf(v[j].y)), fabsf(v[j].z)), fabsf(v[j].w));
        }
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 16));

    // (the lanes that try no ratio go through the loop too: they fetch for the others)
    const bool tries = amax > 0.0f && r < kRatios;
    const float s = tries ? ratio_scale(amax, r) : 1.0f;
    double err = 0.0;
    if (__any(tries)) {
        const float rs = 1.0f / s;
        // What bounds this loop: a lane's error sum is a chain of n additions in element order, and there are only
        // 13 lanes per segment to hide it with (6144 rows: 1.5 wavefronts per SIMD), so everything in front of the
        // addition is worked out for kRun elements at once, independent of each other, and the next run's elements
        // are on their way meanwhile. The correctly rounded division, 11 instructions, is only needed where the
        // quotient lies at a rounding boundary: t = x * (1 / s) differs from x / s by less than 4e-6 here (|x / s| is
        // at most 10: two roundings of half a unit in the last place, 1 / s included), so rint agrees unless t is
        // within 1e-5 of a half-way point; those elements (one in 50,000), infinities, NaNs and scales whose
        // reciprocal is not a normal number take the division.
        // A block goes through LDS, where every lane reads its segment's elements, and is requested three blocks before it is
        // worked on.
        constexpr int kRun = 8;
        const bool normal = reciprocal_holds(rs);
        float4 ahead[2];
        if constexpr (!ONE) {
            ahead[0] = block(1);
            ahead[1] = block(2);
        }
        s_x[0][tid] = block(0);
        for (int k0 = 0; k0 < nv; k0 += 2) {
#pragma unroll
          for (int h = 0; h < (ONE ? 1 : 2); ++h) {
            const int k = k0 + h;
            if (k >= nv) break;   // (uniform)
            if constexpr (!ONE) {
                s_x[h ^ 1][tid] = ahead[h];
                ahead[h] = block(k + 3);
            }
            // (one wavefront: its LDS operations are carried out in order)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int d = 0; d < 64 / kRun; ++d) {
                const float4 x0 = s_x[h][(tid & 48) + 2 * d], x1 = s_x[h][(tid & 48) + 2 * d + 1];
                const float xs[kRun] = { x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w };
                float q[kRun], off[kRun];
#pragma unroll
                for (int j = 0; j < kRun; ++j) {
                    const float t = xs[j] * rs;
                    q[j] = rintf(t);
                    off[j] = t - q[j];
                    q[j] = __builtin_amdgcn_fmed3f(q[j], -8.0f, 7.0f);
                }
                // (a NaN element does not show here and need not: it makes the sum NaN whatever its code)
                float far = absmax3_raw(0.0f, off[0], off[1]);
#pragma unroll
                for (int j = 2; j < kRun; j += 2) far = absmax3_raw(far, off[j], off[j + 1]);
                if (tries && !(normal && far < 0.49999f)) {
#pragma unroll
                    for (int j = 0; j < kRun; ++j) q[j] = fminf(fmaxf(rintf(xs[j] / s), -8.0f), 7.0f);
                }
                // The error e = q s - x in fp32, converted once, instead of the reference's two conversions and a
                // double-precision subtraction: fp32 loses nothing. q is x / s rounded, and |x / s| is at most 10 and
                // clamped to -8 or 7, so q s is 0 or lies between half of x and twice x, and such a difference is exact
                // (a difference that overflows is the same infinity either way). e * e has at most 48 significant bits: exact
                // in double precision, so the one rounding of the fused form is the reference's rounding of the sum.
                double e[kRun];
#pragma unroll
                for (int j = 0; j < kRun; ++j) e[j] = (double) (q[j] * s - xs[j]);
#pragma unroll
                for (int j = 0; j < kRun; ++j) err = __builtin_fma(e[j], e[j], err);
            }
          }
        }
    }
    if (!tries) err = INFINITY;
    // first smallest error in ratio order, as the reference's `err < best_err` scan
    const int base = (tid & 63) & ~15;
    float best_s = 0.0f;
    double best_err = INFINITY;
#pragma unroll
    for (int k = 0; k < kRatios; ++k) {
        const double ek = __shfl(err, base + k, 64);
        const float sk = __shfl(s, base + k, 64);
        if (ek < best_err) {
            best_err = ek;
            best_s = sk;
        }
    }
    if (live && r == 0) a.scale[seg] = best_s;
}

// every segment
template <bool ONE>
__global__ void __launch_bounds__(kSearchThreads) rq_wsearch_kernel(const SearchArgs a) {
    __shared__ float4 s_x[ONE ? 1 : 2][kSearchThreads];   // two blocks of 64 elements of each of the four segments
    const int64_t seg = (int64_t) blockIdx.x * (kSearchThreads / 16) + (threadIdx.x >> 4);
    const bool live = seg < a.segments;
    search_in_order<ONE>(a, live ? seg : a.segments - 1, live, s_x);
}

// The segments that the kernels above left open: a wavefront looks through CHUNK segments and takes the open ones four at a time. (A
// wavefront for 64 groups: with 16 the look alone costs gaussian tensors 2 to 3 %, 6144 x 5120, groups of 64, 134.8 -> 139.1 us.)
template <bool ONE, int CHUNK>
__global__ void __launch_bounds__(kSearchThreads) rq_wsearch_open_kernel(const SearchArgs a) {
    __shared__ float4 s_x[ONE ? 1 : 2][kSearchThreads];
    const int tid = threadIdx.x;
    const int64_t seg0 = (int64_t) blockIdx.x * CHUNK;
    const bool mine = tid < CHUNK && seg0 + tid < a.segments;
    uint64_t open = __ballot(mine && a.scale[seg0 + (mine ? tid : 0)] < 0.0f);
    while (open != 0) {
        // the first four; a row of lanes without one follows the first
        int64_t seg = seg0 + __builtin_ctzll(open);
        bool live = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (open != 0 && k == tid >> 4) {
                seg = seg0 + __builtin_ctzll(open);
                live = true;
            }
            open &= open - 1;   // (zero stays zero)
        }
        search_in_order<ONE>(a, seg, live, s_x);
    }
}

struct EncodeArgs {
    const float *x;
    int64_t ld;
    int K;
    int per_row;        // scales per row: 1, K / 256 or K / 64
    int groups;         // 0: one scale per row, legacy header; 1: weight groups (multiplier headers)
    const float *scale; // [rows * per_row]
    rq_block_w4a4 *blocks;
    int32_t len_field;  // pad[0]: the row length, or the Hadamard length of a W4A4H tensor
};

__device__ __forceinline__ int code_for(float x, float s) {
    return s > 0.0f ? (int) fminf(fmaxf(rintf(x / s), -8.0f), 7.0f) : 0;
}

__global__ void __launch_bounds__(256) rq_wencode_kernel(const EncodeArgs a) {
    __shared__ int s_mult[512];   // multiplier of every weight group of the row (K <= 32768: at most 512 groups)
    __shared__ float s_red[4];
    __shared__ int s_sum;
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int K = a.K, nb = K / RQ_BLOCK_CODES, nw = K >> 3;
    const float *x = a.x + row * a.ld;
    rq_block_w4a4 *out = a.blocks + row * nb;
    float unit;   // the row's d
    if (!a.groups) {
        unit = a.scale[row];
        if (tid == 0) s_sum = 0;
        __syncthreads();
    } else {
        // the row's unit is the largest group scale / 15; every group scale becomes a multiple 1..15 of it
        const float *sb = a.scale + row * a.per_row;
        float smax = 0.0f;
        for (int g = tid; g < a.per_row; g += 256) smax = fmaxf(smax, sb[g]);
        smax = wave_max(smax);
        if ((tid & 63) == 0) s_red[tid >> 6] = smax;
        __syncthreads();
        smax = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
        unit = smax / 15.0f;
        for (int g = tid; g < a.per_row; g += 256) {
            s_mult[g] = unit > 0.0f ? (int) fminf(fmaxf(rintf(sb[g] / unit), 1.0f), 15.0f) : 1;
        }
        __syncthreads();
    }
    const int lgw = nw / a.per_row;   // code words per weight group (8 or 32)
    int sum = 0;
    for (int w = tid; w < nw; w += 256) {
        const float s = !a.groups ? unit : (float) s_mult[w / lgw] * unit;
        const float4 v0 = *reinterpret_cast<const float4 *>(x + 8 * w);
        const float4 v1 = *reinterpret_cast<const float4 *>(x + 8 * w + 4);
        const float xs[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int c = code_for(xs[j], s);
            sum += c;
            word |= (uint32_t) (c & 0xF) << (4 * j);
        }
        out[w >> 5].qs[w & 31] = word;
    }
    if (!a.groups) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if ((tid & 63) == 0) atomicAdd(&s_sum, sum);
        __syncthreads();
    }
    for (int b = tid; b < nb; b += 256) {
        int32_t header;
        if (!a.groups) {
            header = s_sum;   // legacy header: the row's code sum (multiplier 1)
        } else if (a.per_row == nb) {
            header = (int32_t) (1u << 30 | (uint32_t) s_mult[b]);
        } else {
            header = (int32_t) (3u << 29 | (uint32_t) s_mult[4 * b] | (uint32_t) s_mult[4 * b + 1] << 4 |
                                (uint32_t) s_mult[4 * b + 2] << 8 | (uint32_t) s_mult[4 * b + 3] << 12);
        }
        out[b].d = unit;
        out[b].sum = header;
        out[b].pad[0] = a.len_field;
        out[b].pad[1] = 0;
    }
}

// ---- dequantizers ------------------------------------------------------------------------------------------------

struct DequantArgs {
    const rq_block_w4a4 *blocks;
    int K;
    int act;       // 0: weight blocks (multiplier per 64 from the header); 1: activation blocks (zero point + multiplier)
    int rotate;    // the inverse rotation follows
    int n_rot, m;
    float scale;   // 1 / sqrtf(n_rot)
    float *out;
    int64_t ldo;
};

__device__ __forceinline__ int nibble(uint32_t word, int j) { return (int) (((word >> (4 * j)) & 0xF) ^ 8) - 8; }

__device__ __forceinline__ int weight_mult(int32_t sum, int g) {
    const uint32_t s = (uint32_t) sum;
    if ((s >> 29) == 3) return (int) ((s >> (4 * g)) & 0xF);
    if ((s >> 30) == 1) return (int) (s & 0xF);
    return 1;
}

// WIDE: the columns of a long Paley stage by four threads each (paley_row), 1024 threads; see launch_dequant for where.
template <int P, bool WIDE>
__global__ void __launch_bounds__(WIDE ? 1024 : 512) rq_dequant_rows_kernel(const DequantArgs a) {
    constexpr int kNT = WIDE ? 1024 : 512;
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int K = a.K, nb = K / RQ_BLOCK_CODES, nw = K >> 3;
    const rq_block_w4a4 *in = a.blocks + row * nb;
    float *o = a.out + row * a.ldo;
    float *buf = smem;

    for (int w = tid; w < nw; w += kNT) {
        const rq_block_w4a4 &blk = in[w >> 5];
        const int ww = w & 31;
        const uint32_t word = blk.qs[ww];
        float f;
        int bias = 0;
        if (a.act) {
            // reference lines 2744-2753: group of the word from the header's sub-group shift
            const int lsub = (blk.sum >> 16) & 3;
            const int sg = (8 * ww) >> (8 - lsub);
            const int z = (blk.sum >> (4 * sg)) & 0xF;
            const int mg = (int) (((uint32_t) blk.pad[0] >> (8 * sg)) & 0xFF);
            f = (float) mg * blk.d;
            bias = 8 - z;
        } else {
            f = (float) weight_mult(blk.sum, ww >> 3) * blk.d;
        }
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (float) (nibble(word, j) + bias) * f;
        if (a.rotate) {
            float *d = buf + padi(8 * w);   // 8 w % 8 == 0: the eight land in one run of 16
#pragma unroll
            for (int j = 0; j < 8; ++j) d[j] = v[j];
        } else {
            *reinterpret_cast<float4 *>(o + 8 * w) = make_float4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<float4 *>(o + 8 * w + 4) = make_float4(v[4], v[5], v[6], v[7]);
        }
    }
    if (!a.rotate) return;
    __syncthreads();

    const int m = a.m;
    const int lm = __ffs(m) - 1;
    fwht_row(buf, K, lm, tid, kNT);
    if constexpr (WIDE) {
        paley_row<P, kNT, true>(buf, K, m, a.n_rot, a.scale, tid);
    } else if constexpr (P > 1) {
        const int ncols = K / P;
        const bool m16 = (m & 15) == 0;
        const int pm = m + (m >> 4);
        for (int cidx = tid; cidx < ncols; cidx += kNT) {
            const int rb = cidx / m, j = cidx - rb * m;
            const int b0 = rb * a.n_rot + j;
            float col[P];
            if (m16) {
                float *src = buf + padi(b0);
#pragma unroll
                for (int i = 0; i < P; ++i) col[i] = src[i * pm];
                paley_column<P, 0, true>(col, src, pm, a.scale);
            } else {
#pragma unroll
                for (int i = 0; i < P; ++i) col[i] = buf[padi(b0 + i * m)];
                paley_column_generic<P, 0, true>(col, buf, b0, m, a.scale);
            }
        }
    } else {
        for (int i = tid; i < K; i += kNT) buf[padi(i)] = buf[padi(i)] * a.scale;
    }
    __syncthreads();
    for (int i = tid * 4; i < K; i += kNT * 4) {
        const float *sp = buf + padi(i);
        *reinterpret_cast<float4 *>(o + i) = make_float4(sp[0], sp[1], sp[2], sp[3]);
    }
}

template <int P, bool WIDE>
hipError_t launch_dequant_form(const DequantArgs &a, int64_t rows, hipStream_t stream) {
    const size_t lds = a.rotate ? (size_t) (a.K + (a.K >> 4) + 1) * sizeof(float) : 0;
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&rq_dequant_rows_kernel<P, WIDE>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 64);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    hipLaunchKernelGGL((rq_dequant_rows_kernel<P, WIDE>), dim3((unsigned) rows), dim3(WIDE ? 1024 : 512), lds, stream, a);
    return hipGetLastError();
}

// Four threads per column where a thread each leaves half of 512 threads without one, 256 columns: K = 17408, p = 68, 64 rows
// 16.3 -> 12.0 us, 427 rows 34.3 -> 23.4, 2048 rows 128 -> 82; K = 27648, p = 108, 2048 rows 252 -> 174 (p = 44, K = 11264: 427 rows
// 13.3 -> 14.4, so it stays). With more columns the fourfold reads of LDS cost more than the idle threads: 600 rows of K = 29952
// (104 x 288, chunks of 8 / 32) 91.7 -> 108.7 / 96.7 -> 101.9, K = 32256 (84 x 384) 77.9 -> 81.5, (72 x 448, chunks of 8) 63.0 ->
// 76.7, K = 27648 (72 x 384) 63.1 -> 66.2; but for two whole runs in chunks of 256 or more, whose strides are constants: K = 30720 (60 x
// 512) 68.5 -> 65.2, 60.1 -> 55.8 in two chunks of 256.
template <int P>
hipError_t launch_dequant(const DequantArgs &a, int64_t rows, hipStream_t stream) {
    if constexpr (P >= 60) {
        const int columns = a.K / P;
        if (columns == 256 || (columns == 512 && a.m >= 256)) return launch_dequant_form<P, true>(a, rows, stream);
    }
    return launch_dequant_form<P, false>(a, rows, stream);
}

bool factor(int64_t n, int &p, int &m) { return rq_w4a4_hadamard_factor(n, &p, &m) != 0; }

struct QuantWorkspace {
    size_t off_rot, off_scale, bytes;
};

QuantWorkspace quant_workspace(int type, int64_t K, int64_t N, int wgroup) {
    QuantWorkspace w;
    size_t off = 0;
    w.off_rot = off;
    if (type == RQ_TYPE_W4A4H) off = align_up(off + (size_t) N * K * sizeof(float), 256);
    w.off_scale = off;
    const int64_t per_row = wgroup == 0 ? 1 : K / wgroup;
    off = align_up(off + (size_t) N * per_row * sizeof(float), 256);
    w.bytes = off;
    return w;
}

}  // namespace
}  // namespace rq

using namespace rq;

extern "C" {

size_t rq_w4a4_quantize_weights_workspace_bytes(int type, int64_t K, int64_t N, int wgroup) {
    if ((type != RQ_TYPE_W4A4 && type != RQ_TYPE_W4A4H) || K <= 0 || K % RQ_BLOCK_CODES != 0 || K > RQ_MAX_K || N <= 0) return 0;
    if (wgroup != 0 && wgroup != 64 && wgroup != RQ_BLOCK_CODES) return 0;
    return quant_workspace(type, K, N, wgroup).bytes;
}

int rq_w4a4_quantize_weights(int type, const float *w_dev, int64_t ldw, int64_t N, int64_t K, int64_t n_rot, int wgroup,
                             void *blocks_dev, void *workspace_dev, size_t workspace_bytes, rq_stream_t stream) {
    if (!w_dev || !blocks_dev || !workspace_dev) return RQ_E_ARGUMENT;
    if (type != RQ_TYPE_W4A4 && type != RQ_TYPE_W4A4H) return RQ_E_UNSUPPORTED;
    if (K <= 0 || K % RQ_BLOCK_CODES != 0 || K > RQ_MAX_K || N < 0 || N > 0x7fffffff) return RQ_E_UNSUPPORTED;
    if (wgroup != 0 && wgroup != 64 && wgroup != RQ_BLOCK_CODES) return RQ_E_ARGUMENT;
    if (ldw < K || (ldw * 4) % 16 != 0 || (reinterpret_cast<uintptr_t>(w_dev) & 15) != 0) return RQ_E_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(blocks_dev) & 15) != 0 || (reinterpret_cast<uintptr_t>(workspace_dev) & 255) != 0) return RQ_E_ARGUMENT;
    if (N == 0) return 0;
    const QuantWorkspace ws = quant_workspace(type, K, N, wgroup);
    if (workspace_bytes < ws.bytes) return RQ_E_WORKSPACE;
    char *base = reinterpret_cast<char *>(workspace_dev);
    hipStream_t st = (hipStream_t) stream;

    const float *src = w_dev;
    int64_t ld = ldw;
    int32_t len_field = (int32_t) K;
    if (type == RQ_TYPE_W4A4H) {
        // stores Q(W H): the forward rotation of every row, block-diagonal when n_rot < K (reference lines 2701-2710)
        int p, m;
        if (n_rot <= 0 || K % n_rot != 0 || !factor(n_rot, p, m)) return RQ_E_ARGUMENT;
        float *rot = reinterpret_cast<float *>(base + ws.off_rot);
        RotQuantArgs q;
        memset(&q, 0, sizeof q);
        q.x = w_dev;
        q.ldx = ldw;
        q.M = (int) N;
        q.K = (int) K;
        q.rotate = 1;
        q.n_rot = (int) n_rot;
        q.p = p;
        q.m = m;
        q.scale = 1.0f / sqrtf((float) n_rot);
        q.clip = 1.0f;
        q.G = kGroup;
        q.mode = kActRotateOnly;
        q.out_f32 = rot;
        q.ldo = K;
        hipError_t e = launch_rotate_quant(q, st);
        if (e != hipSuccess) return (int) e;
        src = rot;
        ld = K;
        len_field = (int32_t) n_rot;
    }

    const int per_row = wgroup == 0 ? 1 : (int) (K / wgroup);
    SearchArgs s;
    s.x = src;
    s.ld = ld;
    s.per_row = per_row;
    s.segments = N * per_row;
    s.n = (int) (K / per_row);
    s.scale = reinterpret_cast<float *>(base + ws.off_scale);
    auto blocks_of = [&](int64_t per) { return dim3((unsigned) ((s.segments + per - 1) / per)); };
    // (the kernels that decide nearly all of them, then the one for what they leave open)
    if (s.n <= 256 && N * K <= few_floats(s.n)) {
        if (s.n == 64) hipLaunchKernelGGL(rq_wsearch_kernel<true>, blocks_of(kSearchThreads / 16), dim3(kSearchThreads), 0, st, s);
        else hipLaunchKernelGGL(rq_wsearch_kernel<false>, blocks_of(kSearchThreads / 16), dim3(kSearchThreads), 0, st, s);
    } else if (s.n == 64) {
        hipLaunchKernelGGL((rq_wsearch_groups_kernel<1>), blocks_of(kSearchThreads / 16), dim3(kSearchThreads), 0, st, s);
        hipLaunchKernelGGL((rq_wsearch_open_kernel<true, 64>), blocks_of(64), dim3(kSearchThreads), 0, st, s);
    } else if (s.n == 256) {
        hipLaunchKernelGGL((rq_wsearch_groups_kernel<4>), blocks_of(kSearchThreads / 16), dim3(kSearchThreads), 0, st, s);
        hipLaunchKernelGGL((rq_wsearch_open_kernel<false, 64>), blocks_of(64), dim3(kSearchThreads), 0, st, s);
    } else {
        hipLaunchKernelGGL(rq_wsearch_rows_kernel, dim3((unsigned) N), dim3(kRowThreads), 0, st, s);
        hipLaunchKernelGGL((rq_wsearch_open_kernel<false, 4>), blocks_of(4), dim3(kSearchThreads), 0, st, s);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int) e;

    EncodeArgs c;
    c.x = src;
    c.ld = ld;
    c.K = (int) K;
    c.per_row = per_row;
    c.groups = wgroup != 0;
    c.scale = s.scale;
    c.blocks = reinterpret_cast<rq_block_w4a4 *>(blocks_dev);
    c.len_field = len_field;
    hipLaunchKernelGGL(rq_wencode_kernel, dim3((unsigned) N), dim3(256), 0, st, c);
    return (int) hipGetLastError();
}

int rq_w4a4_dequantize(int type, const void *blocks_dev, int64_t rows, int64_t K, int64_t n_rot, float *out_dev,
                       int64_t ldo, rq_stream_t stream) {
    if (!blocks_dev || !out_dev) return RQ_E_ARGUMENT;
    if (type < RQ_TYPE_W4A4 || type > RQ_TYPE_A4H) return RQ_E_UNSUPPORTED;
    if (K <= 0 || K % RQ_BLOCK_CODES != 0 || K > RQ_MAX_K || rows < 0 || rows > 0x7fffffff) return RQ_E_UNSUPPORTED;
    if (ldo < K || (ldo * 4) % 16 != 0 || (reinterpret_cast<uintptr_t>(out_dev) & 15) != 0) return RQ_E_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(blocks_dev) & 15) != 0) return RQ_E_ARGUMENT;
    if (rows == 0) return 0;
    DequantArgs a;
    memset(&a, 0, sizeof a);
    a.blocks = reinterpret_cast<const rq_block_w4a4 *>(blocks_dev);
    a.K = (int) K;
    a.act = type == RQ_TYPE_A4 || type == RQ_TYPE_A4H;
    a.rotate = type == RQ_TYPE_W4A4H || type == RQ_TYPE_A4H;
    a.out = out_dev;
    a.ldo = ldo;
    int p = 1, m = 1;
    if (a.rotate) {
        if (n_rot <= 0 || K % n_rot != 0 || !factor(n_rot, p, m)) return RQ_E_ARGUMENT;
        a.n_rot = (int) n_rot;
        a.m = m;
        a.scale = 1.0f / sqrtf((float) n_rot);
    }
    hipStream_t st = (hipStream_t) stream;
    switch (p) {
        case 1:   return (int) launch_dequant<1>(a, rows, st);
        case 12:  return (int) launch_dequant<12>(a, rows, st);
        case 20:  return (int) launch_dequant<20>(a, rows, st);
        case 44:  return (int) launch_dequant<44>(a, rows, st);
        case 60:  return (int) launch_dequant<60>(a, rows, st);
        case 68:  return (int) launch_dequant<68>(a, rows, st);
        case 72:  return (int) launch_dequant<72>(a, rows, st);
        case 84:  return (int) launch_dequant<84>(a, rows, st);
        case 104: return (int) launch_dequant<104>(a, rows, st);
        case 108: return (int) launch_dequant<108>(a, rows, st);
        default:  return RQ_E_UNSUPPORTED;
    }
}

}  // extern "C"
