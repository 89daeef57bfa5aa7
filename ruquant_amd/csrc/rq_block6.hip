// The fp6 product (rq_gemm6.hip) for launches that are small for the chip: few tokens above 64, few rows, or the tiles
// that are left over behind whole rounds of the tiled kernel.
//
// The tiled kernel's unit of work is 256 rows x 128 tokens, 200 us of one compute unit at long rows; a launch of few tiles
// has to cut them along K across workgroups, whose partial totals meet in memory one after the other, and takes 19 us at
// K = 5120 however little there is to do. Here the unit is one panel of 64 rows x 64 tokens, an eighth of a tile, with its
// whole K: the eight wavefronts of a workgroup take the activation groups in turn (each all 64 x 64 outputs of its groups),
// and their totals meet in LDS. No workspace, no arrival counts, nothing that waits for another workgroup.
//
// Arithmetic and operands are the tiled kernel's: one v_mfma_f32_32x32x64_f8f6f4 on fp6 fragments per 32 x 32 outputs and
// group, and the floor as one FMA rounded toward minus infinity (see there for why both are exact; reference patch lines
// 148-177). The fragments go from memory (L2, after the first reader) straight into registers, four groups of a wavefront
// in flight (non-temporal hints and deeper or shallower rings change nothing). Measured, with the weights in the memory-side
// cache: 4.2 us + 0.52 us per group of a wavefront (K = 5120: ten of them, 9.3 us; the tiled kernel 19.5). Eight groups are 48 KB
// through the compute unit's 64 bytes per cycle, 0.32 us; 112 vector instructions each, 0.37 us of the SIMDs' time, and four
// MFMAs, 0.11 (counters: 1.144 M vector instructions and 1.31 M MFMA cycles for 128 units of 80 groups). From memory the weights'
// 24 KB are the longest, 1.0 to 1.2 us. Beyond two rounds of the chip the tiled kernel's twofold reuse out of LDS wins.
//
// A last round that leaves half of the compute units without a unit, or three quarters, cuts its units in pieces, two of 32 rows x
// 64 tokens or four of 32 x 32, with the whole K as before: a compute unit's share of the loads (which bind it, from memory by the
// weights' rows) and of the vector instructions is halved, and nothing has to meet in memory. Product kernel in us, whole units
// -> pieces, weights from the memory-side cache, then from memory: K = 5120, 32 units 9.2 -> 5.9, 10.9 -> 7.2; 94 units 9.7 -> 8.2,
// 13.4 -> 11.2; K = 17408, 32 units 22.1 -> 12.6, 32.0 -> 17.7; 94 units 23.6 -> 19.1, 32.3 -> 25.7; K = 10240, 128 units 15.6 -> 13.1,
// 20.4 -> 16.6; behind a round, 64 tokens, 256 + 16 units, whole call 27.3 -> 23.8.
#include "rq_common.h"

#pragma clang fp contract(off)

namespace rq {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kTok = 64;                       // tokens of a unit
constexpr int kUnitsPerTile = 8;               // 4 panels x 2 runs of 64 tokens of a tile of 256 x 128
// groups of a wavefront whose operands are on their way (with weight multipliers the registers end there; pieces with 3 and 7 are
// 1 % slower at K = 5120)
constexpr int depth_of(bool hask) { return hask ? 2 : 4; }
constexpr int kTokStride = kPanelRows + 4;     // ints between tokens of a wavefront's totals in LDS
constexpr float kBias = 12582912.0f;           // 1.5 x 2^23
constexpr uint32_t kBiasBits = 0x4B400000;
constexpr int kFlushGroups = 28;               // (and the tile of one more that is folded late): less than 2^22

// RA, RB: fragments of 32 rows and of 32 tokens that the workgroup's unit or piece of one has
template <bool HASK, int RA, int RB>
struct Frag {
    v8i A[RA], B[RB];     // this lane's parts of the fragments of rows and of tokens (six registers each)
    float m4[RB];         // 4 m of this lane's tokens
    uint32_t kw[HASK ? 4 * RA : 1];   // weight multipliers of the lane's rows (32 a + 8 q + 4 (lane / 32) + 0 .. 3), a byte each
};

// (global memory, said so: the plane's address comes out of memory, and the loads the compiler makes for a pointer of unknown
// kind may be LDS accesses too, which it waits out whole, everything in flight behind them included)
typedef const __attribute__((address_space(1))) uint8_t gbyte;
typedef const __attribute__((address_space(1))) float gfloat;
typedef const __attribute__((address_space(1))) uint32_t gword;
typedef const __attribute__((address_space(1))) v4u gv4u;
typedef const __attribute__((address_space(1))) v2u gv2u;

struct Src {
    gbyte *a, *b, *k;           // (wave-uniform) the unit's or piece's operands of group 0
    gfloat *m4;
    size_t b_step;              // bytes between groups of the activation plane
    int Mp;
};

__device__ __forceinline__ v8i operand(gbyte *frag, uint32_t l) {
    const v4u lo = *reinterpret_cast<gv4u *>(frag + l * 16);
    const v2u hi = *reinterpret_cast<gv2u *>(frag + 1024 + l * 8);
    v8i v;
    v[0] = (int) lo.x; v[1] = (int) lo.y; v[2] = (int) lo.z; v[3] = (int) lo.w;
    v[4] = (int) hi.x; v[5] = (int) hi.y;
    // (the fp6 form reads six registers: elements 6 and 7 are left undefined)
    return v;
}

// The wavefront's group j of n. Past the end of its share a wavefront's loads read group 0 again, from offset 0 in
// every lane (the loop stays branch-free, so the wait counts stay exact), and nothing consumes them
template <bool HASK, int RA, int RB>
__device__ __forceinline__ void load_frag(Frag<HASK, RA, RB> &f, const Src &s, int wave, int lane, int j, int n) {
    const int g = wave + j * kWaves;
    // (a mask: on a condition the compiler branches around the address arithmetic, and the folds sink into the blocks behind)
    const int keep = __builtin_amdgcn_readfirstlane((j - n) >> 31);
    const uint32_t gk = (uint32_t) (g & keep), l = (uint32_t) (lane & keep);
    gbyte *a = s.a + (size_t) gk * (8 * kFrag6);
    gbyte *b = s.b + gk * s.b_step;
    gfloat *m4 = s.m4 + (size_t) gk * s.Mp;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (i < RA) f.A[i] = operand(a + i * kFrag6, l);
        if (i < RB) {
            f.B[i] = operand(b + i * kFrag6, l);
            f.m4[i] = m4[32 * i + (l & 31)];
        }
    }
    if constexpr (HASK) {
        gbyte *k = s.k + (size_t) gk * kPanelRows + 4 * (l >> 5);
#pragma unroll
        for (int q = 0; q < 4 * RA; ++q) f.kw[q] = *reinterpret_cast<gword *>(k + 8 * q);
    }
}

// What a wavefront carries from group to group: the totals of its 64 x 64 outputs and the tile whose fold is still due.
// Without weight multipliers `acc` is the biased float accumulator of the tiled kernel; with them a group's term, which may
// be 15 times as large, is formed on the bias by an FMA of its own and its bit pattern is added up in integers
// (acc holds those; the bias of every term comes off at the end). The sum of the patterns passes 2^32 from the fourth group on:
// unsigned, modulo 2^32, which gives the total back, since that is small: at most 64 groups of a wavefront x 15 x 122,400 =
// 117.5 M, and 940 M over the eight.
template <int RA, int RB>
struct State {
    float acc[RA][RB][16];
    v16f P;
    float pm;
    float bias;   // kBias (with weight multipliers; taken from behind the change of the rounding mode, like acc)
};

// the tiles of one group; a tile's fold runs behind the next tile's MFMA
template <int RA, int RB>
__device__ __forceinline__ void group_units(const Frag<false, RA, RB> &f, State<RA, RB> &st) {
    const v16f zero = {};
#pragma unroll
    for (int un = 0; un < RA * RB; ++un) {
        const int a = un / RB, b = un % RB;
        const int pu = (un + RA * RB - 1) % (RA * RB), pa = pu / RB, pb = pu % RB;
        const v16f S = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.A[a], f.B[b], zero, 2, 2, 0, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) st.acc[pa][pb][r] = __builtin_fmaf(st.P[r], st.pm, st.acc[pa][pb][r]);
        st.P = S;
        // (a register of its own, which is not the ring's: renamed into it, the ring's newest load would be moved at the head
        // of the loop and waited for with everything in flight)
        asm volatile("v_mov_b32 %0, %1" : "=v"(st.pm) : "v"(f.m4[b]));
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);   // VALU: the fold of the tile before
        __builtin_amdgcn_sched_barrier(0);
    }
}
// with weight multipliers: the two tiles of a row block together, which share the multipliers as floats (a group is folded
// whole, so that the next one does not need its multipliers)
template <int RA, int RB>
__device__ __forceinline__ void group_units(const Frag<true, RA, RB> &f, State<RA, RB> &st) {
    const v16f zero = {};
#pragma unroll
    for (int a = 0; a < RA; ++a) {
        v16f S[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) S[b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.A[a], f.B[b], zero, 2, 2, 0, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float kf = (float) ((f.kw[4 * a + (r >> 2)] >> (8 * (r & 3))) & 0xFFu);
#pragma unroll
            for (int b = 0; b < RB; ++b) {
                const float term = __builtin_fmaf(S[b][r], kf * f.m4[b], st.bias);
                st.acc[a][b][r] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, st.acc[a][b][r]) + __builtin_bit_cast(uint32_t, term));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// the totals of this wavefront into its own part of LDS, [token][row]; FRESH: nothing is there yet
template <bool FRESH, int RA, int RB>
__device__ __forceinline__ void flush(State<RA, RB> &st, int *part, int lane) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
#pragma unroll
        for (int a = 0; a < RA; ++a) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v4i *dst = reinterpret_cast<v4i *>(part + (32 * b + (lane & 31)) * kTokStride + 32 * a + 8 * q + 4 * (lane >> 5));
                v4i v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = (int) (__builtin_bit_cast(uint32_t, st.acc[a][b][4 * q + e]) - kBiasBits);
                    st.acc[a][b][4 * q + e] = kBias;
                }
                *dst = FRESH ? v : *dst + v;
            }
        }
    }
}

template <bool HASK, int RA, int RB>
__device__ __forceinline__ void stream(const Src &s, int wave, int lane, int n, int *part) {
    State<RA, RB> st;
    st.P = v16f{};
    st.pm = 0.0f;
#pragma unroll
    for (int a = 0; a < RA; ++a) {
#pragma unroll
        for (int b = 0; b < RB; ++b) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                st.acc[a][b][r] = HASK ? 0.0f : kBias;
                asm volatile("" : "+v"(st.acc[a][b][r]));   // (behind the change of the rounding mode)
            }
        }
    }
    constexpr int kDepth = depth_of(HASK);
    st.bias = kBias;
    asm volatile("" : "+s"(st.bias));
    Frag<HASK, RA, RB> ring[kDepth];
#pragma unroll
    for (int i = 0; i < kDepth; ++i) {
        load_frag<HASK, RA, RB>(ring[i], s, wave, lane, i, n);
        __builtin_amdgcn_sched_barrier(0);   // (group by group: a wait counts the loads behind the one it is for)
    }
    const int rounds = n / kDepth;
    bool fresh = true;
    for (int r = 0; r < rounds; ++r) {
#pragma unroll
        for (int i = 0; i < kDepth; ++i) {
            const int j = r * kDepth + i + kDepth;
            group_units(ring[i], st);
            __builtin_amdgcn_sched_barrier(0);
            load_frag<HASK, RA, RB>(ring[i], s, wave, lane, j, n);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!HASK && (r + 1) % (kFlushGroups / kDepth) == 0) {
            if (fresh) flush<true>(st, part, lane);
            else flush<false>(st, part, lane);
            fresh = false;
        }
    }
    const int rem = n - rounds * kDepth;   // the last n % kDepth groups are already here
#pragma unroll
    for (int i = 0; i < kDepth - 1; ++i) {
        if (i < rem) group_units(ring[i], st);
    }
    if constexpr (HASK) {
        // n terms, each with the bias's bit pattern on it
        const uint32_t off = (uint32_t) n * kBiasBits - kBiasBits;   // (flush takes one off)
#pragma unroll
        for (int a = 0; a < RA; ++a) {
#pragma unroll
            for (int b = 0; b < RB; ++b) {
#pragma unroll
                for (int r = 0; r < 16; ++r) st.acc[a][b][r] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, st.acc[a][b][r]) - off);
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) st.acc[RA - 1][RB - 1][r] = __builtin_fmaf(st.P[r], st.pm, st.acc[RA - 1][RB - 1][r]);
    }
    if (fresh) flush<true>(st, part, lane);
    else flush<false>(st, part, lane);
}

struct BlockSet {
    const float   *s_w[kMaxFused];
    const uint8_t *kmul[kMaxFused];
    const int32_t *flags[kMaxFused];
    float         *y[kMaxFused];
    int64_t        ldy[kMaxFused];
    int64_t        N[kMaxFused];
    int            n_panels[kMaxFused];
    int            first[kMaxFused];   // first panel, or row tile of 256 rows; unused slots hold the total, so none selects them
};

// CUT: the launch has units in pieces.
template <bool CUT>
__global__ void __launch_bounds__(kThreads, 2)
rq_block6_kernel(const BlockSet ts, const uint8_t *__restrict__ act6, const float *__restrict__ m4,
                 const float *__restrict__ u, int M, int Mp, int ng, int n_runs, int super_tiles, int first_tile,
                 int n_whole, int n_cut, int pieces) {
    __shared__ __align__(16) int s_part[kWaves][kTok * kTokStride];
    // The first n_whole workgroups have a unit each, the others a piece of one of the n_cut units behind those.
    // An XCD gets a contiguous run of the units, so that those that share a panel or a run of tokens read them from one L2.
    const bool whole = !CUT || (int) blockIdx.x < n_whole;
    int v = whole ? blockIdx.x : blockIdx.x - n_whole;
    const int per_xcd = (whole ? n_whole : n_cut * pieces) / kXcds;
    if (v < per_xcd * kXcds) v = (v % kXcds) * per_xcd + v / kXcds;
    int ra = 0, rb = 0;   // (of a piece) which 32 of the unit's rows, and in quarters which 32 of its tokens
    const bool quarter = pieces == 4;
    if (!whole) {
        rb = quarter ? v & 1 : 0;
        ra = (v >> (quarter ? 1 : 0)) & 1;
        v = n_whole + (v >> (quarter ? 2 : 1));
    }
    int wsel, panel, t0;   // which weight, which of its panels, first token
    if (first_tile < 0) {
        // the whole product: panel by panel, the runs of tokens running fastest. (No unit is without rows or tokens: workgroups
        // are dealt to the shader engines in turn, and with every second one empty the others queue on half of them. 160
        // units and 160 empty ones, K = 5120: 18.8 us.)
        panel = v / n_runs;
        t0 = (v - panel * n_runs) * kTok;
        wsel = (panel >= ts.first[1]) + (panel >= ts.first[2]);
        panel -= wsel == 0 ? 0 : wsel == 1 ? ts.first[1] : ts.first[2];   // now of its weight
    } else {
        // the tiles (256 rows x 128 tokens) from first_tile on in the tiled kernel's order, eight units each
        const int sub = v & 7;
        int row_tile;
        gemm6_tile(first_tile + (v >> 3), Mp / kGemmTokens, super_tiles, row_tile, t0);
        t0 += (sub & 1) * kTok;
        wsel = (row_tile >= ts.first[1]) + (row_tile >= ts.first[2]);
        row_tile -= wsel == 0 ? 0 : wsel == 1 ? ts.first[1] : ts.first[2];
        panel = row_tile * 4 + (sub >> 1);
    }
    auto of_weight = [&](const auto &w) { return wsel == 0 ? w[0] : wsel == 1 ? w[1] : w[2]; };
    if (t0 >= M || panel >= of_weight(ts.n_panels)) return;
    const float *__restrict__ s_w = of_weight(ts.s_w);
    const uint8_t *__restrict__ kmul = of_weight(ts.kmul);
    const int32_t *__restrict__ flags = of_weight(ts.flags);
    float *__restrict__ y = of_weight(ts.y);
    const int64_t ldy = of_weight(ts.ldy);
    const int64_t N = of_weight(ts.N);
    // (a piece without rows or tokens)
    if (t0 + 32 * rb >= M || (int64_t) panel * kPanelRows + 32 * ra >= N) return;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint8_t *w6 = plane6_of(flags);
    const bool hask = flags[0] & 1;
    Src s;
    s.a = (gbyte *) (w6 + ((size_t) (panel >> 2) * ng * 8 + 2 * (panel & 3) + ra) * kFrag6);
    s.b_step = (size_t) (Mp / 32) * kFrag6;
    s.b = (gbyte *) (act6 + (size_t) (t0 / 32 + rb) * kFrag6);
    s.m4 = (gfloat *) (m4 + t0 + 32 * rb);
    s.k = (gbyte *) (kmul + (size_t) panel * ng * kPanelRows + 32 * ra);
    s.Mp = Mp;
    // what the epilogue needs from memory is asked for first: a thread ends with four rows of two tokens
    const int quad = tid & 15, tok = tid >> 4;
    const float4 sw = *reinterpret_cast<const float4 *>(s_w + panel * kPanelRows + 4 * quad);   // rows past N are stored as zero
    float ut[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) ut[i] = u[min(t0 + tok + 32 * i, M - 1)];

    const int n = wave < ng ? (ng - wave + kWaves - 1) / kWaves : 0;   // groups wave, wave + 8, ...
    // fp32 rounding toward minus infinity for the folds (MODE bits 1:0); the MFMA sums are exact in any mode
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2" ::: "memory");
    int *part = s_part[wave] + 32 * rb * kTokStride + 32 * ra;
    if (whole) {
        if (hask) stream<true, 2, 2>(s, wave, lane, n, part);
        else stream<false, 2, 2>(s, wave, lane, n, part);
    } else if (quarter) {
        if (hask) stream<true, 1, 1>(s, wave, lane, n, part);
        else stream<false, 1, 1>(s, wave, lane, n, part);
    } else {
        if (hask) stream<true, 1, 2>(s, wave, lane, n, part);
        else stream<false, 1, 2>(s, wave, lane, n, part);
    }
    // (the totals are in LDS when the mode goes back to round to nearest even, and the conversions below read them from there)
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0" ::: "memory");
    __syncthreads();

    // y = ((float(total) * 16) * u) * s_w (reference patch line 176)
    const int64_t row = (int64_t) panel * kPanelRows + 4 * quad;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (!whole && ((quad >> 3) != ra || (quarter && i != rb))) continue;
        const int t = t0 + tok + 32 * i;
        v4i tot = *reinterpret_cast<const v4i *>(&s_part[0][(tok + 32 * i) * kTokStride + 4 * quad]);
#pragma unroll
        for (int w = 1; w < kWaves; ++w) tot += *reinterpret_cast<const v4i *>(&s_part[w][(tok + 32 * i) * kTokStride + 4 * quad]);
        if (t >= M) continue;
        const float o[4] = { (((float) tot.x * 16.0f) * ut[i]) * sw.x, (((float) tot.y * 16.0f) * ut[i]) * sw.y,
                             (((float) tot.z * 16.0f) * ut[i]) * sw.z, (((float) tot.w * 16.0f) * ut[i]) * sw.w };
        float *dst = y + (int64_t) t * ldy + row;
        if (row + 3 < N && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
            typedef float v4f __attribute__((ext_vector_type(4)));
            __builtin_nontemporal_store(v4f{ o[0], o[1], o[2], o[3] }, reinterpret_cast<v4f *>(dst));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (row + e < N) dst[e] = o[e];
            }
        }
    }
}

}  // namespace

namespace {

hipError_t launch(const Gemm6Args &a, int super_tiles, int first_tile, int n_units, hipStream_t stream) {
    BlockSet ts;
    int first = 0;
    for (int i = 0; i < kMaxFused; ++i) {
        const int k = i < a.w.n ? i : a.w.n - 1;   // unused slots repeat the last weight (never selected)
        const PreparedLayout &L = a.w.L[k];
        const uint8_t *p = a.w.prepared[k];
        ts.s_w[i] = reinterpret_cast<const float *>(p + L.off_sw);
        ts.kmul[i] = p + L.off_kmul;
        ts.flags[i] = reinterpret_cast<const int32_t *>(p + L.off_flags);
        ts.y[i] = a.w.y[k];
        ts.ldy[i] = a.w.ldy[k];
        ts.N[i] = L.N;
        ts.n_panels[i] = L.n_panels;
        ts.first[i] = first;
        if (i < a.w.n) first += first_tile < 0 ? L.n_panels : L.n_rtiles;
    }
    const int ng = a.w.L[0].ng;
    const float *m4 = reinterpret_cast<const float *>(a.act6 + act6_plane_bytes(ng, a.Mp));
    // units of the last round in four pieces where the chip has room for them, in two, or whole (160 units are no faster in pieces,
    // which would be a second round)
    const int last = n_units % kPlanUnits;
    const int pieces = last <= kPlanUnits / 4 ? 4 : last <= kPlanUnits / 2 ? 2 : 1;
    const int n_cut = pieces > 1 ? last : 0, n_whole = n_units - n_cut;
#define RQ_LAUNCH_BLOCK6(CUT)                                                                                              \
    hipLaunchKernelGGL(rq_block6_kernel<CUT>, dim3(n_whole + n_cut * pieces), dim3(kThreads), 0, stream, ts, a.act6, m4,   \
                       a.u, a.M, a.Mp, ng, (a.M + kTok - 1) / kTok, super_tiles, first_tile, n_whole, n_cut, pieces)
    if (n_cut > 0) RQ_LAUNCH_BLOCK6(true);
    else RQ_LAUNCH_BLOCK6(false);
#undef RQ_LAUNCH_BLOCK6
    return hipGetLastError();
}

}  // namespace

hipError_t launch_block6(const Gemm6Args &a, hipStream_t stream) {
    int n_panels = 0;
    for (int i = 0; i < a.w.n; ++i) n_panels += a.w.L[i].n_panels;
    return launch(a, 0, -1, n_panels * ((a.M + kTok - 1) / kTok), stream);
}

hipError_t launch_block6_tiles(const Gemm6Args &a, int super_tiles, int first_tile, int n_tiles, hipStream_t stream) {
    return launch(a, super_tiles, first_tile, (n_tiles - first_tile) * kUnitsPerTile, stream);
}

// 33 .. 64 tokens. The skinny kernel reads two thirds of the bytes (int4 codes) but runs 16 x 16 MFMAs with three vector
// instructions per output behind each, where this one has 32 x 32 and one. So this one is faster on weights that the
// memory-side cache holds and loses on weights that come from memory, as those of a whole model do: a unit's 3 KB a group
// then arrive at 20 KB per microsecond, whatever the other compute units do. The line lies where it is faster from the cache
// and at most 6 % slower from memory. (64 tokens, whole call in us, skinny / here; in front from the cache, behind from memory.)
// - Up to 64 panels, a unit in four pieces: K = 1024, N = 4096 8.8 / 8.1, 9.4 / 8.9 (40 tokens); K = 5120, N = 1024 11.6 / 10.4,
//   12.6 / 12.2, N = 4096 14.1 / 10.4, 15.6 / 13.5; K = 10240 21.6 / 14.2, 23.4 / 18.8; K = 17408, N = 1024 20.2 / 18.6, 22.0 / 25.1,
//   N = 4096 27.3 / 19.7, 28.6 / 27.0; K = 32768, N = 1024 28.7 / 30.3, 28.6 / 40.0. Here up to K = 10240, but for a few panels of
//   rows that long, where the skinny kernel has slices along K instead and the fp6 quantizer, a thread per 32 values, takes longer
//   (33 / 64 tokens, here as a part of the skinny kernel's time, cache; memory, weights in turn from 330 MB of codes): K = 5632 at most
//   1.01; K = 6144 N = 256 1.01 / 1.00; 1.05 / 1.05, N = 512 1.00 / 1.00; 1.07 / 1.05, N = 1165 0.97 / 0.92; 1.01 / 0.97, N = 1344 0.94 / 0.89; 1.05 /
//   0.97. K = 8192 N = 256 0.98 / 0.96; 0.96 / 0.95, N = 1024 0.95 / 0.89; 1.04 / 0.99, N = 2048 0.88 / 0.85; 1.03 / 0.99. K = 9216 (48 / 64
//   tokens; up to 40 its rotation is a launch of its own and the skinny kernel follows) N = 64 1.03 / 1.03; 1.06 / 1.06, N = 1165 1.00 / 0.97; 1.08 /
//   1.07, N = 2048 0.99 / 0.93; 1.06 / 1.04, N = 2238 0.98 / 0.91; 1.04 / 1.03. Without a rotation, whose launch hides some of that: K = 6144 N = 512
//   0.99 / 1.00; 1.08 / 1.07, N = 1165 0.97 / 0.92; 1.01 / 0.97, K = 7168 N = 1165 0.96 / 0.92; 1.06 / 1.02, K = 8192 N = 1165 0.99 / 0.95; 1.12 / 1.08,
//   N = 2048 0.92 / 0.88; 1.10 / 1.06, N = 2560 0.88 / 0.84; 1.04 / 1.01, K = 9216 N = 1165 0.98 / 0.94; 1.14 / 1.12, N = 2048 0.90 / 0.87; 1.11 / 1.07,
//   N = 2560 0.84 / 0.81; 1.04 / 1.01. K = 10240 is the skinny kernel's second step: N = 256 1.01 / 0.91; 1.06 / 0.96 (48 tokens 0.99; 1.02),
//   N = 1165 0.92 / 0.79; 1.08 / 0.92 (48 tokens 1.04), N = 1792 0.88 / 0.76; 1.08 / 0.91, N = 2048 0.84 / 0.71; 1.00 / 0.88.
// - 65 to 128 panels (half the chip: the skinny kernel has two workgroups of 32 tokens a panel): K = 5120, N = 8192 14.8 / 15.0,
//   16.1 / 19.6; K = 17408, N = 8192 47.6 / 39.4, 38.4 / 46.6. The skinny kernel.
// - 129 to 256 panels, a round of units, and two of the skinny kernel's: N = 12288, K = 1024 15.6 / 9.5, 16.3 / 10.9; K = 5120
//   24.4 / 16.4, 25.6 / 20.5; K = 10240 32.0 / 24.6, 32.8 / 32.9; K = 17408 48.1 / 35.5, 48.4 / 50.7; K = 32768 81 / 85 in both.
//   Here up to K = 17408.
// - More: N = 17408 (272), K = 3072 25.7 / 20.0, 27.1 / 24.3; K = 5120 30.7 / 25.9, 31.8 / 32.5; K = 10240 44.5 / 41.1, 45.3 / 53.7;
//   K = 17408 63.0 / 61.7, 63.6 / 83.1; K = 32768 100 / 147. N = 24576 (384), K = 10240 55.7 / 42.2, 56.7 / 55.8; N = 34816 (544)
//   73.7 / 65.7, 74.5 / 79.8. Here up to K = 5120, and up to K = 10240 where the last round is at least half full. (All in whole units.
//   With the 16 units of a second round in four pieces N = 17408, K = 5120 is 23.7 from the cache and 29.5 from memory, and longer rows might
//   win too: the line is from before.)
// - Weight multipliers cost the skinny kernel more: 96 to 128 panels, N = 8192, K = 1024 9.8 / 10.3, K = 3072 N = 6144 14.1 / 13.8,
//   15.3 / 15.8, K = 5120 18.3 / 17.9, 20.0 / 21.3, K = 10240 33.9 / 26.6, 34.9 / 33.4, K = 17408 58.2 / 45.9, 48.4 / 50.7 (and 8 % more
//   at 33 tokens); N = 12288, K = 5120 29.7 / 18.9, 31.2 / 22.4, K = 32768 128 / 91, 128 / 95; N = 17408, K = 17408 86 / 71, 87 / 91,
//   K = 32768 145 / 160. Here from K = 3072 to 10240 with 96 panels, any length in one round of units, up to K = 17408 beyond.
// 33 tokens are within a tenth of 64 on both sides.
bool block6_takes(int64_t n_panels, int64_t M, int ng, bool weight_multipliers, bool rotate) {
    if (M <= 32) return false;
    if (n_panels <= kPlanUnits / 4) {
        if (ng < 96) return true;
        if (ng < 128) return n_panels > (rotate ? 12 : 16);
        if (ng <= 144) return n_panels > (!rotate ? 36 : ng > 128 ? 32 : 0);
        return ng <= 160 && (n_panels > 28 || M > 40);
    }
    if (n_panels <= kPlanUnits / 2) return weight_multipliers && n_panels >= 96 && ng >= 48 && ng <= 160;
    if (n_panels <= kPlanUnits) return ng <= 272 || weight_multipliers;
    if (weight_multipliers) return ng <= 272;
    const int64_t last = n_panels % kPlanUnits;
    return ng <= 80 || (ng <= 160 && (last == 0 || last >= kPlanUnits / 2));
}

}  // namespace rq
