// int4 x int4 GEMM for wide token batches on the gfx950 matrix cores, through v_mfma_f32_32x32x64_f8f6f4 with fp6
// (E2M3) operands: the MFMA form that runs at twice the rate of the int8 one and whose K = 64 is exactly one
// activation group.
//
// Why fp6 is exact here. An E2M3 value with sign s and the five exponent / mantissa bits read as the integer n
// (0 .. 31) is n / 8 for n <= 15 (subnormals 0 .. 7 / 8, then 1 .. 1.875 in steps of 1 / 8): the sign-magnitude code
// of an integer |v| <= 15 IS the fp6 encoding of v / 8. Weight codes w (-8 .. 7) and activation values q - z
// (-15 .. 15) both fit, every product w (q - z) / 64 is a multiple of 1 / 64 below 2, and a group's sum
// S / 64 (|S| <= 7680) is exact in the fp32 accumulator. One MFMA per 32 x 32 outputs and group yields
// S_g = sum_k w_k (q_k - z_g), which equals the reference's acc + (8 - z) colsum (ggml_vec_dot_w4a4_a4, reference
// patch lines 160-172).
//
// The per-group floor. The reference adds floor(m_g S_g / 16) per group (reference patch lines 35-39, 173). With the
// wavefront's fp32 rounding mode set toward minus infinity, acc = fma(S / 64, 4 m, acc) on an accumulator that
// holds an integer in [2^23, 2^24) (where one unit in the last place is 1) is acc + floor(m S / 16): the FMA forms
// m S / 16 + acc exactly and rounds once, downwards, to an integer. One full-rate vector instruction per output and
// group. The accumulator starts at 1.5 x 2^23; a group moves it by at most 255 x 7680 / 16 = 122,400, so after 32
// groups (3,916,800 < 2^22) its offset from the start is moved into an int32 total (two integer instructions per
// value: the float's bit pattern minus the bit pattern of 1.5 x 2^23 is that offset) and it starts again.
//
// Tensors with integer weight multipliers k (uniform branch on the prepared flag) fold 4 m k instead of 4 m, on the bias itself,
// and add the bit patterns up in integers. Activation groups of 128 / 256 (RQ_ACT_GROUP) chain the 2 or 4 MFMAs of a
// group through the accumulator operand before the one fold (and multipliers in integers).
//
// Data movement: a workgroup of eight wavefronts owns 256 rows x 128 tokens; wavefront (wr, wc) owns rows 64 wr .. and
// tokens 64 wc .. as 2 x 2 MFMA tiles of 32 x 32. Operands go from global memory straight into LDS
// (global_load_lds_dwordx4), two groups per ring stage, four stages. Both the fp6 weight plane that
// rq_w4a4_prepare writes and the activation plane of the quantizer are stored as MFMA fragments (32 rows or tokens x
// 64 inputs = 1536 bytes: a 16-byte and an 8-byte piece per lane, each piece contiguous across the lanes), so a
// stage is filled by whole 1 KiB runs and read back without bank conflicts.
//
// What bounds it: the issue of vector instructions, 16 FMAs of four cycles and three others per MFMA. Counters at K = 10240,
// N = 16384, 2048 tokens (four whole rounds): the vector ALU issues in 393,000 of the 515,000 cycles, and in 98,000 more a matrix
// core works without it (its 32 cycles per MFMA share 13 with a vector instruction). Above that, the clock, which the matrix cores, the
// vector ALU and LDS together pull down: 1.9 GHz there, 2.0 at K = 5120 and N = 17408, 2.3 in a launch of one round. With weight
// multipliers the vector ALU issues in 98 % of the cycles. 16 MFMAs of a SIMD, a step, take 0.72 us (in a timing-only build without LDS
// reads and fetches 0.53); a tile costs 9.4 us besides its steps. Product kernels in us since a wavefront waits for its operands where
// it uses them and every read of the ring has a fixed base, weights from the memory-side cache, then from memory: K = 5120,
// N = 17408, 2048 tokens 179.5 -> 170, 192 -> 181 (on another card 190 -> 187); K = 17408, N = 5120 156 -> 147, 170 -> 155; N = 17408, 300
// tokens 102 -> 90, 112 -> 105; with weight multipliers, K = 5120, N = 8192 140 -> 127, 141 -> 129.
#include "rq_common.h"

#include <string.h>

#pragma clang fp contract(off)

namespace rq {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kThreads = 512;
constexpr int kTileRows = 256;                 // rows of a workgroup's tile
constexpr int kTileTok = 128;                  // tokens of a workgroup's tile
constexpr int kCellsA = 8 * kFrag6 / 16;       // 768 cells: eight weight fragments of one group
constexpr int kCellsB = 4 * kFrag6 / 16;       // 384 cells: four activation fragments of one group
constexpr int kCellsM = kTileTok * 4 / 16;     // 32 cells: the 128 tokens' multipliers of one group (4 m as float)
constexpr int kCellsK = kTileRows / 16;         // 16 cells: the 256 rows' weight multipliers of one group (a byte each)
// A ring stage is two groups. The stages of the two operands stand apart, those of the activations first, each [B g0][B g1][m g0]
// [m g1][k g0][k g1], behind them those of the weights, [A g0][A g1]: a lane's reads then reach every stage from few base
// registers (an instruction's offset is 64 KB): one for the activations' 16-byte pieces, one for their 8-byte pieces, one for
// the multipliers, and two each for the weights'.
constexpr int kRing = 4;
constexpr int kStageA = 2 * kCellsA * 16;
constexpr int kOffM = 2 * kCellsB * 16, kOffK = kOffM + 2 * kCellsM * 16;   // in a stage of the activations
constexpr int kStageB = kOffK + 1024;                                       // (k is 512 bytes, moved by a whole wavefront)
constexpr int kOffA = kRing * kStageB;
constexpr int kRingBytes = kOffA + kRing * kStageA;
// Each wavefront moves five runs of 1 KiB per step: three of the weights' 24, one of the activations' first eight, and of the
// rest of their stage wavefronts 0 .. 3 the last four, 4 the tokens' multipliers, 5 the rows'; 6 and 7 the same as 4 and 5 (so
// that every wavefront has the same number of loads in flight).
static_assert(kStageA == 24 * 1024 && kOffM == 12 * 1024 && kStageB == 14 * 1024, "split of a step's loads");
constexpr int kLoadsPerStep = 5;

constexpr int kXposeStride = 36;               // floats between tokens of a wavefront's output block in LDS (32 rows + 4)
constexpr float kBias = 12582912.0f;           // 1.5 x 2^23
constexpr int kBiasBits = 0x4B400000;
constexpr int kFlushSteps = 16;                // 32 groups
constexpr int kRsrcWord3 = 0x00020000;         // last word of a raw buffer descriptor on this target (32-bit data format)
constexpr int kDeviceScope = 16;               // cache policy of a buffer access: the sc1 bit

// a wave-uniform address, said so explicitly: the compiler then keeps it in scalar registers
__device__ __forceinline__ const uint8_t *uniform(const uint8_t *p) {
    const uint64_t b = (uint64_t) (uintptr_t) p;
    return reinterpret_cast<const uint8_t *>(
        (uintptr_t) ((uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) b) |
                     (uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (b >> 32)) << 32));
}

// 64 lanes x 16 bytes from base + lane offset to 1 KiB of LDS at `lds` + OFF (wave-uniform; the hardware adds lane * 16). OFF is added
// on the way into M0. Assembly, so that the count of outstanding loads stays under this file's control (the s_waitcnt of the steps).
template <int OFF>
__device__ __forceinline__ void load_run(const uint8_t *base, uint32_t lane_off, uint32_t lds) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(lane_off), "s"(base), "s"(lds), "n"(OFF)
                 : "memory", "m0", "scc");
}

__device__ __forceinline__ void load_to_lds_dword(const float *gptr, float *lds) {
    const uint32_t lds_addr = (uint32_t) (uintptr_t) (lds_void *) lds;
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
                 :
                 : "v"(gptr), "s"(lds_addr)
                 : "memory", "m0");
}

struct Ctx {
    // what this wavefront moves per step (wave-uniform): three runs of the weights, 8 KB apart, one of the activations, a fifth
    // with lane offsets of its own; and where to, in the first stage
    const uint8_t *a_src, *b_src, *t_src;
    uint32_t b_step, t_step;       // their advance per step (bytes: under 4 GiB for any batch the workspace can hold)
    uint32_t t_off;
    uint32_t lds_run, lds_t;
    // this lane's places in the first stage of the ring: 16- and 8-byte pieces of the activations, the tokens' and the rows'
    // multipliers, and the pieces of the weights in stages 0 and 2
    uint32_t b16, b8, m, k, a16[2], a8[2];
    const uint8_t *k_src;    // weight multipliers of this wavefront's panel, row offset of the lane's first quad
    int wave, wr, wc, lane;
    int n_steps;             // steps (two groups each) of this workgroup
    int g0;                  // its first group
};

// fetch of step `st` (two groups) into stage S, then advance the sources; past the last step they stay where they
// are (the last step is fetched again, into cells nobody reads), so every step issues the same number of loads.
// In pieces, so that the loop can deal them out between its MFMAs: five loads issued back to back by all eight
// wavefronts right behind the barrier queue up in front of the memory pipeline, and a wavefront that waits to issue a
// load issues no MFMA either. Piece 0 .. 2 the weights, 3 and 4 the activations' stage.
template <int S, int PIECE>
__device__ __forceinline__ void fetch_piece(Ctx &c, int st) {
    const bool more = st + 1 < c.n_steps;
    if constexpr (PIECE < 3) {
        load_run<kOffA + S * kStageA + PIECE * 8192>(uniform(c.a_src + PIECE * 8192), (uint32_t) c.lane * 16, c.lds_run);
        if (PIECE == 2) c.a_src = uniform(c.a_src + (more ? kStageA : 0));
    } else if constexpr (PIECE == 3) {
        load_run<S * kStageB>(c.b_src, (uint32_t) c.lane * 16, c.lds_run);
        c.b_src = uniform(c.b_src + (more ? c.b_step : 0));
    } else {
        load_run<S * kStageB>(c.t_src, c.t_off, c.lds_t);
        c.t_src = uniform(c.t_src + (more ? c.t_step : 0));
    }
}
template <int S>
__device__ __forceinline__ void fetch(Ctx &c, int st) {
    fetch_piece<S, 0>(c, st);
    fetch_piece<S, 1>(c, st);
    fetch_piece<S, 2>(c, st);
    fetch_piece<S, 3>(c, st);
    fetch_piece<S, 4>(c, st);
}

typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
template <class T>
__device__ __forceinline__ const __attribute__((address_space(3))) T *lds_at(uint32_t addr, int off) {
    return reinterpret_cast<const __attribute__((address_space(3))) T *>((const __attribute__((address_space(3))) uint8_t *) addr + off);
}
// The two pieces of a fragment straight into the six registers of the operand. (The 8-byte piece by a volatile read: two
// ordinary ones become one ds_read2st64_b64, whose results have to be moved into the operands' registers, and a wavefront
// waits for its reads where the moves stand, right behind them, instead of in front of the MFMA a group later.)
__device__ __forceinline__ v8i fragment(uint32_t p16, uint32_t p8, int off) {
    const v4u lo = *lds_at<v4u>(p16, off);
    const v2u hi = *reinterpret_cast<const volatile __attribute__((address_space(3))) v2u *>(lds_at<v2u>(p8, off));
    v8i v;
    v[0] = (int) lo.x; v[1] = (int) lo.y; v[2] = (int) lo.z; v[3] = (int) lo.w;
    v[4] = (int) hi.x; v[5] = (int) hi.y;
    // (the fp6 form reads six registers: elements 6 and 7 are left undefined)
    return v;
}
__device__ __forceinline__ v8i read_a(const Ctx &c, int stage, int gi, int i) {
    return fragment(c.a16[stage >> 1], c.a8[stage >> 1], (stage & 1) * kStageA + gi * (kCellsA * 16) + i * kFrag6);
}
__device__ __forceinline__ v8i read_b(const Ctx &c, int stage, int gi, int i) {
    return fragment(c.b16, c.b8, stage * kStageB + gi * (kCellsB * 16) + i * kFrag6);
}
__device__ __forceinline__ float read_m(const Ctx &c, int stage, int gi, int i) {
    return *lds_at<float>(c.m, stage * kStageB + gi * (kCellsM * 16) + i * 128);
}

// fast path: acc += floor(m S / 16) for the 16 outputs of one tile (round toward minus infinity is set)
__device__ __forceinline__ void fold_fast(const v16f &S, float m4, float (&acc)[16]) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = __builtin_fmaf(S[r], m4, acc[r]);
}

// weight multipliers (reference patch lines 169-173): floor(k m S / 16) by the same FMA with 4 m k in place of 4 m, on the bias
// itself: a term may be 15 times as large, so its bit pattern is added up in integers, and the bias of every term comes off at
// the end. (The sum of the patterns passes 2^32 from the fourth group on: unsigned, modulo 2^32, which gives the total back, since
// that is small: at most 512 groups x 15 x 122,400 = 940 M.)
__device__ __forceinline__ void fold_km(const v16f &S, float m4, const float (&kf)[16], float bias, float (&acc)[16]) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float term = __builtin_fmaf(S[r], kf[r] * m4, bias);
        acc[r] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, acc[r]) + __builtin_bit_cast(uint32_t, term));
        asm volatile("" : "+v"(acc[r]));   // (formed here, not sunk into the blocks behind)
    }
}
// the sixteen multipliers a lane needs for row block a (rows 32 a + 8 q + 4 (lane / 32) + 0 .. 3, q = 0 .. 3) of group gi
__device__ __forceinline__ void read_kw(const Ctx &c, int stage, int gi, int a, uint32_t (&kw)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) kw[q] = *lds_at<uint32_t>(c.k, stage * kStageB + gi * (kCellsK * 16) + 32 * a + 8 * q);
}

// the same in integers, from multipliers in global memory (the forms for activation groups of 128 / 256)
__device__ __forceinline__ void fold_k(const v16f &S, float m4, const int (&kk)[16], int32_t (&tot)[16]) {
    const int mi = (int) (m4 * 0.25f);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int Si = (int) (S[r] * 64.0f);
        tot[r] += (kk[r] * mi * Si) >> kTermShift;
    }
}

// One step (two groups of 64 inputs) of one wavefront: 64 rows x 64 tokens as 2 x 2 tiles. GS = runs of 64 per
// activation group (1, 2, 4). A unit = one tile x one activation group's runs inside this step: its MFMAs chain through
// the accumulator operand; the fold of unit i runs behind the MFMAs of unit i + 1.
template <bool HASK, int GS, int S0>
__device__ __forceinline__ void compute(const Ctx &c, int st, float (&acc)[2][2][16],
                                        int32_t (&tot)[2][2][16], v16f (&carry)[2][2]) {
    constexpr int kRuns = GS == 1 ? 1 : 2;        // runs of a unit inside one step
    constexpr int kUnits = GS == 1 ? 8 : 4;
    v8i A[2][2], B[2][2];
    float m4[2][2];
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            A[gi][i] = read_a(c, S0, gi, i);
            B[gi][i] = read_b(c, S0, gi, i);
            m4[gi][i] = read_m(c, S0, gi, i);
        }
    }
    // with groups of 256 a unit spans two steps: the even step leaves its half in `carry`, the odd step folds
    const bool folds = GS < 4 || (st & 1);
    const bool starts = GS < 4 || !(st & 1);
    const v16f zero = {};
    v16f S[2];
    int prev_a = 0, prev_b = 0, prev_gi = 0;
#pragma unroll
    for (int un = 0; un < kUnits + 1; ++un) {
        if (un < kUnits) {
            const int gi = GS == 1 ? un >> 2 : 0, a = (un >> 1) & 1, b = un & 1;
            v16f C = GS == 4 && !starts ? carry[a][b] : zero;
#pragma unroll
            for (int run = 0; run < kRuns; ++run) {
                C = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A[gi + run][a], B[gi + run][b], C, 2, 2, 0, 0, 0, 0);
            }
            if (GS == 4 && !folds) carry[a][b] = C;
            S[un & 1] = C;
        }
        if (un > 0 && folds) {
            const v16f &P = S[(un - 1) & 1];
            if (!HASK) {
                fold_fast(P, m4[prev_gi][prev_b], acc[prev_a][prev_b]);
            } else {
                // the multiplier of the group's first run (reference patch line 171: RQ_W_MULT_G(sum, sg << (2 - lsub)))
                const int g = c.g0 + (GS == 4 ? 2 * (st & ~1) : 2 * st) + prev_gi;
                int k16[16];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t k4 = *reinterpret_cast<const uint32_t *>(c.k_src + (size_t) g * kPanelRows + 32 * prev_a + 8 * q);
#pragma unroll
                    for (int i = 0; i < 4; ++i) k16[4 * q + i] = (k4 >> (8 * i)) & 0xFF;
                }
                fold_k(P, m4[prev_gi][prev_b], k16, tot[prev_a][prev_b]);
            }
        }
        if (un < kUnits) {
            prev_gi = GS == 1 ? un >> 2 : 0;
            prev_a = (un >> 1) & 1;
            prev_b = un & 1;
        }
        // A unit's MFMAs and the previous unit's fold stay together, MFMAs first: the fold then runs while the matrix
        // pipe works on the next unit. (Left alone, the scheduler issues all the independent MFMAs of a step first and
        // their results, 16 registers each, spill; with a plain barrier it puts the fold in front of the MFMA, so that
        // every fold waits for the MFMA issued right before it.)
        if (un < kUnits) __builtin_amdgcn_sched_group_barrier(0x008, kRuns, 0);   // MFMA
        if (un > 0 && folds && !HASK) __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);   // VALU
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <bool HASK, int GS, int S>
__device__ __forceinline__ void step(Ctx &c, int st, float (&acc)[2][2][16],
                                     int32_t (&tot)[2][2][16], v16f (&carry)[2][2]) {
    // the loads of steps st + 1 and st + 2 may still be in flight
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kLoadsPerStep) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch<(S + 3) % kRing>(c, st + 3);
    compute<HASK, GS, S>(c, st, acc, tot, carry);
}

__device__ __forceinline__ void flush(float (&acc)[2][2][16], int32_t (&tot)[2][2][16]) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                tot[a][b][r] += __builtin_bit_cast(int, acc[a][b][r]) - kBiasBits;
                acc[a][b][r] = kBias;
            }
        }
    }
}

template <bool HASK, int GS>
__device__ __forceinline__ void body(Ctx &c, int32_t (&tot)[2][2][16]) {
    v16f carry[2][2] = {};
    float acc[2][2][16];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[a][b][r] = kBias;
                tot[a][b][r] = 0;
            }
        }
    }
    fetch<0>(c, 0);
    fetch<1>(c, 1);
    fetch<2>(c, 2);
    for (int st = 0; st < c.n_steps; st += kRing) {
        // (K is a multiple of 256: the number of steps is even, so steps come in pairs)
        step<HASK, GS, 0>(c, st, acc, tot, carry);
        step<HASK, GS, 1>(c, st + 1, acc, tot, carry);
        if (st + 2 < c.n_steps) {
            step<HASK, GS, 2>(c, st + 2, acc, tot, carry);
            step<HASK, GS, 3>(c, st + 3, acc, tot, carry);
        }
        if (!HASK && ((st / kRing + 1) % (kFlushSteps / kRing)) == 0) flush(acc, tot);
    }
    flush(acc, tot);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the refetches of the last steps
}

// ---- groups of 64 (the common case): the same steps with the LDS reads taken out of the critical path.
// The operands of a group are read from LDS while the group before is being computed, a piece behind each of its MFMAs
// (fragment pairs in the order in which the next group's MFMAs take them), and the wait for the next stage (vmcnt + barrier)
// sits between the two groups of a step, so that the next step's first group can be read behind the second group's MFMAs.
struct Operands {
    v8i A[2], B[2];
    float m4[2];
};

__device__ __forceinline__ void read_piece(const Ctx &c, int stage, int gi, int piece, Operands &o) {
    if (piece == 0) {
        o.A[0] = read_a(c, stage, gi, 0);
        o.B[0] = read_b(c, stage, gi, 0);
    } else if (piece == 1) {
        o.B[1] = read_b(c, stage, gi, 1);
    } else if (piece == 2) {
        o.A[1] = read_a(c, stage, gi, 1);
        o.m4[0] = read_m(c, stage, gi, 0);
        o.m4[1] = read_m(c, stage, gi, 1);
    }
}

// What a wavefront carries from group to group: the accumulators (without weight multipliers the biased floats above, with them
// the sums of bit patterns), the tile whose fold is still due, always (1, 1), its tokens' multipliers, and its rows'.
template <bool HASK>
struct State {
    float acc[2][2][16];
    v16f P;
    float pm;
    float kf[HASK ? 16 : 1];
    uint32_t kw[HASK ? 2 : 1][2][4];   // bytes of both groups of a step: [group][row block]
    float bias;
};

// the four tiles of one group; the fold of a tile runs behind the MFMA of the next one, the last tile's result is
// handed to the next group. With weight multipliers the two tiles of a row block share its multipliers, converted once.
template <bool HASK, class Between>
__device__ __forceinline__ void group_units(const Operands &o, int gi, State<HASK> &s, Between between) {
    const v16f zero = {};
#pragma unroll
    for (int un = 0; un < 4; ++un) {
        const int a = un >> 1, b = un & 1;
        const int pa = un == 0 ? 1 : (un - 1) >> 1, pb = un == 0 ? 1 : (un - 1) & 1;
        // (The two statements around the MFMA pin the order MFMA, load, fold: without them the compiler moves the load in front of
        // the MFMA, which then waits behind the load's issue. A raised issue priority for the MFMA costs 1.5 %.)
        __builtin_amdgcn_sched_barrier(0);
        const v16f S = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(o.A[a], o.B[b], zero, 2, 2, 0, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        between(un);   // (pieces of the next operands' reads and of the next stages' fetch: behind the MFMA, in front of the fold)
        if constexpr (HASK) {
            if (b == 1) {   // (the fold below is the first one of row block a)
#pragma unroll
                for (int r = 0; r < 16; ++r) s.kf[r] = (float) ((s.kw[gi][a][r >> 2] >> (8 * (r & 3))) & 0xFFu);
            }
            fold_km(s.P, s.pm, s.kf, s.bias, s.acc[pa][pb]);   // (a workgroup's first fold adds nothing but the bias)
        } else {
            fold_fast(s.P, s.pm, s.acc[pa][pb]);
        }
        s.P = S;
        s.pm = o.m4[b];
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                // MFMA
        if (!HASK) __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);    // VALU: the fold
        __builtin_amdgcn_sched_barrier(0);
    }
}

// step st, whose stage is S
template <bool HASK, int S>
__device__ __forceinline__ void step64(Ctx &c, int st, Operands &X, Operands &Y, State<HASK> &state) {
    constexpr int kNext = (S + 1) % kRing, kPrev = (S + 3) % kRing;
    group_units<HASK>(X, 0, state, [&](int un) {
        read_piece(c, S, 1, un, Y);
        // (both groups' multipliers in this half: behind the barrier their stage belongs to a later step)
        if constexpr (HASK) read_kw(c, S, un & 1, un >> 1, state.kw[un & 1][un >> 1]);
        if (un == 0) fetch_piece<kPrev, 3>(c, st + 3);
        if (un == 2) fetch_piece<kPrev, 4>(c, st + 3);
    });
    // Stage st + 1 is whole once every wavefront has seen its own loads of it arrive (those of steps st + 2 and st + 3
    // may still be in flight). This step's stage has been read by then, a wavefront's last reads of it included, and is free
    // for step st + 4: a load is three steps ahead of its use.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * kLoadsPerStep) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    group_units<HASK>(Y, 1, state, [&](int un) {
        read_piece(c, kNext, 0, un, X);   // (past the last step: stale cells, never used)
        if (un == 0) fetch_piece<S, 0>(c, st + 4);
        if (un == 1) fetch_piece<S, 1>(c, st + 4);
        if (un == 2) fetch_piece<S, 2>(c, st + 4);
    });
}

template <bool HASK>
__device__ __forceinline__ void body64(Ctx &c, int32_t (&tot)[2][2][16]) {
    Operands X, Y;
    State<HASK> s;
    s.P = v16f{};
    s.pm = 0.0f;
    s.bias = kBias;
    asm volatile("" : "+s"(s.bias));
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s.acc[a][b][r] = HASK ? 0.0f : kBias;
                tot[a][b][r] = 0;
            }
        }
    }
    if constexpr (HASK) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s.kf[r] = 0.0f;
    }
    // stages 0 to 2 whole, of stage 3 the weights: its other two loads and everything after them is dealt
    // out between the MFMAs of the loop (three runs of step st + 4 behind the barrier of step st, the fourth and the
    // fifth in the first half of step st + 1)
    fetch<0>(c, 0);
    fetch<1>(c, 1);
    fetch<2>(c, 2);
    fetch_piece<3, 0>(c, 3);
    fetch_piece<3, 1>(c, 3);
    fetch_piece<3, 2>(c, 3);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * kLoadsPerStep - 2) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i) read_piece(c, 0, 0, i, X);
    for (int st = 0; st < c.n_steps; st += kRing) {
        step64<HASK, 0>(c, st, X, Y, s);
        if (st + 1 >= c.n_steps) break;   // (wave-uniform)
        step64<HASK, 1>(c, st + 1, X, Y, s);
        if (st + 2 >= c.n_steps) break;
        step64<HASK, 2>(c, st + 2, X, Y, s);
        if (st + 3 >= c.n_steps) break;
        step64<HASK, 3>(c, st + 3, X, Y, s);
        if (!HASK && ((st / kRing + 1) % (kFlushSteps / kRing)) == 0) flush(s.acc, tot);
    }
    // the last tile of the last group
    if constexpr (HASK) {
        fold_km(s.P, s.pm, s.kf, s.bias, s.acc[1][1]);
        // a bias for every group (and, in tile (1, 1), one of the first fold)
        const uint32_t off = 2 * (uint32_t) c.n_steps * (uint32_t) kBiasBits;
#pragma unroll
        for (int a = 0; a < 2; ++a) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    tot[a][b][r] = (int32_t) (__builtin_bit_cast(uint32_t, s.acc[a][b][r]) - off - (a & b ? (uint32_t) kBiasBits : 0u));
                }
            }
        }
    } else {
        fold_fast(s.P, s.pm, s.acc[1][1]);
        flush(s.acc, tot);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the refetches of the last steps
}

// Up to three weights of one K in one launch: row tile r of the launch belongs to weight w with first[w] <= r <
// first[w + 1]. (What a launch loses is its end: the tiles beyond whole rounds of the chip, cut along K, and the wait for
// the last of them. One launch over q + k + v at K = 5120, N = 6144 + 1024 + 1024, 2048 tokens, has 512 tiles, two whole
// rounds.)
// (a single weight's launch, SET = false, carries one entry)
template <bool SET>
struct TileSet {
    static constexpr int kN = SET ? kMaxFused : 1;
    const float   *s_w[kN];
    const uint8_t *kmul[kN];
    const int32_t *flags[kN];
    float         *y[kN];
    int64_t        ldy[kN];
    int64_t        N[kN];
    int            n_panels[kN];
    int            first[kN];   // unused slots hold the total, so no tile selects them
};

// SET: a launch over several weights (a form of its own: a single weight's launch would pay 1 % for the selection)
template <int GS, bool SET>
__global__ void __launch_bounds__(kThreads)
rq_gemm6_kernel(const TileSet<SET> ts, const uint8_t *__restrict__ act6, const float *__restrict__ m4,
                const float *__restrict__ u, int M, int Mp, int ng, int n_tok_tiles, int n_tiles, int super_tiles,
                int n_whole, int parts, int *__restrict__ counters, unsigned long long *__restrict__ slabs) {
    __shared__ __align__(16) uint8_t ring[kRingBytes];
    constexpr int kXpose = kRingBytes - 8 * 32 * kXposeStride * 4;   // the epilogue's output blocks
    static_assert(kXpose >= kOffA, "fit the weights' stages");
    // the epilogue's operands, fetched ahead of the first groups: the scales of the tile's 256 rows, then the units of
    // its 128 tokens
    __shared__ __align__(16) float s_pre[kTileRows + kTileTok + 4];   // (+ a word for the arrival count of a slice)

    // Workgroups go to the eight XCDs round robin: every XCD gets a contiguous run of tiles, visited in super-tiles of
    // 8 row tiles x 4 token tiles (the 32 workgroups an XCD runs at a time then share 8 weight tiles and 4 activation
    // tiles in its L2), or with the token tiles running fastest where the launch is not made of whole super-tiles.
    // The first n_whole workgroups take a whole tile each. The tiles after them (fewer than would fill the chip once)
    // are cut along K into `parts` slices each, one workgroup per slice, which meet through memory (see the epilogue).
    int row_tile, t0, part = 0, slot = 0;
    {
        int v = blockIdx.x;
        if (v < n_whole) {
            const int per_xcd = n_whole / kXcds;
            if (v < per_xcd * kXcds) v = (v % kXcds) * per_xcd + v / kXcds;
        } else {
            // slices: an XCD gets a contiguous run of (tile, part) pairs, parts running slowest within the run, so that
            // neighbouring tiles' slices of the same stretch of K are resident together
            int j = v - n_whole;
            const int n_sl = (n_tiles - n_whole) * parts, per_xcd = n_sl / kXcds;
            if (j < per_xcd * kXcds) j = (j % kXcds) * per_xcd + j / kXcds;
            v = n_whole + j / parts;
            part = j - (j / parts) * parts;
        }
        gemm6_tile(v, n_tok_tiles, super_tiles, row_tile, t0);
        slot = v - n_whole;
    }
    int wsel = 0;
    if constexpr (SET) {
        wsel = (row_tile >= ts.first[1]) + (row_tile >= ts.first[2]);
        row_tile -= wsel == 0 ? 0 : wsel == 1 ? ts.first[1] : ts.first[2];   // now of its weight
    }
    auto of_weight = [&](const auto &v) {
        if constexpr (SET) return wsel == 0 ? v[0] : wsel == 1 ? v[1] : v[2];
        else return v[0];
    };
    const float *__restrict__ s_w = of_weight(ts.s_w);
    const uint8_t *__restrict__ kmul = of_weight(ts.kmul);
    const int32_t *__restrict__ flags = of_weight(ts.flags);
    float *__restrict__ y = of_weight(ts.y);
    const int64_t ldy = of_weight(ts.ldy);
    const int64_t N = of_weight(ts.N);
    const int n_panels = of_weight(ts.n_panels);
    const bool sliced = (int) blockIdx.x >= n_whole;
    // this workgroup's steps (two groups each) of the tile's ng / 2
    const int s_begin = sliced ? (int) ((int64_t) (ng / 2) * part / parts) : 0;
    const int s_end = sliced ? (int) ((int64_t) (ng / 2) * (part + 1) / parts) : ng / 2;
    const int tid = threadIdx.x;
    const uint8_t *w6 = plane6_of(flags);
    // (read up here, in front of the assembly statements: behind them the compiler takes the word as possibly overwritten
    // and fetches it with a vector load, whose wait stands for a trip to memory between the set-up and the first group, 0.4
    // to 1 us of every launch)
    const bool hask = flags[0] & 1;
    Ctx c;
    c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    c.wr = c.wave & 3;
    c.wc = c.wave >> 2;
    c.lane = tid & 63;
    c.n_steps = s_end - s_begin;
    c.g0 = 2 * s_begin;
    const uint8_t *w_tile = w6 + (size_t) row_tile * ng * (kCellsA * 16);   // this tile's rows, group 0
    const size_t a_step = (size_t) (Mp / 32) * kFrag6;                       // bytes between groups of the activation plane
    const uint8_t *a_tile = act6 + (size_t) (t0 / 32) * kFrag6;              // this tile's tokens, group 0
    // (the weights of a step's two groups are 24 runs of 1 KiB one behind the other, the activations' 6 and 6: a wavefront takes
    // runs w, w + 8, w + 16 of the one and run w of the other)
    c.a_src = uniform(w_tile + (size_t) s_begin * kStageA + c.wave * 1024);
    c.b_step = (uint32_t) (2 * a_step);
    c.b_src = uniform(a_tile + (size_t) (c.wave / 6) * a_step + (size_t) (c.wave % 6) * 1024 + (size_t) s_begin * c.b_step);
    if (c.wave < 4) {          // the last 4 KB of the second group's activations
        c.t_step = c.b_step;
        c.t_off = (uint32_t) c.lane * 16;
        c.t_src = a_tile + a_step + (size_t) (2 + c.wave) * 1024 + (size_t) s_begin * c.t_step;
    } else if (!(c.wave & 1)) { // the tokens' multipliers of the two groups, half a wavefront each
        c.t_step = (uint32_t) (2 * Mp * sizeof(float));
        c.t_off = (uint32_t) (c.lane >> 5) * (uint32_t) (Mp * sizeof(float)) + (uint32_t) (c.lane & 31) * 16;
        c.t_src = reinterpret_cast<const uint8_t *>(m4 + t0) + (size_t) s_begin * c.t_step;
    } else {                    // the weight multipliers of the tile's 256 rows (a byte per row: 64 bytes per panel of 64 rows), a
                                // quarter of a wavefront a group; the other half fetches them once more, into cells nobody reads
        const int x = c.lane & 15, pnl = min(row_tile * 4 + (x >> 2), n_panels - 1) - row_tile * 4;
        c.t_step = 2 * kPanelRows;
        c.t_off = (uint32_t) ((pnl * ng + ((c.lane >> 4) & 1)) * kPanelRows + (x & 3) * 16);
        c.t_src = kmul + (size_t) row_tile * 4 * ng * kPanelRows + (size_t) s_begin * c.t_step;
    }
    c.t_src = uniform(c.t_src);
    const uint32_t lds0 = (uint32_t) (uintptr_t) (lds_void *) ring;
    c.lds_run = lds0 + c.wave * 1024;
    c.lds_t = lds0 + (c.wave < 4 ? 8192 + c.wave * 1024 : c.wave & 1 ? kOffK : kOffM);
    c.b16 = lds0 + 2 * c.wc * kFrag6 + 16 * c.lane;
    c.b8 = lds0 + 2 * c.wc * kFrag6 + 1024 + 8 * c.lane;
    c.m = lds0 + kOffM + 256 * c.wc + 4 * (c.lane & 31);
    c.k = lds0 + kOffK + 64 * c.wr + 4 * (c.lane >> 5);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        c.a16[i] = lds0 + kOffA + 2 * i * kStageA + 2 * c.wr * kFrag6 + 16 * c.lane;
        c.a8[i] = lds0 + kOffA + 2 * i * kStageA + 2 * c.wr * kFrag6 + 1024 + 8 * c.lane;
        // (registers of their own: without these statements the compiler forms an address per stage)
        asm volatile("" : "+v"(c.a16[i]), "+v"(c.a8[i]));
    }
    asm volatile("" : "+v"(c.b16), "+v"(c.b8), "+v"(c.m), "+v"(c.k));
    const int panel = min(row_tile * 4 + c.wr, n_panels - 1);
    c.k_src = kmul + (size_t) panel * ng * kPanelRows + 4 * (c.lane >> 5);

    if (c.wave < 4) {
        const int64_t n = (int64_t) row_tile * kTileRows + 64 * c.wave + c.lane;
        load_to_lds_dword(s_w + (n < N ? n : N - 1), &s_pre[64 * c.wave]);
    } else if (c.wave < 6) {
        const int t = t0 + 64 * (c.wave - 4) + c.lane;
        load_to_lds_dword(u + (t < M ? t : M - 1), &s_pre[kTileRows + 64 * (c.wave - 4)]);
    }

    int32_t tot[2][2][16];
    // fp32 rounding toward minus infinity for the folds (MODE bits 1:0); the MFMA sums are exact in any mode
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2" ::: "memory");
    if (hask) {
        if constexpr (GS == 1) body64<true>(c, tot);
        else body<true, GS>(c, tot);
    } else {
        if constexpr (GS == 1) body64<false>(c, tot);
        else body<false, GS>(c, tot);
    }
    // Back to round to nearest even for the epilogue. The compiler does not know that fp32 arithmetic reads MODE, so
    // the totals pass through a statement on either side of the change: the one in front keeps the last folds (which
    // the totals depend on) from being scheduled behind it, the one behind keeps the conversions below from being
    // scheduled in front of it.
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(tot[a][b][r]));
        }
    }
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0" ::: "memory");
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(tot[a][b][r]));
        }
    }

    if (sliced) {
        // A slice of K: its totals go to a slab of their own (64 ints per thread, written through to memory at
        // device scope: the slices of a tile run on different XCDs, each with its own L2), then one atomic per
        // workgroup counts the arrival. The workgroup that completes the count adds the other slices' slabs to the
        // totals it still holds and goes on to the epilogue; the others are done. (An atomic per output instead,
        // accumulating in 64-bit arrival cells, cost more than the slicing gained: 8 M device-scope atomics.)
        // (Slabs move as 16 bytes per lane with the cache policy of a device-scope access: written through to memory,
        // read past this XCD's L2.)
        constexpr int kSlabBytes = kTileRows * kTileTok * (int) sizeof(int32_t);
        uint8_t *slab_base = reinterpret_cast<uint8_t *>(slabs) + (size_t) slot * parts * kSlabBytes;
        const uint32_t lane_off = (uint32_t) tid * 16;
        {
            const __amdgpu_buffer_rsrc_t mine = __builtin_amdgcn_make_buffer_rsrc(slab_base + (size_t) part * kSlabBytes, 0, kSlabBytes, kRsrcWord3);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int a = i >> 3, b = (i >> 2) & 1, r = 4 * (i & 3);
                __builtin_amdgcn_raw_buffer_store_b128(v4i{ tot[a][b][r], tot[a][b][r + 1], tot[a][b][r + 2], tot[a][b][r + 3] }, mine,
                                                       lane_off + i * (kThreads * 16), 0, kDeviceScope);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's stores have reached memory
        __syncthreads();                                    // ... and everybody else's
        int *s_flag = reinterpret_cast<int *>(&s_pre[kTileRows + kTileTok]);
        if (tid == 0) {
            const int before = __hip_atomic_fetch_add(counters + slot, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (before == parts - 1) __hip_atomic_store(counters + slot, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *s_flag = before;
        }
        __syncthreads();
        if (*s_flag != parts - 1) return;
        // the other parts' slabs, the loads of the next one in flight while one is added
        v4i in[2][16];
        auto load_part = [&](int k, v4i (&dst)[16]) {   // k-th of the other parts
            const int pp = k < part ? k : k + 1;
            const __amdgpu_buffer_rsrc_t other = __builtin_amdgcn_make_buffer_rsrc(slab_base + (size_t) pp * kSlabBytes, 0, kSlabBytes, kRsrcWord3);
#pragma unroll
            for (int i = 0; i < 16; ++i) dst[i] = __builtin_amdgcn_raw_buffer_load_b128(other, lane_off + i * (kThreads * 16), 0, kDeviceScope);
        };
        auto add_part = [&](const v4i (&src)[16]) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int a = i >> 3, b = (i >> 2) & 1, r = 4 * (i & 3);
#pragma unroll
                for (int e = 0; e < 4; ++e) tot[a][b][r + e] += src[i][e];
            }
        };
        const int others = parts - 1;
        load_part(0, in[0]);
        for (int k = 0; k < others; k += 2) {
            if (k + 1 < others) load_part(k + 1, in[1]);
            add_part(in[0]);
            if (k + 1 < others) {
                if (k + 2 < others) load_part(k + 2, in[0]);
                add_part(in[1]);
            }
        }
    }

    // epilogue (reference patch line 176): y = ((float(total) * 16) * u) * s_w. In the MFMA result a lane holds one
    // token (column) and, per tile, rows 8 q + 4 (lane / 32) + 0 .. 3 for q = 0 .. 3: stored as they are, a wavefront's
    // stores would be 32-byte pieces of 32 different rows of y (a third of the kernel's time went there). So every
    // wavefront turns its four 32 x 32 blocks through LDS one after the other and writes 128 contiguous bytes per token. The
    // eight wavefronts' 36 KiB lie over the weights of the last stage and half of those of the one before, at which the refetches
    // of the last steps are aimed: every wavefront has waited for all its loads (the vmcnt(0) that ends body and body64)
    // before it comes to this barrier, and that wait may not go.
    __syncthreads();   // every wavefront is done reading the ring
    float *xp = reinterpret_cast<float *>(ring + kXpose) + c.wave * (32 * kXposeStride);
    const int h = c.lane >> 5;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const float ut = s_pre[kTileRows + 64 * c.wc + 32 * b + (c.lane & 31)];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int rw = 8 * q + 4 * h;   // row within the block
                const float4 sw = *reinterpret_cast<const float4 *>(&s_pre[64 * c.wr + 32 * a + rw]);
                float4 o;
                o.x = (((float) tot[a][b][4 * q + 0] * 16.0f) * ut) * sw.x;
                o.y = (((float) tot[a][b][4 * q + 1] * 16.0f) * ut) * sw.y;
                o.z = (((float) tot[a][b][4 * q + 2] * 16.0f) * ut) * sw.z;
                o.w = (((float) tot[a][b][4 * q + 3] * 16.0f) * ut) * sw.w;
                *reinterpret_cast<float4 *>(&xp[(c.lane & 31) * kXposeStride + rw]) = o;
            }
            // (a wavefront reads back only what it wrote itself, and its LDS operations complete in order)
            const int64_t n = (int64_t) row_tile * kTileRows + 64 * c.wr + 32 * a + 4 * (c.lane & 7);
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                const int tw = 8 * it + (c.lane >> 3);   // token within the block
                const int t = t0 + 64 * c.wc + 32 * b + tw;
                const float4 o = *reinterpret_cast<const float4 *>(&xp[tw * kXposeStride + 4 * (c.lane & 7)]);
                if (t >= M) continue;
                float *dst = y + (int64_t) t * ldy + n;
                if (n + 3 < N && ((reinterpret_cast<uintptr_t>(dst) & 15) == 0)) {
                    // the output is written once and not read back by this launch: non-temporal
                    typedef float v4f __attribute__((ext_vector_type(4)));
                    __builtin_nontemporal_store(v4f{ o.x, o.y, o.z, o.w }, reinterpret_cast<v4f *>(dst));
                } else {
                    const float ov[4] = { o.x, o.y, o.z, o.w };
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (n + i < N) dst[i] = ov[i];
                    }
                }
            }
        }
    }
}

template <bool SET>
void set_weight(TileSet<SET> &ts, int slot, const FusedWeights &w, int k, int first) {
    const PreparedLayout &L = w.L[k];
    const uint8_t *p = w.prepared[k];
    ts.s_w[slot] = reinterpret_cast<const float *>(p + L.off_sw);
    ts.kmul[slot] = p + L.off_kmul;
    ts.flags[slot] = reinterpret_cast<const int32_t *>(p + L.off_flags);
    ts.y[slot] = w.y[k];
    ts.ldy[slot] = w.ldy[k];
    ts.N[slot] = L.N;
    ts.n_panels[slot] = L.n_panels;
    ts.first[slot] = first;
}

}  // namespace

Gemm6Plan gemm6_plan(int n_row_tiles, int64_t M, int ng, int groups_per_fold) {
    Gemm6Plan pl;
    const int n_tok_tiles = (int) ((M + kTileTok - 1) / kTileTok);
    pl.n_tiles = n_row_tiles * n_tok_tiles;
    pl.n_whole = pl.n_tiles;
    pl.parts = 1;
    // Whole rounds of the chip run a tile per workgroup. What is left over (fewer tiles than compute units) would
    // keep the chip busy for one more whole tile time; cut along K into `parts` slices per tile it takes 1 / parts of
    // that. (The count of compute units is taken as the 256 of the part this library is written for: the plan must
    // not depend on the device, because the workspace is sized from it.)
    const int left = pl.n_tiles % kPlanUnits;
    if (left > 0 && kPlanUnits / left >= 2) {
        // more slices = less work per slice, but the workgroup that completes a tile reads the other slices' slabs one
        // after the other (about 2 us each) and every slice pays its own start (about 5 us): per step 1.1 us
        const int steps = ng / 2;
        int best = 1;
        double best_cost = 1.1 * steps;
        for (int parts = 2; parts <= kPlanUnits / left && parts <= steps / 2; ++parts) {
            // wider activation groups: a slice holds whole groups and an even number of steps
            if (groups_per_fold > 1 && steps % (2 * parts) != 0) continue;
            const double cost = 1.1 * ((steps + parts - 1) / parts) + 5.0 + 2.0 * (parts - 1);
            if (cost < best_cost) {
                best_cost = cost;
                best = parts;
            }
        }
        if (best >= 2) {   // (left * parts <= kPlanUnits slices: the workspace holds a slab for each)
            pl.parts = best;
            pl.n_whole = pl.n_tiles - left;
        }
    }
    // one arrival counter per cut tile, then a slab of 256 x 128 ints per slice
    pl.cell_bytes = pl.parts > 1 ? kGemm6CounterBytes + (size_t) (pl.n_tiles - pl.n_whole) * pl.parts * kTileRows * kTileTok * sizeof(int32_t) : 0;
    return pl;
}

namespace {

// Microseconds of a launch by its plan: a round of whole tiles and, behind it, the slices of the tiles that are cut, by
// steps of two groups. Fitted to 112 sets of two and three weights (K = 2560 to 32768, 5 to 750 tiles), in one launch and
// in one each; it gives the ratio of the two within 7 % where that is near 1.
double tiled_price(const Gemm6Plan &pl, int ng, bool weight_multipliers) {
    const int steps = ng / 2;
    const int rounds = (pl.n_whole + kPlanUnits - 1) / kPlanUnits;
    const double whole = weight_multipliers ? 5.8 + 1.53 * steps : 7.4 + 0.72 * steps;
    const int slice = (steps + pl.parts - 1) / pl.parts;
    const double cut = weight_multipliers ? 11.5 + 1.56 * slice + 0.8 * (pl.parts - 1) : 12.3 + 0.85 * slice + 1.1 * (pl.parts - 1);
    return rounds * whole + (pl.parts > 1 ? cut : 0.0);
}

// The same for the kernel of small launches (rq_block6.hip), by rounds of its units and the groups of one wavefront: of whole units.
// K = 1024 / 5120 / 17408: 192 units 5.1 / 10.4 / 25.9 us, with weight groups of 64, K = 5120 / 17408, 13.6 / 35.7. A last round that goes
// in pieces takes less than it is priced: 16 units 3.6 / 5.7 / 12.5, groups of 64 6.5 / 14.6 (whole 5.2 / 9.3 / 21.2, 12.2 / 29.6); 384 units 10.0 /
// 18.4 at K = 1024 / 5120, groups of 64, K = 5120 23.4 (the second round's 128 in halves; whole 9.5 / 18.7, 24.2). So what goes to units by
// this price is at least as fast there, and some of what goes to slices would be faster in units.
double block_price(int64_t units, int ng, bool weight_multipliers) {
    const double rounds = (double) ((units + kPlanUnits - 1) / kPlanUnits);
    const int per_wave = (ng + 7) / 8;
    return rounds * (weight_multipliers ? 5.2 + 0.75 * per_wave : 4.2 + 0.53 * per_wave);
}

}  // namespace

// The cheapest of three. Few tiles: all of them in small units, as long as those are at most two rounds of the chip (K = 5120:
// 2 tiles 19.5 us in slices and 9.9 in whole units, 5.7 in the pieces that they go in; 48 tiles 24.4 and 19.4, 18.4 with the second
// round in halves; 96 tiles, three rounds, 27.7 and 28.6; K = 17408: 2 tiles 29.2 and 22.1, 12.5 in pieces, 48 tiles 39.2 and 47.3, all of it
// in whole units). Whole rounds and a few tiles over: those few in units behind the rounds (K = 5120, N = 17408, 512 tokens, 256 + 16
// tiles: 60.8 us with the 16 in slices, 54.4 with them in 128 whole units; 8.5 of the call's 55 now, in halves). Everything else: tiles,
// the rest in slices.
// The prices are of weights in the memory-side cache. From memory a unit gets its rows at 20 KB per microsecond, whatever the
// others do, while K slices spread a tile's over compute units, so units end where the rows are long: without multipliers
// at K = 17408 in one round and K = 6144 in two (with them the fold is slow enough to hide it). The lines are those of whole units: 64 and
// fewer, in four pieces, get their rows from four compute units (K = 17408, 32 units from memory 17.7 us instead of 32.0), so that for them, and
// for a second round of at most 128, units could go on to longer rows. Whole call in us, slices / whole units, from the cache, then from memory. One round, 128 tokens: K = 17408, N = 1000 39.4 / 32.4, 40.6 / 42.1, N = 6000 42.0 / 33.4,
// 47.4 / 44.0; K = 22528, N = 1000 44.0 / 39.5, 45.1 / 51.7; K = 32768 51.5 / 52.5, 52.7 / 69.7. Two: K = 5120, N = 3000, 400 tokens
// 31.4 / 26.2, 32.8 / 30.9; K = 10240 40.5 / 41.0, 41.7 / 48.8, N = 6000, 256 tokens 38.3 / 38.5, 39.7 / 48.3.
Gemm6Route gemm6_route(const FusedWeights &w, int64_t M, int groups_per_fold, bool weight_multipliers, bool have_slabs) {
    int n_row_tiles = 0;
    int64_t n_panels = 0;
    for (int i = 0; i < w.n; ++i) {
        n_row_tiles += w.L[i].n_rtiles;
        n_panels += w.L[i].n_panels;
    }
    const int ng = w.L[0].ng;
    Gemm6Route r;
    r.plan = gemm6_plan(n_row_tiles, M, ng, groups_per_fold);
    r.n_tiles = r.first_block = r.plan.n_tiles;
    r.units = 0;
    if (!have_slabs) {   // a workspace without slabs: every tile whole
        r.plan.n_whole = r.plan.n_tiles;
        r.plan.parts = 1;
    }
    r.price = tiled_price(r.plan, ng, weight_multipliers);
    if (groups_per_fold != 1) return r;   // (the small units fold groups of 64)
    const int64_t units = n_panels * ((M + 63) / 64);
    const double all = block_price(units, ng, weight_multipliers);
    // (a workspace without slabs: the choice is between units and whole tiles, K = 32768 200 us)
    const bool short_rows = weight_multipliers || !have_slabs || ng <= (units <= kPlanUnits ? 272 : 96);
    if (units <= 2 * kPlanUnits && short_rows && all < r.price) {
        r.plan.n_tiles = r.plan.n_whole = r.first_block = 0;
        r.plan.parts = 1;
        r.units = units;
        r.price = all;
        return r;
    }
    const int left = r.n_tiles % kPlanUnits, rounds = r.n_tiles - left;
    if (left > 0 && rounds > 0) {
        Gemm6Plan whole = r.plan;
        whole.n_tiles = whole.n_whole = rounds;
        whole.parts = 1;
        const double both = tiled_price(whole, ng, weight_multipliers) + 2.0 + block_price((int64_t) left * 8, ng, weight_multipliers);
        if (left * 8 <= 2 * kPlanUnits && both < r.price) {
            r.plan = whole;
            r.first_block = rounds;
            r.units = (int64_t) left * 8;
            r.price = both;
        }
    }
    return r;
}

// One launch has at most the rounds of all the separate ones, but what it has left over may be too many tiles to cut (more
// than half a round), where each weight's own tiles can be. With long rows that is the greater loss: K = 17408,
// N = 4134 + 2216, 525 tokens (85 + 45 tiles) 123.4 us in one launch, 116.4 in two; K = 32768, 66 + 82 tiles 204 and 196.
// The other way round K = 5120, N = 6144 + 1024 + 1024, 512 tokens is 40 and 79 us. (3 % apart is what the prices tell.)
bool gemm6_one_launch(const FusedWeights &w, int64_t M, bool weight_multipliers) {
    double each = 0.0;
    for (int i = 0; i < w.n; ++i) {
        FusedWeights one = {};
        one.n = 1;
        one.L[0] = w.L[i];
        each += gemm6_route(one, M, 1, weight_multipliers, true).price;
    }
    return gemm6_route(w, M, 1, weight_multipliers, true).price <= 1.03 * each;
}

hipError_t launch_gemm6(const Gemm6Args &a, hipStream_t stream) {
    TileSet<true> ts;
    TileSet<false> t1;
    int n_row_tiles = 0;
    for (int i = 0; i < kMaxFused; ++i) {
        const int k = i < a.w.n ? i : a.w.n - 1;   // unused slots repeat the last weight (never selected)
        set_weight(ts, i, a.w, k, n_row_tiles);
        if (i == 0) set_weight(t1, 0, a.w, 0, 0);
        if (i < a.w.n) n_row_tiles += a.w.L[k].n_rtiles;
    }
    const int ng = a.w.L[0].ng;
    const int n_tok_tiles = a.Mp / kTileTok;
    const Gemm6Route route = gemm6_route(a.w, a.M, a.groups_per_fold, a.weight_multipliers, a.cells != nullptr);
    const Gemm6Plan &pl = route.plan;
    if (route.n_tiles != n_row_tiles * n_tok_tiles) return hipErrorInvalidValue;
    if (a.w.n > 1 && a.groups_per_fold != 1) return hipErrorInvalidValue;   // (wider groups go weight by weight)
    const int super_tiles = n_tok_tiles % 4 == 0 && n_row_tiles % 8 == 0;
    if (pl.n_tiles == 0) return launch_block6(a, stream);
    const int grid = pl.n_whole + (pl.n_tiles - pl.n_whole) * pl.parts;
    const float *m4 = reinterpret_cast<const float *>(a.act6 + act6_plane_bytes(ng, a.Mp));
#define RQ_LAUNCH6(GS, SET, TS)                                                                                            \
    hipLaunchKernelGGL((rq_gemm6_kernel<GS, SET>), dim3(grid), dim3(kThreads), 0, stream, TS, a.act6, m4, a.u, a.M,  \
                       a.Mp, ng, n_tok_tiles, pl.n_tiles, super_tiles, pl.n_whole, pl.parts,                         \
                       reinterpret_cast<int *>(a.cells),                                                             \
                       reinterpret_cast<unsigned long long *>(reinterpret_cast<uint8_t *>(a.cells) + kGemm6CounterBytes))
    // (The kernels lie in the code object in the order in which they stand here. Behind the 57 KB of the H68 rotation a
    // launch starts with a cold instruction cache, and how much of it the two share depends on the place: with the sets'
    // kernels first, K = 17408, N = 5120 takes 60.1 us at 256 tokens and 77.9 at 512, with the single weights' first 58.7
    // and 76.9; each kernel by itself takes the same time either way.)
    if (a.w.n == 1) {
        if (a.groups_per_fold == 1) RQ_LAUNCH6(1, false, t1);
        else if (a.groups_per_fold == 2) RQ_LAUNCH6(2, false, t1);
        else RQ_LAUNCH6(4, false, t1);
    } else {
        RQ_LAUNCH6(1, true, ts);
    }
#undef RQ_LAUNCH6
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || route.first_block == route.n_tiles) return e;
    return launch_block6_tiles(a, super_tiles, route.first_block, route.n_tiles, stream);
}

}  // namespace rq
