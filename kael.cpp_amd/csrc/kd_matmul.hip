// kd_matmul.hip - batched matrix products for gfx950.
//
// Contract of reference include/kael/device_kernels.h:111-112 / src/cuda/backend.cu:142-171:
// out[b] = a[b] . b[b] for `batches` row-major matrices, `out` overwritten (never accumulated).
// f32 and f64 are floating point, i64 wraps (kernels.inl:160-169), bool is rejected
// (src/ops/linalg.cpp:72). The reference computes a 4x4 register tile per thread straight from
// global memory (kernels.inl:136-177). Here, per shape:
//
//   pieces f32, the main family: each operand as three bf16 pieces, products on the bf16 matrix
//          cores accumulated in f32; tiles from 64x64 to 256x128 and a K split chosen by size.
//   small  f32, few tiles and a short K (C1's 512^3, small MLP layers): 32x32 tiles, one workgroup of 16
//          waves each, the waves splitting K and reading their operands straight from global memory,
//          their partial tiles added in LDS in wave order. Many batches of tiles that fill less than 64x64 too.
//   rowdot f32, at most 4 columns: a wave per output row.
//   skinny f32, at most 8 rows and a short K: a wave per 256 columns and a quarter of K.
//   parts  f32, split-K partials for the GPT-2 engine's short prompts.
//   general f32 operands whose strides pieces cannot address, on the f32 matrix cores.
//   f64    64x64 tiles on the FP64 matrix cores.
//   tiled  i64: 64x64 LDS tiles, 4x4 outputs per lane (exact wrapping).
//
// Every kernel takes per-operand element strides (batch, row, column), which is how
// kd_matmul_strided reads transposed or batch-broadcast operands in place.
#include <algorithm>
#include <type_traits>

#include "kd_internal.h"
#include "kd_pieces.h"

namespace kd {

namespace {

struct Strides3 {
    int64_t b, r, c;
};

// Batches address the operands on one level (batch b at b * sa.b) or, with heads > 1, on two:
// b = o * heads + h at o * sa.b + h * ha (attention's [batch, head] views of a [batch, token,
// head, dim] tensor, which no single batch stride describes).
struct MatmulArgs {
    int64_t batches, M, K, N;
    Strides3 sa, sb, so;
    int64_t heads = 1;
    int64_t ha = 0, hb = 0, ho = 0;
    const void* bias = nullptr;  // element n added to column n of every output row (element type)
};

// out = v, or v + bias[col] rounded once (wrapping for i64): the bias add of kael's Linear
// (product + bias) as the epilogue of the product that precedes it.
template <typename T> __device__ __forceinline__ T plus_bias(T v, const void* bias, int64_t col) {
    if (bias == nullptr) return v;
    const T b = static_cast<const T*>(bias)[col];
    if constexpr (std::is_same_v<T, int64_t>) return wrap_add(v, b);
    else return add_sep(v, b);
}

// Element offset of batch `batch` in an operand with outer / head strides `outer` / `inner`.
__host__ __device__ __forceinline__ int64_t batch_offset(const MatmulArgs& p, int64_t batch, int64_t outer,
                                                         int64_t inner) {
    if (p.heads == 1) return batch * outer;
    const int64_t o = static_cast<uint32_t>(batch) / static_cast<uint32_t>(p.heads);
    return o * outer + (batch - o * p.heads) * inner;
}

constexpr int kThreads = 256;

// ---- tile order ---------------------------------------------------------------------------------

typedef float v16f __attribute__((ext_vector_type(16)));

// Maps the linear workgroup id to a (tile_m, tile_n) pair so that the workgroups that one XCD
// runs (ids congruent mod 8 are dispatched to the same XCD) cover a compact block of tiles,
// sharing A rows and B columns in that XCD's L2.
__device__ __forceinline__ void tile_of(int64_t id, int64_t tiles_m, int64_t tiles_n, int64_t& tm, int64_t& tn) {
    const int64_t total = tiles_m * tiles_n;
    int64_t local = id;
    if (total % 8 == 0) local = (id % 8) * (total / 8) + id / 8;
    // Grouped order: columns of 8 tile-rows walked along N.
    constexpr int64_t kGroup = 8;
    const int64_t group_size = kGroup * tiles_n;
    const int64_t group = local / group_size;
    const int64_t first_m = group * kGroup;
    const int64_t rows_in_group = std::min<int64_t>(kGroup, tiles_m - first_m);
    const int64_t in_group = local % group_size;
    tm = first_m + in_group % rows_in_group;
    tn = in_group / rows_in_group;
}

// ---- pieces family (f32 on the bf16 matrix cores) ---------------------------------------------
//
// An f32 value, scaled by 2^16, is the exact sum of three bf16 values (kd_pieces.h), so a product of
// two f32 values is 2^-32 times the sum of nine bf16 products, of which the six above 2^-27 of it are taken: hi.hi on one accumulator, and lo.hi, hi.lo, mid.mid,
// mid.hi, hi.mid on a second, both in f32 by v_mfma_f32_32x32x16_bf16, added at the end. The dropped
// three are below half an f32 rounding of the product; what bounds the error is the rounding of the
// running sum, and hi.hi's takes two roundings per 16 K where v_mfma_f32_32x32x2f32 takes sixteen.
// Error against 64 bits, 2-norm, normal inputs, beside v_mfma_f32_32x32x2f32: K = 96 5.8e-8 (1.8e-7),
// 256 8.9e-8 (2.1e-7), 2048 2.7e-7 (8.1e-7), 4096 1.9e-7 in splits (5.7e-7); of the column sums of
// the result likewise, which the second accumulator is for: the bf16 instructions cut the low bits
// of what they align below the accumulator towards minus infinity, and six products on one
// accumulator leave a bias (2048: column sums 4.9e-6). The matrix cores keep bf16 subnormals, so with the
// scale every value below 2^112 splits; larger ones, infinities and NaN, and sums from 2^96 on, see the end.
//
// The rate: 2.5 PFLOP/s / 6 = 417 TFLOP/s of f32 products against 157 on the f32 matrix cores.
// Measured at 4096^3: 662 us (208 TFLOP/s: 1.25 PFLOP/s of bf16 products, where the vendor's bf16
// product reaches 1.13 at this size and 1.36 at 8192^3; the clock falls to ~2.1 GHz under either, and the scaling
// of the operands, one operation in 6.5 of the split, costs 3.5 %) against 966 us (142 TFLOP/s) on the f32
// matrix cores.
//
// A workgroup owns a TM x TN tile and stages both operands through LDS as pieces: each 8-deep K group
// of a row is one 16-byte unit per piece, [piece][group][row], so that a lane's MFMA operand is one
// conflict-free 16-byte read. The split into pieces (6.5 VALU operations per element) runs between
// the MFMAs of the step before. Global loads run two steps ahead (one step: 4096 x 256 x 768 on
// 128 x 128 tiles 24 us, two 17). A partial K step comes first, with guarded loads; rows past M or N
// repeat the last one and are not stored, so ragged sizes cost no tests in the loop. Element
// alignment is all that the loads need (a global 16-byte load takes any 4-byte address).

typedef float f4any __attribute__((ext_vector_type(4), aligned(4)));

// The LDS image of Rows (m of A, n of B) x BK of one operand. The 64 bytes after each group keep the
// writes of a K-contiguous operand, whose neighbouring lanes hold neighbouring groups, off one
// another's banks.
template <int Rows, int BK> struct PieceTile {
    static constexpr int kGroups = BK / 8;
    static constexpr int kUnits = Rows * kGroups;
    static constexpr int kGroup = Rows * 16 + 64;  // bytes
    static constexpr int kPiece = kGroups * kGroup;
    static constexpr int kBytes = 3 * kPiece;
};

// Row and group of unit `u`: neighbouring lanes along K where K is contiguous, along the rows elsewhere.
template <bool KContig, int Rows, int BK> __device__ __forceinline__ void unit_of(int u, int& row, int& g) {
    if constexpr (KContig) {
        g = u % (BK / 8);
        row = u / (BK / 8);
    } else {
        row = u % Rows;
        g = u / Rows;
    }
}

// One unit from `base` + `offset`; `ks` is the stride along K.
template <bool KContig>
__device__ __forceinline__ void load_unit(float (&x)[8], const float* base, int64_t offset, int64_t ks) {
    if constexpr (KContig) {
        const f4any v0 = *reinterpret_cast<const f4any*>(base + offset);
        const f4any v1 = *reinterpret_cast<const f4any*>(base + offset + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = v0[e];
            x[4 + e] = v1[e];
        }
    } else {
        const uint32_t off = static_cast<uint32_t>(offset);  // the host checks that it fits
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (base + e * ks)[off];
    }
}

// Its first `left` elements, then zeros.
__device__ __forceinline__ void load_unit_part(float (&x)[8], const float* base, int64_t offset, int64_t ks, int left) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = e < left ? base[offset + e * ks] : 0.f;
}

// AK / BK_: K is contiguous in A / B; elsewhere any strides. WM x WN waves of (TM / WM) x (TN / WN)
// outputs each. blockIdx.z is the K split: `k_split` deep, its partial sums `split_o` floats further
// into `out`.
template <bool AK, bool BKc, int TM, int TN, int WM, int WN, int BK, int Occ>
__global__ __launch_bounds__(WM * WN * 64, Occ) void pieces_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                                   float* __restrict__ out, MatmulArgs p, int k_split,
                                                                   int64_t split_o) {
    constexpr int kLanes = WM * WN * 64;
    using TA = PieceTile<TM, BK>;
    using TB = PieceTile<TN, BK>;
    constexpr int kUnits = TA::kUnits + TB::kUnits;
    constexpr int kPer = (kUnits + kLanes - 1) / kLanes;
    static_assert(TA::kUnits % 64 == 0 && TB::kUnits % 64 == 0);  // a wave's units are all of one operand
    constexpr int IM = TM / WM / 32, JN = TN / WN / 32;
    constexpr int kStage = TA::kBytes + TB::kBytes;
    __shared__ __attribute__((aligned(16))) char lds[2 * kStage];

    const int M = static_cast<int>(p.M), N = static_cast<int>(p.N);
    int64_t tm, tn;
    tile_of(blockIdx.x, (M + TM - 1) / TM, (N + TN - 1) / TN, tm, tn);
    const int m0 = static_cast<int>(tm) * TM, n0 = static_cast<int>(tn) * TN;
    const int64_t k_begin = static_cast<int64_t>(blockIdx.z) * k_split;
    const int k_len = static_cast<int>(std::min<int64_t>(k_split, p.K - k_begin));
    a += batch_offset(p, blockIdx.y, p.sa.b, p.ha) + k_begin * p.sa.c;
    b += batch_offset(p, blockIdx.y, p.sb.b, p.hb) + k_begin * p.sb.r;
    out += batch_offset(p, blockIdx.y, p.so.b, p.ho) + blockIdx.z * split_o;

    const int t = threadIdx.x;
    const int lane = t % 64, wave = t / 64;
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane % 32, lh = lane / 32;

    // This thread's units: element offset from the tile's corner, and LDS offset.
    int64_t src[kPer];
    int dst[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int u = t + kLanes * i;
        int row, g;
        if (u < TA::kUnits) {
            unit_of<AK, TM, BK>(u, row, g);
            dst[i] = g * TA::kGroup + row * 16;
            src[i] = std::min(row, M - 1 - m0) * p.sa.r + 8 * g * p.sa.c;
        } else {
            unit_of<BKc, TN, BK>(u - TA::kUnits, row, g);
            dst[i] = TA::kBytes + g * TB::kGroup + row * 16;
            src[i] = std::min(row, N - 1 - n0) * p.sb.c + 8 * g * p.sb.r;
        }
    }
    const auto has = [&](int i) {
        return kLanes * (i + 1) <= kUnits || __builtin_amdgcn_readfirstlane(t) + kLanes * i < kUnits;
    };
    const auto is_a = [&](int i) {
        if (TA::kUnits % kLanes == 0) return kLanes * i < TA::kUnits;
        return __builtin_amdgcn_readfirstlane(t) + kLanes * i < TA::kUnits;
    };
    const int64_t a_step = BK * p.sa.c, b_step = BK * p.sb.r;
    const float* at = a + m0 * p.sa.r;
    const float* bt = b + n0 * p.sb.c;
    typedef float Regs[kPer][8];
    const auto fetch = [&](Regs& x) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (!has(i)) continue;
            if (is_a(i)) load_unit<AK>(x[i], at, src[i], p.sa.c);
            else load_unit<BKc>(x[i], bt, src[i], p.sb.r);
        }
    };
    const auto fetch_part = [&](Regs& x, int whole, int left) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (!has(i)) continue;
            int row, g;
            if (is_a(i)) {
                unit_of<AK, TM, BK>(t + kLanes * i, row, g);
                load_unit_part(x[i], at + whole * a_step, src[i], p.sa.c, left - 8 * g);
            } else {
                unit_of<BKc, TN, BK>(t + kLanes * i - TA::kUnits, row, g);
                load_unit_part(x[i], bt + whole * b_step, src[i], p.sb.r, left - 8 * g);
            }
        }
    };
    const auto stash = [&](const Regs& x, char* stage) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (!has(i)) continue;
            bf8 hi, mid, lo;
            split_pieces(x[i], hi, mid, lo);
            const int piece = is_a(i) ? TA::kPiece : TB::kPiece;
            char* d = stage + dst[i];
            *reinterpret_cast<bf8*>(d) = hi;
            *reinterpret_cast<bf8*>(d + piece) = mid;
            *reinterpret_cast<bf8*>(d + 2 * piece) = lo;
        }
    };

    v16f acc[IM][JN], small[IM][JN];
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = small[i][j][r] = 0.f;

    // MFMA operands of lane (li, lh): row li of its block, k = 8 lh .. 8 lh + 7.
    const int a_rd = lh * TA::kGroup + (wm * IM * 32 + li) * 16;
    const int b_rd = TA::kBytes + lh * TB::kGroup + (wn * JN * 32 + li) * 16;
    const auto multiply = [&](const char* stage) {
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            bf8 bf[JN][3];
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    bf[j][q] = *reinterpret_cast<const bf8*>(stage + b_rd + j * 512 + q * TB::kPiece + 2 * kk * TB::kGroup);
            constexpr int kA[5] = {2, 0, 1, 1, 0}, kB[5] = {0, 2, 1, 0, 1};
#pragma unroll
            for (int i = 0; i < IM; ++i) {
                bf8 af[3];
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    af[q] = *reinterpret_cast<const bf8*>(stage + a_rd + i * 512 + q * TA::kPiece + 2 * kk * TA::kGroup);
#pragma unroll
                for (int s = 0; s < 5; ++s)
#pragma unroll
                    for (int j = 0; j < JN; ++j)
                        small[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kA[s]], bf[j][kB[s]], small[i][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < JN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[0], bf[j][0], acc[i][j], 0, 0, 0);
            }
        }
    };
    // The end of a step in which the next stage was also split and stored: its VALU work, 52 operations a unit,
    // spread over the MFMAs (999 x 768 x 3072: 34 us; four after each 37.5).
    constexpr int kProducts = IM * JN * 6 * (BK / 16);
    const auto mix = [&]() {
#pragma unroll
        for (int q = 0; q < kProducts; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (52 * kPer + kProducts - 1) / kProducts, 0);
        }
        __syncthreads();
    };

    const int whole = k_len / BK;
    const int part = k_len - whole * BK;
    int ahead = whole;  // whole steps not fetched yet
    // The next whole step's elements; past the last one, that one again (unused).
    const auto next = [&](Regs& x) {
        fetch(x);
        if (--ahead > 0) {
            at += a_step;
            bt += b_step;
        }
    };
    Regs x0, x1;
    if (part > 0) fetch_part(x0, whole, part);
    else next(x0);
    int steps = ahead;  // stages after the first
    if (steps > 0) next(x1);
    stash(x0, lds);
    if (steps > 1) next(x0);
    __syncthreads();
    char* const s0 = lds;
    char* const s1 = lds + kStage;
    for (; steps > 1; steps -= 2) {
        multiply(s0);
        stash(x1, s1);
        next(x1);
        mix();
        multiply(s1);
        stash(x0, s0);
        next(x0);
        mix();
    }
    multiply(s0);
    if (steps > 0) {
        stash(x1, s1);
        __syncthreads();
        multiply(s1);
    }

    const int row0 = m0 + wm * IM * 32, col0 = n0 + wn * JN * 32;
    // A sum that is not finite means an infinity or a NaN among the inputs, or an overflow of the scaled sum or
    // of a piece (values from 2^112 = 5e33 on, sums from 2^96 = 8e28 on). The wave's outputs are then computed
    // again from the f32 operands on the f32 matrix cores.
    bool odd = false;
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] += small[i][j][r];
                odd |= !(__builtin_fabsf(acc[i][j][r]) < __builtin_inff());
                acc[i][j][r] *= kUnscale;
            }
    if (__any(odd)) {
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int j = 0; j < JN; ++j) {
                const float* ra = a + std::min(row0 + i * 32 + li, M - 1) * p.sa.r;
                const float* rb = b + std::min(col0 + j * 32 + li, N - 1) * p.sb.c;
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
                for (int k = lh; k - lh < k_len; k += 2) {
                    const float av = k < k_len ? ra[k * p.sa.c] : 0.f;
                    const float bv = k < k_len ? rb[k * p.sb.r] : 0.f;
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc[i][j], 0, 0, 0);
                }
            }
    }
    // Accumulator element r of lane (li, lh) is row 8*(r/4) + 4*lh + r%4, column li of its 32x32 block.
#pragma unroll
    for (int j = 0; j < JN; ++j) {
        const int col = col0 + j * 32 + li;
        if (col >= N) continue;
        const float bv = p.bias != nullptr ? static_cast<const float*>(p.bias)[col] : 0.f;
#pragma unroll
        for (int i = 0; i < IM; ++i) {
            const int first = row0 + i * 32 + 4 * lh;
            float* to = out + first * p.so.r + col * p.so.c;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int up = 8 * (r / 4) + r % 4;
                if (first + up < M) to[up * p.so.r] = p.bias != nullptr ? add_sep(acc[i][j][r], bv) : acc[i][j][r];
            }
        }
    }
}

// ---- general family (f32, strides beyond 32-bit tile offsets) -----------------------------------

constexpr int kBM = 128;
constexpr int kBN = 128;
constexpr int kBK = 16;
constexpr int kAld = kBK + 4;   // A tile [m][k]: row stride 20 floats, conflict-free 16-byte reads
constexpr int kBld = kBN + 4;   // B tile [k][n]

// What pieces_kernel does not address (negative or very large strides): 128x128 workgroup tiles, four
// waves of 2x2 v_mfma_f32_32x32x2f32 accumulators, K 16 at a time through double-buffered LDS, every
// element loaded by its own 64-bit offset behind a bounds check.
__global__ __launch_bounds__(kThreads) void general_f32_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                               float* __restrict__ out, MatmulArgs p) {
    __shared__ float As[2][kBM * kAld];
    __shared__ float Bs[2][kBK * kBld];

    int64_t tm, tn;
    tile_of(blockIdx.x, (p.M + kBM - 1) / kBM, (p.N + kBN - 1) / kBN, tm, tn);
    const int64_t m0 = tm * kBM;
    const int64_t n0 = tn * kBN;
    a += batch_offset(p, blockIdx.y, p.sa.b, p.ha);
    b += batch_offset(p, blockIdx.y, p.sb.b, p.hb);
    out += batch_offset(p, blockIdx.y, p.so.b, p.ho);

    const int t = threadIdx.x;
    const int lane = t % 64;
    const int wave = t / 64;
    const int wm = wave / 2;  // wave tile row (0..1), 64 rows each
    const int wn = wave % 2;  // wave tile col (0..1), 64 cols each
    const int li = lane % 32;
    const int lh = lane / 32;

    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    float ra[8], rb[8];
    const auto fetch = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = t + kThreads * i;
            const int64_t m = m0 + idx / kBK, ka = k0 + idx % kBK;
            ra[i] = (m < p.M && ka < p.K) ? a[m * p.sa.r + ka * p.sa.c] : 0.f;
            const int64_t kb = k0 + idx / kBN, n = n0 + idx % kBN;
            rb[i] = (kb < p.K && n < p.N) ? b[kb * p.sb.r + n * p.sb.c] : 0.f;
        }
    };
    const auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = t + kThreads * i;
            As[buf][(idx / kBK) * kAld + idx % kBK] = ra[i];
            Bs[buf][(idx / kBN) * kBld + idx % kBN] = rb[i];
        }
    };
    fetch(0);
    stash(0);
    __syncthreads();
    const int64_t ksteps = (p.K + kBK - 1) / kBK;
    for (int64_t ks = 0; ks < ksteps; ++ks) {
        const int cur = ks & 1;
        const bool more = ks + 1 < ksteps;
        if (more) fetch((ks + 1) * kBK);
        const float* as = As[cur];
        const float* bs = Bs[cur];
#pragma unroll
        for (int kg = 0; kg < kBK; kg += 8) {
            // Lane (li, lh) feeds k = kg + 4*lh + s to MFMA step s (s = 0..3): the same k for
            // its A element and its B element, so the 2-deep MFMA sums cover k = kg..kg+7.
            float4 af[2];
            float bf[2][4];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                af[i] = *reinterpret_cast<const float4*>(as + (wm * 64 + i * 32 + li) * kAld + kg + 4 * lh);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int s = 0; s < 4; ++s) bf[j][s] = bs[(kg + 4 * lh + s) * kBld + wn * 64 + j * 32 + li];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float av = s == 0 ? af[i].x : s == 1 ? af[i].y : s == 2 ? af[i].z : af[i].w;
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bf[j][s], acc[i][j], 0, 0, 0);
                }
            }
        }
        if (more) stash(cur ^ 1);
        __syncthreads();
    }

#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int64_t col = n0 + wn * 64 + j * 32 + li;
            if (col >= p.N) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = m0 + wm * 64 + i * 32 + 8 * (r / 4) + 4 * lh + (r % 4);
                if (row < p.M) out[row * p.so.r + col * p.so.c] = plus_bias(acc[i][j][r], p.bias, col);
            }
        }
}

// ---- small family (f32, few output tiles) -----------------------------------------------------

constexpr int kSmallTile = 32;
constexpr int kSmallWaves = 16;

// Products of few output tiles and a short K (C1's 512^3, small MLP layers), where a launch and the
// first loads are most of the time: one workgroup of 16 waves per 32x32 output tile, in one launch. Wave
// w multiplies the 8-deep K groups g = w, w + 16, ... straight from global memory on the f32 matrix
// cores - lane (li, lh) reads row li of A and column li of B at k = 8g + 4lh .. 8g + 4lh + 3, the
// operands of four v_mfma_f32_32x32x2f32 steps - with the next group's loads in flight during the
// current group's MFMAs. The 16 partial tiles are then added through LDS in wave order, so the result
// does not depend on timing. AVec / BVec: K is contiguous in A / B (one 16-byte load per lane and group,
// at any 4-byte address).
template <bool AVec, bool BVec>
__global__ __launch_bounds__(kSmallWaves * 64) void small_kernel(const float* __restrict__ a,
                                                                 const float* __restrict__ b,
                                                                 float* __restrict__ out, MatmulArgs p) {
    __shared__ float red[kSmallWaves][16 * 64];
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int64_t batch = blockIdx.z;
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kSmallTile;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * kSmallTile;
    const int lane = threadIdx.x % 64;
    const int w = threadIdx.x / 64;
    const int li = lane % 32;
    const int lh = lane / 32;
    // K steps in 32-bit element offsets (the host checks that K times the K strides fits).
    const int K = static_cast<int>(p.K);
    const int a_k = static_cast<int>(p.sa.c);
    const int b_k = static_cast<int>(p.sb.r);
    const int groups = (K + 7) / 8;
    const int64_t m = m0 + li;
    const int64_t n = n0 + li;
    const bool mok = m < p.M;
    const bool nok = n < p.N;
    const float* arow = a + batch_offset(p, batch, p.sa.b, p.ha) + (mok ? m : 0) * p.sa.r;
    const float* bcol = b + batch_offset(p, batch, p.sb.b, p.hb) + (nok ? n : 0) * p.sb.c;
    // Group g's operands, zero past the edges of A, B and K.
    const auto load = [&](int g, f4& av, f4& bv) {
        av = f4{0.f, 0.f, 0.f, 0.f};
        bv = f4{0.f, 0.f, 0.f, 0.f};
        if (g >= groups) return;
        const int k = g * 8 + 4 * lh;
        if (AVec && k + 3 < K) {
            if (mok) av = *reinterpret_cast<const f4any*>(arow + k);
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (mok && k + s < K) av[s] = arow[(k + s) * a_k];
        }
        if (BVec && k + 3 < K) {
            if (nok) bv = *reinterpret_cast<const f4any*>(bcol + k);
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (nok && k + s < K) bv[s] = bcol[(k + s) * b_k];
        }
    };
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    f4 ca, cb, na, nb;
    load(w, ca, cb);
    for (int g = w; g < groups; g += kSmallWaves) {
        load(g + kSmallWaves, na, nb);
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ca[s], cb[s], acc, 0, 0, 0);
        ca = na;
        cb = nb;
    }
    // Accumulator element r of lane (li, lh) is row 8*(r/4) + 4*lh + r%4, column li of the tile.
#pragma unroll
    for (int r = 0; r < 16; ++r) red[w][r * 64 + lane] = acc[r];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * 64; e += kSmallWaves * 64) {
        float v = red[0][e];
#pragma unroll
        for (int q = 1; q < kSmallWaves; ++q) v += red[q][e];
        const int r = e / 64;
        const int l = e % 64;
        const int64_t row = m0 + 8 * (r / 4) + 4 * (l / 32) + (r % 4);
        const int64_t col = n0 + l % 32;
        if (row < p.M && col < p.N)
            out[batch_offset(p, batch, p.so.b, p.ho) + row * p.so.r + col * p.so.c] = plus_bias(v, p.bias, col);
    }
}

// ---- parts family (f32, the GPT-2 engine's short prompts) ---------------------------------------

constexpr int kPartTile = 64;
constexpr int kPartStages = 2;  // stages of loads in flight

// Split-K partial products x . W^T of prompts of 33 to 128 positions on the f32 matrix cores: 64x64
// tiles, blockIdx.y the K split, `k_split` deep (a multiple of Deep). Such a product streams its weights
// once and is a chain of a few loads, so what counts is the time from the first load to the last store:
// four waves of one 32x32 accumulator, K 64 at a time through double-buffered LDS, so that a row's load
// is 256 contiguous bytes (32 at a time, 128 bytes: 9.1 us a launch against 8.3), loads two stages ahead
// (three: no change). GPT-2 small, 64 positions: a prefill 0.75 ms on this kernel, 0.85 on the pieces of
// 64x64 tiles, whose split takes 2 us of such a launch, and 0.86 on the small tiles, which win up to 32
// positions (0.60 against 0.67). Waves 0-1 load A, waves 2-3 load B; rows past M and N repeat the last
// and are not stored.
template <int Deep>
__global__ __launch_bounds__(kThreads) void parts_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                         float* __restrict__ parts, int M, int N, int k_split, int lda,
                                                         int ldb) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int kLd = Deep + 4;       // tiles [row][k]: conflict-free 16-byte reads and writes
    constexpr int kLanes = Deep / 4;    // lanes that load a row's stage
    constexpr int kRows = kThreads / 2 / kLanes, kLoads = kPartTile / kRows;
    __shared__ __attribute__((aligned(16))) float As[kPartStages][kPartTile * kLd];
    __shared__ __attribute__((aligned(16))) float Bs[kPartStages][kPartTile * kLd];
    int64_t tm, tn;
    tile_of(blockIdx.x, (M + kPartTile - 1) / kPartTile, (N + kPartTile - 1) / kPartTile, tm, tn);
    const int m0 = static_cast<int>(tm) * kPartTile;
    const int n0 = static_cast<int>(tn) * kPartTile;
    const int64_t k_begin = static_cast<int64_t>(blockIdx.y) * k_split;
    parts += static_cast<int64_t>(blockIdx.y) * M * N;

    const int t = threadIdx.x;
    const int lane = t % 64;
    const int wave = t / 64;
    const int wm = wave / 2;
    const int wn = wave % 2;
    const int li = lane % 32;
    const int lh = lane / 32;
    const bool loads_a = t < kThreads / 2;
    const int u = loads_a ? t : t - kThreads / 2;
    // load j of this thread: row u / kLanes + kRows * j of its operand, columns k = 4 (u % kLanes) .. +3
    const float* src[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int row = u / kLanes + kRows * j;
        src[j] = (loads_a ? a + static_cast<int64_t>(std::min(m0 + row, M - 1)) * lda
                          : b + static_cast<int64_t>(std::min(n0 + row, N - 1)) * ldb) + k_begin + 4 * (u % kLanes);
    }
    const auto fetch = [&](f4 (&r)[kLoads], int ks) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) r[j] = *reinterpret_cast<const f4any*>(src[j] + ks * Deep);
    };
    const auto stash = [&](const f4 (&r)[kLoads], int buf) {
        float* tile = loads_a ? As[buf] : Bs[buf];
#pragma unroll
        for (int j = 0; j < kLoads; ++j) *reinterpret_cast<f4*>(&tile[(u / kLanes + kRows * j) * kLd + 4 * (u % kLanes)]) = r[j];
    };
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const int a_rd = (wm * 32 + li) * kLd + 4 * lh, b_rd = (wn * 32 + li) * kLd + 4 * lh;
    const auto step = [&](int cur) {
#pragma unroll
        for (int kg = 0; kg < Deep; kg += 8) {
            const f4 af = *reinterpret_cast<const f4*>(&As[cur][a_rd + kg]);
            const f4 bf = *reinterpret_cast<const f4*>(&Bs[cur][b_rd + kg]);
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(af[s], bf[s], acc, 0, 0, 0);
        }
    };
    const int steps = k_split / Deep;
    f4 r[kPartStages][kLoads];
#pragma unroll
    for (int q = 0; q < kPartStages; ++q)
        if (q < steps) fetch(r[q], q);
    stash(r[0], 0);
    __syncthreads();
    for (int s0 = 0; s0 < steps; s0 += kPartStages) {
#pragma unroll
        for (int q = 0; q < kPartStages; ++q) {
            const int s = s0 + q;
            if (s >= steps) break;
            if (s + kPartStages < steps) fetch(r[q], s + kPartStages);
            step(q);
            if (s + 1 < steps) stash(r[(q + 1) % kPartStages], (q + 1) % kPartStages);
            __syncthreads();
        }
    }
    const int col = n0 + wn * 32 + li;
    if (col >= N) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm * 32 + 8 * (r / 4) + 4 * lh + (r % 4);
        if (row < M) parts[static_cast<int64_t>(row) * N + col] = acc[r];
    }
}

// ---- sums of split partials ---------------------------------------------------------------------

// Adds the split partials in split order and writes the output.
__global__ __launch_bounds__(kThreads) void split_sum_kernel(const float* __restrict__ partial, float* __restrict__ out,
                                                             MatmulArgs p, int64_t splits) {
    const int64_t per_batch = p.M * p.N;
    const int64_t total = p.batches * per_batch;
    for (int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; idx < total;
         idx += static_cast<int64_t>(gridDim.x) * kThreads) {
        const int64_t batch = idx / per_batch;
        const int64_t mn = idx % per_batch;
        // The partials come from memory (written by other XCDs): a batch of them is loaded before
        // the first add, one round trip per batch (C4's products split K at most 16 ways); they
        // are added in split order.
        constexpr int kBatch = 16;
        float v = 0.f;
        for (int64_t s0 = 0; s0 < splits; s0 += kBatch) {
            float x[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (s0 + u < splits) x[u] = partial[(batch * splits + s0 + u) * per_batch + mn];
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (s0 + u < splits) v += x[u];
        }
        const int64_t m = mn / p.N;
        const int64_t n = mn % p.N;
        out[batch_offset(p, batch, p.so.b, p.ho) + m * p.so.r + n * p.so.c] = plus_bias(v, p.bias, n);
    }
}

// The same where the outputs are contiguous (rows of a multiple of 4, 16-byte aligned): four outputs
// per thread and 32-bit indices. `total`, `per` (one batch's) and `n4` (a row's) are counts of four.
__global__ __launch_bounds__(kThreads) void split_sum_flat_kernel(const float* __restrict__ partial,
                                                                  float* __restrict__ out,
                                                                  const float* __restrict__ bias, int total, int per,
                                                                  int n4, int splits) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const f4* in = reinterpret_cast<const f4*>(partial);
    for (int idx = blockIdx.x * kThreads + threadIdx.x; idx < total; idx += gridDim.x * kThreads) {
        const int batch = per == total ? 0 : idx / per;
        const f4* from = in + batch * splits * per + (idx - batch * per);
        constexpr int kBatch = 8;  // in flight before the first add
        f4 v = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < splits; s0 += kBatch) {
            f4 x[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (s0 + u < splits) x[u] = from[(s0 + u) * per];
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (s0 + u < splits) v += x[u];
        }
        if (bias != nullptr) {
            const f4 bv = reinterpret_cast<const f4*>(bias)[idx % n4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = add_sep(v[e], bv[e]);
        }
        reinterpret_cast<f4*>(out)[idx] = v;
    }
}

// ---- skinny family (f32, few rows) ------------------------------------------------------------

constexpr int kSkinnyMaxM = 8;
constexpr int kSkinnyCols = 256;  // 64 lanes x 4 columns

// Rows [0, M) x 256 columns: the four waves take interleaved k, then combine in LDS in wave order. Nothing is staged,
// so that a product that is its traffic runs at memory's rate: 4096 x (1 x 64 x 1024) takes 182 us (5.9 TB/s) where
// the 64x64 tiles take 510, 65535 x (1 x 16 x 64) 107 where they take 315.
template <int MT, bool BVec>
__global__ __launch_bounds__(kThreads) void skinny_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                          float* __restrict__ out, MatmulArgs p) {
    __shared__ float red[4][MT][kSkinnyCols];
    const int lane = threadIdx.x % 64;
    const int wave = threadIdx.x / 64;
    const int64_t batch = blockIdx.y;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * kSkinnyCols + lane * 4;
    a += batch_offset(p, batch, p.sa.b, p.ha);
    b += batch_offset(p, batch, p.sb.b, p.hb);

    float total[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) total[m][c] = 0.f;

    // a sum per 64 of K, so that a long one rounds less (K = 256: 1.5e-7 of the result, 2-norm, in one sum)
    for (int64_t k0 = wave; k0 < p.K; k0 += 64) {
        const int64_t end = std::min<int64_t>(p.K, k0 + 64);
        float acc[MT][4];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[m][c] = 0.f;
        for (int64_t k = k0; k < end; k += 4) {
            float bv[4];
            if (BVec && n0 + 3 < p.N) {
                const float4 v = *reinterpret_cast<const float4*>(b + k * p.sb.r + n0);
                bv[0] = v.x;
                bv[1] = v.y;
                bv[2] = v.z;
                bv[3] = v.w;
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) bv[c] = n0 + c < p.N ? b[k * p.sb.r + (n0 + c) * p.sb.c] : 0.f;
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (m < p.M) {
                    const float av = a[m * p.sa.r + k * p.sa.c];
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[m][c] += av * bv[c];
                }
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < 4; ++c) total[m][c] += acc[m][c];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) red[wave][m][lane * 4 + c] = total[m][c];
    __syncthreads();
    for (int idx = threadIdx.x; idx < MT * kSkinnyCols; idx += kThreads) {
        const int m = idx / kSkinnyCols;
        const int col = idx % kSkinnyCols;
        const int64_t n = static_cast<int64_t>(blockIdx.x) * kSkinnyCols + col;
        if (m >= p.M || n >= p.N) continue;
        const float v = ((red[0][m][col] + red[1][m][col]) + red[2][m][col]) + red[3][m][col];
        out[batch_offset(p, batch, p.so.b, p.ho) + m * p.so.r + n * p.so.c] = plus_bias(v, p.bias, n);
    }
}

// ---- rowdot family (f32, few columns) ---------------------------------------------------------------

constexpr int kRowdotMaxN = 4;
constexpr int64_t kGridBatches = 65535;

// One wave per (batch, row), all in the grid's first dimension; lanes stride along K. 65535 x (1 x 256 x 1) takes 24 us
// here and 500 on the small tiles, 1 x 1024 x 1 3.1 and 6.7 on the pieces; 1 x 50257 x 1, a serial chain, 107 and 21.
template <bool AVec>
__global__ __launch_bounds__(kThreads) void rowdot_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                          float* __restrict__ out, MatmulArgs p) {
    const int lane = threadIdx.x % 64;
    const int64_t row_id = static_cast<int64_t>(blockIdx.x) * (kThreads / 64) + threadIdx.x / 64;
    if (row_id >= p.batches * p.M) return;
    const int64_t batch = row_id / p.M;
    const int64_t m = row_id % p.M;
    const float* arow = a + batch_offset(p, batch, p.sa.b, p.ha) + m * p.sa.r;
    const float* bb = b + batch_offset(p, batch, p.sb.b, p.hb);
    float acc[kRowdotMaxN] = {0.f, 0.f, 0.f, 0.f};
    if (AVec) {
        const int64_t vecs = p.K / 4;
        for (int64_t v = lane; v < vecs; v += 64) {
            const float4 x = *reinterpret_cast<const float4*>(arow + 4 * v);
            const int64_t k = 4 * v;
#pragma unroll
            for (int n = 0; n < kRowdotMaxN; ++n) {
                if (n < p.N) {
                    const float* bc = bb + n * p.sb.c;
                    acc[n] += x.x * bc[k * p.sb.r] + x.y * bc[(k + 1) * p.sb.r] + x.z * bc[(k + 2) * p.sb.r] +
                              x.w * bc[(k + 3) * p.sb.r];
                }
            }
        }
        for (int64_t k = vecs * 4 + lane; k < p.K; k += 64) {
#pragma unroll
            for (int n = 0; n < kRowdotMaxN; ++n)
                if (n < p.N) acc[n] += arow[k] * bb[k * p.sb.r + n * p.sb.c];
        }
    } else {
        for (int64_t k = lane; k < p.K; k += 64) {
            const float x = arow[k * p.sa.c];
#pragma unroll
            for (int n = 0; n < kRowdotMaxN; ++n)
                if (n < p.N) acc[n] += x * bb[k * p.sb.r + n * p.sb.c];
        }
    }
#pragma unroll
    for (int n = 0; n < kRowdotMaxN; ++n) {
#pragma unroll
        for (int off = 32; off > 0; off /= 2) acc[n] += __shfl_xor(acc[n], off, 64);
    }
    if (lane == 0) {
#pragma unroll
        for (int n = 0; n < kRowdotMaxN; ++n)
            if (n < p.N) out[batch_offset(p, batch, p.so.b, p.ho) + m * p.so.r + n * p.so.c] = plus_bias(acc[n], p.bias, n);
    }
}

// ---- tiled family (f64 / i64) ----------------------------------------------------------------------

constexpr int kTT = 64;  // tile edge
constexpr int kTK = 16;

template <typename T> __device__ __forceinline__ T mul_add(T acc, T x, T y) {
    if constexpr (std::is_same_v<T, int64_t>) return wrap_add(acc, wrap_mul(x, y));
    else return acc + x * y;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void tiled_kernel(const T* __restrict__ a, const T* __restrict__ b,
                                                         T* __restrict__ out, MatmulArgs p) {
    __shared__ T As[kTK][kTT + 1];
    __shared__ T Bs[kTK][kTT + 1];
    const int64_t batch = blockIdx.z;
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kTT;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * kTT;
    a += batch_offset(p, batch, p.sa.b, p.ha);
    b += batch_offset(p, batch, p.sb.b, p.hb);
    const int tr = threadIdx.x / 16;  // 0..15 -> rows tr*4 .. +3
    const int tc = threadIdx.x % 16;  // cols tc + 16*j
    T acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = T(0);
    for (int64_t k0 = 0; k0 < p.K; k0 += kTK) {
        for (int idx = threadIdx.x; idx < kTK * kTT; idx += kThreads) {
            const int kk = idx % kTK;
            const int mm = idx / kTK;
            const int64_t m = m0 + mm, k = k0 + kk;
            As[kk][mm] = (m < p.M && k < p.K) ? a[m * p.sa.r + k * p.sa.c] : T(0);
            const int nn = idx % kTT;
            const int kb = idx / kTT;
            const int64_t n = n0 + nn, k2 = k0 + kb;
            Bs[kb][nn] = (n < p.N && k2 < p.K) ? b[k2 * p.sb.r + n * p.sb.c] : T(0);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kTK; ++kk) {
            T av[4], bv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = As[kk][tr * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) bv[j] = Bs[kk][tc + 16 * j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mul_add(acc[i][j], av[i], bv[j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t m = m0 + tr * 4 + i;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t n = n0 + tc + 16 * j;
            if (n < p.N) out[batch_offset(p, batch, p.so.b, p.ho) + m * p.so.r + n * p.so.c] = plus_bias(acc[i][j], p.bias, n);
        }
    }
}

// ---- dispatch ----------------------------------------------------------------------------------

bool aligned16(const void* ptr) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0; }

// Status of the launch just issued (KD_LAUNCH_CHECK for callers that report through a pointer).
int launch_status() {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? KD_OK : ::kd::hip_fail(e, "kernel launch", __FILE__, __LINE__);
}

// ---- choosing the tiles of the pieces family ----------------------------------------------------

// One instantiation of pieces_kernel. `alone_us` is what a 32-deep K step of one workgroup takes when
// it has a CU to itself, `crowded_us` the CU's time per such step when `per_cu` of them share it (the
// throughput), `end_us` the prologue and epilogue that nothing overlaps. Measured on 2^20-2^24-output
// products with K of 256 to 50257, uniform inputs.
struct Tiling {
    int tm, tn, bk, per_cu, most_splits;
    double alone_us, crowded_us, end_us;
};
constexpr Tiling kTilings[] = {
    {256, 128, 16, 1, 64, 2.30, 2.48, 7.0},  // 8 waves of 64 x 64: the best rate (4096^3: 662 us; 128 x 128 below 690)
    {128, 128, 16, 2, 64, 1.35, 1.29, 5.0},  // two workgroups hide one another's ends (999 x 768 x 50257: 427 us; above 468)
    {128, 128, 32, 1, 64, 1.10, 1.37, 8.0},  // one workgroup per CU (2048^3: 94 us; 999 x 768 x 3072: 33)
    {128, 64, 32, 2, 64, 0.80, 0.76, 5.5},   // 1024 x 4096 x 256 in 8 splits: 21 us (128 x 128: 27)
    {64, 64, 32, 3, 64, 0.54, 0.44, 5.0},    // grids of a few hundred tiles (4096 x 256 x 256: 9.4 us; 128 x 128: 15)
    {64, 64, 16, 5, 1, 0.80, 0.52, 4.6},    // a short K over many tiles, whose ends five workgroups hide (4096 x (40 x 16 x 1024): 314 us; above 613): no splits
};
constexpr int kTilingCount = sizeof kTilings / sizeof kTilings[0];

template <bool AK, bool BKc>
void launch_pieces(int tiling, dim3 grid, const float* a, const float* b, float* out, const MatmulArgs& p, int k_split,
                   int64_t split_o) {
    hipStream_t s = stream();
    switch (tiling) {
    case 0: hipLaunchKernelGGL((pieces_kernel<AK, BKc, 256, 128, 4, 2, 16, 2>), grid, dim3(512), 0, s, a, b, out, p, k_split, split_o); break;
    case 1: hipLaunchKernelGGL((pieces_kernel<AK, BKc, 128, 128, 4, 2, 16, 4>), grid, dim3(512), 0, s, a, b, out, p, k_split, split_o); break;
    case 2: hipLaunchKernelGGL((pieces_kernel<AK, BKc, 128, 128, 4, 2, 32, 2>), grid, dim3(512), 0, s, a, b, out, p, k_split, split_o); break;
    case 3: hipLaunchKernelGGL((pieces_kernel<AK, BKc, 128, 64, 4, 2, 32, 4>), grid, dim3(512), 0, s, a, b, out, p, k_split, split_o); break;
    case 4: hipLaunchKernelGGL((pieces_kernel<AK, BKc, 64, 64, 2, 2, 32, 3>), grid, dim3(256), 0, s, a, b, out, p, k_split, split_o); break;
    default: hipLaunchKernelGGL((pieces_kernel<AK, BKc, 64, 64, 2, 2, 16, 5>), grid, dim3(256), 0, s, a, b, out, p, k_split, split_o); break;
    }
}

// A tiling, the number of K splits and their depth (a multiple of 32) for M x N x K, `batches` times.
struct Plan {
    int tiling;
    int64_t splits, k_split;
    double us;
};

// The cheapest by the times above: n workgroups per CU take steps * n * crowded (one alone its own
// time), and the ends of those that run at once overlap. Splitting K adds the sum of the partials: a
// launch and their way from memory (10 x 768 x 256: 3.9 us).
Plan plan_pieces(int64_t M, int64_t N, int64_t K, int64_t batches, int64_t most_splits = 64) {
    constexpr int kSplits[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 24, 32, 48, 64};
    const int64_t cus = compute_units();
    const double outputs = static_cast<double>(M) * static_cast<double>(N) * static_cast<double>(batches);
    Plan best{-1, 1, (K + 31) / 32 * 32, 0.0};
    for (int c = 0; c < kTilingCount; ++c) {
        const Tiling& tl = kTilings[c];
        const int64_t tiles = (M + tl.tm - 1) / tl.tm * ((N + tl.tn - 1) / tl.tn) * batches;
        const int64_t most = std::min<int64_t>(most_splits, tl.most_splits);
        int64_t last_k = 0;
        for (const int want : kSplits) {
            // at least 64 deep, at most four rounds of workgroups, and partials of at most 256 MiB
            if (want > 1 && (want > most || K < want * 64 || tiles * want > 4 * cus * tl.per_cu || want * outputs > 0x1p26)) break;
            const int64_t k_split = ((K + want - 1) / want + 31) / 32 * 32;
            if (k_split == last_k) continue;
            last_k = k_split;
            const int64_t splits = want == 1 ? 1 : (K + k_split - 1) / k_split;
            const double n = static_cast<double>((tiles * splits + cus - 1) / cus);
            const double steps = static_cast<double>(k_split / 32);
            double us = steps * (n > 1 ? std::max(tl.alone_us, n * tl.crowded_us) : tl.alone_us) +
                        tl.end_us * std::ceil(n / tl.per_cu);
            if (splits > 1) us += 2.5 + static_cast<double>(splits + 1) * outputs * 0.9e-6;
            if (best.tiling < 0 || us < best.us) best = Plan{c, splits, k_split, us};
        }
    }
    return best;
}

template <typename F> auto with_k_modes(bool ak, bool bk, F&& f) {
    if (ak) return bk ? f(std::true_type{}, std::true_type{}) : f(std::true_type{}, std::false_type{});
    return bk ? f(std::false_type{}, std::true_type{}) : f(std::false_type{}, std::false_type{});
}

// Enqueues split_sum_kernel over `p`'s outputs.
int launch_split_sum(const float* partial, float* out, const MatmulArgs& p, int64_t splits) {
    const int64_t total = p.batches * p.M * p.N;
    const bool flat = p.heads == 1 && p.so.c == 1 && p.so.r == p.N && (p.batches == 1 || p.so.b == p.M * p.N) &&
                      p.N % 4 == 0 && p.batches * splits * p.M * p.N < (int64_t{1} << 31) && aligned16(out) &&
                      (p.bias == nullptr || aligned16(p.bias));
    const int64_t items = flat ? total / 4 : total;
    const int64_t blocks = std::min<int64_t>((items + kThreads - 1) / kThreads, int64_t{compute_units()} * 16);
    if (flat)
        hipLaunchKernelGGL(split_sum_flat_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kThreads), 0, stream(), partial, out,
                           static_cast<const float*>(p.bias), static_cast<int>(total / 4), static_cast<int>(p.M * p.N / 4),
                           static_cast<int>(p.N / 4), static_cast<int>(splits));
    else
        hipLaunchKernelGGL(split_sum_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kThreads), 0, stream(), partial, out, p,
                           splits);
    return launch_status();
}

// Whether pieces_kernel addresses the operands: 32-bit sizes, and for an operand whose K is not
// contiguous offsets from its tile's corner that are not negative and fit 32 bits.
bool pieces_addressable(const MatmulArgs& p) {
    constexpr int64_t kMax = int64_t{1} << 31;
    const auto fits = [](int64_t rows, int64_t k) { return rows >= 0 && k >= 0 && rows < (kMax >> 9) && k < (kMax >> 6); };
    return p.M < kMax - 256 && p.N < kMax - 256 && p.K < kMax - 256 && p.batches <= kGridBatches &&
           (p.sa.c == 1 || fits(p.sa.r, p.sa.c)) && (p.sb.r == 1 || fits(p.sb.c, p.sb.r));
}

// Enqueues `plan` for p; split s writes split_o * s floats into `out`.
int launch_plan(const Plan& plan, const float* a, const float* b, float* out, const MatmulArgs& p, int64_t split_o) {
    const Tiling& tl = kTilings[plan.tiling];
    const int64_t tiles = (p.M + tl.tm - 1) / tl.tm * ((p.N + tl.tn - 1) / tl.tn);
    if (tiles > (int64_t{1} << 31) - 1) return fail(KD_E_INVALID, "kd_matmul: too many tiles");
    const dim3 grid(static_cast<uint32_t>(tiles), static_cast<uint32_t>(p.batches), static_cast<uint32_t>(plan.splits));
    with_k_modes(p.sa.c == 1, p.sb.r == 1, [&](auto ak, auto bk) {
        launch_pieces<decltype(ak)::value, decltype(bk)::value>(plan.tiling, grid, a, b, out, p, static_cast<int>(plan.k_split),
                                                                split_o);
    });
    return launch_status();
}

int matmul_pieces(const float* a, const float* b, float* out, const MatmulArgs& p, const Plan& plan) {
    if (plan.splits == 1) return launch_plan(plan, a, b, out, p, 0);
    Workspace ws;  // held until the sum is enqueued
    const int64_t per = p.M * p.N;
    if (int rc = workspace(ws, static_cast<size_t>(plan.splits * p.batches * per) * sizeof(float))) return rc;
    MatmulArgs partial = p;
    partial.bias = nullptr;
    partial.ho = plan.splits * per;
    partial.so = Strides3{p.heads * partial.ho, p.N, 1};
    if (int rc = launch_plan(plan, a, b, static_cast<float*>(ws.ptr), partial, per)) return rc;
    return launch_split_sum(static_cast<const float*>(ws.ptr), out, p, plan.splits);
}

// ---- choosing the family ------------------------------------------------------------------------
//
// Estimates in us beside plan_pieces', fitted to 3300 products of 1 to 40 rows or 1 to 16 columns, 1 to 65535 batches
// and K of 8 to 4096, each family on each of them (half of the estimates within 8 %, nine tenths within 30 %). The
// family that they choose took at most 1.06 times the quickest's time for nine tenths of the products.

// A launch, a chain of loads along K, and the waves (each a row of A and N columns of B).
double rowdot_us(const MatmulArgs& p, bool avec) {
    const double n = static_cast<double>(p.N), k = static_cast<double>(p.K);
    const double rows = static_cast<double>(p.batches) * static_cast<double>(p.M);
    const double steps = std::ceil(k / (avec ? 256 : 64));
    double chain = p.N == 1 ? (avec ? 0.16 : 0.13) : n * 0.09;
    if (avec && p.N > 1) chain = n * (p.sb.r == 1 ? 0.18 : 0.07 + 0.09 * std::min(rows, 4.0));  // a workgroup's waves share its loads
    const double element = avec && p.N == 1 ? 5e-7 : n * (avec && p.sb.r == 1 ? 7e-7 : 1.2e-6);
    return 2.7 + chain * steps + rows * (2.3e-4 + k * element);
}

// A launch, the chain of k, the workgroups' LDS sums and multiplications, and B's and the output's traffic.
double skinny_us(const MatmulArgs& p) {
    const double m = static_cast<double>(p.M), n = static_cast<double>(p.N), k = static_cast<double>(p.K);
    const double batches = static_cast<double>(p.batches);
    const double groups = batches * static_cast<double>((p.N + kSkinnyCols - 1) / kSkinnyCols);
    return 2.5 + k * (0.029 + 0.018 * m) + groups * (1.1e-4 * (p.M <= 1 ? 1 : p.M <= 4 ? 4 : 8) + 3.1e-5 * k * (m + 1)) +
           batches * n * (k * (p.sb.c == 1 ? 4.4e-7 : 2.2e-6) + m * 3.9e-7);
}

// Up to two tiles a CU a launch and its ends, and 0.85 us per 128 of K (16 waves of 8), 2 where a CU has two. Beyond, the
// tiles' share of a CU and their loads and stores. Small / pieces: 512^3 6.5 / 11.4 us, 256^3 4.3 / 8.3, 128 x 64 x 784
// 2.9 / 6.0, 64 x 784 x 128 with B transposed 7.5 / 9.2, 600^3 10.3 / 14.5; 300 x 2000 x 300 18.3 / 14.0, 128 x 2048 x 128
// 17.3 / 10.7, 400 x 768 x 768 14.4 / 13.2; 4096 x (32 x 128 x 32) 26.5 / 36, 1000 x (24 x 64 x 24) 5.9 / 8.5.
double small_us(const MatmulArgs& p) {
    const double gm = static_cast<double>((p.M + kSmallTile - 1) / kSmallTile), gn = static_cast<double>((p.N + kSmallTile - 1) / kSmallTile);
    const double batches = static_cast<double>(p.batches), tiles = gm * gn * batches, k = static_cast<double>(p.K);
    const double m = static_cast<double>(p.M), n = static_cast<double>(p.N), cus = compute_units();
    if (tiles <= 2 * cus) return 2.0 + static_cast<double>((p.K + 127) / 128) * (tiles <= cus ? 0.85 : 2.0);
    return 2.2 + tiles * (2.3e-3 + 2.7e-5 * k) + batches * (1.8e-7 * k * (m * gn + n * gm) + 8.4e-7 * m * n);
}

int launch_small(const float* a, const float* b, float* out, const MatmulArgs& p) {
    const dim3 grid(static_cast<uint32_t>((p.N + kSmallTile - 1) / kSmallTile), static_cast<uint32_t>((p.M + kSmallTile - 1) / kSmallTile),
                    static_cast<uint32_t>(p.batches));
    with_k_modes(p.sa.c == 1, p.sb.r == 1, [&](auto ak, auto bk) {
        hipLaunchKernelGGL((small_kernel<decltype(ak)::value, decltype(bk)::value>), grid, dim3(kSmallWaves * 64), 0, stream(), a, b,
                           out, p);
    });
    return launch_status();
}

int matmul_f32(const float* a, const float* b, float* out, MatmulArgs p) {
    enum { kRowdot, kSkinny, kSmall, kPieces, kGeneral };
    if (p.batches > kGridBatches && p.N > kRowdotMaxN) return fail(KD_E_INVALID, "kd_matmul: too many batches");
    // the batches fold into M when they share B and lie back to back in A and the output
    if (p.batches > 1 && p.heads == 1 && p.sb.b == 0 && p.sa.b == p.M * p.sa.r && p.so.b == p.M * p.so.r &&
        p.M * p.batches < (int64_t{1} << 31) - 256) {
        p.M *= p.batches;
        p.batches = 1;
    }
    const bool avec = p.sa.c == 1 && p.sa.r % 4 == 0 && p.sa.b % 4 == 0 && p.ha % 4 == 0 && aligned16(a);
    const int64_t gm = (p.M + kSmallTile - 1) / kSmallTile, gn = (p.N + kSmallTile - 1) / kSmallTile;
    const bool grid = p.batches <= kGridBatches;
    int family = kGeneral;
    double us = 0.0;
    const auto consider = [&](int f, double estimate) {
        if (family == kGeneral || estimate < us) {
            family = f;
            us = estimate;
        }
    };
    // (a launch holds fewer than 2^32 threads in its first dimension)
    if (p.N <= kRowdotMaxN && p.batches * p.M < (int64_t{1} << 26) - 4) consider(kRowdot, rowdot_us(p, avec));
    if (grid && p.M <= kSkinnyMaxM && p.N < (int64_t{1} << 31)) consider(kSkinny, skinny_us(p));
    const bool pieces = pieces_addressable(p);
    const bool fits32 = p.K * std::abs(p.sa.c) < (int64_t{1} << 31) && p.K * std::abs(p.sb.r) < (int64_t{1} << 31);
    // (what the pieces cannot take has no estimate: beyond two tiles a CU it is the general kernel's)
    if (grid && fits32 && gm <= 65535 && gn < (int64_t{1} << 22) && (pieces || gm * gn * p.batches <= 2 * int64_t{compute_units()}))
        consider(kSmall, small_us(p));
    Plan plan{};
    // Where many tiles leave the choice close the pieces' sums have fewer roundings: small tiles if a quarter quicker.
    if (family == kSmall && pieces && gm * gn * p.batches > 2 * int64_t{compute_units()}) us *= 1.25;
    if (pieces && (family == kGeneral || us >= 5.3)) {  // (no plan takes less)
        // A graph would hold on to partials in the shared workspace, which a later call may free to grow it, and
        // growing it is no call to make under capture: a captured product is not split.
        hipStreamCaptureStatus captured = hipStreamCaptureStatusNone;
        if (stream() != nullptr) KD_HIP(hipStreamIsCapturing(stream(), &captured));
        plan = plan_pieces(p.M, p.N, p.K, p.batches, captured == hipStreamCaptureStatusNone ? 64 : 1);
        consider(kPieces, plan.us);
    }
    switch (family) {
    case kRowdot: {
        const dim3 groups(static_cast<uint32_t>((p.batches * p.M + 3) / 4));
        if (avec) hipLaunchKernelGGL((rowdot_kernel<true>), groups, dim3(kThreads), 0, stream(), a, b, out, p);
        else hipLaunchKernelGGL((rowdot_kernel<false>), groups, dim3(kThreads), 0, stream(), a, b, out, p);
        return launch_status();
    }
    case kSkinny: {
        const dim3 groups(static_cast<uint32_t>((p.N + kSkinnyCols - 1) / kSkinnyCols), static_cast<uint32_t>(p.batches));
        const bool bvec = p.sb.c == 1 && p.sb.r % 4 == 0 && p.sb.b % 4 == 0 && p.hb % 4 == 0 && aligned16(b);
        const auto launch = [&](auto mt) {
            constexpr int kRows = decltype(mt)::value;
            if (bvec) hipLaunchKernelGGL((skinny_kernel<kRows, true>), groups, dim3(kThreads), 0, stream(), a, b, out, p);
            else hipLaunchKernelGGL((skinny_kernel<kRows, false>), groups, dim3(kThreads), 0, stream(), a, b, out, p);
        };
        if (p.M <= 1) launch(std::integral_constant<int, 1>{});
        else if (p.M <= 4) launch(std::integral_constant<int, 4>{});
        else launch(std::integral_constant<int, kSkinnyMaxM>{});
        return launch_status();
    }
    case kSmall: return launch_small(a, b, out, p);
    case kPieces: return matmul_pieces(a, b, out, p, plan);
    default: break;
    }
    if (!grid) return fail(KD_E_INVALID, "kd_matmul: too many batches");
    const int64_t tiles = ((p.M + kBM - 1) / kBM) * ((p.N + kBN - 1) / kBN);
    hipLaunchKernelGGL(general_f32_kernel, dim3(static_cast<uint32_t>(tiles), static_cast<uint32_t>(p.batches)), dim3(kThreads),
                       0, stream(), a, b, out, p);
    return launch_status();
}

// ---- f64 on the FP64 matrix cores ------------------------------------------------------------
//
// 64x64 output tiles, four waves each a 2x2 grid of 16x16 v_mfma_f64_16x16x4f64 accumulators;
// K advances 16 at a time through double-buffered LDS, the next stage's elements in registers
// while the current one multiplies. Any operand strides (each thread loads 4 elements of A and 4
// of B per stage, one at a time), batches with one or two stride levels, the bias epilogue; Full
// drops the bounds checks for whole tiles. Lane layout of the 16x16x4 f64 MFMA (measured with
// random operands on gfx950): A[i][k] and B[k][j] come from lane i + 16 k (j + 16 k), and
// register r of lane l holds D[l / 16 + 4 r][l % 16].
constexpr int kD = 64;
constexpr int kDK = 16;
constexpr int kDAld = kDK + 1;  // A tile [m][k]: odd stride, the 16 rows a wave reads spread over the banks
constexpr int kDBld = kD + 1;   // B tile [k][n]
typedef double v4d __attribute__((ext_vector_type(4)));

template <bool Full>
__global__ __launch_bounds__(kThreads) void mfma_f64_kernel(const double* __restrict__ a, const double* __restrict__ b,
                                                            double* __restrict__ out, MatmulArgs p) {
    __shared__ double As[2][kD * kDAld];
    __shared__ double Bs[2][kDK * kDBld];
    const int64_t tiles_m = (p.M + kD - 1) / kD;
    const int64_t tiles_n = (p.N + kD - 1) / kD;
    int64_t tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int64_t batch = blockIdx.y;
    const int64_t m0 = tm * kD;
    const int64_t n0 = tn * kD;
    a += batch_offset(p, batch, p.sa.b, p.ha);
    b += batch_offset(p, batch, p.sb.b, p.hb);
    out += batch_offset(p, batch, p.so.b, p.ho);

    const int t = threadIdx.x;
    const int lane = t % 64;
    const int wave = t / 64;
    const int wm = wave / 2;
    const int wn = wave % 2;
    const int li = lane % 16;
    const int lk = lane / 16;

    v4d acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

    double ra[4], rb[4];
    const auto fetch = [&](int64_t k0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int idx = t + kThreads * e;
            const int64_t m = m0 + idx / kDK, ka = k0 + idx % kDK;
            ra[e] = (Full || (m < p.M && ka < p.K)) ? a[m * p.sa.r + ka * p.sa.c] : 0.0;
            const int64_t kb = k0 + idx / kD, n = n0 + idx % kD;
            rb[e] = (Full || (kb < p.K && n < p.N)) ? b[kb * p.sb.r + n * p.sb.c] : 0.0;
        }
    };
    const auto stash = [&](int buf) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int idx = t + kThreads * e;
            As[buf][(idx / kDK) * kDAld + idx % kDK] = ra[e];
            Bs[buf][(idx / kD) * kDBld + idx % kD] = rb[e];
        }
    };
    fetch(0);
    stash(0);
    __syncthreads();
    const int64_t ksteps = (p.K + kDK - 1) / kDK;
    for (int64_t ks = 0; ks < ksteps; ++ks) {
        const int cur = static_cast<int>(ks & 1);
        const bool more = ks + 1 < ksteps;
        if (more) fetch((ks + 1) * kDK);
        const double* as = As[cur];
        const double* bs = Bs[cur];
#pragma unroll
        for (int kk = 0; kk < kDK; kk += 4) {
            double av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) av[i] = as[(wm * 32 + i * 16 + li) * kDAld + kk + lk];
#pragma unroll
            for (int j = 0; j < 2; ++j) bv[j] = bs[(kk + lk) * kDBld + wn * 32 + j * 16 + li];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        if (more) stash(cur ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int64_t col = n0 + wn * 32 + j * 16 + li;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = m0 + wm * 32 + i * 16 + lk + 4 * r;
                if (Full || (row < p.M && col < p.N))
                    out[row * p.so.r + col * p.so.c] = plus_bias(acc[i][j][r], p.bias, col);
            }
        }
}

int matmul_f64(const double* a, const double* b, double* out, const MatmulArgs& p) {
    if (p.batches > 65535) return fail(KD_E_INVALID, "kd_matmul: too many batches");
    const int64_t tiles = ((p.M + kD - 1) / kD) * ((p.N + kD - 1) / kD);
    if (tiles > (int64_t{1} << 31) - 1) return fail(KD_E_INVALID, "kd_matmul: too many tiles");
    const dim3 grid(static_cast<uint32_t>(tiles), static_cast<uint32_t>(p.batches));
    const bool full = p.M % kD == 0 && p.N % kD == 0 && p.K % kDK == 0;
    if (full) hipLaunchKernelGGL((mfma_f64_kernel<true>), grid, dim3(kThreads), 0, stream(), a, b, out, p);
    else hipLaunchKernelGGL((mfma_f64_kernel<false>), grid, dim3(kThreads), 0, stream(), a, b, out, p);
    KD_LAUNCH_CHECK();
    return KD_OK;
}

template <typename T> int matmul_tiled(const T* a, const T* b, T* out, const MatmulArgs& p) {
    if (p.batches > 65535) return fail(KD_E_INVALID, "kd_matmul: too many batches");
    const int64_t gm = (p.M + kTT - 1) / kTT, gn = (p.N + kTT - 1) / kTT;
    if (gm > 65535) return fail(KD_E_INVALID, "kd_matmul: too many rows");
    hipLaunchKernelGGL((tiled_kernel<T>), dim3(static_cast<uint32_t>(gn), static_cast<uint32_t>(gm), static_cast<uint32_t>(p.batches)),
                       dim3(kThreads), 0, stream(), a, b, out, p);
    KD_LAUNCH_CHECK();
    return KD_OK;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void zero_kernel(T* out, MatmulArgs p) {
    const int64_t total = p.batches * p.M * p.N;
    for (int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; idx < total;
         idx += static_cast<int64_t>(gridDim.x) * kThreads) {
        const int64_t batch = idx / (p.M * p.N);
        const int64_t m = (idx / p.N) % p.M;
        const int64_t n = idx % p.N;
        out[batch_offset(p, batch, p.so.b, p.ho) + m * p.so.r + n * p.so.c] = plus_bias(T(0), p.bias, n);
    }
}

int dispatch(int dtype, const void* a, const void* b, void* out, const MatmulArgs& p) {
    if (dtype == KD_BOOL) return fail(KD_E_UNSUPPORTED, "matmul does not support dtype bool");
    if (dtype_size(dtype) == 0) return fail(KD_E_INVALID, "kd_matmul: unknown dtype");
    if (p.batches < 0 || p.M < 0 || p.K < 0 || p.N < 0) return fail(KD_E_INVALID, "kd_matmul: negative size");
    if (p.batches == 0 || p.M == 0 || p.N == 0) return KD_OK;
    if (int rc = ensure_device()) return rc;
    if (p.K == 0) {
        // An empty inner dimension yields zeros (the reference's accumulators start at zero).
        const int64_t total = p.batches * p.M * p.N;
        const int64_t blocks = std::min<int64_t>((total + kThreads - 1) / kThreads, int64_t{compute_units()} * 16);
        const dim3 grid(static_cast<uint32_t>(blocks));
        if (dtype == KD_F32) hipLaunchKernelGGL((zero_kernel<float>), grid, dim3(kThreads), 0, stream(), static_cast<float*>(out), p);
        else if (dtype == KD_F64) hipLaunchKernelGGL((zero_kernel<double>), grid, dim3(kThreads), 0, stream(), static_cast<double*>(out), p);
        else hipLaunchKernelGGL((zero_kernel<int64_t>), grid, dim3(kThreads), 0, stream(), static_cast<int64_t*>(out), p);
        KD_LAUNCH_CHECK();
        return KD_OK;
    }
    switch (dtype) {
    case KD_F32: return matmul_f32(static_cast<const float*>(a), static_cast<const float*>(b), static_cast<float*>(out), p);
    case KD_F64: return matmul_f64(static_cast<const double*>(a), static_cast<const double*>(b), static_cast<double*>(out), p);
    default: return matmul_tiled<int64_t>(static_cast<const int64_t*>(a), static_cast<const int64_t*>(b), static_cast<int64_t*>(out), p);
    }
}

} // namespace

int matmul_split_parts(const float* a, const float* b, float* parts, int64_t M, int64_t N, int64_t K, int64_t lda,
                       int64_t ldb, int64_t splits) {
    constexpr int64_t kMax = (int64_t{1} << 31) - 256;
    if (M <= 0 || N <= 0 || K <= 0 || M >= kMax || N >= kMax || K >= kMax || lda >= kMax || ldb >= kMax || splits < 1 ||
        splits > 65535 || K % (32 * splits) != 0)
        return fail(KD_E_INVALID, "matmul_split_parts: operands outside the split-K kernel's bounds");
    if (M <= kSmallTile) {  // the small tiles, the splits as batches: their K offsets as batch strides
        MatmulArgs p;
        p.batches = splits;
        p.M = M;
        p.K = K / splits;
        p.N = N;
        p.sa = {p.K, lda, 1};
        p.sb = {p.K, 1, ldb};
        p.so = {M * N, N, 1};
        hipLaunchKernelGGL((small_kernel<true, true>),
                           dim3(static_cast<uint32_t>((N + kSmallTile - 1) / kSmallTile), 1, static_cast<uint32_t>(splits)),
                           dim3(kSmallWaves * 64), 0, stream(), a, b, parts, p);
        return launch_status();
    }
    const int64_t tiles = (M + kPartTile - 1) / kPartTile * ((N + kPartTile - 1) / kPartTile);
    const dim3 grid(static_cast<uint32_t>(tiles), static_cast<uint32_t>(splits));
    const int m = static_cast<int>(M), n = static_cast<int>(N), deep = static_cast<int>(K / splits);
    const int la = static_cast<int>(lda), lb = static_cast<int>(ldb);
    if (deep % 64 == 0) hipLaunchKernelGGL((parts_kernel<64>), grid, dim3(kThreads), 0, stream(), a, b, parts, m, n, deep, la, lb);
    else hipLaunchKernelGGL((parts_kernel<32>), grid, dim3(kThreads), 0, stream(), a, b, parts, m, n, deep, la, lb);
    return launch_status();
}

int matmul_linear_parts(const float* a, const float* b, float* parts, int64_t capacity, int64_t M, int64_t N, int64_t K,
                        int64_t* splits) {
    MatmulArgs p;
    p.batches = 1;
    p.M = M;
    p.K = K;
    p.N = N;
    p.sa = {0, K, 1};
    p.sb = {0, 1, K};
    p.so = {0, N, 1};
    if (M <= 0 || N <= 0 || K <= 0 || capacity < M * N || !pieces_addressable(p))
        return fail(KD_E_INVALID, "matmul_linear_parts: operands outside the product's bounds");
    const Plan plan = plan_pieces(M, N, K, 1, capacity / (M * N));
    const int64_t small_tiles = (M + kSmallTile - 1) / kSmallTile * ((N + kSmallTile - 1) / kSmallTile);
    if (small_tiles <= 2 * int64_t{compute_units()} && small_us(p) < plan.us) {
        *splits = 1;
        return launch_small(a, b, parts, p);
    }
    *splits = plan.splits;
    return launch_plan(plan, a, b, parts, p, M * N);
}

} // namespace kd

using namespace kd;

extern "C" int kd_matmul(int dtype, const void* a, const void* b, void* out, const kd_matmul_sizes* sizes) {
    if (sizes == nullptr) return fail(KD_E_INVALID, "kd_matmul: null sizes");
    MatmulArgs p;
    p.batches = sizes->batches;
    p.M = sizes->rows;
    p.K = sizes->inner;
    p.N = sizes->columns;
    p.sa = {p.M * p.K, p.K, 1};
    p.sb = {p.K * p.N, p.N, 1};
    p.so = {p.M * p.N, p.N, 1};
    return dispatch(dtype, a, b, out, p);
}

extern "C" int kd_matmul_strided(int dtype, const void* a, const void* b, void* out, const kd_matmul_sizes* sizes,
                                 const kd_matmul_strides* strides) {
    if (sizes == nullptr || strides == nullptr) return fail(KD_E_INVALID, "kd_matmul_strided: null argument");
    MatmulArgs p;
    p.batches = sizes->batches;
    p.M = sizes->rows;
    p.K = sizes->inner;
    p.N = sizes->columns;
    p.sa = {strides->a[0], strides->a[1], strides->a[2]};
    p.sb = {strides->b[0], strides->b[1], strides->b[2]};
    p.so = {strides->out[0], strides->out[1], strides->out[2]};
    return dispatch(dtype, a, b, out, p);
}

extern "C" int kd_matmul_strided_bias(int dtype, const void* a, const void* b, void* out, const kd_matmul_sizes* sizes,
                                      const kd_matmul_strides* strides, const void* bias) {
    if (sizes == nullptr || strides == nullptr) return fail(KD_E_INVALID, "kd_matmul_strided_bias: null argument");
    if (bias == nullptr && sizes->batches > 0 && sizes->rows > 0 && sizes->columns > 0)
        return fail(KD_E_INVALID, "kd_matmul_strided_bias: null bias");
    MatmulArgs p;
    p.batches = sizes->batches;
    p.M = sizes->rows;
    p.K = sizes->inner;
    p.N = sizes->columns;
    p.sa = {strides->a[0], strides->a[1], strides->a[2]};
    p.sb = {strides->b[0], strides->b[1], strides->b[2]};
    p.so = {strides->out[0], strides->out[1], strides->out[2]};
    p.bias = bias;
    return dispatch(dtype, a, b, out, p);
}

extern "C" int kd_matmul_strided_heads(int dtype, const void* a, const void* b, void* out, const kd_matmul_sizes* sizes,
                                       const kd_matmul_strides* strides, const kd_matmul_heads* heads) {
    if (sizes == nullptr || strides == nullptr || heads == nullptr)
        return fail(KD_E_INVALID, "kd_matmul_strided_heads: null argument");
    if (heads->heads < 1) return fail(KD_E_INVALID, "kd_matmul_strided_heads: heads must be >= 1");
    if (sizes->batches > 0 && sizes->batches % heads->heads != 0)
        return fail(KD_E_INVALID, "kd_matmul_strided_heads: batches is not a multiple of heads");
    if (sizes->batches > (int64_t{1} << 31)) return fail(KD_E_INVALID, "kd_matmul_strided_heads: too many batches");
    MatmulArgs p;
    p.batches = sizes->batches;
    p.M = sizes->rows;
    p.K = sizes->inner;
    p.N = sizes->columns;
    p.sa = {strides->a[0], strides->a[1], strides->a[2]};
    p.sb = {strides->b[0], strides->b[1], strides->b[2]};
    p.so = {strides->out[0], strides->out[1], strides->out[2]};
    if (heads->heads > 1) {
        p.heads = heads->heads;
        p.ha = heads->a;
        p.hb = heads->b;
        p.ho = heads->out;
    }
    return dispatch(dtype, a, b, out, p);
}
