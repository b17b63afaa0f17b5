// kd_split_gemm.h - f32 products on the bf16 matrix cores, three bf16 pieces per operand.
#pragma once

#include "kd_internal.h"

namespace kd {
namespace split_gemm {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4a __attribute__((ext_vector_type(4), aligned(4)));  // any f32 address
typedef float v16 __attribute__((ext_vector_type(16)));

struct Operand {
    const float* base;
    int64_t ld;     // elements between consecutive rows of the contiguous dim's other index
    int64_t batch;  // elements between outer batches
    int64_t head;   // elements between inner batches (heads)
};

struct Args {
    Operand a, b;
    float* out;
    int64_t ldo, batch_o, head_o;
    int64_t split_o;  // elements between split partials in `out`
    const float* bias;
    int M, N, K;
    int k_split;      // K per split (a multiple of the K step)
    uint32_t heads;
};

// x = hi + mid + lo exactly (8 + 8 + 8 significant bits, each piece rounded to nearest). The
// remainders x - piece come from the two-term bf16 dot product, which takes the piece from its half
// of a packed pair without unpacking it.
__device__ __forceinline__ void split3(const float (&x)[8], bf8& hi, bf8& mid, bf8& lo) {
    const bf2 low = {static_cast<__bf16>(-1.f), static_cast<__bf16>(0.f)};
    const bf2 high = {static_cast<__bf16>(0.f), static_cast<__bf16>(-1.f)};
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const f2 v{x[e], x[e + 1]};
        const bf2 h = __builtin_convertvector(v, bf2);
#ifdef DOT2
        const f2 r{__builtin_amdgcn_fdot2_f32_bf16(h, low, v[0], false), __builtin_amdgcn_fdot2_f32_bf16(h, high, v[1], false)};
#else
        const f2 r{v[0] - static_cast<float>(h[0]), v[1] - static_cast<float>(h[1])};
#endif
        const bf2 m = __builtin_convertvector(r, bf2);
#ifdef DOT2
        const f2 q{__builtin_amdgcn_fdot2_f32_bf16(m, low, r[0], false), __builtin_amdgcn_fdot2_f32_bf16(m, high, r[1], false)};
#else
        const f2 q{r[0] - static_cast<float>(m[0]), r[1] - static_cast<float>(m[1])};
#endif
        const bf2 l = __builtin_convertvector(q, bf2);
        hi[e] = h[0];
        hi[e + 1] = h[1];
        mid[e] = m[0];
        mid[e + 1] = m[1];
        lo[e] = l[0];
        lo[e + 1] = l[1];
    }
}

// Rows (m of A, n of B) x BK of one operand: the 8-deep K groups of each row are 16-byte units.
template <int Rows, int BK> struct Tile {
    static constexpr int kGroups = BK / 8;
    static constexpr int kUnits = Rows * kGroups;
    static constexpr int kGroupBytes = Rows * 16 + 64;
    static constexpr int kPlane = kGroups * kGroupBytes;
    static constexpr int kBytes = 3 * kPlane;
};

template <bool KContig, int Rows, int BK> __device__ __forceinline__ void unit_of(int u, int& row, int& g) {
    if constexpr (KContig) {
        g = u % (BK / 8);
        row = u / (BK / 8);
    } else {
        row = u % Rows;
        g = u / Rows;
    }
}

template <bool KContig> __device__ __forceinline__ void load_unit(float (&x)[8], const float* p, int ld) {
    if constexpr (KContig) {
        const f4a v0 = *reinterpret_cast<const f4a*>(p);
        const f4a v1 = *reinterpret_cast<const f4a*>(p + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = v0[e];
            x[4 + e] = v1[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = p[static_cast<uint32_t>(e * ld)];
    }
}

template <bool KContig> __device__ __forceinline__ void load_unit_tail(float (&x)[8], const float* p, int ld, int left) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = e < left ? p[KContig ? e : e * ld] : 0.f;
}

__device__ __forceinline__ void tile_order(int id, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n;
    int local = id;
    if (total % 8 == 0) local = (id % 8) * (total / 8) + id / 8;
    constexpr int kGroup = 8;
    const int group_size = kGroup * tiles_n;
    const int group = local / group_size;
    const int first_m = group * kGroup;
    const int rows_in_group = min(kGroup, tiles_m - first_m);
    const int in_group = local - group * group_size;
    tm = first_m + in_group % rows_in_group;
    tn = in_group / rows_in_group;
}

// AT: A is M-contiguous; BT: B is K-contiguous.
template <bool AT, bool BT, int TM, int TN, int WM, int WN, int BK, int Occ, int Depth = 2>
__global__ __launch_bounds__(WM * WN * 64, Occ) void kernel(Args p) {
    constexpr int kThreads = WM * WN * 64;
    constexpr bool kAK = !AT, kBKc = BT;  // K-contiguous?
    using TA = Tile<TM, BK>;
    using TB = Tile<TN, BK>;
    constexpr int kUnits = TA::kUnits + TB::kUnits;
    constexpr int kPer = (kUnits + kThreads - 1) / kThreads;
    static_assert(TA::kUnits % 64 == 0 && TB::kUnits % 64 == 0);  // a wave's units are all of one operand
    constexpr int IM = TM / WM / 32, JN = TN / WN / 32;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int kStage = TA::kBytes + TB::kBytes;

    const int tiles_m = (p.M + TM - 1) / TM, tiles_n = (p.N + TN - 1) / TN;
    int tm, tn;
    tile_order(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * TM, n0 = tn * TN;
    const uint32_t outer = blockIdx.y / p.heads, head = blockIdx.y - outer * p.heads;
    const int k_begin = blockIdx.z * p.k_split;
    const int k_len = min(p.k_split, p.K - k_begin);
    const int lda = static_cast<int>(p.a.ld), ldb = static_cast<int>(p.b.ld);
    const float* a = p.a.base + outer * p.a.batch + head * p.a.head +
                     (AT ? k_begin * p.a.ld + m0 : m0 * p.a.ld + k_begin);
    const float* b = p.b.base + outer * p.b.batch + head * p.b.head +
                     (BT ? n0 * p.b.ld + k_begin : k_begin * p.b.ld + n0);
    float* out = p.out + outer * p.batch_o + head * p.head_o + blockIdx.z * p.split_o;

    const int t = threadIdx.x;
    const int lane = t % 64, wave = t / 64;
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane % 32, lh = lane / 32;

    // This thread's units: source offset (elements from the tile's corner) and LDS offset.
    uint32_t src[kPer];
    int dst[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int u = t + kThreads * i;
        int row, g;
        if (u < TA::kUnits) {
            unit_of<kAK, TM, BK>(u, row, g);
            dst[i] = g * TA::kGroupBytes + row * 16;
            const int r = min(row, p.M - 1 - m0);
            src[i] = AT ? 8u * g * lda + r : static_cast<uint32_t>(r) * lda + 8 * g;
        } else {
            unit_of<kBKc, TN, BK>(u - TA::kUnits, row, g);
            dst[i] = TA::kBytes + g * TB::kGroupBytes + row * 16;
            const int r = min(row, p.N - 1 - n0);
            src[i] = BT ? static_cast<uint32_t>(r) * ldb + 8 * g : 8u * g * ldb + r;
        }
    }
    const auto has = [&](int i) {
        if (kThreads * (i + 1) <= kUnits) return true;
        return __builtin_amdgcn_readfirstlane(t) + kThreads * i < kUnits;
    };
    const auto is_a = [&](int i) {
        if (TA::kUnits % kThreads == 0) return kThreads * i < TA::kUnits;
        return __builtin_amdgcn_readfirstlane(t) + kThreads * i < TA::kUnits;
    };
    const int64_t a_step = AT ? static_cast<int64_t>(BK) * lda : BK;
    const int64_t b_step = BT ? BK : static_cast<int64_t>(BK) * ldb;
    typedef float Regs[kPer][8];
    Regs x0, x1;
    const auto fetch = [&](Regs& x) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (!has(i)) continue;
            if (is_a(i)) load_unit<kAK>(x[i], a + src[i], lda);
            else load_unit<kBKc>(x[i], b + src[i], ldb);
        }
    };
    const auto fetch_tail = [&](Regs& x, int whole, int left) {
        const float* ta = a + whole * a_step;
        const float* tb = b + whole * b_step;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (!has(i)) continue;
            const int u = t + kThreads * i;
            int row, g;
            if (is_a(i)) {
                unit_of<kAK, TM, BK>(u, row, g);
                load_unit_tail<kAK>(x[i], ta + src[i], lda, left - 8 * g);
            } else {
                unit_of<kBKc, TN, BK>(u - TA::kUnits, row, g);
                load_unit_tail<kBKc>(x[i], tb + src[i], ldb, left - 8 * g);
            }
        }
    };
    const auto stash = [&](const Regs& x, char* stage) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            if (!has(i)) continue;
            bf8 hi, mid, lo;
            split3(x[i], hi, mid, lo);
            const int plane = is_a(i) ? TA::kPlane : TB::kPlane;
            char* d = stage + dst[i];
            *reinterpret_cast<bf8*>(d) = hi;
            *reinterpret_cast<bf8*>(d + plane) = mid;
            *reinterpret_cast<bf8*>(d + 2 * plane) = lo;
        }
    };

    v16 acc[IM][JN];
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const int a_rd = lh * TA::kGroupBytes + (wm * IM * 32 + li) * 16;
    const int b_rd = TA::kBytes + lh * TB::kGroupBytes + (wn * JN * 32 + li) * 16;
    const auto multiply = [&](const char* stage) {
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            bf8 bf[JN][3];
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    bf[j][q] = *reinterpret_cast<const bf8*>(stage + b_rd + j * 512 + q * TB::kPlane + 2 * kk * TB::kGroupBytes);
            constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int i = 0; i < IM; ++i) {
                bf8 af[3];
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    af[q] = *reinterpret_cast<const bf8*>(stage + a_rd + i * 512 + q * TA::kPlane + 2 * kk * TA::kGroupBytes);
#pragma unroll
                for (int s = 0; s < 6; ++s)
#pragma unroll
                    for (int j = 0; j < JN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kA[s]], bf[j][kB[s]], acc[i][j], 0, 0, 0);
            }
        }
    };

    const int whole = k_len / BK;
    const int tail = k_len - whole * BK;
    int ahead = whole;  // whole steps not fetched yet
    // The next whole step's elements; past the last one, that one again (unused).
    const auto next = [&](Regs& x) {
        fetch(x);
        if (--ahead > 0) {
            a += a_step;
            b += b_step;
        }
    };
    // a partial step comes first
    if (tail > 0) fetch_tail(x0, whole, tail);
    else next(x0);
    int steps = ahead;  // stages to come after the first
    if (Depth == 2 && steps > 0) next(x1);
    stash(x0, lds);
    if (steps > 1 || (Depth == 1 && steps > 0)) next(x0);
    __syncthreads();
    char* const s0 = lds;
    char* const s1 = lds + kStage;
    const auto mix = [&]() {
#ifdef SGB
        constexpr int kMfma = IM * JN * 6 * (BK / 16);
#pragma unroll
        for (int q = 0; q < kMfma; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, SGB, 0);
        }
#endif
        __syncthreads();
    };
    if constexpr (Depth == 2) {
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
    } else {
        char *cur = s0, *nxt = s1;
        for (; steps > 0; --steps) {
            multiply(cur);
            stash(x0, nxt);
            next(x0);
            mix();
            char* const swap = cur;
            cur = nxt;
            nxt = swap;
        }
        multiply(cur);
    }

    const int row0 = m0 + wm * IM * 32, col0 = n0 + wn * JN * 32;
    // Non-finite sums: an infinity or NaN among the inputs, or an overflow; the pieces of an
    // infinity are not its product's (inf - inf), so this wave's blocks are computed again in f32.
    bool odd = false;
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) odd |= !(__builtin_fabsf(acc[i][j][r]) < __builtin_inff());
    if (__any(odd)) {
        const float* fa = p.a.base + outer * p.a.batch + head * p.a.head + (AT ? k_begin * p.a.ld : k_begin);
        const float* fb = p.b.base + outer * p.b.batch + head * p.b.head + (BT ? k_begin : k_begin * p.b.ld);
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int j = 0; j < JN; ++j) {
                const int64_t m = min(row0 + i * 32 + li, p.M - 1), n = min(col0 + j * 32 + li, p.N - 1);
                const float* ra = fa + (AT ? m : m * p.a.ld);
                const float* rb = fb + (BT ? n * p.b.ld : n);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
                for (int k = lh; k - lh < k_len; k += 2) {
                    const float av = k < k_len ? ra[AT ? k * p.a.ld : k] : 0.f;
                    const float bv = k < k_len ? rb[BT ? k : k * p.b.ld] : 0.f;
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc[i][j], 0, 0, 0);
                }
            }
    }
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j) {
            const int col = col0 + j * 32 + li;
            const bool in = col < p.N;
            const float bv = p.bias != nullptr && in ? p.bias[col] : 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = row0 + i * 32 + 8 * (r / 4) + 4 * lh + (r % 4);
                if (in && row < p.M) out[row * p.ldo + col] = p.bias != nullptr ? add_sep(acc[i][j][r], bv) : acc[i][j][r];
            }
        }
}

} // namespace split_gemm
} // namespace kd
