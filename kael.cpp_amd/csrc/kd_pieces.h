// kd_pieces.h - an f32 value as three bf16 pieces, for products on the bf16 matrix cores.
//
// The pieces' exact sum is 2^16 times the value (8 + 8 + 8 significant bits, each piece the remainder rounded to
// nearest), so a product's sums are multiplied by kUnscale at the end. bf16 ends at 2^-133, f32 at 2^-149: unscaled, the
// pieces of a value below about 2^-110 would lose its low bits (4e-5 of it at 1e-36, 4e-3 at 1e-38). Values from 2^112
// on have an infinite piece, and their products are NaN. How the products of pieces make an f32 product, with what
// error, stands in kd_matmul.hip.
#pragma once

namespace kd {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));

constexpr float kPieceScale = 0x1p16f;
constexpr float kUnscale = 0x1p-32f;

__device__ __forceinline__ void split_pieces(const float (&x)[8], bf8& hi, bf8& mid, bf8& lo) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const f2v s{x[e] * kPieceScale, x[e + 1] * kPieceScale};
        const bf2 h = __builtin_convertvector(s, bf2);
        const f2v r{s[0] - static_cast<float>(h[0]), s[1] - static_cast<float>(h[1])};
        const bf2 m = __builtin_convertvector(r, bf2);
        const f2v q{r[0] - static_cast<float>(m[0]), r[1] - static_cast<float>(m[1])};
        const bf2 l = __builtin_convertvector(q, bf2);
        hi[e] = h[0];
        hi[e + 1] = h[1];
        mid[e] = m[0];
        mid[e + 1] = m[1];
        lo[e] = l[0];
        lo[e + 1] = l[1];
    }
}

} // namespace kd
