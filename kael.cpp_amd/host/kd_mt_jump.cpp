// kd_mt_jump.cpp - the polynomials that jump ahead in MT19937-64's word sequence.
//
// A generator whose state transition is linear over GF(2) reaches the state n + J by the polynomial
// t^J modulo the transition's characteristic polynomial phi, evaluated at the transition (Haramoto,
// Matsumoto, Nishimura, Panneton and L'Ecuyer, "Efficient jump ahead for F2-linear random number
// generators", INFORMS Journal on Computing 20(3), 2008): s[n + J] is the sum of the s[n + k] with a
// set coefficient k. MT19937-64's state holds the upper 33 bits of its oldest word and the 311 whole
// words after it, so the sums hold word by word from the second word of the window on: hence the
// exponents one below a multiple of 312.
//
// phi in closed form (Matsumoto and Nishimura, "Mersenne twister", ACM Transactions on Modeling and
// Computer Simulation 8(1), 1998, on the characteristic polynomial): with n = 312, m = 156, w = 64, r = 31,
// X = t^n + t^m, Y = t^(n-1) + t^(m-1) and a_i bit i of the twist's matrix,
//   phi = X^(w-r) Y^r + sum over i < r of a_i X^(w-r) Y^(r-1-i) + sum over i >= r of a_i X^(w-1-i).
// It has 285 terms, the second highest 311 below t^19937, so that 256 bits above t^19937 reduce at once.
#include "kd_mt_jump.h"

#include <cstring>
#include <mutex>

namespace kd {

namespace {

constexpr int kMiddle = 156, kWordBits = 64, kLowBits = 31;
constexpr uint64_t kMatrixA = 0xB5026F5AA96619E9ull;
constexpr int kPolyWords = kMtWords + 1;
constexpr int kTop = kMtDegree / 64, kTopShift = kMtDegree % 64;  // word and bit of t^19937
constexpr int kLow = 4;                                           // words that one step reduces

struct Poly {
    uint64_t w[kPolyWords];
};

// to ^= from << shift (what leaves the polynomial is lost)
void add_shifted(Poly& to, const Poly& from, int shift) {
    const int words = shift / 64, bits = shift % 64;
    for (int i = kPolyWords - 1; i >= words; --i) {
        uint64_t x = from.w[i - words] << bits;
        if (bits != 0 && i > words) x |= from.w[i - words - 1] >> (64 - bits);
        to.w[i] ^= x;
    }
}

// p (t^high + t^low)
Poly times_binomial(const Poly& p, int high, int low) {
    Poly out{};
    add_shifted(out, p, high);
    add_shifted(out, p, low);
    return out;
}

Poly characteristic_polynomial() {
    Poly phi{}, x{};  // x: X^0, X^1, ...
    x.w[0] = 1;
    for (int i = kWordBits - 1; i >= kLowBits; --i) {
        if ((kMatrixA >> i) & 1) add_shifted(phi, x, 0);  // a_i X^(w-1-i)
        x = times_binomial(x, kMtWords, kMiddle);
    }
    for (int i = kLowBits - 1; i >= 0; --i) {  // x: X^(w-r) Y^(r-1-i)
        if ((kMatrixA >> i) & 1) add_shifted(phi, x, 0);
        x = times_binomial(x, kMtWords - 1, kMiddle - 1);
    }
    add_shifted(phi, x, 0);
    return phi;
}

// The chains' polynomials so far, and the state of their computation.
struct Jumps {
    std::mutex mutex;
    int count = 0;  // polynomials there are
    Poly phi{};
    int words[400], shifts[400];  // of phi's terms below t^19937, by their exponents modulo 64
    int terms = 0;
    uint64_t power[2 * kMtWords + kLow];  // t^(19968 count) modulo phi in its first 312 words
    uint64_t polynomials[(kJumpChains - 1) * kMtWords];
};

void start(Jumps& j) {
    j.phi = characteristic_polynomial();
    for (int bit = 0; bit < 64; ++bit)
        for (int k = bit; k < kMtDegree; k += 64)
            if ((j.phi.w[k / 64] >> bit) & 1) {
                j.words[j.terms] = k / 64;
                j.shifts[j.terms++] = bit;
            }
    std::memset(j.power, 0, sizeof j.power);
    j.power[0] = 1;
}

// power := power t^19968 modulo phi: 312 words up, then 256 bits at a time from the top down, each 256 bits m above
// t^19937 replaced by m times phi's other terms.
void next_power(Jumps& j) {
    static_assert(kJumpBlocks * kMtWords == 64 * kMtWords && kMtWords % kLow == 0);
    uint64_t* p = j.power;
    std::memcpy(p + kMtWords, p, kMtWords * sizeof *p);
    std::memset(p, 0, kMtWords * sizeof *p);
    for (int k = kMtWords / kLow - 1; k >= 0; --k) {
        uint64_t* from = p + kTop + kLow * k;
        uint64_t m[kLow];
        for (int i = 0; i < kLow; ++i) m[i] = (from[i] >> kTopShift) | (from[i + 1] << (64 - kTopShift));
        from[0] &= (uint64_t{1} << kTopShift) - 1;
        for (int i = 1; i <= kLow; ++i) from[i] = 0;
        uint64_t shifted[kLow + 1] = {};
        int bits = -1;
        for (int t = 0; t < j.terms; ++t) {
            if (bits != j.shifts[t]) {
                bits = j.shifts[t];
                const auto carry = [&](int i) { return bits == 0 ? 0 : m[i] >> (64 - bits); };
                shifted[0] = m[0] << bits;
                for (int i = 1; i < kLow; ++i) shifted[i] = (m[i] << bits) | carry(i - 1);
                shifted[kLow] = carry(kLow - 1);
            }
            uint64_t* to = p + kLow * k + j.words[t];
            for (int i = 0; i <= kLow; ++i) to[i] ^= shifted[i];
        }
    }
}

} // namespace

const uint64_t* mt_jump_polynomials(int count) {
    static Jumps j;
    std::lock_guard<std::mutex> lock(j.mutex);
    if (j.terms == 0) start(j);
    for (; j.count < count; ++j.count) {
        next_power(j);
        // divided by t: phi(0) = 1, so an odd power becomes even by adding phi
        uint64_t* out = j.polynomials + j.count * kMtWords;
        const uint64_t odd = (j.power[0] & 1) ? ~uint64_t{0} : 0;
        const auto word = [&](int w) { return w < kMtWords ? j.power[w] ^ (odd & j.phi.w[w]) : 0; };
        for (int w = 0; w < kMtWords; ++w) out[w] = (word(w) >> 1) | (word(w + 1) << 63);
    }
    return j.polynomials;
}

} // namespace kd
