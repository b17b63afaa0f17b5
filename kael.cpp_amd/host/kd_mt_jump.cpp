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
// phi comes from the generator's own output: Massey's algorithm ("Shift-register synthesis and BCH
// decoding", IEEE Transactions on Information Theory 15(1), 1969) on one bit of 2 * 19937 words gives
// the shortest recurrence, and phi is prime, so every nonzero bit sequence has it whole.
#include "kd_mt_jump.h"

#include <algorithm>
#include <cstring>
#include <vector>

namespace kd {

namespace {

using Poly = std::vector<uint64_t>;  // kMtWords words, or one more for degree 19968 and up

constexpr int kShift = 156;
constexpr uint64_t kMatrixA = 0xB5026F5AA96619E9ull;
constexpr uint64_t kUpperMask = 0xFFFFFFFF80000000ull;
constexpr uint64_t kLowerMask = 0x000000007FFFFFFFull;

bool bit(const Poly& p, int k) { return (p[k / 64] >> (k % 64)) & 1; }

// Bit 0 of the words of a generator, from its second word on.
std::vector<uint8_t> output_bits(int count) {
    std::vector<uint64_t> x(kMtWords);
    x[0] = 5489;
    for (int i = 1; i < kMtWords; ++i)
        x[i] = 6364136223846793005ull * (x[i - 1] ^ (x[i - 1] >> 62)) + static_cast<uint64_t>(i);
    x.reserve(count + 1 + kMtWords);
    for (int n = 0; static_cast<int>(x.size()) < count + 1; ++n) {
        const uint64_t y = (x[n] & kUpperMask) | (x[n + 1] & kLowerMask);
        x.push_back(x[n + kShift] ^ (y >> 1) ^ ((y & 1) ? kMatrixA : 0));
    }
    std::vector<uint8_t> bits(count);
    for (int n = 0; n < count; ++n) bits[n] = x[n + 1] & 1;
    return bits;
}

// x ^= y << shift
void add_shifted(Poly& x, const Poly& y, int shift) {
    const int words = shift / 64, bits = shift % 64;
    const int n = static_cast<int>(x.size());
    if (bits == 0) {
        for (int i = n - 1; i >= words; --i) x[i] ^= y[i - words];
        return;
    }
    for (int i = n - 1; i > words; --i) x[i] ^= (y[i - words] << bits) | (y[i - words - 1] >> (64 - bits));
    if (words < n) x[words] ^= y[0] << bits;
}

// The connection polynomial 1 + c1 x + ... of `bits` and its length.
int shortest_recurrence(const std::vector<uint8_t>& bits, Poly& c) {
    const int words = kMtWords + 1;
    Poly b(words, 0), recent(words, 0);  // recent: bit i is bits[n - i]
    c.assign(words, 0);
    c[0] = b[0] = 1;
    int length = 0, gap = 1;
    for (int n = 0; n < static_cast<int>(bits.size()); ++n) {
        for (int i = words - 1; i > 0; --i) recent[i] = (recent[i] << 1) | (recent[i - 1] >> 63);
        recent[0] = (recent[0] << 1) | bits[n];
        uint64_t sum = 0;
        const int used = std::min(words, length / 64 + 1);
        for (int i = 0; i < used; ++i) sum ^= c[i] & recent[i];
        if (__builtin_parityll(sum) == 0) {
            ++gap;
        } else if (2 * length <= n) {
            const Poly old = c;
            if (gap < words * 64) add_shifted(c, b, gap);
            length = n + 1 - length;
            b = old;
            gap = 1;
            if (length > kMtDegree) return length;
        } else {
            if (gap < words * 64) add_shifted(c, b, gap);
            ++gap;
        }
    }
    return length;
}

std::vector<uint64_t> make_polynomials() {
    Poly c;
    if (shortest_recurrence(output_bits(2 * kMtDegree), c) != kMtDegree) return {};
    Poly phi(kMtWords, 0);  // phi(t) = t^19937 c(1 / t)
    for (int k = 0; k <= kMtDegree; ++k)
        if (bit(c, kMtDegree - k)) phi[k / 64] |= uint64_t{1} << (k % 64);
    // Multiples of phi by every polynomial m of degree below 8, as the remainder's correction for m's top
    // bits: row m cancels the 8 bits m above t^19937 (t^19937 m + row m = 0 modulo phi).
    Poly low = phi;  // phi without its leading term
    low[kMtDegree / 64] ^= uint64_t{1} << (kMtDegree % 64);
    constexpr int kBytes = kMtWords * 8;
    std::vector<Poly> power(8, Poly(kMtWords, 0));  // t^(19937 + i) modulo phi
    power[0] = low;
    for (int i = 1; i < 8; ++i) {
        Poly& p = power[i];
        add_shifted(p, power[i - 1], 1);
        if (bit(p, kMtDegree)) {
            p[kMtDegree / 64] ^= uint64_t{1} << (kMtDegree % 64);
            for (int w = 0; w < kMtWords; ++w) p[w] ^= low[w];
        }
    }
    std::vector<Poly> rows(256, Poly(kMtWords, 0));
    for (int m = 1; m < 256; ++m) {
        const int top = 31 - __builtin_clz(static_cast<unsigned>(m));
        for (int w = 0; w < kMtWords; ++w) rows[m][w] = rows[m ^ (1 << top)][w] ^ power[top][w];
    }
    // p := p t^8 modulo phi, kJumpBlocks * 312 / 8 times for each chain
    const auto times_t8 = [&](Poly& p) {
        // the 8 bits of p at t^19929 .. t^19936 become t^19937 .. t^19944
        const int at = kMtDegree - 8;
        const unsigned m = static_cast<unsigned>((p[at / 64] >> (at % 64)) | (at % 64 > 56 ? p[at / 64 + 1] << (64 - at % 64) : 0)) & 255u;
        uint8_t* bytes = reinterpret_cast<uint8_t*>(p.data());
        std::memmove(bytes + 1, bytes, kBytes - 1);
        bytes[0] = 0;
        p[kMtWords - 1] &= (uint64_t{1} << (kMtDegree % 64)) - 1;
        const uint64_t* row = rows[m].data();
        for (int w = 0; w < kMtWords; ++w) p[w] ^= row[w];
    };
    std::vector<uint64_t> out;
    out.reserve(static_cast<size_t>(kJumpChains - 1) * kMtWords);
    Poly p(kMtWords, 0);
    p[0] = 1;
    static_assert(kMtWords * kJumpBlocks % 8 == 0);
    for (int chain = 1; chain < kJumpChains; ++chain) {
        for (int i = 0; i < kMtWords * kJumpBlocks / 8; ++i) times_t8(p);
        // divided by t: phi(0) = 1, so an odd p becomes even by adding phi
        Poly q = p;
        if (q[0] & 1)
            for (int w = 0; w < kMtWords; ++w) q[w] ^= phi[w];
        for (int w = 0; w < kMtWords; ++w) q[w] = (q[w] >> 1) | (w + 1 < kMtWords ? q[w + 1] << 63 : 0);
        out.insert(out.end(), q.begin(), q.end());
    }
    return out;
}

} // namespace

const uint64_t* mt_jump_polynomials() {
    try {
        static const std::vector<uint64_t> polynomials = make_polynomials();  // once, by the first caller
        return polynomials.empty() ? nullptr : polynomials.data();
    } catch (...) {  // no memory: the callers draw serially
        return nullptr;
    }
}

} // namespace kd
