// kd_random.hip - kael's bernoulli masks and dropout drawn on the device from kael's generator.
//
// Reference: kael::bernoulli (src/random.cpp:106-110) is (rand(shape, F64) < p).to(dtype), where
// rand draws one std::uniform_real_distribution<double>(0, 1) value per element from the global
// std::mt19937_64 (src/random.cpp:66-84); kael::nn::functional::dropout (src/nn/functional.cpp:32-39)
// is input * bernoulli(shape, keep, dtype) / keep, each op rounded to the element type, the scalar
// `keep` converted to it. kael draws the mask on the host and copies it over; here the draws, the
// compare and the two element ops run in one launch, and the generator state comes back advanced
// by exactly `count` draws, so the caller's later draws continue kael's stream.
//
// The state is passed as libstdc++ streams a mersenne_twister_engine (operator<<): the 312 state
// words, then the index of the next word to temper (0..312).
//
// MT19937-64 (Matsumoto and Nishimura; the C++ standard's mt19937_64 parameters). The state is
// regenerated 312 words at a time (a twist): new word k mixes old words k and k + 1 into
// y = (upper bit of old[k]) | (lower 31 bits of old[k + 1]) and is
// old[k + 156] ^ (y >> 1) ^ (y odd ? A : 0) for k < 156, and new[k - 156] ^ ... for k >= 156 (word
// 311 takes new word 0 as its second input), so a twist is two parallel phases of 156 words. A
// draw is the tempered next word x; libstdc++'s generate_canonical<double, 53> over a 64-bit engine
// uses one word and returns double(x) / 2^64 (the conversion rounded to nearest), or the largest
// double below 1 when that rounds up to 1; uniform_real_distribution(0, 1) returns it unchanged.
//
// Device layout: draw e is element e. The draws split into blocks that follow the twists: block 0
// is what is left of the current state (words pos..311), block j >= 1 the 312 words of the j-th
// twist. The twists are a serial chain: in a workgroup three waves twist from one half of an LDS buffer
// into the other while five temper, compare, load and store the elements of the current block, with one
// barrier a block (0.24 us; with all waves twisting behind two barriers 0.37, and the elements after it).
//
// Few draws (up to kSerialBlocks blocks): every workgroup runs the chain and handles the blocks j with
// j % gridDim.x == blockIdx.x. The workgroup of the last block writes the final state to a second
// buffer (others may still be reading the first).
//
// More: rounds of up to 64 chains of 64 blocks, each chain's first words reached by a jump
// (kd_mt_jump.h): one workgroup writes the round's first 65 blocks of words; the words that each other
// chain starts from are sums of about 10^4 of them, taken by 16 workgroups a chain that each add
// the words of a range of coefficients (exclusive or: any order gives the same); then a workgroup
// per chain walks its own 64 blocks. 2^20 draws: 1.26 ms on one chain, 0.13 ms so, of which the three
// kernels take 20, 50 (LDS reads: 17 MB a chain) and 39 us. At 300 blocks the two are even (0.10 ms). A process's
// first such call also computes and copies the polynomials: 1.37 ms.
#include "kd_mt_jump.h"

#include <algorithm>
#include <mutex>

#include "kd_internal.h"

namespace kd {

namespace {

constexpr int kWords = 312;
constexpr int kShift = 156;
constexpr uint64_t kMatrixA = 0xB5026F5AA96619E9ull;
constexpr uint64_t kUpperMask = 0xFFFFFFFF80000000ull;  // the top 33 bits
constexpr uint64_t kLowerMask = 0x000000007FFFFFFFull;  // the low 31 bits
constexpr int kRngThreads = 320;                         // 312 words, rounded up to whole waves
constexpr int kTwistThreads = 192;                       // the waves that twist (156 words)
constexpr int kChainThreads = kTwistThreads + kRngThreads;
constexpr int64_t kSerialBlocks = 300;
constexpr int64_t kRoundBlocks = int64_t{kJumpBlocks} * kJumpChains;
constexpr int kJumpSplits = 16;                          // workgroups that share a chain's jump
constexpr int kJumpWords = (kWords + kJumpSplits - 1) / kJumpSplits;  // coefficient words of each
static_assert(kWords == kMtWords && kJumpBlocks * kWords >= kMtDegree + 1);  // 65 blocks hold every word a jump adds

// The jump polynomials, copied here before the first launch that reads them.
__device__ uint64_t g_jump[(kJumpChains - 1) * kWords];

__host__ __device__ __forceinline__ uint64_t twist_word(uint64_t first, uint64_t second, uint64_t far) {
    const uint64_t y = (first & kUpperMask) | (second & kLowerMask);
    return far ^ (y >> 1) ^ ((y & 1) ? kMatrixA : 0);
}

__device__ __forceinline__ uint64_t temper(uint64_t x) {
    x ^= (x >> 29) & 0x5555555555555555ull;
    x ^= (x << 17) & 0x71D67FFFEDA60000ull;
    x ^= (x << 37) & 0xFFF7EEE000000000ull;
    x ^= x >> 43;
    return x;
}

// generate_canonical<double, 53>: one 64-bit word, double(x) * 2^-64, kept below 1.
__device__ __forceinline__ double canonical(uint64_t x) {
    const double u = static_cast<double>(x) * 0x1p-64;
    return u >= 1.0 ? 0x1.fffffffffffffp-1 : u;
}

template <typename T> __device__ __forceinline__ T dropped(T x, bool keep, T keep_t);
template <> __device__ __forceinline__ float dropped<float>(float x, bool keep, float keep_t) {
    return __fdiv_rn(__fmul_rn(x, keep ? 1.0f : 0.0f), keep_t);
}
template <> __device__ __forceinline__ double dropped<double>(double x, bool keep, double keep_t) {
    return __ddiv_rn(__dmul_rn(x, keep ? 1.0 : 0.0), keep_t);
}

struct RngArgs {
    void* out;
    void* mask;          // dropout: the mask as T(1) / T(0) too, or nullptr
    const void* in;      // dropout input (nullptr for a mask)
    const uint64_t* state;  // device copy: 312 words, then the position
    uint64_t* next;         // the state after the draws, same layout
    int64_t count;
    int64_t blocks;      // blocks of draws (block 0: the rest of the current state)
    int64_t first;       // draws in block 0
    double p;            // the compare threshold (keep for dropout)
};

// The next 312 words after `old`, into `nw`, by three waves: thread k < 156 makes words k and k + 156. A
// word's second half mixes the same thread's word of the first half (the last one also word 0, which its
// thread makes too), so a twist is one round of LDS reads, without a barrier inside.
__device__ __forceinline__ void twist(const uint64_t* __restrict__ old, uint64_t* __restrict__ nw, int k) {
    if (k >= kShift) return;
    const uint64_t m0 = old[k + kShift];
    const uint64_t first = twist_word(old[k], old[k + 1], m0);
    const uint64_t second = k + 1 < kShift ? old[k + kShift + 1] : twist_word(old[0], old[1], old[kShift]);
    nw[k] = first;
    nw[k + kShift] = twist_word(m0, second, first);
}

// One workgroup's walk from the words of block `first` in mt[0] to block `last`: the first three waves
// twist to the next block while the others (t = 0 .. 319) visit the current one, then all meet. Returns
// which half of `mt` holds the last block's words.
template <class Visit>
__device__ __forceinline__ int walk(uint64_t (&mt)[2][kWords], int64_t first, int64_t last, const Visit& visit) {
    int cur = 0;
    for (int64_t j = first;; ++j) {
        if (threadIdx.x >= kTwistThreads) visit(j, mt[cur]);
        else if (j < last) twist(mt[cur], mt[cur ^ 1], threadIdx.x);
        if (j >= last) return cur;
        __syncthreads();
        cur ^= 1;
    }
}

// A thread's elements of the blocks that its workgroup handles: thread t element t of each. Dropout =
// true: out = in * (u < p) / T(p) (and mask = T(u < p) when asked for). Dropout = false: out = T(u < p).
template <typename T, bool Dropout> struct Elements {
    const RngArgs& a;
    const int t;
    const T keep;
    const int64_t pos, last;
    T x = T(0), y = T(0);  // the inputs of the next two blocks (a block takes less than a load's way from memory)

    __device__ __forceinline__ int64_t start(int64_t j) const { return j == 0 ? int64_t{0} : a.first + (j - 1) * kWords; }
    __device__ __forceinline__ int64_t size(int64_t j) const {
        return j == 0 ? a.first : std::min<int64_t>(kWords, a.count - start(j));
    }
    __device__ __forceinline__ T input(int64_t j) const {
        if constexpr (Dropout) {
            if (j <= last && t < size(j)) return static_cast<const T*>(a.in)[start(j) + t];
        }
        return T(0);
    }
    // before the first block, `step` apart
    __device__ __forceinline__ void begin(int64_t j, int64_t step) {
        x = input(j);
        y = input(j + step);
    }
    // block j from its words; `next` is the block after the next, whose input is loaded meanwhile
    __device__ __forceinline__ void draw(int64_t j, const uint64_t* words, int64_t next) {
        const T mine = x;
        x = y;
        y = input(next);
        if (t >= size(j)) return;
        const int64_t e = start(j) + t;
        const bool hit = canonical(temper(words[(j == 0 ? pos : 0) + t])) < a.p;
        if constexpr (Dropout) {
            static_cast<T*>(a.out)[e] = dropped<T>(mine, hit, keep);
            if (a.mask != nullptr) static_cast<T*>(a.mask)[e] = hit ? T(1) : T(0);
        } else {
            static_cast<T*>(a.out)[e] = hit ? T(1) : T(0);
        }
    }
};

// The state after the last draw: the current words and the index past the last one used.
__device__ __forceinline__ void store_state(const RngArgs& a, const uint64_t (&words)[kWords], int64_t pos, int t) {
    const int64_t last = a.blocks - 1;
    if (t < kWords) a.next[t] = words[t];
    if (t == 0)
        a.next[kWords] = static_cast<uint64_t>(last == 0 ? pos + a.first
                                                         : std::min<int64_t>(kWords, a.count - (a.first + (last - 1) * kWords)));
}

template <typename T, bool Dropout>
__global__ __launch_bounds__(kChainThreads) void mt_kernel(RngArgs a, T keep_t) {
    __shared__ uint64_t mt[2][kWords];
    const int t = static_cast<int>(threadIdx.x) - kTwistThreads;  // below 0: a twisting wave
    if (t >= 0 && t < kWords) mt[0][t] = a.state[t];
    const int64_t pos = static_cast<int64_t>(a.state[kWords]);
    const int64_t G = gridDim.x, mine = blockIdx.x, last = a.blocks - 1;
    if (mine > last) return;
    const int64_t own_last = last - (last - mine) % G;  // this workgroup's last block
    Elements<T, Dropout> elements{a, t, keep_t, pos, own_last};
    if (t >= 0) elements.begin(mine, G);
    int64_t next = mine;
    __syncthreads();
    const int cur = walk(mt, 0, own_last, [&](int64_t j, const uint64_t* words) {
        if (j != next) return;
        next += G;
        elements.draw(j, words, j + 2 * G);
    });
    if (own_last == last && t >= 0) store_state(a, mt[cur], pos, t);
}

// The words of a round's first 65 blocks, from its first block's in a.state (first round) or the block
// before it in `before`, and zeros for the chains' starts.
__global__ __launch_bounds__(kChainThreads) void round_words_kernel(RngArgs a, const uint64_t* before, uint64_t* words,
                                                                    uint64_t* starts, int chains) {
    __shared__ uint64_t mt[2][kWords];
    const int t = static_cast<int>(threadIdx.x) - kTwistThreads;
    for (int i = threadIdx.x; i < (chains - 1) * kWords; i += kChainThreads) starts[i] = 0;
    const int skip = before != nullptr ? 1 : 0;
    if (t >= 0 && t < kWords) mt[0][t] = skip ? before[t] : a.state[t];
    __syncthreads();
    walk(mt, 0, kJumpBlocks + skip, [&](int64_t j, const uint64_t* block) {
        if (j >= skip && t < kWords) words[(j - skip) * kWords + t] = block[t];
    });
}

// Workgroup (s, c): the sum of the words that coefficient words s * kJumpWords .. of chain c + 1's
// polynomial select, added to the chain's start.
__global__ __launch_bounds__(kRngThreads) void jump_kernel(const uint64_t* words, uint64_t* starts) {
    constexpr int kSpan = kJumpWords * 64 + kWords;
    __shared__ uint64_t w[kSpan];
    const int t = threadIdx.x;
    const int first = blockIdx.x * kJumpWords;
    // coefficient k selects words k + 1 .. k + 312, all within the 65 blocks; past them no coefficient is set
    for (int i = t; i < kSpan; i += kRngThreads) {
        const int at = first * 64 + 1 + i;
        w[i] = at < (kJumpBlocks + 1) * kWords ? words[at] : 0;
    }
    __syncthreads();
    const uint64_t* p = g_jump + blockIdx.y * kWords;
    uint64_t sum = 0;
    const int mine = t < kWords ? t : 0;
    for (int q = 0; q < kJumpWords && first + q < kWords; ++q) {
        const uint64_t coefficients = p[first + q];  // the same for every lane: scalar, as are its bit numbers
        uint64_t bits = (uint64_t{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(coefficients >> 32)))} << 32) |
                        static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(coefficients)));
        const uint64_t* from = w + q * 64 + mine;
        const auto lowest = [&]() {
            const int k = __ffsll(static_cast<unsigned long long>(bits)) - 1;
            bits &= bits - 1;
            return k;
        };
        for (int n = __popcll(bits) / 8; n > 0; --n) {  // eight reads in flight
            uint64_t x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = from[lowest()];
#pragma unroll
            for (int i = 0; i < 8; ++i) sum ^= x[i];
        }
        while (bits != 0) sum ^= from[lowest()];
    }
    if (t < kWords)
        atomicXor(reinterpret_cast<unsigned long long*>(starts + blockIdx.y * kWords + t), static_cast<unsigned long long>(sum));
}

// Chain blockIdx.x of the round that starts at block `round`: its own blocks, and the last chain's last
// words for the next round.
template <typename T, bool Dropout>
__global__ __launch_bounds__(kChainThreads) void chain_kernel(RngArgs a, T keep_t, int64_t round, const uint64_t* words,
                                                              const uint64_t* starts, uint64_t* after) {
    __shared__ uint64_t mt[2][kWords];
    const int t = static_cast<int>(threadIdx.x) - kTwistThreads;
    const int64_t chain = blockIdx.x;
    if (t >= 0 && t < kWords) mt[0][t] = chain == 0 ? words[t] : starts[(chain - 1) * kWords + t];
    const int64_t pos = static_cast<int64_t>(a.state[kWords]);
    const int64_t first = round + chain * kJumpBlocks, last = std::min<int64_t>(a.blocks, first + kJumpBlocks) - 1;
    Elements<T, Dropout> elements{a, t, keep_t, pos, last};
    if (t >= 0) elements.begin(first, 1);
    __syncthreads();
    const int cur = walk(mt, first, last, [&](int64_t j, const uint64_t* block) { elements.draw(j, block, j + 2); });
    if (t < 0) return;
    if (last == a.blocks - 1) store_state(a, mt[cur], pos, t);
    else if (chain == kJumpChains - 1 && t < kWords) after[t] = mt[cur][t];
}

// At least `count` polynomials on the device (the backend has one device a process): each computed and copied once, by
// the first call that draws as many chains (kd_dropout and kd_bernoulli block).
int ensure_jump(int count) {
    static std::mutex mutex;
    static int ready = 0;
    std::lock_guard<std::mutex> lock(mutex);
    if (ready >= count) return KD_OK;
    constexpr size_t kBytes = kWords * sizeof(uint64_t);
    const uint64_t* polynomials = mt_jump_polynomials(count);
    while (ready < count) {  // 10 KB at a time: a process's first copy of more than 16 KB takes 5 to 10 ms
        const int n = std::min(count - ready, 4);
        KD_HIP(hipMemcpyToSymbol(HIP_SYMBOL(g_jump), polynomials + ready * kWords, n * kBytes, ready * kBytes, hipMemcpyHostToDevice));
        ready += n;
    }
    return KD_OK;
}

template <typename T, bool Dropout>
int run_rng(void* out, void* mask, const void* in, int64_t count, double p, uint64_t* host_state) {
    const int64_t pos = static_cast<int64_t>(host_state[kWords]);
    RngArgs a{};
    a.out = out;
    a.mask = mask;
    a.in = in;
    a.count = count;
    a.first = std::min<int64_t>(kWords - pos, count);
    a.blocks = 1 + (count - a.first + kWords - 1) / kWords;
    a.p = p;
    const bool rounds = a.blocks > kSerialBlocks;
    if (rounds)
        if (int rc = ensure_jump(static_cast<int>((std::min(a.blocks, kRoundBlocks) + kJumpBlocks - 1) / kJumpBlocks) - 1)) return rc;
    // the state, the state after, then (for rounds) a round's words, its chains' starts, and its last words
    constexpr int64_t kRoundWords = int64_t{kJumpBlocks + 1} * kWords;
    const int64_t words = 2 * (kWords + 1) + (rounds ? kRoundWords + int64_t{kJumpChains} * kWords : 0);
    Workspace lease;
    if (int rc = workspace(lease, static_cast<size_t>(words) * sizeof(uint64_t))) return rc;
    uint64_t* dev_state = static_cast<uint64_t*>(lease.ptr);
    a.state = dev_state;
    a.next = dev_state + kWords + 1;
    hipStream_t s = stream();
    KD_HIP(hipMemcpyAsync(dev_state, host_state, (kWords + 1) * sizeof(uint64_t), hipMemcpyHostToDevice, s));
    if (rounds) {
        uint64_t* round_words = dev_state + 2 * (kWords + 1);
        uint64_t* starts = round_words + kRoundWords;
        uint64_t* after = starts + (kJumpChains - 1) * kWords;
        for (int64_t round = 0; round < a.blocks; round += kRoundBlocks) {
            const int64_t left = std::min<int64_t>(kRoundBlocks, a.blocks - round);
            const int chains = static_cast<int>((left + kJumpBlocks - 1) / kJumpBlocks);
            hipLaunchKernelGGL(round_words_kernel, dim3(1), dim3(kChainThreads), 0, s, a, round == 0 ? nullptr : after,
                               round_words, starts, chains);
            if (chains > 1)
                hipLaunchKernelGGL(jump_kernel, dim3(kJumpSplits, static_cast<uint32_t>(chains - 1)), dim3(kRngThreads), 0, s,
                                   round_words, starts);
            hipLaunchKernelGGL((chain_kernel<T, Dropout>), dim3(static_cast<uint32_t>(chains)), dim3(kChainThreads), 0, s, a,
                               static_cast<T>(p), round, round_words, starts, after);
        }
    } else {
        // Enough workgroups that each handles a few blocks, at most two per CU.
        const int64_t grid = std::max<int64_t>(1, std::min<int64_t>(a.blocks, 2 * int64_t{compute_units()}));
        hipLaunchKernelGGL((mt_kernel<T, Dropout>), dim3(static_cast<uint32_t>(grid)), dim3(kChainThreads), 0, s, a,
                           static_cast<T>(p));
    }
    KD_LAUNCH_CHECK();
    KD_HIP(hipMemcpyAsync(host_state, a.next, (kWords + 1) * sizeof(uint64_t), hipMemcpyDeviceToHost, s));
    KD_HIP(hipStreamSynchronize(s));
    return KD_OK;
}

int check_state(const uint64_t* state, const char* what) {
    if (state == nullptr) return fail(KD_E_INVALID, std::string(what) + ": null generator state");
    if (state[kWords] > kWords)
        return fail(KD_E_INVALID, std::string(what) + ": generator position " + std::to_string(state[kWords]) +
                                      " outside [0, 312]");
    return KD_OK;
}

} // namespace

} // namespace kd

using namespace kd;

extern "C" void kd_mt19937_64_seed(uint64_t* state, uint64_t seed) {
    // std::mt19937_64(seed): x0 = seed, x_i = f * (x_{i-1} ^ (x_{i-1} >> 62)) + i, position 312 (the
    // first draw twists).
    state[0] = seed;
    for (int i = 1; i < kWords; ++i)
        state[i] = 6364136223846793005ull * (state[i - 1] ^ (state[i - 1] >> 62)) + static_cast<uint64_t>(i);
    state[kWords] = kWords;
}

extern "C" int kd_bernoulli(int dtype, void* out, int64_t count, double probability, uint64_t* state) {
    if (count < 0) return fail(KD_E_INVALID, "kd_bernoulli: negative count");
    if (!(probability >= 0.0 && probability <= 1.0))
        return fail(KD_E_INVALID, "kd_bernoulli: probability must be in [0, 1]");
    if (dtype_size(dtype) == 0) return fail(KD_E_INVALID, "kd_bernoulli: unknown dtype");
    if (int rc = check_state(state, "kd_bernoulli")) return rc;
    if (count == 0) return KD_OK;
    if (out == nullptr) return fail(KD_E_INVALID, "kd_bernoulli: null output");
    if (int rc = ensure_device()) return rc;
    switch (dtype) {
    case KD_F32: return run_rng<float, false>(out, nullptr, nullptr, count, probability, state);
    case KD_F64: return run_rng<double, false>(out, nullptr, nullptr, count, probability, state);
    case KD_I64: return run_rng<int64_t, false>(out, nullptr, nullptr, count, probability, state);
    default: return run_rng<uint8_t, false>(out, nullptr, nullptr, count, probability, state);
    }
}

extern "C" int kd_dropout(int dtype, void* out, void* mask, const void* in, int64_t count, double keep,
                          uint64_t* state) {
    if (count < 0) return fail(KD_E_INVALID, "kd_dropout: negative count");
    if (!(keep > 0.0 && keep <= 1.0)) return fail(KD_E_INVALID, "kd_dropout: keep probability must be in (0, 1]");
    if (dtype != KD_F32 && dtype != KD_F64) return fail(KD_E_INVALID, "kd_dropout: dtype must be f32 or f64");
    if (int rc = check_state(state, "kd_dropout")) return rc;
    if (count == 0) return KD_OK;
    if (out == nullptr || in == nullptr) return fail(KD_E_INVALID, "kd_dropout: null operand");
    if (int rc = ensure_device()) return rc;
    return dtype == KD_F32 ? run_rng<float, true>(out, mask, in, count, keep, state)
                           : run_rng<double, true>(out, mask, in, count, keep, state);
}
