// Host-side noise sampler shared by key generation and encryption.
//
// Discrete Gaussian of standard deviation sigma on [-12 sigma, 12 sigma]:
// weights w_0 = 1, w_k = 2 exp(-k^2 / (2 sigma^2)); thresholds
// T[k] = (uint64)(cumulative_k / total * 2^63); draw r = rng() >> 1, take the
// first k with r < T[k] (the last index if none), then a sign bit rng() & 1
// when k > 0.  The reference rounds std::normal_distribution draws
// (src/keygen.cpp:61,83), whose values are implementation-defined; this fixed
// table sampler makes keys and ciphertexts reproducible everywhere.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <vector>

namespace gf {

class GaussSampler {
public:
    explicit GaussSampler(double sigma) {
        K_ = (int)std::ceil(sigma * 12.0);
        if (K_ > 256) K_ = 256;
        std::vector<double> w(K_ + 1);
        double total = 0.0, cum = 0.0;
        for (int k = 0; k <= K_; ++k) {
            w[k] = k == 0 ? 1.0 : 2.0 * std::exp(-(double)k * (double)k / (2.0 * sigma * sigma));
            total += w[k];
        }
        T_.resize(K_ + 1);
        for (int k = 0; k <= K_; ++k) {
            cum += w[k];
            T_[k] = (uint64_t)std::ldexp(cum / total, 63);
        }
        G_.resize((size_t)1 << GUIDE_BITS);
        int k = 0;
        for (size_t b = 0; b < G_.size(); ++b) {
            while (k < K_ && ((uint64_t)b << (63 - GUIDE_BITS)) >= T_[k]) ++k;
            G_[b] = (uint16_t)k;
        }
    }
    int64_t operator()(std::mt19937_64& g) const {
        const uint64_t r = g() >> 1;
        int k = 0;
        while (k < K_ && r >= T_[k]) ++k;
        if (k == 0) return 0;
        return (g() & 1) ? -(int64_t)k : (int64_t)k;
    }

    // the index k of a 63-bit draw r: operator()'s search, started from the
    // index of r's leading bits (a few of 4096 prefixes hold a threshold, so
    // the search rarely takes a step)
    int index(uint64_t r) const {
        int k = G_[r >> (63 - GUIDE_BITS)];
        while (k < K_ && r >= T_[k]) ++k;
        return k;
    }

    // the thresholds T[0..K] (the counter sampler uses T[0..K-1])
    const std::vector<uint64_t>& table() const { return T_; }
    int K() const { return K_; }

private:
    enum { GUIDE_BITS = 12 };
    int K_ = 0;
    std::vector<uint64_t> T_;
    std::vector<uint16_t> G_;
};

// The draws of std::mt19937_64 (MT19937-64, Nishimura and Matsumoto), a block
// of 312 at a time: both loops of the recurrence and the tempering are free of
// dependences within a vector, so the compiler runs them several words at
// once (1.07 -> 0.69 ns a draw on the measuring machine's host).
class Mt64Block {
public:
    enum { N = 312, M = 156 };
    explicit Mt64Block(uint64_t seed) {
        s_[0] = seed;
        for (int i = 1; i < N; ++i) s_[i] = 6364136223846793005ull * (s_[i - 1] ^ (s_[i - 1] >> 62)) + (uint64_t)i;
    }
    void next(uint64_t* out) {
        const uint64_t UP = ~0ull << 31, LOW = ~UP, A = 0xB5026F5AA96619E9ull;
        auto mix = [&](uint64_t a, uint64_t b, uint64_t m) {
            const uint64_t y = (a & UP) | (b & LOW);
            return m ^ (y >> 1) ^ ((0 - (y & 1)) & A);
        };
        for (int i = 0; i < N - M; ++i) s_[i] = mix(s_[i], s_[i + 1], s_[i + M]);
        for (int i = N - M; i < N - 1; ++i) s_[i] = mix(s_[i], s_[i + 1], s_[i + M - N]);
        s_[N - 1] = mix(s_[N - 1], s_[0], s_[M - 1]);
        for (int i = 0; i < N; ++i) {
            uint64_t z = s_[i];
            z ^= (z >> 29) & 0x5555555555555555ull;
            z ^= (z << 17) & 0x71D67FFFEDA60000ull;
            z ^= (z << 37) & 0xFFF7EEE000000000ull;
            out[i] = z ^ (z >> 43);
        }
    }

private:
    uint64_t s_[N];
};

// the per-part draws of a switching key (src/evalkeygen.cpp:62-66): for each
// coefficient u (ternary), e0, e1 (Gaussian), parts in order (cnt = parts n
// coefficients; |e| <= 256, so any signed type of 16 bits or more holds them)
//
// The draws come from blocks and the next draw's place depends on the last
// one only through whether it took a sign: no branch on a drawn value but the
// rare steps of index(), so nothing is mispredicted (2^15 coefficients: 639 ->
// 215 us on one core of the measuring machine's host).
template <class V>
inline void sample_switch_key(size_t cnt, double sigma, uint64_t seed, V* u, V* e0, V* e1) {
    Mt64Block g(seed);
    const GaussSampler gauss(sigma);
    const uint64_t T0 = gauss.K() > 0 ? gauss.table()[0] : ~0ull;   // a draw below it has index 0 and no sign
    uint64_t buf[2 * Mt64Block::N];
    size_t at = 0, have = 0;
    auto draw = [&] {
        const uint64_t r = buf[at] >> 1;
        const int64_t k = gauss.index(r), s = -(int64_t)(buf[at + 1] & 1);
        at += 1 + (r >= T0 ? 1 : 0);
        return (k ^ s) - s;   // index 0 has no sign to take
    };
    for (size_t x = 0; x < cnt; ++x) {
        if (have - at < 5) {   // a coefficient takes at most 5 draws
            std::memmove(buf, buf + at, (have - at) * sizeof(uint64_t));
            have -= at;
            at = 0;
            g.next(buf + have);
            have += Mt64Block::N;
        }
        u[x] = (V)((int64_t)(buf[at++] % 3) - 1);
        e0[x] = (V)draw();
        e1[x] = (V)draw();
    }
}
inline void sample_switch_key(uint32_t n, uint32_t parts, double sigma, uint64_t seed, std::vector<int64_t>& u,
                              std::vector<int64_t>& e0, std::vector<int64_t>& e1) {
    const size_t cnt = (size_t)parts * n;
    u.resize(cnt);
    e0.resize(cnt);
    e1.resize(cnt);
    sample_switch_key(cnt, sigma, seed, u.data(), e0.data(), e1.data());
}

// the draws of one encryption (src/encdec.cpp:47-53): for each coefficient
// v (ternary), e0, e1 (Gaussian)
inline void sample_encrypt(uint32_t n, double sigma, uint64_t seed, std::vector<int64_t>& v,
                           std::vector<int64_t>& e0, std::vector<int64_t>& e1) {
    sample_switch_key(n, 1, sigma, seed, v, e0, e1);
}

}  // namespace gf
