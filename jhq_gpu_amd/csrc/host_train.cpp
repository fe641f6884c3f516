// host_train.cpp — host-side training math (see host_train.h).
#include "host_train.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <limits>
#include <random>
#include <thread>

namespace jhq {

// libstdc++ generate_canonical<float, 24>(mt19937): one draw, float(u)/2^32,
// clamped below 1.
static inline float canonical(std::mt19937& g) {
    const float s = static_cast<float>(static_cast<uint32_t>(g()));
    float r = s / 4294967296.0f;
    if (r >= 1.0f) r = std::nextafter(1.0f, 0.0f);
    return r;
}

// libstdc++ normal_distribution<float>: Marsaglia polar method, y*mult first,
// x*mult cached for the next draw.  The reference instantiates it in a
// -march=native translation unit, where x*x + y*y becomes fma(x, x, y*y).
void normal_fill(uint32_t seed, float* out, int64_t n) {
    std::mt19937 g(seed);
    int64_t i = 0;
    while (i < n) {
        float x, y, r2;
        do {
            x = static_cast<float>(static_cast<double>(2.0f * canonical(g)) - 1.0);
            y = static_cast<float>(static_cast<double>(2.0f * canonical(g)) - 1.0);
            r2 = std::fma(x, x, y * y);
        } while (static_cast<double>(r2) > 1.0 || static_cast<double>(r2) == 0.0);
        const float mult = std::sqrt(-2.0f * std::log(r2) / r2);
        out[i++] = y * mult;
        if (i < n) out[i++] = x * mult;
    }
}

float erfinv_f(float x) {
    if (x >= 1.0f) return std::numeric_limits<float>::infinity();
    if (x <= -1.0f) return -std::numeric_limits<float>::infinity();
    if (x == 0.0f) return 0.0f;
    const float sign = (x > 0.0f) ? 1.0f : -1.0f;
    const float a = std::fabs(x);
    const float kC = 0.147f;
    const float k2Pi = 2.0f / 3.14159265358979f;
    // 1 - a*a, k2Pi/kC + 0.5*ln1 and t*t - ln1/kC are contracted by the
    // reference build.
    const float ln1 = std::log(std::fma(-a, a, 1.0f));
    const float t = std::fma(0.5f, ln1, k2Pi / kC);
    float z = sign * std::sqrt(std::sqrt(std::fma(t, t, -(ln1 / kC))) - t);
    const float err = std::erf(z) - x;
    const float der = (2.0f / std::sqrt(static_cast<float>(M_PI))) * std::exp(-z * z);
    z -= err / der;
    return z;
}

std::vector<float> lloyd_max_c1d(float sigma, int K1D) {
    std::vector<float> c(K1D);
    for (int i = 0; i < K1D; i++) {
        const float q_i = (static_cast<float>(i) + 0.5f) / static_cast<float>(K1D);
        c[i] = sigma * static_cast<float>(M_SQRT2) * erfinv_f(std::fma(2.0f, q_i, -1.0f));
    }
    return c;
}

float estimate_sigma(const float* x, int64_t n, int d) {
    double sum2 = 0.0;
    const int64_t total = n * static_cast<int64_t>(d);
    for (int64_t i = 0; i < total; i++) sum2 += static_cast<double>(x[i]) * static_cast<double>(x[i]);
    return static_cast<float>(std::sqrt(sum2 / (static_cast<double>(n) * d)));
}

int nearest_sorted(const float* arr, int n, float v) {
    if (n == 1) return 0;
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (v < 0.5f * (arr[mid] + arr[mid + 1])) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

namespace {

// From here on the 1-D k-means shares its work over threads (below, starting
// them costs more than they save: 70 K values take 24 ms on one path, 32 on the other)
constexpr int64_t kManyValues = (int64_t)1 << 19;

// Float order as unsigned order.
uint32_t ord32(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The values of rank rank[0..K) (ascending) of vals[0..n).  Few values:
// nth_element on the remaining suffix for each rank.  Many: a histogram of the
// values' upper 16 bits names the bin of each rank, and only those bins' values
// are ordered.
std::vector<float> order_statistics(const float* vals, int64_t n, const std::vector<int64_t>& rank,
                                    unsigned T) {
    if (n < kManyValues) {
        std::vector<float> work(vals, vals + n), out(rank.size());
        int64_t lo = 0;
        for (size_t i = 0; i < rank.size(); i++) {
            if (rank[i] >= lo) {
                std::nth_element(work.begin() + lo, work.begin() + rank[i], work.end());
                lo = rank[i];
            }
            out[i] = work[rank[i]];
        }
        return out;
    }
    std::vector<std::vector<int64_t>> hist(T, std::vector<int64_t>(1 << 16, 0));
    parallel(T, [&](unsigned t) {
        for (int64_t i = n * t / T; i < n * (t + 1) / T; i++) hist[t][ord32(vals[i]) >> 16]++;
    });
    for (unsigned t = 1; t < T; t++)
        for (int b = 0; b < 1 << 16; b++) hist[0][b] += hist[t][b];
    const int K = static_cast<int>(rank.size());
    std::vector<int> bin(K);
    std::vector<int64_t> below(K);  // values in lower bins
    std::vector<int16_t> slot(1 << 16, -1);
    std::vector<std::vector<float>> held;
    for (int i = 0; i < K; i++) {
        int64_t sum = 0;
        int b = 0;
        while (sum + hist[0][b] <= rank[i]) sum += hist[0][b++];
        bin[i] = b;
        below[i] = sum;
        if (slot[b] < 0) {
            slot[b] = static_cast<int16_t>(held.size());
            held.emplace_back();
        }
    }
    std::vector<std::vector<std::vector<float>>> part(T, std::vector<std::vector<float>>(held.size()));
    parallel(T, [&](unsigned t) {
        for (int64_t i = n * t / T; i < n * (t + 1) / T; i++) {
            const int s = slot[ord32(vals[i]) >> 16];
            if (s >= 0) part[t][s].push_back(vals[i]);
        }
    });
    parallel(std::min<unsigned>(T, static_cast<unsigned>(held.size())), [&](unsigned t) {
        const unsigned Tb = std::min<unsigned>(T, static_cast<unsigned>(held.size()));
        for (size_t s = t; s < held.size(); s += Tb) {
            for (auto& p : part) held[s].insert(held[s].end(), p[s].begin(), p[s].end());
            std::sort(held[s].begin(), held[s].end());
        }
    });
    std::vector<float> out(K);
    for (int i = 0; i < K; i++) out[i] = held[slot[bin[i]]][static_cast<size_t>(rank[i] - below[i])];
    return out;
}

}  // namespace

// The reference sorts a full copy of the n values only to read Kr quantiles
// (cpu/codebook.cpp:13-20, reused for empty clusters at :46-49); order
// statistics are unique values, so selecting just those ranks gives the same
// codewords.  Each Lloyd iteration's cluster sums must add a cluster's values in
// index order in double.  Many values are first brought into cluster order,
// stably (each thread places its share of the values at its offsets), and then
// each cluster is one sequential sum on a thread of its own: 2.56 M values, 16
// words, 16 threads 184 -> 66 ms.
std::vector<float> train_1d_kmeans(const float* vals, int64_t n, int Kr, int max_iter,
                                   unsigned max_threads) {
    if (n <= 0 || Kr <= 0) return {};
    if (n < Kr) Kr = static_cast<int>(n);
    const float nf = static_cast<float>(n);
    unsigned T = std::min(host_threads(), std::max(max_threads, 1u));
    if (n < (int64_t)1 << 16) T = 1;
    std::vector<int64_t> qidx(Kr);
    for (int i = 0; i < Kr; i++) {
        int64_t idx = static_cast<int64_t>((static_cast<float>(i) + 0.5f) / static_cast<float>(Kr) * nf);
        qidx[i] = std::min<int64_t>(idx, n - 1);
    }
    const std::vector<float> quant = order_statistics(vals, n, qidx, T);
    std::vector<float> c(quant);
    std::vector<double> sum(Kr);
    std::vector<int64_t> cnt(Kr);
    const bool wide = Kr > 256;
    std::vector<uint8_t> a8(wide ? 0 : static_cast<size_t>(n));
    std::vector<int32_t> a32(wide ? static_cast<size_t>(n) : 0);
    const bool group = T > 1 && n >= kManyValues;
    std::vector<float> grouped(group ? static_cast<size_t>(n) : 0);
    std::vector<std::vector<int64_t>> at(T, std::vector<int64_t>(Kr));
    std::vector<float> mid(Kr > 1 ? Kr - 1 : 0);
    for (int iter = 0; iter < max_iter; iter++) {
        // nearest_sorted's thresholds; where they ascend, the word it ends at
        // is the number of thresholds that are not above the value
        bool ascending = true;
        for (int i = 0; i + 1 < Kr; i++) {
            mid[i] = 0.5f * (c[i] + c[i + 1]);
            ascending = ascending && (i == 0 ? mid[0] == mid[0] : mid[i - 1] <= mid[i]);
        }
        const bool count = ascending && Kr <= 32;
        auto assign = [&](unsigned t) {
            const int64_t i0 = n * t / T, i1 = n * (t + 1) / T;
            std::vector<int64_t>& k = at[t];
            std::fill(k.begin(), k.end(), 0);
            constexpr int64_t kBlock = 1024;
            int32_t idx[kBlock];
            for (int64_t b = i0; b < i1; b += kBlock) {
                const int m = static_cast<int>(std::min(kBlock, i1 - b));
                const float* v = vals + b;
                if (count) {
                    for (int i = 0; i < m; i++) idx[i] = 0;
                    for (int q = 0; q + 1 < Kr; q++) {
                        const float th = mid[q];
                        for (int i = 0; i < m; i++) idx[i] += !(v[i] < th);
                    }
                } else {
                    for (int i = 0; i < m; i++) idx[i] = nearest_sorted(c.data(), Kr, v[i]);
                }
                for (int i = 0; i < m; i++) {
                    if (wide) a32[b + i] = idx[i];
                    else a8[b + i] = static_cast<uint8_t>(idx[i]);
                    k[idx[i]]++;
                }
            }
        };
        auto word = [&](int64_t i) { return wide ? a32[i] : static_cast<int32_t>(a8[i]); };
        parallel(T, assign);
        for (int q = 0; q < Kr; q++) {
            cnt[q] = 0;
            for (unsigned t = 0; t < T; t++) cnt[q] += at[t][q];
        }
        if (!group) {
            std::fill(sum.begin(), sum.end(), 0.0);
            for (int64_t i = 0; i < n; i++) sum[word(i)] += vals[i];
        } else {
            std::vector<int64_t> start(Kr + 1, 0);
            for (int q = 0; q < Kr; q++) {
                start[q + 1] = start[q] + cnt[q];
                int64_t o = start[q];
                for (unsigned t = 0; t < T; t++) {
                    const int64_t k = at[t][q];
                    at[t][q] = o;
                    o += k;
                }
            }
            parallel(T, [&](unsigned t) {
                std::vector<int64_t>& o = at[t];
                for (int64_t i = n * t / T; i < n * (t + 1) / T; i++) grouped[o[word(i)]++] = vals[i];
            });
            std::atomic<int> next(0);
            parallel(std::min<unsigned>(T, Kr), [&](unsigned) {
                for (int q; (q = next++) < Kr;) {
                    double s = 0.0;
                    for (int64_t i = start[q]; i < start[q + 1]; i++) s += grouped[i];
                    sum[q] = s;
                }
            });
        }
        bool changed = false;
        for (int i = 0; i < Kr; i++) {
            const float new_c = (cnt[i] == 0) ? quant[i]
                                              : static_cast<float>(sum[i] / static_cast<double>(cnt[i]));
            if (new_c != c[i]) { c[i] = new_c; changed = true; }
        }
        std::sort(c.begin(), c.end());
        if (!changed) break;
    }
    return c;
}

std::vector<float> build_rotation(int d, int seed) {
    const int64_t n = d;
    std::vector<float> G(static_cast<size_t>(n * n));
    normal_fill(static_cast<uint32_t>(seed), G.data(), n * n);
    std::vector<double> A(G.begin(), G.end());
    std::vector<double> tau(static_cast<size_t>(n));
    // xGEQR2: column k reflector with beta = -sign(alpha) * ||A(k:n, k)||.
    for (int64_t k = 0; k < n; k++) {
        double* colk = A.data() + k * n;
        const double alpha = colk[k];
        double ss = 0.0;
        for (int64_t i = k + 1; i < n; i++) ss += colk[i] * colk[i];
        if (ss == 0.0) { tau[k] = 0.0; continue; }
        const double nrm = std::sqrt(alpha * alpha + ss);
        const double beta = (alpha >= 0.0) ? -nrm : nrm;
        tau[k] = (beta - alpha) / beta;
        const double scal = 1.0 / (alpha - beta);
        for (int64_t i = k + 1; i < n; i++) colk[i] *= scal;
        colk[k] = beta;
        for (int64_t j = k + 1; j < n; j++) {
            double* colj = A.data() + j * n;
            double w = colj[k];
            for (int64_t i = k + 1; i < n; i++) w += colk[i] * colj[i];
            w *= tau[k];
            colj[k] -= w;
            for (int64_t i = k + 1; i < n; i++) colj[i] -= w * colk[i];
        }
    }
    // xORG2R: Q = H_1 ... H_n applied to the identity, last reflector first.
    for (int64_t i = n - 1; i >= 0; i--) {
        double* coli = A.data() + i * n;
        if (i < n - 1) {
            coli[i] = 1.0;
            for (int64_t j = i + 1; j < n; j++) {
                double* colj = A.data() + j * n;
                double w = 0.0;
                for (int64_t r = i; r < n; r++) w += coli[r] * colj[r];
                w *= tau[i];
                for (int64_t r = i; r < n; r++) colj[r] -= w * coli[r];
            }
            for (int64_t r = i + 1; r < n; r++) coli[r] *= -tau[i];
        }
        coli[i] = 1.0 - tau[i];
        for (int64_t r = 0; r < i; r++) coli[r] = 0.0;
    }
    for (int64_t i = 0; i < n * n; i++) G[i] = static_cast<float>(A[i]);
    return G;
}

}  // namespace jhq
