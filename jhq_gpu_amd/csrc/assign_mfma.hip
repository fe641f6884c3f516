// assign_mfma.hip — IVF assignment on bf16 MFMA with an exact re-check
// (v14/jhq_gpu_index.cu:23-40,367-393: argmin over lists of
// ||c||^2 - 2 <y, c>, ties to the lowest list).
//
// The assignment must equal the fixed-order one (gemm_nt_argmin: each dot an
// fmaf chain in k order, score fmaf(-2, dot, norm), ties to the lowest list)
// bit for bit.  A first pass computes every score on MFMA and keeps per row
// the smallest score s1 (list c1) and the second smallest s2.  The pass
// splits each float into two bf16 (hi = bf16(x), lo = bf16(x - hi), so
// |x - hi - lo| <= 2^-16 |x|) and sums hi*hi + hi*lo + lo*hi with three
// bf16 MFMAs per 32 k (the products are exact in fp32).  Against the
// fixed-order dot F, the first pass's dot A differs by at most
//   e_dot = (2u * 1.02 * 33 * 3 * min(dp/32, 4) + 1.02 u * chunks + 3.01 * 2^-16
//            + (d + 4) u) ||y|| Cmax
// (u = 2^-24, dp = d rounded up to 32).  The MFMAs accumulate over chunks of 4
// steps (128 k) from zero, at most 33 roundings of at most 2u per MFMA over the
// three product sums, each relative to the chunk's own ||y_j|| ||c_j||, which
// add up to at most ||y|| ||c|| over the chunks; one rounding per chunk then
// adds the chunk to the dot.  (One accumulator over all of k takes 33 * 3 *
// dp/32 roundings at the full ||y|| ||c||: three times the bound at d = 1024,
// and with it the near ties below.)  The split's dropped terms are
// hi*E + e*H + r*R <= 3.01 * 2^-16 |y_k c_k|; (d + 4) u is the fixed-order chain's
// own rounding.  The scores then differ by at most 2 e_dot plus one rounding
// each; with a factor 2 of headroom and a term for values the MFMA may flush
// as subnormals,
//   E = 2 (2 e_dot + 2u Nmax + 4u ||y|| Cmax) + 6d (2^-126 (||y|| + Cmax) + 2^-149)
// (Cmax = max ||c||, Nmax = max ||c||^2).  If s2 - s1 > 2E, list c1 is the
// unique fixed-order argmin.  For the other rows (near and exact ties) the
// fixed-order argmin has an MFMA score of at most s1 + 2E: a second MFMA pass
// over those rows alone lists the lists at or below that (two or three as a
// rule), and only their scores are formed in the fixed order.  Rows with more
// than kCand such lists, or with a non-finite score, take the fixed-order
// argmin over every list (gemm_nt_argmin_rows).
//
// Measured (bf16 products counted three times): 65536 x 128 rows against 65536
// lists 9458 -> 2507 us (scores 2334 us, 1.4 PFLOP/s; re-check 102 us), 65536 x
// 1024 against 4096 4302 -> 2159 us (1623 us, 1.0 PFLOP/s; 335 us), 2000 x 768
// against 1024 136 -> 97 us, 1000 x 100 against 1000 76 -> 58 us.  Before, all
// scores of the near ties were formed in the fixed order on the vector ALU
// (1914 and 2062 us of the first two).
#include "kernels.h"

#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstdint>

namespace jhq {

typedef __bf16 bf16x8_a __attribute__((ext_vector_type(8)));
typedef float v4f_a __attribute__((ext_vector_type(4)));

// k per bf16 MFMA
constexpr int kTopBK = 32;
// k steps accumulated in one chunk
constexpr int kChunk = 4;
// candidate lists kept per re-checked row
constexpr int kCand = 16;

__host__ __device__ constexpr int top2_kpad(int d) { return (d + kTopBK - 1) / kTopBK * kTopBK; }

// float -> bf16 bits, round to nearest even (NaN stays NaN)
__device__ __forceinline__ uint32_t bf16_rne(float x) {
    const uint32_t b = __float_as_uint(x);
    if ((b & 0x7fffffffu) > 0x7f800000u) return (b >> 16) | 0x40u;
    return (b + 0x7fffu + ((b >> 16) & 1u)) >> 16;
}

// Operands in fragment order: rows (lists) in groups of 16, and per group and
// k step of 32 one 1 KB block of hi = bf16(x) and one of lo = bf16(x - hi),
// 16 bytes per lane as the MFMA takes them: lane r + 16 g holds row r's k =
// 8 g .. 8 g + 7 of the step.  Every later load, into registers or LDS, is a
// whole contiguous block, and an LDS read of a fragment is lane-linear.
__device__ __forceinline__ int64_t frag_block(int64_t group, int ks, int hl, int KS) {
    return ((group * KS + ks) * 2 + hl) * 64;  // in 16-byte units
}

// One workgroup per group of 16 rows of Y, then of the lists (its waves take
// every fourth k step): the split operands, ||y|| (slightly rounded up) and the
// padded norms (+inf past nlist, so that a padding list is never the best); the
// last workgroup takes Nmax = max ||c||^2 and zeroes the counters.  Rows past n
// and lists past nlist are zero.  Bound by the copy: 65536 x 1024 moves 537 MB.
__global__ void __launch_bounds__(256)
split_kernel(const float* __restrict__ Y, int64_t n, const float* __restrict__ Cm, int nlist, int d,
             int KS, int64_t ygroups, uint4* __restrict__ Yf, uint4* __restrict__ Cf,
             float* __restrict__ ny, const float* __restrict__ norms, float* __restrict__ normsp,
             float* __restrict__ nmax, int32_t* __restrict__ cnt) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ float red[4];
        float m = 0.0f;
        for (int c0 = 0; c0 < nlist; c0 += 256 * 16) {
            float v[16];
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = norms[min(c0 + i * 256 + tid, nlist - 1)];
#pragma unroll
            for (int i = 0; i < 16; i++) m = fmaxf(m, v[i]);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
        if (lane == 0) red[wv] = m;
        __syncthreads();
        if (tid == 0) nmax[0] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        if (tid < 4) cnt[tid] = 0;
        return;
    }
    __shared__ double part[4][16];
    const int64_t u = blockIdx.x;
    const bool isy = u < ygroups;
    const int64_t group = isy ? u : u - ygroups;
    const int r = lane & 15, g = lane >> 4;
    const int64_t row = group * 16 + r, rows = isy ? n : nlist;
    const float* x = (isy ? Y : Cm) + (row < rows ? row : rows - 1) * d;
    uint4* out = isy ? Yf : Cf;
    double ss = 0.0;
#pragma unroll 2
    for (int ks = wv; ks < KS; ks += 4) {
        const int k = ks * kTopBK + 8 * g;
        // d a multiple of 4: four values are inside or past the end together
        float4 a = *(const float4*)(x + min(k, d - 4)), b = *(const float4*)(x + min(k + 4, d - 4));
        if (row >= rows || k >= d) a = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row >= rows || k + 4 >= d) b = make_float4(0.f, 0.f, 0.f, 0.f);
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t h[8], l[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            h[i] = bf16_rne(v[i]);
            l[i] = bf16_rne(v[i] - __uint_as_float(h[i] << 16));
            ss += (double)v[i] * (double)v[i];
        }
        out[frag_block(group, ks, 0, KS) + lane] =
            make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                       h[6] | (h[7] << 16));
        out[frag_block(group, ks, 1, KS) + lane] =
            make_uint4(l[0] | (l[1] << 16), l[2] | (l[3] << 16), l[4] | (l[5] << 16),
                       l[6] | (l[7] << 16));
    }
    if (!isy) {
        if (tid < 16) normsp[row] = row < nlist ? norms[row] : INFINITY;
        return;
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) part[wv][r] = ss;
    __syncthreads();
    if (tid < 16 && row < n)
        ny[row] = (float)(sqrt(part[0][r] + part[1][r] + part[2][r] + part[3][r]) *
                          (1.0 + 8.0 / 16777216.0));
}

// 16 bytes per lane from global memory straight to LDS (lane l at lds + 16 l)
__device__ __forceinline__ void load_block_lds(const uint4* src, uint4* lds, int lane) {
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(src + lane),
        (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// What a row of a score pass is compared with, and where results go: TOP2
// keeps each row's best, its list and the second best; COLLECT lists the lists
// whose score is not above the row's bound.
struct Top2Out {
    int32_t* best;  // [row][slots]
    float *s1, *s2;
    int slots, slot;
};
struct CollectIO {
    const int32_t* rows;   // re-checked rows, *count of them
    const int32_t* count;
    const float* bound;    // per re-checked row
    int32_t* ncand;        // per re-checked row, zeroed
    int32_t* cand;         // [row slot][kCand]
    int32_t* ovf;          // rows with more candidates
    unsigned long long* ovf_keys;
    int32_t* novf;
};

__device__ __forceinline__ void push_candidate(const CollectIO& io, int64_t slot, int col) {
    const int at = atomicAdd(&io.ncand[slot], 1);
    if (at < kCand) {
        io.cand[slot * kCand + at] = col;
    } else if (at == kCand) {
        const int o = atomicAdd(io.novf, 1);
        io.ovf[o] = io.rows[slot];
        io.ovf_keys[o] = ~0ull;
    }
}

// The 16 RT rows of a wave in TOP2: lane (r, g) keeps rows 16 i + 4 g + j over
// its columns (r of every group of 16).  A NaN score is never the best, as in
// the fixed order, where its key is above every number's; s becomes b then
// (v_med3 of a NaN is the smaller of the others), so that the row is
// re-checked unless a score smaller by more than the bound follows.
template <int RT>
struct Top2State {
    float b[RT][4], s[RT][4];
    int c[RT][4];  // column group of b
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                b[i][j] = INFINITY;
                s[i][j] = INFINITY;
                c[i][j] = 0x7fffffff / 16;
            }
    }
    __device__ __forceinline__ void update(int i, const v4f_a& acc, float nc, int grp) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float v = fmaf(-2.0f, acc[j], nc);
            const bool less = v < b[i][j];
            s[i][j] = __builtin_amdgcn_fmed3f(b[i][j], s[i][j], v);
            c[i][j] = less ? grp : c[i][j];
            b[i][j] = less ? v : b[i][j];
        }
    }
    // The best over the 16 lanes r (their rows are the same), 16 (or 8) rows at a
    // time: each round a lane keeps half of its rows and hands the others to its
    // partner, so 15 exchanges do for 16 rows; one lane per row stores.
    __device__ __forceinline__ void store(int r, int g, int64_t row0, int64_t n, const Top2Out& o) {
        constexpr int H = RT < 4 ? RT : 4, Q = 4 * H;  // rows of a block: 8 or 16
#pragma unroll
        for (int i0 = 0; i0 < RT; i0 += H) {
            float bv[Q], sv[Q];
            int bc[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                bv[q] = b[i0 + q / 4][q % 4];
                sv[q] = s[i0 + q / 4][q % 4];
                bc[q] = c[i0 + q / 4][q % 4] * 16 + r;
            }
            auto take = [&](int q, float ob, float os, int oc) {
                const bool mine = (bv[q] < ob) | ((bv[q] == ob) & (bc[q] < oc));
                const float lose = mine ? ob : bv[q], s2 = mine ? sv[q] : os;
                sv[q] = fminf(s2, lose);
                bv[q] = mine ? bv[q] : ob;
                bc[q] = mine ? bc[q] : oc;
            };
#pragma unroll
            for (int h = Q / 2, bit = 8; h >= 1; h /= 2, bit /= 2) {
                const bool up = (r & bit) != 0;
#pragma unroll
                for (int q = 0; q < h; q++) {
                    const float gb = up ? bv[q] : bv[q + h], gs = up ? sv[q] : sv[q + h];
                    const int gc = up ? bc[q] : bc[q + h];
                    bv[q] = up ? bv[q + h] : bv[q];
                    sv[q] = up ? sv[q + h] : sv[q];
                    bc[q] = up ? bc[q + h] : bc[q];
                    take(q, __shfl_xor(gb, bit), __shfl_xor(gs, bit), __shfl_xor(gc, bit));
                }
            }
            if (Q == 8) take(0, __shfl_xor(bv[0], 1), __shfl_xor(sv[0], 1), __shfl_xor(bc[0], 1));
            const int q = Q == 8 ? r >> 1 : r;
            const int64_t row = row0 + 16 * (i0 + q / 4) + 4 * g + q % 4;
            if ((Q == 16 || !(r & 1)) && row < n) {
                const int64_t at = row * o.slots + o.slot;
                o.best[at] = bc[0];
                o.s1[at] = bv[0];
                o.s2[at] = sv[0];
            }
        }
    }
};

// The three product sums of one k step for RT row groups against one column
// group (ah, al [RT], bh, bl).
template <int RT>
__device__ __forceinline__ void mfma3(const bf16x8_a (&ah)[RT], const bf16x8_a (&al)[RT],
                                      const bf16x8_a& bh, const bf16x8_a& bl, v4f_a (&acc)[RT]) {
#pragma unroll
    for (int i = 0; i < RT; i++)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh, acc[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < RT; i++)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl, acc[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < RT; i++)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh, acc[i], 0, 0, 0);
}

// Scores of short vectors (KS k steps of 32, KS <= 8).  A wave keeps its 16 RT
// rows' operands in registers for the whole walk over the lists (8 RT KS of
// them), so only the lists move: in tiles of 16 NG, double-buffered in LDS by
// direct loads, read by all 4 waves.  Restaging the rows with every list tile,
// as the long-vector kernel does, made 65536 x 128 rows against 65536 lists
// wait for the operands (34 GB beyond L2, 7320 us); with two workgroups per
// CU one wave's score updates run beside the other's MFMAs.  Workgroup item:
// row tile item / S, share item % S of the list tiles.
template <int KS>
struct ResidentShape {
    static constexpr int RT = KS <= 4 ? 4 : 2;
    static constexpr int NG = KS <= 4 ? 4 : 2;
    static constexpr int BM = 64 * RT;  // rows per workgroup
};

template <int KS, bool COLLECT>
__global__ void __launch_bounds__(256, 2)
score_resident_kernel(const uint4* __restrict__ Yf, int64_t n, const uint4* __restrict__ Cf,
                      int ntile, const float* __restrict__ normsp, int S, Top2Out out, CollectIO io) {
    constexpr int RT = ResidentShape<KS>::RT, NG = ResidentShape<KS>::NG, BM = 64 * RT;
    constexpr int NB = NG * KS * 2;  // 1 KB blocks per list tile
    __shared__ __align__(16) uint4 Bs[2][NB][64];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    int64_t nrow = n, items = gridDim.x;
    if (COLLECT) {
        nrow = *io.count;
        if (nrow <= 0) return;
        // shares so that the grid is filled whatever the count
        const int64_t rt = (nrow + BM - 1) / BM;
        S = (int)max((int64_t)1, min((int64_t)ntile, (int64_t)gridDim.x / rt));
        items = rt * S;
    }
    for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
        const int64_t row0 = item / S * BM + wv * 16 * RT;
        const int share = (int)(item % S);
        const int t0 = (int)((int64_t)ntile * share / S), t1 = (int)((int64_t)ntile * (share + 1) / S);
        auto fetch = [&](int t, int buf) {
#pragma unroll
            for (int q = 0; q < NB / 4; q++) {
                const int blk = q * 4 + wv;
                load_block_lds(Cf + ((int64_t)t * NB + blk) * 64, Bs[buf][blk], lane);
            }
        };
        __syncthreads();  // (the previous item's reads are done)
        if (t0 < t1) fetch(t0, 0);
        bf16x8_a ah[KS][RT], al[KS][RT];
        float bound[RT][4];
#pragma unroll
        for (int i = 0; i < RT; i++) {
            int64_t row = min(row0 + 16 * i + r, nrow - 1);
            if (COLLECT) row = io.rows[row];
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                ah[ks][i] = *(const bf16x8_a*)(Yf + frag_block(row >> 4, ks, 0, KS) + (row & 15) + 16 * g);
                al[ks][i] = *(const bf16x8_a*)(Yf + frag_block(row >> 4, ks, 1, KS) + (row & 15) + 16 * g);
            }
            if (COLLECT)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int64_t sl = row0 + 16 * i + 4 * g + j;
                    bound[i][j] = sl < nrow ? io.bound[sl] : -INFINITY;
                }
        }
        Top2State<RT> st;
        if (!COLLECT) st.init();
        float nn[NG];  // the next tile's norms
        auto norms_of = [&](int t) {
#pragma unroll
            for (int c = 0; c < NG; c++) nn[c] = normsp[(t * NG + c) * 16 + r];
        };
        if (t0 < t1) norms_of(t0);
        for (int t = t0; t < t1; t++) {
            const int buf = (t - t0) & 1;
            float nc[NG];
#pragma unroll
            for (int c = 0; c < NG; c++) nc[c] = nn[c];
            // this wave's blocks of tile t have arrived, then everyone's; the
            // other buffer's reads (tile t - 1) are done
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (t + 1 < t1) fetch(t + 1, buf ^ 1);
            norms_of(min(t + 1, t1 - 1));
#pragma unroll
            for (int c = 0; c < NG; c++) {
                v4f_a acc[RT], sum[RT];
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    if (ks % kChunk == 0)
#pragma unroll
                        for (int i = 0; i < RT; i++) {
                            if (ks) sum[i] = ks > kChunk ? sum[i] + acc[i] : acc[i];
                            acc[i] = v4f_a{0.f, 0.f, 0.f, 0.f};
                        }
                    const bf16x8_a bh = *(const bf16x8_a*)&Bs[buf][(c * KS + ks) * 2][lane];
                    const bf16x8_a bl = *(const bf16x8_a*)&Bs[buf][(c * KS + ks) * 2 + 1][lane];
                    mfma3<RT>(ah[ks], al[ks], bh, bl, acc);
                }
                if (KS > kChunk)
#pragma unroll
                    for (int i = 0; i < RT; i++) acc[i] = sum[i] + acc[i];
                const int grp = t * NG + c;
                if (!COLLECT) {
#pragma unroll
                    for (int i = 0; i < RT; i++) st.update(i, acc[i], nc[c], grp);
                } else {
                    bool any = false;
#pragma unroll
                    for (int i = 0; i < RT; i++)
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            any |= !(fmaf(-2.0f, acc[i][j], nc[c]) > bound[i][j]);
                    if (any) {
#pragma unroll
                        for (int i = 0; i < RT; i++)
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                const int64_t sl = row0 + 16 * i + 4 * g + j;
                                // (a padding list's score is +inf or NaN)
                                if (!(fmaf(-2.0f, acc[i][j], nc[c]) > bound[i][j]) && sl < nrow &&
                                    nc[c] != INFINITY)
                                    push_candidate(io, sl, grp * 16 + r);
                            }
                    }
                }
            }
        }
        if (!COLLECT) {
            out.slot = share;
            st.store(r, g, row0, n, out);
        }
    }
}

// Scores of long vectors.  One workgroup (4 waves, 2 x 2) per 32 RT rows and
// share of the list tiles of 32 CT; a wave holds RT x CT accumulators of 16 x
// 16.  Both operands pass through a ring of three k steps in LDS by direct
// loads, two steps ahead; one barrier per step.  RT 8, CT 4: a wave's step
// reads 24 KB of LDS for 96 MFMAs (64 x 64 tiles read 16 KB for 48 and with
// the staging stores kept the LDS busy all the time).  65536 x 1024 against 4096
// lists: 1979 -> 1623 us.  RT 4, CT 2 where that leaves CUs without work.
// The two column halves are slots of their own (slot 2 share + half).
// Workgroups go to the 8 XCDs in turn; consecutive slots of an XCD are the
// shares of one row tile, at least 4 (row tiles of 8 XCDs rounded up), so that
// the 32 workgroups of an XCD's L2 step through 8 row tiles x 4 list tiles and
// not through 32 row tiles (whose 1 MB each at d = 1024 came from beyond L2 at
// every list tile).
template <int RT, int CT, bool COLLECT>
__global__ void __launch_bounds__(256, RT == 8 ? 1 : 2)
score_stream_kernel(const uint4* __restrict__ Yf, int64_t n, const uint4* __restrict__ Cf, int ntile,
                    int KS, const float* __restrict__ normsp, int S, Top2Out out, CollectIO io) {
    constexpr int BM = 32 * RT, AB = 4 * RT, NBK = AB + 4 * CT;  // blocks of a step: rows, all
    static_assert(NBK % 4 == 0, "each wave loads NBK / 4 blocks");
    __shared__ __align__(16) uint4 ring[3][NBK][64];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4, wr = wv >> 1, wc = wv & 1;
    int64_t nrow = n, items = gridDim.x;
    if (COLLECT) {
        nrow = *io.count;
        if (nrow <= 0) return;
        const int64_t rt = (nrow + BM - 1) / BM;
        S = (int)min((int64_t)ntile, max((int64_t)4, (int64_t)gridDim.x / rt));
        items = (rt + 7) / 8 * 8 * S;
    }
    for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
        const int64_t slot = item >> 3;
        const int64_t tile0 = ((item & 7) + 8 * (slot / S)) * BM, row0 = tile0 + wr * 16 * RT;
        const int share = (int)(slot % S);
        if (tile0 >= nrow) continue;
        const int t0 = (int)((int64_t)ntile * share / S), t1 = (int)((int64_t)ntile * (share + 1) / S);
        const int nstep = (t1 - t0) * KS;
        // the wave's row blocks: groups 2 q + wv / 2, half wv % 2, of the tile's
        // 2 RT groups (the lane's row, past the end the last one)
        int64_t aofs[RT];
#pragma unroll
        for (int q = 0; q < RT; q++) {
            int64_t row = min(tile0 + 16 * (2 * q + (wv >> 1)) + r, nrow - 1);
            if (COLLECT) row = io.rows[row];
            aofs[q] = frag_block(row >> 4, 0, wv & 1, KS) + (row & 15) + 16 * g;
        }
        // next step to fetch: its k step, and the list tile's first group there
        int fk = 0;
        const uint4* fb = Cf + frag_block((int64_t)t0 * 2 * CT + (wv >> 1), 0, wv & 1, KS);
        auto fetch = [&](int buf) {
#pragma unroll
            for (int q = 0; q < RT; q++)
                load_block_lds(Yf + aofs[q] + fk * 128 - lane, ring[buf][4 * q + wv], lane);
#pragma unroll
            for (int q = 0; q < CT; q++)
                load_block_lds(fb + (int64_t)q * 2 * KS * 128, ring[buf][AB + 4 * q + wv], lane);
            fb += 128;
            if (++fk == KS) {
                fk = 0;
                fb += (int64_t)(2 * CT - 1) * KS * 128;
            }
        };
        float bound[RT][4];
        if (COLLECT)
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int64_t sl = row0 + 16 * i + 4 * g + j;
                    bound[i][j] = sl < nrow ? io.bound[sl] : -INFINITY;
                }
        Top2State<RT> st;
        if (!COLLECT) st.init();
        __syncthreads();  // (the previous item's reads are done)
        if (nstep > 0) fetch(0);
        if (nstep > 1) fetch(1);
        int step = 0, buf = 0;
        for (int t = t0; t < t1; t++) {
            v4f_a sum[CT][RT], acc[CT][RT];
#pragma unroll
            for (int c = 0; c < CT; c++)
#pragma unroll
                for (int i = 0; i < RT; i++) sum[c][i] = v4f_a{0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < KS; k0 += kChunk) {
#pragma unroll
                for (int kc = 0; kc < kChunk; kc++) {
                    if (k0 + kc >= KS) break;
                    // this wave's blocks of the step have arrived (those of the
                    // next step, RT + CT loads, may be on their way), then
                    // everyone's; the reads of the step before are done
                    if (step + 1 < nstep) {
                        if constexpr (RT + CT == 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
                        else asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
                    } else {
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    }
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    if (step + 2 < nstep) fetch(buf == 0 ? 2 : buf - 1);
                    step++;
                    bf16x8_a bh[CT], bl[CT];
#pragma unroll
                    for (int c = 0; c < CT; c++) {
                        bh[c] = *(const bf16x8_a*)&ring[buf][AB + 2 * (wc * CT + c)][lane];
                        bl[c] = *(const bf16x8_a*)&ring[buf][AB + 2 * (wc * CT + c) + 1][lane];
                    }
                    // row operands one group ahead of their MFMAs
                    bf16x8_a a[2][2];
                    auto rows = [&](int i) {
                        a[i & 1][0] = *(const bf16x8_a*)&ring[buf][2 * (wr * RT + i)][lane];
                        a[i & 1][1] = *(const bf16x8_a*)&ring[buf][2 * (wr * RT + i) + 1][lane];
                    };
                    rows(0);
#pragma unroll
                    for (int i = 0; i < RT; i++) {
                        if (i + 1 < RT) rows(i + 1);
                        __builtin_amdgcn_sched_barrier(0);
                        const bf16x8_a ah = a[i & 1][0], al = a[i & 1][1];
#pragma unroll
                        for (int c = 0; c < CT; c++) {
                            if (kc == 0) acc[c][i] = v4f_a{0.f, 0.f, 0.f, 0.f};
                            acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[c], acc[c][i], 0, 0, 0);
                        }
#pragma unroll
                        for (int c = 0; c < CT; c++)
                            acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[c], acc[c][i], 0, 0, 0);
#pragma unroll
                        for (int c = 0; c < CT; c++)
                            acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[c], acc[c][i], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    buf = buf == 2 ? 0 : buf + 1;
                }
#pragma unroll
                for (int c = 0; c < CT; c++)
#pragma unroll
                    for (int i = 0; i < RT; i++) sum[c][i] += acc[c][i];
            }
#pragma unroll
            for (int c = 0; c < CT; c++) {
                const int grp = t * 2 * CT + wc * CT + c;
                const float nc = normsp[grp * 16 + r];
                if (!COLLECT) {
#pragma unroll
                    for (int i = 0; i < RT; i++) st.update(i, sum[c][i], nc, grp);
                } else {
                    bool any = false;
#pragma unroll
                    for (int i = 0; i < RT; i++)
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            any |= !(fmaf(-2.0f, sum[c][i][j], nc) > bound[i][j]);
                    if (any) {
#pragma unroll
                        for (int i = 0; i < RT; i++)
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                const int64_t sl = row0 + 16 * i + 4 * g + j;
                                if (!(fmaf(-2.0f, sum[c][i][j], nc) > bound[i][j]) && sl < nrow &&
                                    nc != INFINITY)
                                    push_candidate(io, sl, grp * 16 + r);
                            }
                    }
                }
            }
        }
        if (!COLLECT) {
            out.slot = 2 * share + wc;
            st.store(r, g, row0, n, out);
        }
    }
}

// L lanes per row (a power of two up to 64): combines the slots' (best, list,
// second; ties to the lower list), accepts the list when the gap clears 2E,
// else puts the row on the re-check list with its bound s1 + 2E (rounded up),
// or, with a score that is not finite, on the list of rows that take every
// list.
__global__ void __launch_bounds__(256)
top2_accept_kernel(int64_t n, int d, int L, const Top2Out in, const float* __restrict__ nyp,
                   const float* __restrict__ nmax, int32_t* __restrict__ assign,
                   int32_t* __restrict__ recheck, float* __restrict__ bound,
                   int32_t* __restrict__ ncand, int32_t* __restrict__ ovf,
                   unsigned long long* __restrict__ ovf_keys, int32_t* __restrict__ cnt) {
    const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / L;
    const int lane = threadIdx.x & 63, j = threadIdx.x & (L - 1);
    bool near = false;
    float top = 0.0f;
    float s1 = INFINITY, s2 = INFINITY;
    int c = 0x7fffffff;
    auto take = [&](float ob, float os, int oc) {
        const bool mine = (s1 < ob) | ((s1 == ob) & (c < oc));
        const float lose = mine ? ob : s1, keep = mine ? s2 : os;
        s2 = fminf(keep, lose);
        s1 = mine ? s1 : ob;
        c = mine ? c : oc;
    };
    if (row < n)
        for (int y = j; y < in.slots; y += L) {
            const int64_t at = row * in.slots + y;
            take(in.s1[at], in.s2[at], in.best[at]);
        }
    for (int off = L / 2; off > 0; off >>= 1)
        take(__shfl_xor(s1, off), __shfl_xor(s2, off), __shfl_xor(c, off));
    if (row < n && j == 0) {
        const double u = 1.0 / 16777216.0;
        const double Nm = (double)nmax[0] * (1.0 + 4.0 * u);
        const double ny = (double)nyp[row], cm = sqrt(Nm);
        const int steps = top2_kpad(d) / kTopBK;
        const double e_dot =
            (2.0 * u * 1.02 * 33.0 * 3.0 * (double)min(steps, kChunk) +
             1.02 * u * (double)((steps + kChunk - 1) / kChunk) + 3.01 / 65536.0 + (d + 4.0) * u) *
            ny * cm;
        const double tiny = 6.0 * d * (0x1p-126 * (ny + cm) + 0x1p-149);
        const double E = 2.0 * (2.0 * e_dot + 2.0 * u * Nm + 4.0 * u * ny * cm) + tiny;
        const double a = (double)s1, b = (double)s2;
        // b = +inf (a single list) passes
        if (isfinite(a) && !isnan(b) && (b - a > 2.0 * E)) {
            assign[row] = c;
        } else if (isfinite(a) && isfinite(E)) {
            near = true;
            top = __double2float_ru(a + 2.0 * E);
        } else {
            const int o = atomicAdd(&cnt[1], 1);
            atomicAdd(&cnt[2], 1);
            ovf[o] = (int32_t)row;
            ovf_keys[o] = ~0ull;
        }
    }
    const unsigned long long m = __ballot(near);
    int at = 0;
    if (lane == 0 && m) at = atomicAdd(&cnt[0], __popcll(m));
    at = __shfl(at, 0) + __popcll(m & ((1ull << lane) - 1ull));
    if (near) {
        recheck[at] = (int32_t)row;
        bound[at] = top;
        ncand[at] = 0;
    }
}

// 16 lanes per re-checked row, one candidate list each: its score in the fixed
// order, the least (score, list) is the row's.  Then the rows that took every
// list.
__global__ void __launch_bounds__(256)
recheck_kernel(const float* __restrict__ Y, int d, const float* __restrict__ Cm,
               const float* __restrict__ norms, const int32_t* __restrict__ cnt,
               const int32_t* __restrict__ recheck, const int32_t* __restrict__ ncand,
               const int32_t* __restrict__ cand, const int32_t* __restrict__ ovf,
               const unsigned long long* __restrict__ ovf_keys, int32_t* __restrict__ assign) {
    const int64_t m = cnt[0], mo = cnt[1];
    const int j = threadIdx.x & 15;
    for (int64_t s0 = (int64_t)blockIdx.x * 16; s0 < m; s0 += (int64_t)gridDim.x * 16) {
        const int64_t slot = s0 + (threadIdx.x >> 4);
        const int nc = slot < m ? ncand[slot] : 0;
        const int64_t row = slot < m ? recheck[slot] : 0;
        unsigned long long key = ~0ull;
        if (nc <= kCand && j < nc) {
            const int c = cand[slot * kCand + j];
            const float* y = Y + row * d;
            const float* cc = Cm + (int64_t)c * d;
            float acc = 0.0f;
            int k = 0;
            for (; k + 64 <= d; k += 64) {
                float4 a[16], b[16];  // all loads of 64 k in flight
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    a[q] = *(const float4*)(y + k + 4 * q);
                    b[q] = *(const float4*)(cc + k + 4 * q);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    acc = fmaf(a[q].x, b[q].x, acc);
                    acc = fmaf(a[q].y, b[q].y, acc);
                    acc = fmaf(a[q].z, b[q].z, acc);
                    acc = fmaf(a[q].w, b[q].w, acc);
                }
            }
            for (; k < d; k += 4) {
                const float4 a = *(const float4*)(y + k), b = *(const float4*)(cc + k);
                acc = fmaf(a.x, b.x, acc);
                acc = fmaf(a.y, b.y, acc);
                acc = fmaf(a.z, b.z, acc);
                acc = fmaf(a.w, b.w, acc);
            }
            const uint32_t u = __float_as_uint(fmaf(-2.0f, acc, norms[c]));
            key = ((unsigned long long)((u & 0x80000000u) ? ~u : (u | 0x80000000u)) << 32) |
                  (uint32_t)c;
        }
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) {
            const unsigned long long o = __shfl_xor(key, off);
            key = o < key ? o : key;
        }
        if (j == 0 && nc > 0 && nc <= kCand) assign[row] = (int32_t)(uint32_t)key;
    }
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < mo; i += (int64_t)gridDim.x * 256)
        assign[ovf[i]] = (int32_t)(uint32_t)(ovf_keys[i] & 0xffffffffull);
}

__global__ void tally_kernel(const int32_t* __restrict__ cnt, unsigned long long* __restrict__ total) {
    if (threadIdx.x == 0) total[0] += (unsigned long long)cnt[0] + (unsigned long long)cnt[2];
}

bool assign_mfma_ok(int d, const float* Y, const float* Cm) {
    return d > 0 && d % 4 == 0 && ((uintptr_t)Y & 15) == 0 && ((uintptr_t)Cm & 15) == 0;
}

namespace {

// The score kernel of a shape: rows and lists per tile, list-tile shares and
// result slots per row, workgroups.
struct Top2Plan {
    bool resident, large;
    int KS, bm, bn, S, slots;
    int64_t rt;  // row tiles
    int ntile;   // list tiles
};

// Vectors of up to 8 k steps (256) stay in registers: 65536 x 256 rows against
// 8192 lists take 723 us there (1844 us before), and past 256 the registers hold
// too few rows per list read.  Shares of the list tiles fill the chip
// (two workgroups per CU, one of the large tiles) when the rows are few.
Top2Plan top2_plan(int64_t n, int d, int nlist) {
    Top2Plan p{};
    p.KS = top2_kpad(d) / kTopBK;
    p.resident = p.KS <= 8;
    int64_t wg = 512;
    if (p.resident) {
        p.bm = p.KS <= 4 ? ResidentShape<4>::BM : ResidentShape<8>::BM;
        p.bn = p.KS <= 4 ? 16 * ResidentShape<4>::NG : 16 * ResidentShape<8>::NG;
    } else {
        p.large = ((n + 255) / 256) * ((nlist + 127) / 128) >= 256;
        p.bm = p.large ? 256 : 128;
        p.bn = p.large ? 128 : 64;
        if (p.large) wg = 256;
    }
    p.rt = (n + p.bm - 1) / p.bm;
    p.ntile = (nlist + p.bn - 1) / p.bn;
    p.S = (int)std::max<int64_t>(1, std::min<int64_t>(p.ntile, wg / p.rt));
    if (!p.resident) p.S = std::min(p.ntile, std::max(p.S, 4));
    p.slots = p.resident ? p.S : 2 * p.S;
    return p;
}

constexpr size_t kAlign = 64;  // words
size_t words(size_t w) { return (w + kAlign - 1) / kAlign * kAlign; }

// The scratch: counters (re-check rows, rows that take every list, those of
// them that were not finite) and Nmax; results per slot; re-check lists;
// padded norms; split operands.
struct Scratch {
    int32_t *cnt, *best, *recheck, *ncand, *cand, *ovf;
    float *nmax, *s1, *s2, *bound, *ny, *normsp;
    uint4 *yf, *cf;
    size_t total;
};

Scratch carve(float* base, int64_t n, const Top2Plan& p) {
    Scratch s{};
    size_t at = 0;
    auto take = [&](size_t w) {
        float* q = base + at;
        at += words(w);
        return q;
    };
    const size_t N = (size_t)n;
    s.cnt = (int32_t*)take(8);
    s.nmax = (float*)s.cnt + 4;
    s.best = (int32_t*)take(N * p.slots);
    s.s1 = take(N * p.slots);
    s.s2 = take(N * p.slots);
    s.recheck = (int32_t*)take(N);
    s.bound = take(N);
    s.ncand = (int32_t*)take(N);
    s.ovf = (int32_t*)take(N);
    s.ny = take(N);
    s.cand = (int32_t*)take(N * kCand);
    s.normsp = take((size_t)p.ntile * p.bn);
    s.yf = (uint4*)take((N + 15) / 16 * 16 * p.KS * kTopBK);
    s.cf = (uint4*)take((size_t)p.ntile * p.bn * p.KS * kTopBK);
    s.total = at;
    return s;
}

template <bool COLLECT>
void launch_scores(const Top2Plan& p, const Scratch& w, int64_t n, const Top2Out& o,
                   const CollectIO& io, hipStream_t s) {
    // the re-check's grid fits any count
    const int64_t tiles = p.resident ? p.rt : (p.rt + 7) / 8 * 8;
    const dim3 grid((unsigned)(COLLECT ? 512 : tiles * p.S)), block(256);
    if (!p.resident) {
        if (!COLLECT && p.large)
            hipLaunchKernelGGL((score_stream_kernel<8, 4, false>), grid, block, 0, s, w.yf, n, w.cf,
                               p.ntile, p.KS, w.normsp, p.S, o, io);
        else
            hipLaunchKernelGGL((score_stream_kernel<4, 2, COLLECT>), grid, block, 0, s, w.yf, n, w.cf,
                               p.ntile * (p.bn / 64), p.KS, w.normsp, p.S, o, io);
        return;
    }
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, grid, block, 0, s, w.yf, n, w.cf, p.ntile, w.normsp, p.S, o, io);
    };
    switch (p.KS) {
        case 1: go(score_resident_kernel<1, COLLECT>); break;
        case 2: go(score_resident_kernel<2, COLLECT>); break;
        case 3: go(score_resident_kernel<3, COLLECT>); break;
        case 4: go(score_resident_kernel<4, COLLECT>); break;
        case 5: go(score_resident_kernel<5, COLLECT>); break;
        case 6: go(score_resident_kernel<6, COLLECT>); break;
        case 7: go(score_resident_kernel<7, COLLECT>); break;
        default: go(score_resident_kernel<8, COLLECT>); break;
    }
}

}  // namespace

size_t assign_mfma_scratch_floats(int64_t n, int d, int nlist) {
    return carve(nullptr, n, top2_plan(n, d, nlist)).total;
}

hipError_t assign_mfma_tally(const float* scratch, unsigned long long* total, hipStream_t s) {
    hipLaunchKernelGGL(tally_kernel, dim3(1), dim3(64), 0, s, (const int32_t*)scratch, total);
    return hipGetLastError();
}

hipError_t assign_mfma(const float* Y, int64_t n, int d, const float* Cm, int nlist,
                       const float* norms, int32_t* assign, float* scratch,
                       size_t scratch_floats, unsigned long long* keys, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (!assign_mfma_ok(d, Y, Cm) || nlist <= 0 || !scratch || !keys ||
        scratch_floats < assign_mfma_scratch_floats(n, d, nlist) || (n + 127) / 128 > 65535)
        return hipErrorInvalidValue;
    const Top2Plan p = top2_plan(n, d, nlist);
    const Scratch w = carve(scratch, n, p);
    const int64_t yg = (n + 15) / 16, cg = (int64_t)p.ntile * p.bn / 16;
    hipLaunchKernelGGL(split_kernel, dim3((unsigned)(yg + cg + 1)), dim3(256), 0, s, Y, n, Cm, nlist,
                       d, p.KS, yg, w.yf, w.cf, w.ny, norms, w.normsp, w.nmax, w.cnt);
    const Top2Out o{w.best, w.s1, w.s2, p.slots, 0};
    const CollectIO io{w.recheck, w.cnt, w.bound, w.ncand, w.cand, w.ovf, keys, w.cnt + 1};
    launch_scores<false>(p, w, n, o, io, s);
    int L = 1;
    while (L < p.slots && L < 64) L *= 2;
    hipLaunchKernelGGL(top2_accept_kernel, dim3((unsigned)((n * L + 255) / 256)), dim3(256), 0, s, n, d,
                       L, o, w.ny, w.nmax, assign, w.recheck, w.bound, w.ncand, w.ovf, keys,
                       w.cnt);
    // the near ties (their count is read on the device)
    launch_scores<true>(p, w, n, o, io, s);
    hipError_t e = gemm_nt_argmin_rows(Y, d, w.ovf, w.cnt + 1, n, Cm, d, nlist, d, norms, keys, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(recheck_kernel, dim3((unsigned)std::min<int64_t>((n + 15) / 16, 2048)),
                       dim3(256), 0, s, Y, d, Cm, norms, w.cnt, w.recheck, w.ncand, w.cand, w.ovf,
                       keys, assign);
    return hipGetLastError();
}

}  // namespace jhq
