// insert.hip — encode and list placement of inserted vectors: primary and
// residual codes (v14/encode.cu:20-86), scatter into the list pool, block
// moves, and the copies of the primary codes that the scans read.
#include "kernels.h"

#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>

namespace jhq {

// ---------------------------------------------------------------------------
// Encode: a workgroup takes kEncV vectors and walks their dimensions in
// chunks of kEncC.  Every thread quantizes dimensions of the chunk (reads of
// consecutive floats of one vector), the digits and residual indices are
// packed into code and residual bytes from LDS, and one lane per vector
// carries that vector's residual correction: a sequential fmaf chain in
// dimension order over the quantized values the chunk left in LDS.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int nearest_mid(const float* mids, int n, float v) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (v < mids[mid]) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

constexpr int kEncV = 16, kEncC = 128, kEncT = 256;
constexpr int kEncPer = kEncV * kEncC / kEncT;  // dimensions a thread quantizes per chunk

__global__ void __launch_bounds__(kEncT)
encode_kernel(const float* __restrict__ y, int64_t n, int d, int M, int Ds, int K1D, int bpd,
              const float* __restrict__ c1d, int Kr, int RC, int Br, int bpv,
              const float* __restrict__ res_c1d, uint8_t* __restrict__ codes,
              uint8_t* __restrict__ res, float* __restrict__ corr, int mode) {
    // RC residual codebooks of Kr words: one shared by every dimension (the
    // reference, v14/jhq_gpu_index.cu:302-330) or one per subspace (RC = M)
    __shared__ float cval[256], cmid[256];
    // the chunk's quantized values (yhat, rhat) per vector; the odd row
    // stride puts the chain lanes' reads of one column in distinct banks
    __shared__ float yh[kEncV][kEncC + 1], rh[kEncV][kEncC + 1];
    __shared__ uint8_t dg[kEncV][kEncC], rq[kEncV][kEncC];
    extern __shared__ float rsh[];  // rval[RC*Kr], rmid[RC*Kr]
    float* rval = rsh;
    float* rmid = rsh + RC * Kr;
    const int tid = threadIdx.x;
    const int64_t v0 = (int64_t)blockIdx.x * kEncV;
    const int nv = (n - v0) < kEncV ? (int)(n - v0) : kEncV;
    if (tid < K1D) cval[tid] = c1d[tid];
    if (mode & 2)
        for (int i = tid; i < RC * Kr; i += kEncT) rval[i] = res_c1d[i];
    __syncthreads();
    if (tid + 1 < K1D) cmid[tid] = 0.5f * (cval[tid] + cval[tid + 1]);
    if (mode & 2)
        for (int i = tid; i < RC * Kr; i += kEncT)
            if ((i % Kr) + 1 < Kr) rmid[i] = 0.5f * (rval[i] + rval[i + 1]);
    __syncthreads();
    const int kmask = K1D - 1;
    float dot = 0.0f;  // lane v < nv: vector v0 + v's chain
    for (int c0 = 0; c0 < d; c0 += kEncC) {
        const int cw = (d - c0) < kEncC ? (d - c0) : kEncC;
        float val[kEncPer];
#pragma unroll
        for (int i = 0; i < kEncPer; i++) {
            const int e = tid + i * kEncT, v = e / kEncC, jj = e % kEncC;
            val[i] = (v < nv && jj < cw) ? y[(v0 + v) * d + c0 + jj] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kEncPer; i++) {
            const int e = tid + i * kEncT, v = e / kEncC, jj = e % kEncC;
            if (v >= nv || jj >= cw) continue;
            const int j = c0 + jj;
            const int m = j / Ds, k = j - m * Ds;
            int dig;
            if (mode & 1) dig = (K1D == 1) ? 0 : nearest_mid(cmid, K1D, val[i]);
            else dig = (codes[(v0 + v) * M + m] >> (k * bpd)) & kmask;
            dg[v][jj] = (uint8_t)dig;
            if (mode & 2) {
                const int cb = (RC == 1) ? 0 : m;
                const float yhat = cval[dig];
                const float r = val[i] - yhat;
                const int ri = (Kr == 1) ? 0 : nearest_mid(rmid + cb * Kr, Kr, r);
                rq[v][jj] = (uint8_t)ri;
                yh[v][jj] = yhat;
                rh[v][jj] = rval[cb * Kr + ri];
            }
        }
        __syncthreads();
        if (mode & 1) {
            // whole subspaces of the chunk (c0 is a multiple of Ds, which divides 32)
            const int ms = cw / Ds;
            for (int e = tid; e < kEncV * ms; e += kEncT) {
                const int v = e / ms, mm = e - v * ms;
                if (v >= nv) continue;
                uint32_t code = 0u;
                for (int k = 0; k < Ds; k++) code |= (uint32_t)dg[v][mm * Ds + k] << (k * bpd);
                codes[(v0 + v) * M + c0 / Ds + mm] = (uint8_t)code;
            }
        }
        if (mode & 2) {
            if (Br == 4) {
                // two dimensions a byte, the even one in the low nibble; an odd
                // last dimension alone in the low nibble of the last byte
                const int nb = (cw + 1) >> 1;
                for (int e = tid; e < kEncV * nb; e += kEncT) {
                    const int v = e / nb, b = e - v * nb;
                    if (v >= nv) continue;
                    const uint32_t lo = rq[v][2 * b] & 0x0Fu;
                    const uint32_t hi = (2 * b + 1 < cw) ? (rq[v][2 * b + 1] & 0x0Fu) : 0u;
                    res[(v0 + v) * bpv + (c0 >> 1) + b] = (uint8_t)(lo | (hi << 4));
                }
            } else {
                for (int e = tid; e < kEncV * cw; e += kEncT) {
                    const int v = e / cw, jj = e - v * cw;
                    if (v >= nv) continue;
                    res[(v0 + v) * bpv + c0 + jj] = rq[v][jj];
                }
            }
            if (tid < nv)
                for (int jj = 0; jj < cw; jj++) dot = fmaf(yh[tid][jj], rh[tid][jj], dot);
        }
        __syncthreads();
    }
    if ((mode & 2) && tid < nv) corr[v0 + tid] = 2.0f * dot;
}

// ---------------------------------------------------------------------------
// The same for the usual shapes (Ds 1, 2, 4 or 8, d a multiple of 4, Br = 4 with
// 16 residual words, or Br = 8): a thread takes 8 consecutive dimensions of a
// vector, 16 lanes a vector's 128, so that code and residual bytes are packed in
// registers and go out as words.  The searches of up to 16 words run in
// registers (the same comparisons as nearest_mid's, by selects); larger
// codebooks stay in LDS.  The correction's chain of one vector is sequential:
// each chunk's (yhat, rhat) pairs go through LDS, double-buffered, and one wave
// (the four in turn) adds a chunk's pairs while all four quantize the next.
// Bound by reading y: 65536 x 1024 in 268 MB (57 us at the rate of a copy).
// ---------------------------------------------------------------------------
// index of nearest_mid(mids, K, v), mids in registers
template <int K>
__device__ __forceinline__ int tree_mid(const float (&m)[K - 1], float v) {
    if constexpr (K == 2) {
        return v < m[0] ? 0 : 1;
    } else {
        // the half that the first comparison leaves, then the same in it
        const bool up = !(v < m[K / 2 - 1]);
        float h[K / 2 - 1];
#pragma unroll
        for (int i = 0; i < K / 2 - 1; i++) h[i] = up ? m[K / 2 + i] : m[i];
        return (up ? K / 2 : 0) + tree_mid<K / 2>(h, v);
    }
}

template <int K>
struct RegBook {
    float m[K - 1];
    __device__ __forceinline__ void load(const float* mids) {
#pragma unroll
        for (int i = 0; i < K - 1; i++) m[i] = mids[i];
    }
    __device__ __forceinline__ int find(const float*, int, float v) const { return tree_mid<K>(m, v); }
};
struct LdsBook {
    __device__ __forceinline__ void load(const float*) {}
    __device__ __forceinline__ int find(const float* mids, int K, float v) const {
        return nearest_mid(mids, K, v);
    }
};

constexpr int kEncLd = 2 * kEncC + 4;  // floats per vector of a chunk's pairs

template <class PBook, class RBook, int DS, int MODE>
__global__ void __launch_bounds__(kEncT)
encode_words_kernel(const float* __restrict__ y, int64_t n, int d, int M, int K1D, int bpd,
                    const float* __restrict__ c1d, int Kr, int RC, int bpv,
                    const float* __restrict__ res_c1d, uint8_t* __restrict__ codes,
                    uint8_t* __restrict__ res, float* __restrict__ corr, int cword, int rword) {
    constexpr int NS = 8 / DS;  // subspaces of a thread's 8 dimensions
    __shared__ float cval[256], cmid[256];
    __shared__ __align__(16) float pair[(MODE & 2) ? 2 : 1][(MODE & 2) ? kEncV : 1][kEncLd];
    __shared__ float sdot[kEncV];
    extern __shared__ float rsh[];  // rval[RC*Kr], rmid[RC*Kr]
    float* rval = rsh;
    float* rmid = rsh + RC * Kr;
    const int tid = threadIdx.x, v = tid >> 4, l = tid & 15, wv = tid >> 6;
    const int64_t row = (int64_t)blockIdx.x * kEncV + v;
    const bool have = row < n;
    const float* yr = y + (have ? row : n - 1) * d;
    for (int i = tid; i < K1D; i += kEncT) cval[i] = c1d[i];
    if (MODE & 2)
        for (int i = tid; i < RC * Kr; i += kEncT) rval[i] = res_c1d[i];
    if (tid < kEncV) sdot[tid] = 0.0f;
    auto fetch = [&](int j0, float (&x)[8]) {
        // d a multiple of 4: four dimensions are inside or past the end together
        const float4 a = *(const float4*)(yr + min(j0, d - 4));
        const float4 b = *(const float4*)(yr + min(j0 + 4, d - 4));
        x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
        x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    };
    float x[8], nx[8];
    fetch(8 * l, nx);
    __syncthreads();
    for (int i = tid; i + 1 < K1D; i += kEncT) cmid[i] = 0.5f * (cval[i] + cval[i + 1]);
    if (MODE & 2)
        for (int i = tid; i < RC * Kr; i += kEncT)
            if ((i % Kr) + 1 < Kr) rmid[i] = 0.5f * (rval[i] + rval[i + 1]);
    __syncthreads();
    PBook pb;
    RBook rb;
    if (MODE & 1) pb.load(cmid);
    if ((MODE & 2) && RC == 1) rb.load(rmid);
    const int nch = (d + kEncC - 1) / kEncC;
    // vector t's chain over chunk c (one wave's first kEncV lanes)
    auto chain = [&](int c) {
        const int t = tid & 63;
        if (t >= kEncV) return;
        const int w = min(d - c * kEncC, kEncC);  // a multiple of 4
        const float* p = pair[c & 1][t];
        float dot = sdot[t];
#pragma unroll 8
        for (int j = 0; j < w; j += 2) {
            const float4 q = *(const float4*)(p + 2 * j);
            dot = fmaf(q.x, q.y, dot);
            dot = fmaf(q.z, q.w, dot);
        }
        sdot[t] = dot;
    };
    for (int c = 0; c < nch; c++) {
        const int j0 = c * kEncC + 8 * l;
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = nx[i];
        if (c + 1 < nch) fetch(j0 + kEncC, nx);
        const int nd = min(d - j0, 8);  // 8, 4, or none left
        if (nd > 0) {
            uint32_t cb[NS];
            const int m0 = j0 / DS;
            if (MODE == 2)
#pragma unroll
                for (int s = 0; s < NS; s++)
                    cb[s] = (have && s * DS < nd) ? codes[row * M + m0 + s] : 0u;
            else
#pragma unroll
                for (int s = 0; s < NS; s++) cb[s] = 0u;
            uint32_t rw[2] = {0u, 0u};  // residual nibbles (or bytes), first dimension lowest
            float2 pr[8];
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const int rc0 = RC == 1 ? 0 : min(m0 + s, M - 1) * Kr;
                if ((MODE & 2) && RC != 1) rb.load(rmid + rc0);
#pragma unroll
                for (int k = 0; k < DS; k++) {
                    const int i = s * DS + k;
                    int dig;
                    if (MODE & 1) {
                        dig = pb.find(cmid, K1D, x[i]);
                        cb[s] |= (uint32_t)dig << (k * bpd);
                    } else {
                        dig = (int)(cb[s] >> (k * bpd)) & (K1D - 1);
                    }
                    if (MODE & 2) {
                        const float yhat = cval[dig];
                        const int ri = rb.find(rmid + rc0, Kr, x[i] - yhat);
                        if (rword == 4) rw[0] |= (uint32_t)(ri & 15) << (4 * i);
                        else rw[i / 4] |= (uint32_t)ri << (8 * (i % 4));
                        pr[i] = make_float2(yhat, rval[rc0 + ri]);
                    }
                }
            }
            if (MODE & 2) {
                float* p = pair[c & 1][v] + 16 * l;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    *(float4*)(p + 4 * i) = make_float4(pr[2 * i].x, pr[2 * i].y, pr[2 * i + 1].x,
                                                        pr[2 * i + 1].y);
            }
            if (have) {
                if (MODE & 1) {
                    uint8_t* o = codes + row * M + m0;
                    if (cword && nd == 8) {
                        if constexpr (NS == 1) *o = (uint8_t)cb[0];
                        if constexpr (NS == 2) *(uint16_t*)o = (uint16_t)(cb[0] | (cb[1] << 8));
                        if constexpr (NS == 4)
                            *(uint32_t*)o = cb[0] | (cb[1] << 8) | (cb[2] << 16) | (cb[3] << 24);
                        if constexpr (NS == 8)
                            *(uint2*)o = make_uint2(cb[0] | (cb[1] << 8) | (cb[2] << 16) | (cb[3] << 24),
                                                    cb[4 % NS] | (cb[5 % NS] << 8) | (cb[6 % NS] << 16) |
                                                        (cb[7 % NS] << 24));
                    } else {
#pragma unroll
                        for (int s = 0; s < NS; s++)
                            if (s * DS < nd) o[s] = (uint8_t)cb[s];
                    }
                }
                if (MODE & 2) {
                    if (rword == 4) {  // Br = 4: two dimensions a byte
                        uint8_t* o = res + row * bpv + j0 / 2;
                        if ((bpv & 3) == 0 && nd == 8) {
                            *(uint32_t*)o = rw[0];
                        } else {  // (bpv is even)
                            *(uint16_t*)o = (uint16_t)rw[0];
                            if (nd == 8) *(uint16_t*)(o + 2) = (uint16_t)(rw[0] >> 16);
                        }
                    } else {
                        uint8_t* o = res + row * bpv + j0;
                        *(uint32_t*)o = rw[0];
                        if (nd == 8) *(uint32_t*)(o + 4) = rw[1];
                    }
                }
            }
        }
        if (MODE & 2) {
            // the chunk before is added by one of the waves while the others
            // are at the next chunk; its buffer is written again after that
            if (c > 0 && wv == (c & 3)) chain(c - 1);
            __syncthreads();
        }
    }
    if (MODE & 2) {
        if (wv == 0) chain(nch - 1);
        if (tid < kEncV && (int64_t)blockIdx.x * kEncV + tid < n)
            corr[(int64_t)blockIdx.x * kEncV + tid] = 2.0f * sdot[tid];
    }
}

template <class PBook, class RBook, int DS>
static hipError_t launch_words(int mode, size_t lds, const float* y, int64_t n, int d, int M, int K1D,
                               int bpd, const float* c1d, int Kr, int RC, int bpv,
                               const float* res_c1d, uint8_t* codes, uint8_t* res, float* corr,
                               int cword, int rword, hipStream_t s) {
    const dim3 grid((unsigned)((n + kEncV - 1) / kEncV));
    auto go = [&](auto* k) -> hipError_t {
        if (lds > 16 * 1024) {  // beside the static 40 KB
            const hipError_t e = hipFuncSetAttribute((const void*)k,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k, grid, dim3(kEncT), lds, s, y, n, d, M, K1D, bpd, c1d, Kr, RC, bpv, res_c1d,
                           codes, res, corr, cword, rword);
        return hipGetLastError();
    };
    if (mode == 1) return go(encode_words_kernel<PBook, RBook, DS, 1>);
    if (mode == 2) return go(encode_words_kernel<PBook, RBook, DS, 2>);
    return go(encode_words_kernel<PBook, RBook, DS, 3>);
}

hipError_t encode(const float* y, int64_t n, int d, int M, int Ds, int K1D, int bpd,
                  const float* c1d, int Kr, int RC, int Br, int bpv, const float* res_c1d,
                  uint8_t* codes, uint8_t* res, float* corr, int mode, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (K1D > 256 || Kr > 256 || (32 % Ds) != 0 || (RC != 1 && RC != M) || Ds * M != d ||
        ((mode & 2) && Br != 4 && Br != 8))
        return hipErrorInvalidValue;
    const size_t lds = (size_t)2 * RC * Kr * sizeof(float);
    if (lds > 96 * 1024) return hipErrorInvalidValue;
    const int64_t blocks = (n + kEncV - 1) / kEncV;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    // One bit at Ds 8, two at 4, four at 2, eight at 1 (the codebook in LDS):
    // the digits of 8-bit codes; residual words in registers with Br = 4, in LDS
    // with Br = 8.  Word stores need aligned rows.
    const bool book = (Ds == 8 && bpd == 1) || (Ds == 4 && bpd == 2) || (Ds == 2 && bpd == 4) ||
                      (Ds == 1 && bpd == 8);
    if (book && d % 4 == 0 && ((uintptr_t)y & 15) == 0 &&
        (!(mode & 2) || (((uintptr_t)res & 3) == 0 && (Br == 8 || Kr == 16)))) {
        const int ns = 8 / Ds;
        const int cword = M % ns == 0 && (uintptr_t)codes % ns == 0, rword = Br == 4 ? 4 : 8;
#define JHQ_WORDS(P, D)                                                                             \
    (Br == 4 ? launch_words<P, RegBook<16>, D>(mode, lds, y, n, d, M, K1D, bpd, c1d, Kr, RC, bpv,   \
                                               res_c1d, codes, res, corr, cword, rword, s)          \
             : launch_words<P, LdsBook, D>(mode, lds, y, n, d, M, K1D, bpd, c1d, Kr, RC, bpv,       \
                                           res_c1d, codes, res, corr, cword, rword, s))
        if (Ds == 8) return JHQ_WORDS(RegBook<2>, 8);
        if (Ds == 4) return JHQ_WORDS(RegBook<4>, 4);
        if (Ds == 2) return JHQ_WORDS(RegBook<16>, 2);
        return JHQ_WORDS(LdsBook, 1);
#undef JHQ_WORDS
    }
    if (lds > 48 * 1024) {
        static const hipError_t e = hipFuncSetAttribute((const void*)encode_kernel,
                                                         hipFuncAttributeMaxDynamicSharedMemorySize,
                                                         96 * 1024);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(encode_kernel, dim3((unsigned)blocks), dim3(kEncT), lds, s, y, n, d, M, Ds,
                       K1D, bpd, c1d, Kr, RC, Br, bpv, res_c1d, codes, res, corr, mode);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// List storage.  The lists live in one pool of padded candidate slots; list l
// is described by ListDesc {start, cap, size, cbase} (int4): it owns slots
// [start, start + cap) (cap a multiple of 16) and holds size candidates.
// Primary codes are code-major inside the block: byte m of candidate i is at
// codes_t[start*M + m*cap + i], so one 32-bit load returns byte m of four
// consecutive candidates.  Residual codes, corrections and ids are indexed by
// slot.  cbase is the list's first canonical position (lists in list order,
// candidates in insertion order), the tag the exact selection breaks ties
// with, so results do not depend on where a list's block sits in the pool.
// ---------------------------------------------------------------------------
// V vectors per workgroup, staged in LDS: their code rows come in as words and
// go out byte by byte with consecutive threads on consecutive vectors (in list
// order: neighbours in their list's block), residual rows are copied 16 bytes
// (or a byte) per thread.  One thread per vector and byte loops over both had
// 2000 x 768 vectors take 57 us; the code bytes are scattered stores by the
// pool's layout.  rows (optional): the row-major copy takes the code rows too.
template <int V>
__global__ void __launch_bounds__(256)
scatter_kernel(const int32_t* __restrict__ order, const int32_t* __restrict__ slist,
               const int32_t* __restrict__ sidx, int64_t n, int64_t id_base,
               const int4* __restrict__ ldesc, const uint8_t* __restrict__ pc,
               const uint8_t* __restrict__ rc, const float* __restrict__ co, int M, int bpv,
               int32_t* __restrict__ ids_out, uint8_t* __restrict__ codes_t,
               uint8_t* __restrict__ res_out, float* __restrict__ corr_out,
               uint8_t* __restrict__ rows) {
    extern __shared__ __align__(16) uint8_t stage[];  // [V][M + 4] code rows
    __shared__ int64_t sbase[V], sslot[V], sid[V];
    __shared__ int scap[V];
    const int tid = threadIdx.x, ld = M + 4;
    const int64_t s0 = (int64_t)blockIdx.x * V;
    const int nv = (int)min((int64_t)V, n - s0);
    if (tid < nv) {
        const int64_t id = order[s0 + tid];
        const int4 L = ldesc[slist[s0 + tid]];
        const int64_t i = sidx[s0 + tid], slot = (int64_t)L.x + i;
        sid[tid] = id;
        sslot[tid] = slot;
        sbase[tid] = (int64_t)L.x * M + i;
        scap[tid] = L.y;
        ids_out[slot] = (int32_t)(id + id_base);
        corr_out[slot] = co[id];
    }
    __syncthreads();
    if (M % 4 == 0) {
        const int w = M / 4;
        for (int e = tid; e < nv * w; e += 256) {
            const int v = e / w, q = e - v * w;
            const uint32_t x = *(const uint32_t*)(pc + sid[v] * M + 4 * q);
            *(uint32_t*)(stage + v * ld + 4 * q) = x;
            if (rows) *(uint32_t*)(rows + sslot[v] * M + 4 * q) = x;
        }
    } else {
        for (int e = tid; e < nv * M; e += 256) {
            const int v = e / M, m = e - v * M;
            stage[v * ld + m] = pc[sid[v] * M + m];
        }
    }
    if (bpv % 16 == 0) {
        const int w = bpv / 16;
        for (int e = tid; e < nv * w; e += 256) {
            const int v = e / w, q = e - v * w;
            *(uint4*)(res_out + sslot[v] * bpv + 16 * q) = *(const uint4*)(rc + sid[v] * bpv + 16 * q);
        }
    } else {
        for (int e = tid; e < nv * bpv; e += 256) {
            const int v = e / bpv, q = e - v * bpv;
            res_out[sslot[v] * bpv + q] = rc[sid[v] * bpv + q];
        }
    }
    __syncthreads();
    const int v = tid % V;
    if (v < nv)
        for (int m = tid / V; m < M; m += 256 / V)
            codes_t[sbase[v] + (int64_t)m * scap[v]] = stage[v * ld + m];
}

// ---------------------------------------------------------------------------
// Lane-skewed copy of the primary codes, for the scan that runs each lane a
// fixed number of subspaces behind its neighbours.  Candidate i of a list
// (pool slot p = start + i) gets M bytes
//   row[t] = code[t - s]                 for t >= s = i mod 32,
//   row[t] = (code[M + t - s] + 1) mod 256 for t < s,
// so that at step t the lane holding i reads subspace t - s from row
// position t.  The tail bytes (t < s, read one period later, with the next
// candidate's head bytes) are raised by one LUT row: their LUT address
// (v + 1) * M + t - s is then the head bytes' formula, and code 255 wraps to
// the copy of row 255's last subspaces kept just below the LUT.
// The rows are stored in blocks of 16 slots (list starts and capacities are
// multiples of 16), piece by piece: the 16 bytes row[16q .. 16q+15] of slot p
// are at skew_piece(p, q) = ((p / 16) * (M / 16) + q) * 256 + (p mod 16) * 16,
// so the 64 lanes of a wave reading one piece of their candidates (four
// blocks of 16 consecutive slots) touch four 256-byte runs.
// Rows from[l] .. size-1 of list l are written (with the rest of the first
// block, whose rows are current anyway); one thread per piece, the codes read
// from the code-major blocks (codes_t[start * M + m * cap + i]).
// ---------------------------------------------------------------------------
__global__ void skew_codes_kernel(const int4* __restrict__ ldesc, const int32_t* __restrict__ from,
                                  const uint8_t* __restrict__ codes_t, int M,
                                  uint8_t* __restrict__ skew) {
    const int4 L = ldesc[blockIdx.x];
    const int q = threadIdx.x >> 4;
    if (q >= M / 16) return;
    // blocks of 16 slots; grid-y strides over the list's blocks
    for (int64_t i = (int64_t)(from[blockIdx.x] & ~15) + (int64_t)blockIdx.y * 16 + (threadIdx.x & 15);
         i < L.z; i += (int64_t)gridDim.y * 16) {
        const uint8_t* src = codes_t + (int64_t)L.x * M + i;
        const int s = (int)(i & 31);
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            w[k] = 0u;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                int m = 16 * q + 4 * k + e - s;
                // tail bytes (t < s) hold code + 1 (mod 256)
                const uint32_t inc = m < 0 ? 1u : 0u;
                if (m < 0) m += M;
                w[k] |= ((src[(int64_t)m * L.y] + inc) & 0xffu) << (8 * e);
            }
        }
        *(uint4*)(skew + skew_piece((int64_t)L.x + i, q, M)) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

int64_t skew_bytes(int64_t pool_cap, int M) { return (pool_cap + 15) / 16 * 16 * M; }

// Row-major copy of the primary codes: slot p's M bytes at rows[p * M], so
// that one vector's codes are one contiguous run (the pre-scan's re-check
// reads whole rows of a few candidates).  Rows from[l] .. size-1 of list l
// (from rounded down to 16); thread (16-byte piece q, slot i % 16).
__global__ void row_codes_kernel(const int4* __restrict__ ldesc, const int32_t* __restrict__ from,
                                 const uint8_t* __restrict__ codes_t, int M,
                                 uint8_t* __restrict__ rows) {
    const int4 L = ldesc[blockIdx.x];
    const int q = threadIdx.x >> 4;
    if (q >= M / 16) return;
    for (int64_t i = (int64_t)(from[blockIdx.x] & ~15) + (int64_t)blockIdx.y * 16 + (threadIdx.x & 15);
         i < L.z; i += (int64_t)gridDim.y * 16) {
        const uint8_t* src = codes_t + (int64_t)L.x * M + i;
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            w[k] = 0u;
#pragma unroll
            for (int e = 0; e < 4; e++)
                w[k] |= (uint32_t)src[(int64_t)(16 * q + 4 * k + e) * L.y] << (8 * e);
        }
        *(uint4*)(rows + ((int64_t)L.x + i) * M + 16 * q) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

hipError_t row_codes(const int4* ldesc, const int32_t* from, int nlist, int max_rows,
                     const uint8_t* codes_t, int M, uint8_t* rows, hipStream_t s) {
    if (nlist <= 0 || max_rows <= 0) return hipSuccess;
    const int64_t gy = std::min<int64_t>(((int64_t)max_rows + 15 + 15) / 16, 65535);
    if (M % 16 != 0 || M > 256) return hipErrorInvalidValue;
    hipLaunchKernelGGL(row_codes_kernel, dim3(nlist, (unsigned)gy), dim3(M), 0, s, ldesc, from,
                       codes_t, M, rows);
    return hipGetLastError();
}

hipError_t skew_codes(const int4* ldesc, const int32_t* from, int nlist, int max_rows,
                      const uint8_t* codes_t, int M, uint8_t* skew, hipStream_t s) {
    if (nlist <= 0 || max_rows <= 0) return hipSuccess;
    // one block of threads per 16 slots; from[l] is rounded down to 16
    // (a list of any length: the kernel strides over grid-y)
    const int64_t gy = std::min<int64_t>(((int64_t)max_rows + 15 + 15) / 16, 65535);
    if (M % 32 != 0 || M > 256) return hipErrorInvalidValue;
    hipLaunchKernelGGL(skew_codes_kernel, dim3(nlist, (unsigned)gy), dim3(M), 0, s, ldesc, from,
                       codes_t, M, skew);
    return hipGetLastError();
}

hipError_t scatter_lists(const int32_t* order, const int32_t* slist, const int32_t* sidx,
                         int64_t n, int64_t id_base, const int4* ldesc, const uint8_t* pc,
                         const uint8_t* rc, const float* co, int M, int bpv, int32_t* ids_out,
                         uint8_t* codes_t, uint8_t* res_out, float* corr_out, uint8_t* rows,
                         hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (rows && M % 4 != 0) return hipErrorInvalidValue;
    // 16 vectors a workgroup fill the chip for an append of a few thousand; 64
    // write whole 64-byte runs of a list when an add() brings it many
    auto go = [&](auto* k, int V) {
        hipLaunchKernelGGL(k, dim3((unsigned)((n + V - 1) / V)), dim3(256), (size_t)V * (M + 4), s,
                           order, slist, sidx, n, id_base, ldesc, pc, rc, co, M, bpv, ids_out, codes_t,
                           res_out, corr_out, rows);
    };
    if (n < 32768 || M > 512) go(scatter_kernel<16>, 16);
    else go(scatter_kernel<64>, 64);
    return hipGetLastError();
}

// Moves list blocks.  moves[2r] = {start, cap, size} of block r's source,
// moves[2r+1] = {start, cap} of its destination; the size candidates are
// copied and the code-major primary codes re-strided.  Source and
// destination blocks never overlap (destinations lie past every live block,
// or in another pool).
// List starts and capacities are multiples of 16, so every copied run (each
// code row of a block, its residual rows, corrections and ids, the row-major
// copy's rows) starts on 16 bytes and goes in 16-byte pieces, the last one over
// the block's padding; several workgroups share a block.  (Byte by byte with a
// division each, one workgroup per list, re-packing 730 K x 768 vectors took
// 40 ms.)
__global__ void __launch_bounds__(256)
relocate_kernel(const int4* __restrict__ moves, int M, int bpv, const uint8_t* __restrict__ codes_src,
                uint8_t* __restrict__ codes_dst, const uint8_t* __restrict__ res_src,
                uint8_t* __restrict__ res_dst, const float* __restrict__ corr_src,
                float* __restrict__ corr_dst, const int32_t* __restrict__ ids_src,
                int32_t* __restrict__ ids_dst, const uint8_t* __restrict__ rows_src,
                uint8_t* __restrict__ rows_dst) {
    const int4 fr = moves[blockIdx.x * 2];
    const int4 to = moves[blockIdx.x * 2 + 1];
    const int size = fr.z;
    if (size <= 0) return;
    const int t = blockIdx.y * 256 + threadIdx.x, T = gridDim.y * 256;
    const int w = (size + 15) / 16;  // 16-byte pieces of a code row
    const uint8_t* cs = codes_src + (int64_t)fr.x * M;
    uint8_t* cd = codes_dst + (int64_t)to.x * M;
    for (int m = t / w, q = t % w, dm = T / w, dq = T % w; m < M; m += dm, q += dq) {
        if (q >= w) {
            q -= w;
            if (++m >= M) break;
        }
        *(uint4*)(cd + (int64_t)m * to.y + 16 * q) = *(const uint4*)(cs + (int64_t)m * fr.y + 16 * q);
    }
    auto run = [&](const void* src, void* dst, int64_t bytes) {
        const uint4* a = (const uint4*)src;
        uint4* b = (uint4*)dst;
        for (int64_t e = t; e < (bytes + 15) / 16; e += T) b[e] = a[e];
    };
    run(res_src + (int64_t)fr.x * bpv, res_dst + (int64_t)to.x * bpv, (int64_t)size * bpv);
    run(corr_src + fr.x, corr_dst + to.x, (int64_t)size * 4);
    run(ids_src + fr.x, ids_dst + to.x, (int64_t)size * 4);
    if (rows_dst) run(rows_src + (int64_t)fr.x * M, rows_dst + (int64_t)to.x * M, (int64_t)size * M);
}

hipError_t relocate_lists(const int4* moves, int nmoves, int M, int bpv, const uint8_t* codes_src,
                          uint8_t* codes_dst, const uint8_t* res_src, uint8_t* res_dst,
                          const float* corr_src, float* corr_dst, const int32_t* ids_src,
                          int32_t* ids_dst, const uint8_t* rows_src, uint8_t* rows_dst,
                          hipStream_t s) {
    if (nmoves <= 0) return hipSuccess;
    const int gy = std::max(1, std::min(64, 4096 / nmoves));
    hipLaunchKernelGGL(relocate_kernel, dim3((unsigned)nmoves, (unsigned)gy), dim3(256), 0, s, moves, M,
                       bpv, codes_src, codes_dst, res_src, res_dst, corr_src, corr_dst, ids_src,
                       ids_dst, rows_src, rows_dst);
    return hipGetLastError();
}

}  // namespace jhq
