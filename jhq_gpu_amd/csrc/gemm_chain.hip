// gemm_chain.hip — fixed-order GEMM C = A * Bm^T on fp32 MFMA (gfx950).
//
// Every output is the fmaf chain acc = fmaf(A[i][k], Bm[j][k], acc) with k
// ascending from 0, the order the CPU restatement of the reference pins for
// the add/train rotation and the IVF assignment (cuBLAS Sgemm in
// v14/jhq_gpu_index.cu:209-225,367-393,444-448).  v_mfma_f32_32x32x2_f32 adds
// its two products one after the other, each with a single rounding and with
// subnormals kept: bit for bit fmaf(a1, b1, fmaf(a0, b0, c)).  So the chain
// runs on the matrix cores at twice the vector ALU's fused multiply-add rate,
// without packed ones (the vector kernel before it reached 43 TFLOP/s).
//
// Measured (rotation, n x d): 65536 x 1024 3199 -> 1054-1081 us (130 TFLOP/s of
// the 157 the unit has), 10000 x 768 310 -> 124-128 us, 2000 x 768 152 -> 34 us,
// 65536 x 128 64 -> 26 us.  The limit at long k is the MFMA issue; a short k
// (64 MFMAs per wave at d = 128) leaves the tile's loads and stores exposed.
#include "kernels.h"

#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>

namespace jhq {

typedef float v4f_c __attribute__((ext_vector_type(4)));
typedef float v16f_c __attribute__((ext_vector_type(16)));

enum { CHAIN_STORE = 0, CHAIN_ARGMIN = 1 };

// k per step, and the LDS row stride in floats: 16-byte reads of 16 rows
// (stride 36 = 9 quads, odd) start in 16 different quads of banks
constexpr int kChainBK = 32, kChainLd = kChainBK + 4;

__device__ __forceinline__ uint32_t chain_ord(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// One workgroup (4 waves, 2 x 2) per 64 T x 64 T tile of C; a wave holds T x T
// accumulators of 32 x 32.  Lane l of the instruction supplies row l % 32 at
// k = 2 step + l / 32, so a row's 8 consecutive k sit in LDS as its 4 even ones
// and then its 4 odd ones and each lane reads the operands of 4 steps with
// one 16-byte read.  The next k step's global loads are in flight while a
// step's 16 T^2 MFMAs (64 cycles each) run.  Rows past n and columns past m
// read the last valid row and are not stored; k past d is zero in both
// operands, which leaves the chain's value.  Workgroups go to the 8 XCDs in
// turn; the column tiles of a row tile take consecutive slots of one XCD, so
// its rows come from that XCD's L2 after the first.
// With ROWS, row i of A is A[rowidx[i]], i < min(n, *ndev) (the count read on the
// device), and the workgroups step over the tiles.
template <int T, int EPI, bool VEC, bool ROWS = false>
__global__ void __launch_bounds__(256, 2)
gemm_chain_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ Bm,
                  int64_t ldb, int64_t n, int m, int d, float* __restrict__ C, int64_t ldc,
                  const float* __restrict__ norms, unsigned long long* __restrict__ keys,
                  const int32_t* __restrict__ rowidx = nullptr,
                  const int32_t* __restrict__ ndev = nullptr) {
    constexpr int BT = 64 * T, L = BT * kChainBK / 4 / 256;  // float4 per thread and operand
    __shared__ __align__(16) float As[BT][kChainLd];
    __shared__ __align__(16) float Bs[BT][kChainLd];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int l32 = lane & 31, h = lane >> 5, wr = wv >> 1, wc = wv & 1;
    const int ncol = (m + BT - 1) / BT;
    if (ROWS) n = min(n, (int64_t)*ndev);
    // (without ROWS the grid covers the tiles: one pass)
    for (int64_t item = blockIdx.x;; item += gridDim.x) {
        const int64_t slot = item >> 3;
        const int64_t row0 = ((item & 7) + 8 * (slot / ncol)) * BT;
        const int col0 = (int)(slot % ncol) * BT;
        if (row0 >= n) {
            if (!ROWS || slot / ncol * 8 * BT >= n) return;
            continue;
        }
        if (ROWS) __syncthreads();  // the previous tile's reads are done

        // thread t stages 4 k from 4 (t % 8) of rows t / 8 + 32 i
        const int lk = 4 * (tid & 7), lr = tid >> 3;
        const float* ap[L];
        const float* bp[L];
#pragma unroll
        for (int i = 0; i < L; i++) {
            const int64_t row = min(row0 + lr + 32 * i, n - 1);
            ap[i] = A + (ROWS ? (int64_t)rowidx[row] : row) * lda;
            bp[i] = Bm + (int64_t)min(col0 + lr + 32 * i, m - 1) * ldb;
        }
        float4 ra[L], rb[L];
        // a whole k step: plain loads, no test behind them, so that they stay in
        // flight over the step before (a zero selected for k past d made the
        // compiler wait for each load: 102 TFLOP/s at 65536 x 1024 x 1024)
        auto load = [&](int k0) {
#pragma unroll
            for (int i = 0; i < L; i++) {
                const float* pa = ap[i] + k0 + lk;
                const float* pb = bp[i] + k0 + lk;
                if (VEC) {
                    ra[i] = *(const float4*)pa;
                    rb[i] = *(const float4*)pb;
                } else {
                    ra[i] = make_float4(pa[0], pa[1], pa[2], pa[3]);
                    rb[i] = make_float4(pb[0], pb[1], pb[2], pb[3]);
                }
            }
        };
        // the last step of d % 32 k
        auto load_tail = [&](int k0) {
            auto at = [&](const float* p, int k) { return k < d ? p[k] : 0.0f; };
            const int k = k0 + lk;
#pragma unroll
            for (int i = 0; i < L; i++) {
                ra[i] = make_float4(at(ap[i], k), at(ap[i], k + 1), at(ap[i], k + 2), at(ap[i], k + 3));
                rb[i] = make_float4(at(bp[i], k), at(bp[i], k + 1), at(bp[i], k + 2), at(bp[i], k + 3));
            }
        };
        // k of a block of 8: even ones at 0..3, odd ones at 4..7
        const int st = (lk & ~7) + (lk & 4) / 2;
        auto store = [&]() {
#pragma unroll
            for (int i = 0; i < L; i++) {
                // the pairs are put together here, not (with a wait) behind the loads
                asm volatile("" : "+v"(ra[i].x), "+v"(ra[i].y), "+v"(ra[i].z), "+v"(ra[i].w));
                asm volatile("" : "+v"(rb[i].x), "+v"(rb[i].y), "+v"(rb[i].z), "+v"(rb[i].w));
                *(float2*)&As[lr + 32 * i][st] = make_float2(ra[i].x, ra[i].z);
                *(float2*)&As[lr + 32 * i][st + 4] = make_float2(ra[i].y, ra[i].w);
                *(float2*)&Bs[lr + 32 * i][st] = make_float2(rb[i].x, rb[i].z);
                *(float2*)&Bs[lr + 32 * i][st + 4] = make_float2(rb[i].y, rb[i].w);
            }
        };

        v16f_c acc[T][T];
#pragma unroll
        for (int i = 0; i < T; i++)
#pragma unroll
            for (int j = 0; j < T; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

        auto step = [&]() {
#pragma unroll
            for (int kk = 0; kk < kChainBK; kk += 8) {
                v4f_c a[T], b[T];
#pragma unroll
                for (int i = 0; i < T; i++)
                    a[i] = *(const v4f_c*)&As[32 * (wr * T + i) + l32][kk + 4 * h];
#pragma unroll
                for (int j = 0; j < T; j++)
                    b[j] = *(const v4f_c*)&Bs[32 * (wc * T + j) + l32][kk + 4 * h];
#pragma unroll
                for (int s = 0; s < 4; s++)
#pragma unroll
                    for (int i = 0; i < T; i++)
#pragma unroll
                        for (int j = 0; j < T; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][s], b[j][s],
                                                                             acc[i][j], 0, 0, 0);
            }
        };
        const int dw = d / kChainBK * kChainBK;  // whole steps
        if (dw > 0) load(0);
        for (int k0 = 0; k0 < dw; k0 += kChainBK) {
            store();
            __syncthreads();
            // (the last pass loads its own step again)
            load(min(k0 + kChainBK, dw - kChainBK));
            __builtin_amdgcn_sched_barrier(0);  // the loads are issued before the MFMAs
            step();
            __syncthreads();
        }
        if (dw < d) {
            load_tail(dw);
            store();
            __syncthreads();
            step();
        }

        // register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
        auto row_of = [&](int i, int r) {
            return row0 + 32 * (wr * T + i) + 8 * (r / 4) + 4 * h + r % 4;
        };
#pragma unroll
        for (int i = 0; i < T; i++) {
            if constexpr (EPI == CHAIN_STORE) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int64_t row = row_of(i, r);
                    if (row < n) {
#pragma unroll
                        for (int j = 0; j < T; j++) {
                            const int col = col0 + 32 * (wc * T + j) + l32;
                            if (col < m) C[row * ldc + col] = acc[i][j][r];
                        }
                    }
                }
            } else {
                unsigned long long best[16];
#pragma unroll
                for (int r = 0; r < 16; r++) best[r] = ~0ull;
#pragma unroll
                for (int j = 0; j < T; j++) {
                    const int col = col0 + 32 * (wc * T + j) + l32;
                    if (col >= m) continue;
                    const float nc = norms[col];
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const float sc = fmaf(-2.0f, acc[i][j][r], nc);
                        const unsigned long long key =
                            ((unsigned long long)chain_ord(sc) << 32) | (uint32_t)col;
                        best[r] = key < best[r] ? key : best[r];
                    }
                }
                // minimum over the 32 columns of a lane half: each round a lane
                // keeps half of its rows and hands the others to its partner
                // (16 exchanges instead of 80)
#pragma unroll
                for (int c = 8; c >= 1; c >>= 1) {
                    const bool up = (l32 & (2 * c)) != 0;
#pragma unroll
                    for (int r = 0; r < c; r++) {
                        const unsigned long long keep = up ? best[r + c] : best[r];
                        const unsigned long long o = __shfl_xor(up ? best[r] : best[r + c], 2 * c);
                        best[r] = o < keep ? o : keep;
                    }
                }
                const unsigned long long o = __shfl_xor(best[0], 1);
                const unsigned long long key = o < best[0] ? o : best[0];
                const int64_t row = row_of(i, l32 >> 1);
                if (!(l32 & 1) && row < n && key != ~0ull) atomicMin(&keys[row], key);
            }
        }
        if (!ROWS) return;
    }
}

template <int T, int EPI>
static hipError_t launch_chain(const float* A, int64_t lda, const float* Bm, int64_t ldb, int64_t n,
                               int m, int d, float* C, int64_t ldc, const float* norms,
                               unsigned long long* keys, hipStream_t s) {
    constexpr int BT = 64 * T;
    const bool vec = d % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 && ((uintptr_t)A & 15) == 0 &&
                     ((uintptr_t)Bm & 15) == 0;
    const int64_t ncol = (m + BT - 1) / BT;
    // at most 2^22 workgroups a launch, whole groups of 8 row tiles
    const int64_t chunk = std::max<int64_t>(8, ((int64_t)1 << 22) / ncol / 8 * 8) * BT;
    for (int64_t r0 = 0; r0 < n; r0 += chunk) {
        const int64_t nr = std::min(n - r0, chunk);
        const int64_t rt = (nr + BT - 1) / BT;
        const dim3 grid((unsigned)((rt + 7) / 8 * 8 * ncol));
        auto* k = vec ? gemm_chain_kernel<T, EPI, true> : gemm_chain_kernel<T, EPI, false>;
        hipLaunchKernelGGL(k, grid, dim3(256), 0, s, A + r0 * lda, lda, Bm, ldb, nr, m, d,
                           C ? C + r0 * ldc : nullptr, ldc, norms, keys ? keys + r0 : nullptr,
                           (const int32_t*)nullptr, (const int32_t*)nullptr);
    }
    return hipGetLastError();
}

// 64 x 64 tiles where 128 x 128 ones would not give each of the 256 CUs two
// workgroups: 2000 x 768 has 96 of the large (a third of the chip, 41 us of MFMAs
// in each) and 384 of the small (34 us measured); from 512 on the large ones win
// by their fewer LDS reads per MFMA (64 x 64: 16 bytes per lane for 4, 128 x 128
// for 8).  The small ones down to one row (a kernel with 1 to 8 rows per thread on
// the vector ALU took, and these take, us: 1 x 1024 24.5 and 23.0, 64 x 1024 25.6
// and 23.8, 512 x 1024 108 and 24, 1 x 128 5.3 and 4.7, 64 x 128 5.7 and 5.1)
static bool chain_small(int64_t n, int m) {
    return ((n + 127) / 128) * ((m + 127) / 128) < 512;
}

hipError_t gemm_nt_store(const float* A, int64_t lda, const float* Bm, int64_t ldb, int64_t n,
                         int m, int d, float* C, int64_t ldc, hipStream_t s) {
    if (n <= 0 || m <= 0) return hipSuccess;
    return chain_small(n, m)
               ? launch_chain<1, CHAIN_STORE>(A, lda, Bm, ldb, n, m, d, C, ldc, nullptr, nullptr, s)
               : launch_chain<2, CHAIN_STORE>(A, lda, Bm, ldb, n, m, d, C, ldc, nullptr, nullptr, s);
}

hipError_t gemm_nt_argmin(const float* A, int64_t lda, const float* Bm, int64_t ldb, int64_t n,
                          int m, int d, const float* norms, unsigned long long* keys,
                          hipStream_t s) {
    if (n <= 0 || m <= 0) return hipSuccess;
    return chain_small(n, m)
               ? launch_chain<1, CHAIN_ARGMIN>(A, lda, Bm, ldb, n, m, d, nullptr, 0, norms, keys, s)
               : launch_chain<2, CHAIN_ARGMIN>(A, lda, Bm, ldb, n, m, d, nullptr, 0, norms, keys, s);
}

// The grid fills the chip for any count; with no row listed it ends at once.
hipError_t gemm_nt_argmin_rows(const float* A, int64_t lda, const int32_t* rowidx,
                               const int32_t* ndev, int64_t n_max, const float* Bm, int64_t ldb,
                               int m, int d, const float* norms, unsigned long long* keys,
                               hipStream_t s) {
    if (n_max <= 0 || m <= 0) return hipSuccess;
    const bool vec = d % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 && ((uintptr_t)A & 15) == 0 &&
                     ((uintptr_t)Bm & 15) == 0;
    auto* k = vec ? gemm_chain_kernel<1, CHAIN_ARGMIN, true, true>
                  : gemm_chain_kernel<1, CHAIN_ARGMIN, false, true>;
    const int64_t tiles = (n_max + 63) / 64 * ((m + 63) / 64);
    hipLaunchKernelGGL(k, dim3((unsigned)std::min<int64_t>((tiles + 7) / 8 * 8, 1024)), dim3(256), 0,
                       s, A, lda, Bm, ldb, n_max, m, d, (float*)nullptr, (int64_t)0, norms, keys,
                       rowidx, ndev);
    return hipGetLastError();
}

}  // namespace jhq
