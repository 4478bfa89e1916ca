// out[m, n] (+)= sum_k a[m, k] * w[n, k]     (src/kernels.cpp:33-57: W is [N, K] row-major)
//
// The plain-precision matrix product: every element is widened to 32-bit, multiplied
// and accumulated with 32-bit FMA, whatever the storage types. It is the whole
// matrix path of the 32-bit model and the fallback of the bfloat16 model for
// operand types or shapes that the MFMA kernels refuse. Any M, N, K. W may also come in the
// MFMA kernels' blocked layout ([N / 16][K / 32] blocks of [4][16][8]; N % 16 == 0, K % 32 == 0).
//
// Up to 16 rows (decoding) go to a kernel of their own that streams the weights once, and more rows of 32-bit
// operands to one on the matrix cores' 32-bit instruction (both further down). Tiling otherwise: a workgroup of 256
// threads makes a 64 x 64 tile of the output, 4 x 4 per thread, stepping through K in slabs of 16 staged in LDS (stored
// k-major so that the inner loop reads consecutive addresses).
#include "gemm_tiles.h"

#include <type_traits>

namespace llme {

constexpr int GB = 64;   // tile edge in m and n
constexpr int GK = 16;   // k slab

template <typename TA, typename TW, typename TO, bool ACC>
__global__ __launch_bounds__(256) void gemm_generic_kernel(const TA* __restrict__ a, const TW* __restrict__ w,
                                                           TO* __restrict__ out, int M, int N, int K, int blocked) {
    __shared__ float As[GK][GB + 4];
    __shared__ float Ws[GK][GB + 4];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * GB;
    const int n0 = blockIdx.x * GB;
    const int tx = tid % 16;      // n direction
    const int ty = tid / 16;      // m direction
    // loader mapping: 64 rows x 16 k per slab = 1024 elements, 4 per thread
    const int lrow = tid / 4;          // 0..63
    const int lk = (tid % 4) * 4;      // 0,4,8,12

    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += GK) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + lk + j;
            const int am = m0 + lrow;
            const int wn = n0 + lrow;
            As[lk + j][lrow] = (am < M && k < K) ? to_float(a[static_cast<size_t>(am) * K + k]) : 0.f;
            const size_t widx = blocked
                ? (static_cast<size_t>(wn / 16) * (K / 32) + k / 32) * 512 + ((k % 32) / 8 * 16 + wn % 16) * 8 + k % 8
                : static_cast<size_t>(wn) * K + k;
            Ws[lk + j][lrow] = (wn < N && k < K) ? to_float(w[widx]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GK; ++k) {
            float av[4], wv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = As[k][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) wv[j] = Ws[k][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            TO* o = out + static_cast<size_t>(m) * N + n;
            if (ACC) *o = from_float<TO>(to_float(*o) + acc[i][j]);
            else *o = from_float<TO>(acc[i][j]);
        }
    }
}

// The same product for up to 16 rows (decoding): nothing to tile, the weight matrix is streamed
// once. A wavefront takes GV_COLS output columns at a time; its lanes split k in groups of four
// (16- or 8-byte loads), each lane keeps a partial sum per row and column, and the lanes' sums are
// added at the end. The rows of a come from the cache (they are read once per GV_COLS columns).
// K a multiple of 4, a and w 16-byte aligned, w row-major.
constexpr int GV_COLS = 4;
constexpr int GV_MAX_ROWS = 16;

// KS wavefronts of a workgroup share the columns and take every KS-th piece of k; their sums meet in LDS, in one order.
// (An output of 2,048 columns is 512 wavefronts of whole columns, half of one per scheduler: two rows times the o-proj's and
// the down-proj's 32-bit weights of the 1B sizes, 16.8 and 67 MB, took 19.6 us on average so, and take 11.9 with k in four;
// q/k/v, 768 wavefronts, 11.7 and 8.5. At 4,096 wavefronts, gate/up, 134 MB take 28.7 us, the rate of memory, without.)
template <typename TA, typename TW, typename TO, bool ACC, int MR, int KS>
__global__ __launch_bounds__(256) void gemv_generic_kernel(const TA* __restrict__ a, const TW* __restrict__ w,
                                                           TO* __restrict__ out, int M, int N, int K) {
    __shared__ float part[KS > 1 ? KS : 1][MR * GV_COLS];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6, share = wave % KS;
    const int n0 = (blockIdx.x * (4 / KS) + wave / KS) * GV_COLS;
    if (n0 >= N) return;                                  // (whole wavefronts; with KS of 4 the whole workgroup)
    float acc[MR][GV_COLS];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int c = 0; c < GV_COLS; ++c) acc[m][c] = 0.f;
#pragma unroll 2
    for (int k = (share * 64 + lane) * 4; k < K; k += KS * 64 * 4) {
        float wv[GV_COLS][4];
#pragma unroll
        for (int c = 0; c < GV_COLS; ++c) {
            const int n = n0 + c < N ? n0 + c : N - 1;     // past the edge: the last column again, not stored
            if constexpr (std::is_same_v<TW, float>) {     // (read once)
                const f32x4 x = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w + static_cast<size_t>(n) * K + k));
#pragma unroll
                for (int i = 0; i < 4; ++i) wv[c][i] = x[i];
            } else {
                load4<TW>(w + static_cast<size_t>(n) * K + k, wv[c]);
            }
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float av[4];
            load4<TA>(a + static_cast<size_t>(m < M ? m : M - 1) * K + k, av);
#pragma unroll
            for (int c = 0; c < GV_COLS; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[m][c] = fmaf(av[i], wv[c][i], acc[m][c]);
        }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int c = 0; c < GV_COLS; ++c) {
            const float s = wave_sum(acc[m][c]);
            if (KS > 1) {
                if (lane == 0) part[share][m * GV_COLS + c] = s;
            } else if (lane == 0 && m < M && n0 + c < N) {
                TO* o = out + static_cast<size_t>(m) * N + n0 + c;
                *o = from_float<TO>(ACC ? to_float(*o) + s : s);
            }
        }
    if (KS == 1) return;
    __syncthreads();
    const int m = threadIdx.x / GV_COLS, c = threadIdx.x % GV_COLS;
    if (m >= MR || m >= M || n0 + c >= N) return;
    float s = part[0][threadIdx.x];
#pragma unroll
    for (int i = 1; i < KS; ++i) s += part[i][threadIdx.x];
    TO* o = out + static_cast<size_t>(m) * N + n0 + c;
    *o = from_float<TO>(ACC ? to_float(*o) + s : s);
}

// The same for 32-bit weights with the norm of the 32-bit rows in front of it, and (GATED) the SiLU gate behind it: a wavefront reads
// whole rows anyway (its share of k), so it adds up their squares beside its products with the norm's weight and scales its sums by
// 1 / rms at the end. GATED: gate and up rows of w alternate in groups of 16; a wavefront makes two units. What this saves is launches
// that wait for each other: nine norms of 4.4 us and four activations of 4.9 in a step of two rows through four layers of the 1B
// sizes and their head, which took 410 us.
template <typename TN, bool GATED, int MR, int KS>
__global__ __launch_bounds__(256) void gemv_norm_f32_kernel(const float* __restrict__ h, const int* __restrict__ rows,
                                                            const TN* __restrict__ norm, float eps, const float* __restrict__ w,
                                                            float* __restrict__ out, int M, int N, int K) {
    constexpr int COLS = GATED ? GV_COLS / 2 : GV_COLS, SUMS = MR * (GV_COLS + 1);
    __shared__ float part[4 / KS][KS][SUMS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, share = wave % KS, set = wave / KS;
    const int n0 = (blockIdx.x * (4 / KS) + set) * COLS;
    const float* wr[GV_COLS];
    const float* hr[MR];
#pragma unroll
    for (int c = 0; c < GV_COLS; ++c) {                    // past the edge: the last column again, not stored
        const int n = n0 + c % COLS < N ? n0 + c % COLS : N - 1;
        wr[c] = w + static_cast<size_t>(GATED ? n / 16 * 32 + n % 16 + c / COLS * 16 : n) * K;
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        const int r = m < M ? m : M - 1;
        hr[m] = h + static_cast<size_t>(rows ? rows[r] : r) * K;
    }
    float acc[MR][GV_COLS], ss[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        ss[m] = 0.f;
#pragma unroll
        for (int c = 0; c < GV_COLS; ++c) acc[m][c] = 0.f;
    }
#pragma unroll 2
    for (int k = (share * 64 + lane) * 4; k < K; k += KS * 64 * 4) {
        float wv[GV_COLS][4], nv[4];
#pragma unroll
        for (int c = 0; c < GV_COLS; ++c) {                // (read once)
            const f32x4 x = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(wr[c] + k));
#pragma unroll
            for (int i = 0; i < 4; ++i) wv[c][i] = x[i];
        }
        load4<TN>(norm + k, nv);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float v[4];
            load4<float>(hr[m] + k, v);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                ss[m] = fmaf(v[i], v[i], ss[m]);
                v[i] *= nv[i];
            }
#pragma unroll
            for (int c = 0; c < GV_COLS; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[m][c] = fmaf(v[i], wv[c][i], acc[m][c]);
        }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        const float s = wave_sum(ss[m]);
        if (lane == 0) part[set][share][m * (GV_COLS + 1) + GV_COLS] = s;
#pragma unroll
        for (int c = 0; c < GV_COLS; ++c) {
            const float p = wave_sum(acc[m][c]);
            if (lane == 0) part[set][share][m * (GV_COLS + 1) + c] = p;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < (4 / KS) * MR * COLS; i += 256) {
        const int of = i / (MR * COLS), m = i % (MR * COLS) / COLS, c = i % COLS, n = (blockIdx.x * (4 / KS) + of) * COLS + c;
        if (m >= M || n >= N) continue;
        const float* p = part[of][0] + m * (GV_COLS + 1);
        float sum = p[c], up = GATED ? p[c + COLS] : 0.f, sq = p[GV_COLS];
#pragma unroll
        for (int s = 1; s < KS; ++s) {
            sum += p[s * SUMS + c];
            if (GATED) up += p[s * SUMS + c + COLS];
            sq += p[s * SUMS + GV_COLS];
        }
        const float inv = 1.0f / sqrtf(sq / static_cast<float>(K) + eps);
        sum *= inv;
        if (GATED) sum = sum / (1.0f + expf(-sum)) * (up * inv);
        out[static_cast<size_t>(m) * N + n] = sum;
    }
}

template <typename TA, typename TW, typename TO>
static int launch_gemv_generic(const void* a, const void* w, void* out, int M, int N, int K, int accumulate,
                               hipStream_t stream) {
    const int waves = (N + GV_COLS - 1) / GV_COLS;
    // (k in four where whole columns are less than two wavefronts for each of a compute unit's four schedulers)
    const bool split = waves < 8 * compute_units() && K >= 1024;
    const dim3 grid(split ? waves : (waves + 3) / 4);
#define LLME_GEMV_KS(ACC, MR, KS)                                                                   \
    hipLaunchKernelGGL((gemv_generic_kernel<TA, TW, TO, ACC, MR, KS>), grid, dim3(256), 0, stream, \
                       static_cast<const TA*>(a), static_cast<const TW*>(w), static_cast<TO*>(out), M, N, K)
#define LLME_GEMV(ACC, MR)                                                                          \
    do {                                                                                            \
        if (split) LLME_GEMV_KS(ACC, MR, 4);                                                        \
        else LLME_GEMV_KS(ACC, MR, 1);                                                              \
    } while (0)
    // (rows in steps: the partial sums live in registers, 4 per row)
#define LLME_GEMV_ROWS(ACC)                                                                         \
    do {                                                                                            \
        if (M <= 1) LLME_GEMV(ACC, 1);                                                              \
        else if (M <= 2) LLME_GEMV(ACC, 2);                                                         \
        else if (M <= 4) LLME_GEMV(ACC, 4);                                                         \
        else if (M <= 8) LLME_GEMV(ACC, 8);                                                         \
        else LLME_GEMV(ACC, 16);                                                                    \
    } while (0)
    if (accumulate) LLME_GEMV_ROWS(true);
    else LLME_GEMV_ROWS(false);
#undef LLME_GEMV_ROWS
#undef LLME_GEMV
#undef LLME_GEMV_KS
    return launch_status();
}

// 32-bit operands, more than 16 rows, where launch_generic does not send them through LDS (gemm_panel.hip):
// v_mfma_f32_16x16x4_f32, whose products and sums are 32-bit like the vector unit's, at twice the rate of its single multiply-adds (32 against 16 a cycle and scheduler: 157 TFLOP/s). At that rate the operands
// need no LDS: a lane loads 8 consecutive k of a row (two loads of 16 bytes; the four lanes of a row take 128 bytes together), and step s of eight
// multiplies element s of every lane, which is k = 8 q + s for lane group q in both operands. A wavefront makes
// 16 WMT x 16 WNT of the output; KW wavefronts share an output and take every KW-th 32 of k, their sums meeting in LDS in one
// order (the same bits in every run). D blocks of 32 k are in flight per wavefront.
// Measured at 149 rows, the 1B sizes (before: the 64 x 64 tile kernel above on 96 to 768 workgroups, one load at a time):
// o-proj and down-proj 587 -> 69 us on average, q/k/v 236 -> 32, gate/up 398 -> 140 (71 TFLOP/s of its 10.0 GFLOP with
// 64 x 64 tiles; 159 with 32 x 64). The error against 64 bits is half the former's (2.4e-6 of the logits, 4.7e-6): more and shorter sums.

template <int WMT, int WNT, int WR, int WC, int KW, int D, bool ACC>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                       float* __restrict__ out, int M, int N, int K, int tiles_m) {
    static_assert(WR * WC * KW == 4, "four wavefronts");
    constexpr int BM = 16 * WMT * WR, BN = 16 * WNT * WC;
    __shared__ f32x4 part[KW > 1 ? KW * WMT * WNT * 64 : 1];
    int pid = blockIdx.x;                               // (a die gets consecutive tiles: they share a tile's rows of W)
    if (gridDim.x % 8 == 0) pid = (pid % 8) * (gridDim.x / 8) + pid / 8;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int kw = wave % KW, wr = wave / KW / WC, wc = wave / KW % WC;
    const int m0 = (pid % tiles_m) * BM + wr * 16 * WMT, n0 = (pid / tiles_m) * BN + wc * 16 * WNT;
    const float *ap[WMT], *wp[WNT];                     // (rows past an edge: the last one again, not stored)
#pragma unroll
    for (int i = 0; i < WMT; ++i) ap[i] = a + static_cast<size_t>(m0 + i * 16 + r < M ? m0 + i * 16 + r : M - 1) * K + q * 8;
#pragma unroll
    for (int j = 0; j < WNT; ++j) wp[j] = w + static_cast<size_t>(n0 + j * 16 + r < N ? n0 + j * 16 + r : N - 1) * K + q * 8;
    f32x4 acc[WMT][WNT];
#pragma unroll
    for (int i = 0; i < WMT; ++i)
#pragma unroll
        for (int j = 0; j < WNT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Block {
        f32x4 a[WMT][2], w[WNT][2];
    };
    const int whole = K / 32;                           // blocks of 32 k
    auto load = [&](int b) {
        Block x;
        const int k = (b < whole ? b : whole - 1) * 32; // (past the end: the last one again, not multiplied)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int i = 0; i < WMT; ++i) x.a[i][u] = *reinterpret_cast<const f32x4*>(ap[i] + k + u * 4);
#pragma unroll
            for (int j = 0; j < WNT; ++j) x.w[j][u] = *reinterpret_cast<const f32x4*>(wp[j] + k + u * 4);
        }
        return x;
    };
    auto multiply = [&](const Block& x) {
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int i = 0; i < WMT; ++i)
#pragma unroll
                for (int j = 0; j < WNT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.a[i][s / 4][s % 4], x.w[j][s / 4][s % 4], acc[i][j], 0, 0, 0);
    };
    if (kw < whole) {
        const int mine = (whole - kw + KW - 1) / KW;    // this wavefront's blocks
        Block x[D];
#pragma unroll
        for (int d = 0; d < D; ++d) x[d] = load(kw + d * KW);
        int at = 0;
        for (; at + D <= mine; at += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                multiply(x[d]);
                x[d] = load(kw + (at + D + d) * KW);
            }
        }
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (at + d < mine) multiply(x[d]);
    }
    if (K % 32 != 0 && kw == whole % KW) {              // what is left of k (a multiple of 4): zeros behind its end
        Block x;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const bool in = whole * 32 + q * 8 + u * 4 < K;
#pragma unroll
            for (int i = 0; i < WMT; ++i)
                x.a[i][u] = in ? *reinterpret_cast<const f32x4*>(ap[i] + whole * 32 + u * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < WNT; ++j)
                x.w[j][u] = in ? *reinterpret_cast<const f32x4*>(wp[j] + whole * 32 + u * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        multiply(x);
    }
    // column r, rows 4 q + e of every tile of 16 x 16
    auto store = [&](int i, int j, const f32x4& v) {
        const int n = n0 + j * 16 + r;
        if (n >= N) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + i * 16 + q * 4 + e;
            if (m >= M) continue;
            float* o = out + static_cast<size_t>(m) * N + n;
            *o = ACC ? *o + v[e] : v[e];
        }
    };
    if (KW == 1) {
#pragma unroll
        for (int i = 0; i < WMT; ++i)
#pragma unroll
            for (int j = 0; j < WNT; ++j) store(i, j, acc[i][j]);
        return;
    }
#pragma unroll
    for (int i = 0; i < WMT; ++i)
#pragma unroll
        for (int j = 0; j < WNT; ++j) part[(kw * WMT * WNT + i * WNT + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    for (int t = kw; t < WMT * WNT; t += KW) {          // (a wavefront adds up and stores every KW-th tile)
        f32x4 v = part[t * 64 + lane];
#pragma unroll
        for (int s = 1; s < KW; ++s) v += part[(s * WMT * WNT + t) * 64 + lane];
        store(t / WNT, t % WNT, v);
    }
}

template <bool ACC>
static int launch_gemm_f32(const float* a, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
    // The tile whose rounds of workgroups over the compute units take the least time: a round is the products of one of a
    // workgroup's wavefronts, over how well its loads are used (a 32 x 32 tile loads twice what a 64 x 64 one does per product).
    // Measured, outputs of 2,048 to 16,384 columns, 17 to 900 rows: with 1, 0.95, 0.9 and 0.8 the rule took smaller tiles in 25 of
    // 128 sizes, and 64 x 64 or 128 x 128 are up to 1.36 times as fast there (200 rows x 3,072 of k 2,048: 60 -> 45 us; 149 x
    // 16,384: 148 -> 133; 200 x 16,384: 206 -> 167) and never more than 4% slower (65 x 16,384: 87 -> 91).
    const int cus = compute_units();
    struct Shape { int bm, bn, products; float eff; };
    constexpr Shape shapes[4] = {{128, 128, 64, 1.0f}, {64, 64, 16, 1.0f}, {32, 64, 8, 0.75f}, {32, 32, 4, 0.65f}};
    int best = 0;
    float least = 0.f;
    for (int c = 0; c < 4; ++c) {
        const long tiles = static_cast<long>((M + shapes[c].bm - 1) / shapes[c].bm) * ((N + shapes[c].bn - 1) / shapes[c].bn);
        const float cost = static_cast<float>((tiles + cus - 1) / cus) * shapes[c].products / shapes[c].eff;
        if (c == 0 || cost < least) {
            least = cost;
            best = c;
        }
    }
    const int tiles_m = (M + shapes[best].bm - 1) / shapes[best].bm, tiles_n = (N + shapes[best].bn - 1) / shapes[best].bn;
    const dim3 grid(tiles_m * tiles_n), block(256);
    switch (best) {
        case 0: hipLaunchKernelGGL((gemm_f32_kernel<4, 4, 2, 2, 1, 2, ACC>), grid, block, 0, stream, a, w, out, M, N, K, tiles_m); break;
        case 1: hipLaunchKernelGGL((gemm_f32_kernel<4, 4, 1, 1, 4, 2, ACC>), grid, block, 0, stream, a, w, out, M, N, K, tiles_m); break;
        case 2: hipLaunchKernelGGL((gemm_f32_kernel<2, 4, 1, 1, 4, 3, ACC>), grid, block, 0, stream, a, w, out, M, N, K, tiles_m); break;
        default: hipLaunchKernelGGL((gemm_f32_kernel<2, 2, 1, 1, 4, 4, ACC>), grid, block, 0, stream, a, w, out, M, N, K, tiles_m); break;
    }
    return launch_status();
}

template <typename TA, typename TW, typename TO>
static int launch_generic(const void* a, const void* w, void* out, int M, int N, int K, int accumulate,
                          int blocked, hipStream_t stream) {
    if (M <= GV_MAX_ROWS && !blocked && K % 4 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(w) % 16 == 0)
        return launch_gemv_generic<TA, TW, TO>(a, w, out, M, N, K, accumulate, stream);
    if constexpr (std::is_same_v<TA, float> && std::is_same_v<TW, float> && std::is_same_v<TO, float>) {
        if (!blocked && K % 4 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0) {
            const float *fa = static_cast<const float*>(a), *fw = static_cast<const float*>(w);
            // Through LDS (gemm_panel.hip) where its pieces of four columns fit: operands straight from memory cost four times their
            // bytes in the loads' path, since the lanes of a quarter lie in four rows. Not where 32 x 32 tiles of few columns are one round
            // over the chip and wait for memory alone: there a ring of slabs only fills and drains. (Measured, us, straight / through LDS:
            // columns x k 64 x 2,048 at 17 rows 16.4 / 19.9, at 300 20.1 / 20.8; 2,048 x 2,048 at 17 rows 18.1 / 20.6, 97: 19.7 / 21.2,
            // 200: 28.0 / 21.8; 2,048 x 8,192 at 65 rows 64.6 / 72.8; 2,560 x 2,048 at 97 rows, 320 tiles, 28.1 / 21.2; 3,072 x 2,048 at 32
            // rows 21.9 / 21.2, 65: 29.7 / 21.8; 6,144 x 4,096 at 32 rows 42.1 / 38.6; 16,384 x 2,048 at 149 rows 137 / 87.)
            const bool one_round = N < 3072 && static_cast<long>((M + 31) / 32) * ((N + 31) / 32) <= compute_units();
            if (!one_round && N % 4 == 0 && K < (1 << 22) && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
                const PanelPlan plan = panel_plan(M, N, K, 1, 0, true);
                return gemm_panel_f32(plan.mt, plan.bn, accumulate ? kAddF32 : kStoreF32, fa, fw, static_cast<float*>(out), M, N, K, 1, stream);
            }
            return accumulate ? launch_gemm_f32<true>(fa, fw, static_cast<float*>(out), M, N, K, stream)
                              : launch_gemm_f32<false>(fa, fw, static_cast<float*>(out), M, N, K, stream);
        }
    }
    const dim3 grid((N + GB - 1) / GB, (M + GB - 1) / GB);
    if (accumulate)
        hipLaunchKernelGGL((gemm_generic_kernel<TA, TW, TO, true>), grid, dim3(256), 0, stream,
                           static_cast<const TA*>(a), static_cast<const TW*>(w), static_cast<TO*>(out), M, N, K, blocked);
    else
        hipLaunchKernelGGL((gemm_generic_kernel<TA, TW, TO, false>), grid, dim3(256), 0, stream,
                           static_cast<const TA*>(a), static_cast<const TW*>(w), static_cast<TO*>(out), M, N, K, blocked);
    return launch_status();
}

}  // namespace llme

using namespace llme;

// a [M, K], w [N, K], out [M, N]; each of f32 or bf16; accumulate adds into out.
extern "C" int llme_gemm_generic(const void* a, int a_dtype, const void* w, int w_dtype, void* out,
                                 int out_dtype, int M, int N, int K, int accumulate, int blocked,
                                 hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return kErrBadArgument;
    if (blocked && (N % 16 != 0 || K % 32 != 0)) return kErrUnsupported;
    const int key = a_dtype * 4 + w_dtype * 2 + out_dtype;
    switch (key) {
        case 0: return launch_generic<float, float, float>(a, w, out, M, N, K, accumulate, blocked, stream);
        case 1: return launch_generic<float, float, bf16>(a, w, out, M, N, K, accumulate, blocked, stream);
        case 2: return launch_generic<float, bf16, float>(a, w, out, M, N, K, accumulate, blocked, stream);
        case 3: return launch_generic<float, bf16, bf16>(a, w, out, M, N, K, accumulate, blocked, stream);
        case 4: return launch_generic<bf16, float, float>(a, w, out, M, N, K, accumulate, blocked, stream);
        case 5: return launch_generic<bf16, float, bf16>(a, w, out, M, N, K, accumulate, blocked, stream);
        case 6: return launch_generic<bf16, bf16, float>(a, w, out, M, N, K, accumulate, blocked, stream);
        case 7: return launch_generic<bf16, bf16, bf16>(a, w, out, M, N, K, accumulate, blocked, stream);
        default: return kErrBadArgument;
    }
}

// out [M, N] = (rows of h, normed) w^T, all 32-bit (the norm's weight 32-bit or bfloat16), M up to 16; gated: w [2 N, K] holds gate and up
// rows alternating in groups of 16 and out is silu(gate) up. K a multiple of 4, h, w and the norm's weight 16-byte aligned.
extern "C" int llme_gemv_norm_f32(const float* h, const int* rows, const void* norm, int norm_dtype, float eps, const float* w, float* out,
                                  int M, int N, int K, int gated, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % 4 != 0 || M > GV_MAX_ROWS || (gated && N % 16 != 0) || reinterpret_cast<uintptr_t>(h) % 16 != 0 ||
        reinterpret_cast<uintptr_t>(w) % 16 != 0 || reinterpret_cast<uintptr_t>(norm) % 16 != 0)
        return kErrUnsupported;
    const int cols = gated ? GV_COLS / 2 : GV_COLS, waves = (N + cols - 1) / cols;
    const bool split = waves < 8 * compute_units() && K >= 1024;        // (as gemv_generic)
    const dim3 grid(split ? waves : (waves + 3) / 4);
#define LLME_GNF(TN, GATED, MR)                                                                                                      \
    do {                                                                                                                             \
        if (split)                                                                                                                   \
            hipLaunchKernelGGL((gemv_norm_f32_kernel<TN, GATED, MR, 4>), grid, dim3(256), 0, stream, h, rows,                        \
                               static_cast<const TN*>(norm), eps, w, out, M, N, K);                                                  \
        else                                                                                                                         \
            hipLaunchKernelGGL((gemv_norm_f32_kernel<TN, GATED, MR, 1>), grid, dim3(256), 0, stream, h, rows,                        \
                               static_cast<const TN*>(norm), eps, w, out, M, N, K);                                                  \
    } while (0)
#define LLME_GNF_ROWS(TN, GATED)                  \
    do {                                          \
        if (M <= 1) LLME_GNF(TN, GATED, 1);       \
        else if (M <= 2) LLME_GNF(TN, GATED, 2);  \
        else if (M <= 4) LLME_GNF(TN, GATED, 4);  \
        else if (M <= 8) LLME_GNF(TN, GATED, 8);  \
        else LLME_GNF(TN, GATED, 16);             \
    } while (0)
    if (norm_dtype == kF32 && gated) LLME_GNF_ROWS(float, true);
    else if (norm_dtype == kF32) LLME_GNF_ROWS(float, false);
    else if (norm_dtype == kBF16 && gated) LLME_GNF_ROWS(bf16, true);
    else if (norm_dtype == kBF16) LLME_GNF_ROWS(bf16, false);
    else return kErrBadArgument;
#undef LLME_GNF_ROWS
#undef LLME_GNF
    return launch_status();
}

LLME_LOAD_ENTRY(gemm_generic)
