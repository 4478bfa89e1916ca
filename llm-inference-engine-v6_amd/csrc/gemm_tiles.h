// What the bfloat16 matrix kernels share: operand types, the modes of their outputs, the epilogues that go through LDS, loads from
// memory straight into LDS.
#pragma once

#include "common.h"

#include <type_traits>

namespace llme {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = static_cast<__bf16>(0.f);
    return z;
}

__device__ __forceinline__ bf16x8 load8(const bf16* p, bool ok) {
    return ok ? *reinterpret_cast<const bf16x8*>(p) : zero8();
}
// The same with the hint that the data is read once (the weights of a product with few rows).
__device__ __forceinline__ bf16x8 load8_once(const bf16* p, bool ok) {
    return ok ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p)) : zero8();
}

typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
// The fourth word of a buffer descriptor for raw 32-bit data on this chip.
constexpr int kBufferFlags = 0x00020000;

enum OutMode : int { kStoreF32 = 0, kAddF32 = 1, kStoreBF16 = 2, kAtomicF32 = 3, kGatedBF16 = 4, kRopeCache = 5,
                     kGatedReluBF16 = 6, kGatedGeluBF16 = 7, kGatedExtraBF16 = 8, kSquaredReluBF16 = 9 };
// Stored in bfloat16 one value a column: as it is, or the square of its positive part (kSquaredReluBF16).
constexpr bool is_stored_bf16(int mode) { return mode == kStoreBF16 || mode == kSquaredReluBF16; }
template <int MODE> __device__ __forceinline__ float stored_value(float v) {
    if (MODE != kSquaredReluBF16) return v;
    v = fmaxf(v, 0.f);
    return v * v;
}
// The gated outputs: act(gate) * up with act = SiLU (kGatedBF16), the rectifier (kGatedReluBF16) or the tanh form of
// GELU (kGatedGeluBF16); kGatedExtraBF16: SiLU or a clamped swish with biases on gate and up (GateExtra).
constexpr bool is_gated(int mode) {
    return mode == kGatedBF16 || mode == kGatedReluBF16 || mode == kGatedGeluBF16 || mode == kGatedExtraBF16;
}
template <int MODE> __device__ __forceinline__ float gate_act(float g) {
    if (MODE == kGatedReluBF16) return fmaxf(g, 0.f);
    if (MODE == kGatedGeluBF16) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
    return g / (1.0f + expf(-g));
}
// What kGatedExtraBF16 does around the activation. bias [N] in the order of w's rows (so in the order of the product's
// columns): added to gate and up first. limit > 0: gate <- min(gate, limit), up <- clamp(up, -limit, limit) and the
// value is gate sigmoid(alpha gate) (up + 1); otherwise silu(gate) up. pair_scale with row_pair: the gate and up sums of
// row m are multiplied by pair_scale[row_pair[m]] first (0 where row_pair[m] < 0), which is the layer run on that multiple
// of its input (an expert whose weight is on its input).
struct GateExtra {
    const bf16* bias = nullptr;
    float limit = 0.f, alpha = 1.f;
    const int* row_pair = nullptr;
    const float* pair_scale = nullptr;
};
__device__ __forceinline__ float gate_row_scale(const GateExtra& gx, int m) {
    if (gx.pair_scale == nullptr) return 1.f;
    const int pair = gx.row_pair[m];
    return pair < 0 ? 0.f : gx.pair_scale[pair];
}
// bg, bu: the biases of this gate and up value (zero where there are none).
template <int MODE> __device__ __forceinline__ float gated_value(float g, float u, const GateExtra& gx, float bg, float bu) {
    if (MODE != kGatedExtraBF16) return gate_act<MODE>(g) * u;
    g += bg;
    u += bu;
    if (gx.limit > 0.f) {
        g = fminf(g, gx.limit);
        u = fminf(fmaxf(u, -gx.limit), gx.limit);
        return g / (1.0f + expf(-gx.alpha * g)) * (u + 1.0f);
    }
    return g / (1.0f + expf(-g)) * u;
}

// Products in groups (the tile kernel's GROUPED instances): every row tile belongs to one group and is multiplied by that
// group's matrix, w + group * w_stride.
//  * tile_group given (experts): tile t holds rows t BM .. of `out`; its group is tile_group[t]; tiles from n_tiles[0] on do
//    not exist; row m of `a` is row_index[m] / gather_div where row_index is given (a negative entry: a row of zeros).
//  * otherwise (heads): every group has rows_per_group rows of `a` and `out`, one group after the other, in tiles_per_group
//    tiles.
struct Groups {
    const int* tile_group = nullptr;
    const int* n_tiles = nullptr;
    const int* row_index = nullptr;
    int gather_div = 1;
    int rows_per_group = 0, tiles_per_group = 1;
    int rows_out = 0;           // heads: `out` is [rows_per_group, groups * N], the groups' results side by side
    int n_groups = 1;
    long w_stride = 0;          // elements
    unsigned a_bytes = 0;       // of the whole of `a`, where rows are gathered
};

// Where the q/k/v projection's epilogue (kRopeCache) puts its result: the columns are the heads
// of q, then k, then v (hd columns each); q and k heads are rotated at the rows' positions (pairs
// (i, i + hd / 2), src/kernels.cpp:189-203), q goes to q_out [M, n_q hd], k and v into the rows'
// cache pages (k_cache [pages, n_kv, page, hd], v_cache [pages, n_kv, hd, page]), all bfloat16.
struct QkvTarget {
    const float* cos_t;         // [max_pos, hd / 2]
    const float* sin_t;
    const int* positions;       // [M]
    const int* seq_idx;         // [M] row of the block table
    const int* block_table;     // [n_seq, max_blocks]
    int max_blocks;
    bf16* q_out;
    bf16* k_cache;
    bf16* v_cache;
    int n_q, n_kv, hd, page;
};

// ----------------------------------------------------------------------------------------
// tile kernel: a workgroup of 2 x 2 wavefronts makes a (32 WMT) x (32 WNT) tile of the output,
// each wavefront WMT x WNT MFMA tiles of 16 x 16. Larger wavefront tiles read fewer LDS bytes
// per product (the 64 x 64 wavefront tile is bound by LDS reads); smaller tiles give more
// workgroups when the output is small.
constexpr int TK = 64;
constexpr int TSTRIDE = TK + 16;                     // elements; 160-byte rows measured fastest (144 had bank conflicts)

template <int WMT, int WNT>
constexpr int tile_lds_bytes() { return 2 * (32 * WMT + 32 * WNT) * TSTRIDE * 2; }   // A and W, two buffers

// Kinds of instruction for the compiler's scheduler, and a hint for it: the next COUNT matrix
// products with one instruction of KIND behind each.
constexpr int kMfma = 0x008, kVmemRead = 0x020, kDsRead = 0x100, kDsWrite = 0x200;
template <int KIND, int COUNT>
__device__ __forceinline__ void deal_between_products() {
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
        __builtin_amdgcn_sched_group_barrier(KIND, 1, 0);
    }
}

// The end of a tile kernel: the wavefronts' accumulators go to `out` in the kernel's mode. The
// result tile (i, j) of a lane is column wn + 16 j + r, rows wm + 16 i + 4 q + e: written straight
// from there, a store instruction touches 4 rows with 64 bytes each. Where the tile fits into the
// LDS that the operand slabs no longer need (LDS_BYTES of it; the caller has passed a barrier), it
// goes through LDS instead, so that every thread stores 16 contiguous bytes of a row.
// The values that an adding epilogue adds to, asked for before the tile's last products and the
// staging (a thread's pieces of four in the order in which the staged epilogue takes them): their
// trip from memory is over when the sums are staged. (Measured at 2,048 rows: the adding down-proj
// of the 1B sizes took 6 us more than the storing one, o-proj 2 us.)
template <int BM, int BN, int NT>
struct AddendsAhead {
    static constexpr int PER_ROW = BN / 4, COUNT = (BM * PER_ROW + NT - 1) / NT;
    float4 v[COUNT];
    __device__ __forceinline__ void load(const void* out, int M, int N, int m0, int n0, int tid) {
#pragma unroll
        for (int it = 0; it < COUNT; ++it) {
            const int idx = tid + it * NT;
            const int m = m0 + idx / PER_ROW, n = n0 + (idx % PER_ROW) * 4;
            const bool in = idx < BM * PER_ROW && m < M && n < N;
            // (N is a multiple of 8 here: a piece of four is in or out whole; out: a place that exists)
            v[it] = *reinterpret_cast<const float4*>(static_cast<const float*>(out) + (in ? static_cast<size_t>(m) * N + n : 0));
        }
    }
};

// A rotated pair (a, b) -> (a c - b s, b c + a s) with the product that is rounded first named: left to the compiler, which of the
// two it is differs from kernel to kernel, and with it the last bit of a row by the tile that made it.
__device__ __forceinline__ float rotated_first(float a, float b, float c, float s) { return __builtin_fmaf(a, c, -(b * s)); }
__device__ __forceinline__ float rotated_second(float a, float b, float c, float s) { return __builtin_fmaf(b, c, a * s); }

// Where row m0 + tid of the tile goes (rotating epilogue): its position and the page that holds it,
// looked up by thread tid while the products run (see the kernel).
struct RowPlace {
    int pos = 0, page = 0;
};

// A tile that lies in LDS in 32 bits (HB rows of BN columns, BN + 4 floats apart; its first row is mp, its first column n0) goes to
// `out` in the kernel's mode, 16 bytes a thread: what the NT threads of a workgroup do behind the barrier that ends the staging.
template <int HB, int BN, int NT, int MODE, bool AHEAD, typename ADDENDS>
__device__ __forceinline__ void store_staged(const float* stage, const int* row_pos, const int* row_page, void* __restrict__ out,
                                             int M, int N, int mp, int n0, int tid, const QkvTarget& qt, const ADDENDS& ahead,
                                             const GateExtra& gx, size_t ld16) {
    constexpr int SS = BN + 4;                           // floats per staged row
    if (MODE == kRopeCache) {
        // The tile holds whole heads (the entry point chose it so). q and k heads: a thread takes 8
        // dims of a head's first half and their partners in the second, of one row.
        const int hd = qt.hd, half = hd / 2, hv = half / 8, rotated = qt.n_q + qt.n_kv;
        const int per_row = (BN / hd) * hv;
        for (int idx = tid; idx < HB * per_row; idx += NT) {
            const int row = idx / per_row, e = idx % per_row;
            const int hh = e / hv, i = (e % hv) * 8;
            const int m = mp + row, head = n0 / hd + hh;
            if (m >= M || head >= rotated) continue;
            const float* sp = stage + row * SS + hh * hd + i;
            const int pos = row_pos[row];
            const float* cs = qt.cos_t + static_cast<size_t>(pos) * half + i;
            const float* sn = qt.sin_t + static_cast<size_t>(pos) * half + i;
            bf16x8 lo, hi;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                lo[j] = static_cast<__bf16>(rotated_first(sp[j], sp[half + j], cs[j], sn[j]));
                hi[j] = static_cast<__bf16>(rotated_second(sp[j], sp[half + j], cs[j], sn[j]));
            }
            bf16* dst;
            if (head < qt.n_q) {
                dst = qt.q_out + (static_cast<size_t>(m) * qt.n_q + head) * hd + i;
            } else {
                const int pg = row_page[row];
                dst = qt.k_cache + ((static_cast<size_t>(pg) * qt.n_kv + (head - qt.n_q)) * qt.page + pos % qt.page) * hd + i;
            }
            *reinterpret_cast<bf16x8*>(dst) = lo;
            *reinterpret_cast<bf16x8*>(dst + half) = hi;
        }
        // v heads: a thread takes one dim of 16 consecutive rows. Where these are 16 consecutive
        // positions of one request that begin at a multiple of 16 (the usual case in a prompt) they
        // lie together in the transposed page and go out as one piece; otherwise one by one.
        for (int idx = tid; idx < (HB / 16) * BN; idx += NT) {
            const int g16 = idx / BN, col = idx % BN;
            const int n = n0 + col, head = n / hd;
            const int mg = mp + g16 * 16;
            if (head < rotated || n >= N || mg >= M) continue;
            const int kvh = head - rotated, d = n % hd;
            const int nt = M - mg < 16 ? M - mg : 16;
            const float* sp = stage + (g16 * 16) * SS + col;
            // (a page belongs to one request: the same page and 15 positions further on is the same request)
            const int pos0 = row_pos[g16 * 16];
            const bool together = nt == 16 && row_page[g16 * 16] == row_page[g16 * 16 + 15] && pos0 % 16 == 0 &&
                                  qt.page % 16 == 0 && row_pos[g16 * 16 + 15] == pos0 + 15;
            if (together) {
                const int pg = row_page[g16 * 16];
                bf16* dst = qt.v_cache + ((static_cast<size_t>(pg) * qt.n_kv + kvh) * hd + d) * qt.page + pos0 % qt.page;
                bf16x8 lo, hi;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    lo[j] = static_cast<__bf16>(sp[j * SS]);
                    hi[j] = static_cast<__bf16>(sp[(j + 8) * SS]);
                }
                *reinterpret_cast<bf16x8*>(dst) = lo;
                *reinterpret_cast<bf16x8*>(dst + 8) = hi;
            } else {
                for (int j = 0; j < nt; ++j) {
                    const int pos = row_pos[g16 * 16 + j];
                    const int pg = row_page[g16 * 16 + j];
                    qt.v_cache[((static_cast<size_t>(pg) * qt.n_kv + kvh) * hd + d) * qt.page + pos % qt.page] =
                        static_cast<__bf16>(sp[j * SS]);
                }
            }
        }
    } else if (is_gated(MODE)) {
        // a thread makes 8 units: their gates and ups lie 16 columns apart in a group of 32
        constexpr int PER_ROW = BN / 16;             // 8-unit pieces per row
        for (int idx = tid; idx < HB * PER_ROW; idx += NT) {
            const int row = idx / PER_ROW, piece = idx % PER_ROW;
            const int col = (piece / 2) * 32 + (piece % 2) * 8;
            const int m = mp + row, n = n0 + col;
            if (m >= M || n >= N) continue;
            const float* gp = stage + row * SS + col;
            bf16x8 o, bgv = zero8(), buv = zero8();
            if (MODE == kGatedExtraBF16 && gx.bias != nullptr) {    // (a piece's gates are columns n .., its ups 16 on)
                bgv = *reinterpret_cast<const bf16x8*>(gx.bias + n);
                buv = *reinterpret_cast<const bf16x8*>(gx.bias + n + 16);
            }
            const float rs = MODE == kGatedExtraBF16 ? gate_row_scale(gx, m) : 1.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float gt = gp[e] * rs, up = gp[16 + e] * rs;
                o[e] = static_cast<__bf16>(gated_value<MODE>(gt, up, gx, static_cast<float>(bgv[e]), static_cast<float>(buv[e])));
            }
            const int unit = (n0 + (piece / 2) * 32) / 2 + (piece % 2) * 8;
            *reinterpret_cast<bf16x8*>(static_cast<bf16*>(out) + static_cast<size_t>(m) * (N / 2) + unit) = o;
        }
    } else if (is_stored_bf16(MODE)) {
        constexpr int PER_ROW = BN / 8;
        for (int idx = tid; idx < HB * PER_ROW; idx += NT) {
            const int row = idx / PER_ROW, col = (idx % PER_ROW) * 8;
            const int m = mp + row, n = n0 + col;
            if (m >= M || n >= N) continue;
            const float* sp = stage + row * SS + col;
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = static_cast<__bf16>(stored_value<MODE>(sp[e]));
            *reinterpret_cast<bf16x8*>(static_cast<bf16*>(out) + static_cast<size_t>(m) * ld16 + n) = o;
        }
    } else if constexpr (MODE == kAddF32 && AHEAD) {
        constexpr int PER_ROW = BN / 4;
#pragma unroll
        for (int it = 0; it < (HB * PER_ROW + NT - 1) / NT; ++it) {
            const int idx = tid + it * NT;
            const int row = idx / PER_ROW, col = (idx % PER_ROW) * 4;
            const int m = mp + row, n = n0 + col;
            if (idx >= HB * PER_ROW || m >= M || n >= N) continue;
            const float4 v = *reinterpret_cast<const float4*>(stage + row * SS + col);
            float4 cur = ahead.v[it];
            cur.x += v.x; cur.y += v.y; cur.z += v.z; cur.w += v.w;
            *reinterpret_cast<float4*>(static_cast<float*>(out) + static_cast<size_t>(m) * N + n) = cur;
        }
    } else {
        constexpr int PER_ROW = BN / 4;
        for (int idx = tid; idx < HB * PER_ROW; idx += NT) {
            const int row = idx / PER_ROW, col = (idx % PER_ROW) * 4;
            const int m = mp + row, n = n0 + col;
            if (m >= M || n >= N) continue;
            const float4 v = *reinterpret_cast<const float4*>(stage + row * SS + col);
            float* op = static_cast<float*>(out) + static_cast<size_t>(m) * N + n;
            if (MODE == kStoreF32) {
                *reinterpret_cast<float4*>(op) = v;
            } else if (MODE == kAddF32) {
                float4 cur = *reinterpret_cast<const float4*>(op);
                cur.x += v.x; cur.y += v.y; cur.z += v.z; cur.w += v.w;
                *reinterpret_cast<float4*>(op) = cur;
            } else {
                atomicAdd(op, v.x); atomicAdd(op + 1, v.y); atomicAdd(op + 2, v.z); atomicAdd(op + 3, v.w);
            }
        }
    }
}

template <int WMT, int WNT, int MODE, int LDS_BYTES, int WR = 2, int WC = 2, bool AHEAD = false>
__device__ __forceinline__ void tile_epilogue(f32x4 (&acc)[WMT][WNT], unsigned char* lds_raw, void* __restrict__ out,
                                              int M, int N, int m0, int n0, int wm, int wn, int tid, int r, int q,
                                              const QkvTarget& qt = QkvTarget{},
                                              const AddendsAhead<WR * 16 * WMT, WC * 16 * WNT, 64 * WR * WC>& ahead = {},
                                              const RowPlace& place = RowPlace{}, const GateExtra& gx = GateExtra{},
                                              int stored_ld = 0) {
    constexpr int BM = WR * 16 * WMT, BN = WC * 16 * WNT, NT = 64 * WR * WC;
    // (a result stored in bfloat16 may lie in rows further apart than its columns: heads side by side)
    const size_t ld16 = static_cast<size_t>(stored_ld > 0 ? stored_ld : N);

    constexpr int SS = BN + 4;                           // floats per staged row
    // A tile that is larger than the LDS goes through it in 2 or 4 passes of whole wavefront rows.
    constexpr int WAVE_ROWS = 16 * WMT;
    constexpr auto fits = [](int passes) {
        return (BM / passes) % WAVE_ROWS == 0 && static_cast<size_t>(BM / passes) * SS * 4 <= static_cast<size_t>(LDS_BYTES);
    };
    constexpr int PASSES = fits(1) ? 1 : (WR % 2 == 0 && fits(2)) ? 2 : (WR % 4 == 0 && fits(4)) ? 4 : 0;
    // (Atomic adds are faster scattered than packed into the same cache lines: they stay direct.)
    constexpr bool STAGED = MODE != kAtomicF32 && PASSES > 0;
    if (STAGED && N % 8 == 0) {
        constexpr int HB = PASSES > 0 ? BM / (PASSES > 0 ? PASSES : 1) : BM;     // rows of a pass
        float* stage = reinterpret_cast<float*>(lds_raw);
        // the rows' positions and pages, behind the stage: [BM] each (the rotating epilogue has one pass)
        int* row_pos = reinterpret_cast<int*>(lds_raw + static_cast<size_t>(HB) * SS * 4);
        int* row_page = row_pos + BM;
        if (MODE == kRopeCache) {
            static_assert(MODE != kRopeCache || (PASSES == 1 && static_cast<size_t>(BM) * SS * 4 + BM * 8 <= static_cast<size_t>(LDS_BYTES)),
                          "the rows' places fit behind the stage");
            if (tid < BM) {
                row_pos[tid] = place.pos;
                row_page[tid] = place.page;
            }
        }
#pragma unroll
        for (int pass = 0; pass < PASSES; ++pass) {
        if (pass > 0) __syncthreads();                  // the pass before has been stored
        if (wm / HB == pass) {
#pragma unroll
            for (int i = 0; i < WMT; ++i)
#pragma unroll
                for (int j = 0; j < WNT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        stage[(wm - pass * HB + i * 16 + q * 4 + e) * SS + wn + j * 16 + r] = acc[i][j][e];
        }
        __syncthreads();
        store_staged<HB, BN, NT, MODE, PASSES == 1 && AHEAD>(stage, row_pos, row_page, out, M, N, m0 + pass * HB, n0, tid, qt,
                                                             ahead, gx, ld16);
        }
        return;
    }
    if (MODE == kRopeCache) return;                     // (always staged: its columns are whole heads of 16 dims and more)
#pragma unroll
    for (int i = 0; i < WMT; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + wm + i * 16 + q * 4 + e;
            if (m >= M) continue;
            if (is_gated(MODE)) {
#pragma unroll
                for (int j = 0; j + 1 < WNT; j += 2) {
                    const int unit = (n0 + wn + j * 16) / 2 + r;        // tile column pair (gate, up)
                    if (2 * unit >= N) continue;
                    const float rs = MODE == kGatedExtraBF16 ? gate_row_scale(gx, m) : 1.f;
                    const float gt = acc[i][j][e] * rs, up = acc[i][j + 1][e] * rs;
                    float bg = 0.f, bu = 0.f;
                    if (MODE == kGatedExtraBF16 && gx.bias != nullptr) {
                        bg = static_cast<float>(gx.bias[n0 + wn + j * 16 + r]);
                        bu = static_cast<float>(gx.bias[n0 + wn + j * 16 + r + 16]);
                    }
                    static_cast<bf16*>(out)[static_cast<size_t>(m) * (N / 2) + unit] =
                        static_cast<bf16>(gated_value<MODE>(gt, up, gx, bg, bu));
                }
            } else {
#pragma unroll
                for (int j = 0; j < WNT; ++j) {
                    const int n = n0 + wn + j * 16 + r;
                    if (n >= N) continue;
                    const size_t idx = static_cast<size_t>(m) * N + n;
                    const float v = acc[i][j][e];
                    if (MODE == kStoreF32) static_cast<float*>(out)[idx] = v;
                    else if (MODE == kAddF32) static_cast<float*>(out)[idx] += v;
                    else if (MODE == kAtomicF32) atomicAdd(static_cast<float*>(out) + idx, v);
                    else static_cast<bf16*>(out)[static_cast<size_t>(m) * ld16 + n] = static_cast<bf16>(stored_value<MODE>(v));
                }
            }
        }
    }
}

// Waits until at most N of this wavefront's vector memory loads are still on their way.
template <int N> __device__ __forceinline__ void wait_vm() { __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14)); }

// A buffer descriptor for raw data, as four words (what __builtin_amdgcn_make_buffer_rsrc makes).
__device__ __forceinline__ u32x4 raw_descriptor(const void* base, unsigned bytes) {
    const unsigned long long p = reinterpret_cast<unsigned long long>(base);
    return u32x4{static_cast<unsigned>(p), static_cast<unsigned>(p >> 32) & 0xFFFFu, bytes, static_cast<unsigned>(kBufferFlags)};
}
// 16 bytes per lane from rsrc at voffset (per lane) + soffset (scalar), straight into LDS: lane l's
// bytes land at lds_base + 16 l (lds_base: the same in every lane, a byte address within LDS).
// Written as assembly because the compiler, which cannot tell which LDS reads such a load may
// alias, would wait for every load in flight in front of every LDS read.
__device__ __forceinline__ void load_b128_to_lds(u32x4 rsrc, unsigned lds_base, unsigned voffset, unsigned soffset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_base), "v"(voffset), "s"(rsrc), "s"(soffset)
                 : "memory", "m0");
}

// gemm_panel.hip: tiles of BM = 16 mt rows x bn columns, ksplit parts over k (kStoreF32 only, each a matrix of its own).
struct PanelPlan {
    int mt, bn, ksplit;
    int rounds;                 // of workgroups over the chip
    float us;                   // as estimated
};
PanelPlan panel_plan(int M, int N, int K, int ks_only, int heads, bool wide = false, bool pairs = false);
int gemm_panel_f32(int mt, int bn, int mode, const float* A, const float* W, float* out, int M, int N, int K, int ksplit, hipStream_t stream);
int gemm_panel(int mt, int bn, int mode, const bf16* A, const bf16* W, void* out, int M, int N, int K, int ksplit, const QkvTarget& qt,
               const GateExtra& gx, hipStream_t stream);

}  // namespace llme
