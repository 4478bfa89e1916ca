// out[m, n] (+)= sum_k a[m, k] * w[n, k] for a few dozen to some thousand rows: bfloat16 with a blocked W, or 32-bit with a row-major W.
//
// Between the kernels that stream W for up to 16 rows and the tiles of 256 x 256 for prompts lie products whose rows are one or two
// tiles high, and outputs of few columns. Tiles through staging registers (gemm_tile_kernel) read 2.6 times the bytes there that
// they must (273 rows x 16,384 columns in tiles of 96 x 64: 503 MB over the chip), and a compute unit gets 55 to 90 bytes a ns.
// So the tile takes its height from the rows (BM = 16 MT, up to 192) x BN = 64 or 128 columns (bfloat16: 192 and 256 too), one workgroup of
// eight wavefronts a compute unit, with as many bytes on their way as LDS holds:
//  * BN / 32 wavefronts share out the columns (32 each; of a tile of 192 or 256 four wavefronts 48 or 64 each). bfloat16: the KS wavefronts of a group of columns (256 / BN;
//    two with 192 and 256) share out its rows of tiles, and each adds up all of k in turn, so that a sum has the one order that every other tile kernel gives it: whichever tile
//    a product's rows are given, its results are the same bits. (Sharing out k instead, with the parts joined through LDS at
//    the end, reads a fifth less of LDS and was no faster: parts of the 1B o-proj at 273 rows 8.2 / 8.0 us, of its down-proj 17.6 / 16.5,
//    of the 8B down-proj at 528 rows 69.9 / 70.0, and with other orders of sums a prompt's bfloat16 logits moved by their rounding
//    with the number of its rows. Wavefronts of 64 columns by a quarter of the rows: 0 to 2 % slower.) 32-bit: the wavefronts share out the
//    steps of k, which is even for any number of rows; there the products take the time.
//  * a slab is A's BM rows and W's BN columns of KS steps of k (64 bytes a row each), all straight from memory into LDS.
//  * NS slabs lie in LDS as a ring, all but the one that is read and the one that is multiplied on their way.
// A slab's operands are in registers when its turn starts. The turn waits for the slab behind it, meets the barrier, and, step of k
// by step of k and row of tiles by row of tiles, multiplies, reads the next slab's operand into the same registers and asks for a share of the slab NS - 1
// ahead, into the buffer of the slab before, which everybody has multiplied. A wavefront passes the barrier with LDS reads on their
// way: the buffer that they read is asked for again only behind the next one.
// LDS holds A's chunks (8 rows x 64 k, lane 8 r + p: piece p ^ r of row r) and W's blocks as the kernel of 256 x 256 tiles does. In the
// order of the operand, neighbouring lanes in neighbouring rows, a load of A took four times as long and a slab of 160 + 128 rows
// 0.62 us instead of 0.38; half the wavefronts asking for A and half for W lost 15 % (a wavefront can only ask so fast).
// Measured (us, weights from memory, tiles through registers / these): gate/up of the 1B sizes at 150 rows 22.1 / 20.2, 273:
// 34.5 / 25.5, 528: 51.3 / 46.5; of the 8B sizes at 150 rows 63.9 / 49.3; sums: 1B down-proj at 2,048 rows 84.4 / 73.8, 2,995 rows of
// k = 12,288 209 / 129; in parts (see below) against atomics at 96 rows 14.3 / 10.7, at 273 25.8 / 16.5.
#include "gemm_tiles.h"

namespace llme {

// CG x KS wavefronts; a slab is KS steps of 64 bytes of k. bfloat16: W in blocks, the wavefronts of a column group share out the rows (ROWS).
// 32-bit: W row-major, its chunks loaded and read as A's, and they share out the steps of k.
template <typename T, int MT, int CG, int KS, int WT = 2, bool HALF = false>
struct PanelSizes {
    static constexpr bool BLOCKED = sizeof(T) == 2, ROWS = BLOCKED;
    static constexpr int WNT = WT;                              // tiles of 16 columns a wavefront (HALF: slabs of 32 k)
    static constexpr int NW = CG * KS, BM = 16 * MT, BN = 16 * WNT * CG, SK = HALF ? 32 : 32 * KS;
    static constexpr int A_STAGE = BM * SK * 2, W_STAGE = BN * SK * 2, STAGE = A_STAGE + W_STAGE;
    static constexpr int NS_MOST = 160 * 1024 / STAGE, NS = NS_MOST > 6 ? 6 : NS_MOST;
    static constexpr int JOIN_MOST = 160 / (NW * WNT), JOIN_ROWS = MT < JOIN_MOST ? MT : JOIN_MOST;   // rows of tiles that join at a time
    static constexpr int JOIN = ROWS ? 0 : NW * JOIN_ROWS * WNT * 1024, TURNED = BM * (BN + 4) * 4 + BM * 8;
    static constexpr int LDS = NS * STAGE > JOIN ? NS * STAGE : JOIN;
    static constexpr bool TURNS = TURNED <= 160 * 1024;         // the rotating epilogue's tile and its rows' places fit
    static_assert(NS >= 3 && LDS <= 160 * 1024, "LDS");
};

// A lane's 16 bytes of an operand: 8 bfloat16 of k 8 q .., or 4 floats of k 4 q .., of which the s-th of every lane makes the k of
// the s-th of four products (the same k in both operands).
template <typename T> struct PanelOperand;
template <> struct PanelOperand<bf16> {
    using Type = bf16x8;
    static __device__ __forceinline__ void multiply(const Type& w, const Type& a, f32x4& acc) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, acc, 0, 0, 0);
    }
};
template <> struct PanelOperand<float> {
    using Type = f32x4;
    static __device__ __forceinline__ void multiply(const Type& w, const Type& a, f32x4& acc) {
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], a[s], acc, 0, 0, 0);
    }
};

template <typename T, int MT, int CG, int KS, int WT, bool HALF, int MODE>
__global__ __launch_bounds__(64 * CG * KS, 1) void gemm_panel_kernel(const T* __restrict__ a, const T* __restrict__ w,
                                                            void* __restrict__ out, int M, int N, int K, int tiles_m, int tiles_n,
                                                            int ksplit, QkvTarget qt, GateExtra gx) {
    using S = PanelSizes<T, MT, CG, KS, WT, HALF>;
    constexpr int NW = S::NW, WNT = S::WNT, BM = S::BM, BN = S::BN, NS = S::NS;
    constexpr bool BLOCKED = S::BLOCKED, ROWS = S::ROWS;
    // a wavefront multiplies KW of a slab's steps of k with MTW rows of tiles, of which place i is row i RG + part (ROWS) or i
    constexpr int KW = ROWS && !HALF ? KS : 1, RG = ROWS ? KS : 1, MTW = (MT + RG - 1) / RG;
    constexpr int SLAB = HALF ? 64 : 64 * KS;                   // bytes of a row in a slab
    using Operand = typename PanelOperand<T>::Type;
    constexpr int ROWS8 = BM / 8, CHUNKS = ROWS8 * (KS / 2);    // of A's slab: 8 rows x 64 k each
    constexpr int JOBS = HALF ? MT + BN / 16 : CHUNKS;          // (a slab of 32 k: all its loads in one row, A's chunks of 16 rows x 32 k first)
    constexpr int LA = JOBS / NW, REST = JOBS % NW, LW = HALF ? 0 : WNT;  // a wavefront's: LA, the first REST wavefronts one more
    extern __shared__ __align__(16) unsigned char lds_raw[];

    // A die gets consecutive tiles, rows fastest (up to 8 tiles of them), so that tiles which read the same W share its L2.
    const int total = tiles_m * tiles_n * ksplit;
    const int die = blockIdx.x % 8, per_die = total / 8, more = total % 8;
    const int place_in = die * per_die + (die < more ? die : more) + blockIdx.x / 8;
    const int split = place_in / (tiles_m * tiles_n), pid = place_in % (tiles_m * tiles_n);
    constexpr int GROUP = 8;
    const int g = pid / (GROUP * tiles_n), first_m = g * GROUP;
    const int gsize = tiles_m - first_m < GROUP ? tiles_m - first_m : GROUP;
    const int m0 = (first_m + pid % (GROUP * tiles_n) % gsize) * BM, n0 = pid % (GROUP * tiles_n) / gsize * BN;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int cg = wave % CG, part = wave / CG;

    // this workgroup's share of k, in slabs
    const unsigned row = static_cast<unsigned>(K) * sizeof(T);  // bytes
    const int ns_all = static_cast<int>((row + SLAB - 1) / SLAB), ns_per = (ns_all + ksplit - 1) / ksplit;
    const int s_begin = split * ns_per, s_end = s_begin + ns_per < ns_all ? s_begin + ns_per : ns_all;

    const int a_rows = M - m0 < BM ? M - m0 : BM, w_rows = N - n0 < BN ? N - n0 : BN;
    const u32x4 a_rsrc = raw_descriptor(a + static_cast<size_t>(m0) * K, a_rows * row);
    const u32x4 w_rsrc = raw_descriptor(w + static_cast<size_t>(n0) * K, w_rows * row);
    const unsigned lds_origin = static_cast<unsigned>(reinterpret_cast<size_t>(
        (__attribute__((address_space(3))) unsigned char*)lds_raw));
    constexpr unsigned kNowhere = 0xFFFFFF00u;                  // behind every descriptor's end: zeros, without a fetch
    const unsigned last_at = (ns_all - 1) * SLAB;               // (k may end in the last slab: 16 bytes of a row are in or out whole)
    // A's chunk j: rows 8 (j % ROWS8) .., bytes 128 (j / ROWS8) .. of the slab; lane 8 r' + p: row r', piece p ^ r' of its 128 bytes
    unsigned a_off[LA + 1], a_last[LA + 1], w_off[WNT], w_last[WNT];
    auto place_chunk = [&](int j, int rows8, unsigned& off, unsigned& last) {
        const unsigned at = j / rows8 * 128 + ((lane & 7) ^ (lane >> 3)) * 16;
        off = (j % rows8 * 8 + (lane >> 3)) * row + at;
        last = last_at + at < row ? off : kNowhere;
    };
#pragma unroll
    for (int i = 0; i <= LA; ++i) place_chunk(wave + NW * i, ROWS8, a_off[i], a_last[i]);
#pragma unroll
    for (int j = 0; j < WNT; ++j) {
        if (BLOCKED) {
            w_off[j] = (static_cast<unsigned>(cg * WNT + j) * (K / 32) + part) * 1024u + lane * 16u;
            w_last[j] = last_at + part * 64 < row ? w_off[j] : kNowhere;
        } else {
            place_chunk(wave + NW * j, BN / 8, w_off[j], w_last[j]);
        }
    }
    u32x4 job_rsrc[LA + 1];                                     // HALF: where job wave + NW t reads, and how far a slab is
    unsigned job_step[LA + 1];
    if constexpr (HALF) {
#pragma unroll
        for (int t = 0; t <= LA; ++t) {
            const int j = wave + NW * t;
            const bool of_a = j < MT;
            job_rsrc[t] = of_a ? a_rsrc : w_rsrc;
            job_step[t] = of_a ? SLAB : 1024;
            // A's chunk j: rows 16 j .., lane 4 r + p: row r, piece p ^ (r / 4's place in 0 2 3 1) of its 64 bytes
            a_off[t] = of_a ? (j * 16 + (lane >> 2)) * row + (((lane & 3) ^ ((0x78 >> (lane >> 4) * 2) & 3)) * 16)
                            : static_cast<unsigned>(j - MT) * (K / 32) * 1024u + lane * 16u;
        }
    }
    const bool one_more = wave < REST;
    auto ask = [&](int s, int stage, int t) {                   // load t of slab s: W's blocks of this wavefront, then A's chunks
        // (past the share's end nothing is fetched: the offset of no lane is inside, and the scalar one is 0, since a descriptor's end less
        // a scalar offset that lies behind it, which is what a lane's offset is held against, would wrap around)
        const bool past = s >= s_end, last = s == ns_all - 1;
        const unsigned to = lds_origin + stage * S::STAGE, slab = past ? 0 : s;
        if constexpr (HALF) {
            if (t < LA || one_more) load_b128_to_lds(job_rsrc[t], to + (wave + NW * t) * 1024, past ? kNowhere : a_off[t], slab * job_step[t]);
        } else if (t < WNT) {
            load_b128_to_lds(w_rsrc, to + S::A_STAGE + (BLOCKED ? wave * WNT + t : wave + NW * t) * 1024,
                             past ? kNowhere : last ? w_last[t] : w_off[t], slab * (BLOCKED ? KS * 1024 : SLAB));
        } else if (t < LA + WNT || one_more) {
            const int i = t - WNT;
            load_b128_to_lds(a_rsrc, to + (wave + NW * i) * 1024, past ? kNowhere : last ? a_last[i] : a_off[i], slab * SLAB);
        }
    };
    constexpr int LOADS = LA + LW + (REST > 0 ? 1 : 0);
    // at most `slabs` slabs of this wavefront's loads still on their way
    auto wait_slabs = [&](auto slabs) {
        constexpr int n = decltype(slabs)::value;
        static_assert(n * (LA + LW + 1) < 64, "the count of loads in flight has six bits");
        if (REST > 0 && one_more) wait_vm<n * (LA + LW + 1)>();
        else wait_vm<n * (LA + LW)>();
    };
    // The barrier of a turn: what a wavefront's LDS reads wait for is its own business (see below), the compiler keeps its order.
    auto meet = [&] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    auto mine = [&](int i) { return MT % RG == 0 || i < MTW - 1 || i * RG + part < MT; };   // (the same in a whole wavefront)
    f32x4 acc[MTW][WNT];
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int j = 0; j < WNT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    if (s_begin < s_end) {
#pragma unroll
        for (int d = 0; d < NS - 1; ++d)
#pragma unroll
            for (int t = 0; t < LOADS; ++t) ask(s_begin + d, d, t);
        // this lane's place in an operand of A: chunk 2 g + r / 8 of column k / 64, row r % 8 of it, piece 4 (k / 32 % 2) + q
        const unsigned in_chunk = (r >> 3) * 1024 + (r & 7) * 128 + ((((ROWS ? 0 : part & 1) * 4 + q) ^ (r & 7)) * 16);
        const unsigned a_first = in_chunk + (ROWS ? part * 2048 : (part >> 1) * (ROWS8 * 1024)), a_lane[2] = {a_first, a_first ^ 64};
        const unsigned half_lane = part * 1024 + r * 64 + (q ^ ((0x78 >> (r >> 2) * 2) & 3)) * 16;
        const unsigned w_lane = S::A_STAGE + (BLOCKED ? (ROWS ? cg : wave) * (WNT * 1024) + lane * 16
                                                      : in_chunk + ((part >> 1) * (BN / 8) + cg * (2 * WNT)) * 1024);
        auto read_a = [&](int stage, int k, int i) {
            if constexpr (HALF) return *reinterpret_cast<const Operand*>(lds_raw + stage * S::STAGE + half_lane + i * (RG * 1024));
            else
            return *reinterpret_cast<const Operand*>(lds_raw + stage * S::STAGE + a_lane[k & 1] + (k >> 1) * (ROWS8 * 1024) + i * (RG * 2048));
        };
        auto read_w = [&](int stage, int k, int j) {
            return *reinterpret_cast<const Operand*>(lds_raw + stage * S::STAGE + w_lane + k * (CG * WNT * 1024) + j * (BLOCKED ? 1024 : 2048));
        };
        wait_slabs(std::integral_constant<int, NS - 2>{});
        meet();
        // (read in the order in which a turn reads: the compiler's waits for LDS then hold on both ways into the loop)
        Operand fa[KW][MTW], fw0[KW][WNT], fw1[KW][WNT];
        auto read_row = [&](int stage, int k, int i, Operand (&into)[KW][WNT]) {
            if (mine(i)) fa[k][i] = read_a(stage, k, i);
#pragma unroll
            for (int j = 0; j < WNT; ++j)
                if (j / 2 == i) into[k][j] = read_w(stage, k, j);
        };
#pragma unroll
        for (int k = 0; k < KW; ++k)
#pragma unroll
            for (int i = 0; i < MTW; ++i) {
                read_row(0, k, i, fw0);
                __builtin_amdgcn_sched_barrier(0);
            }
        int st = 0, before = NS - 1;                            // the ring's places of slabs s and s - 1
        auto turn = [&](int s, const Operand (&now)[KW][WNT], Operand (&next)[KW][WNT]) {
            wait_slabs(std::integral_constant<int, NS - 3>{});  // slab s + 1 has landed ..
            meet();                                             // .. everybody's share of it, and everybody has multiplied slab s - 1
            const int behind = st + 1 == NS ? 0 : st + 1;
#pragma unroll
            for (int k = 0; k < KW; ++k)
#pragma unroll
                for (int i = 0; i < MTW; ++i) {
                    if (mine(i))
#pragma unroll
                        for (int j = 0; j < WNT; ++j) PanelOperand<T>::multiply(now[k][j], fa[k][i], acc[i][j]);
                    read_row(behind, k, i, next);
#pragma unroll
                    for (int t = 0; t < LOADS; ++t)
                        if (t * (KW * MTW) / LOADS == k * MTW + i) ask(s + NS - 1, before, t);
                    __builtin_amdgcn_sched_barrier(0);
                }
            before = st;
            st = behind;
        };
        int s = s_begin;
        for (; s + 1 < s_end; s += 2) {
            turn(s, fw0, fw1);
            turn(s + 1, fw1, fw0);
        }
        if (s < s_end) turn(s, fw0, fw1);
    }
    const int nw = n0 + cg * (16 * WNT) + q * 4;                // this lane's four columns of tile j: nw + 16 j ..; its row of tile i: m0 + 16 i + r
    // what the sums are added to is asked for before they join (places past an edge ask for one that exists)
    constexpr int OWN = (MT + KS - 1) / KS;                     // rows of tiles that a wavefront ends up with: those of part, part + KS, ..
    f32x4 had[MODE == kAddF32 ? OWN : 1][WNT];
    if constexpr (MODE == kAddF32) {
#pragma unroll
        for (int i = 0; i < OWN; ++i)
#pragma unroll
            for (int j = 0; j < WNT; ++j) {
                const int m = m0 + (i * KS + part) * 16 + r, n = nw + j * 16;
                had[i][j] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(out) + (i * KS + part < MT && m < M && n < N ? static_cast<size_t>(m) * N + n : 0));
            }
    }
    RowPlace place;
    if constexpr (MODE == kRopeCache) {                         // where row m0 + tid goes
        const int mrow = m0 + tid < M ? m0 + tid : M - 1;
        place.pos = qt.positions[mrow];
        place.page = qt.block_table[static_cast<size_t>(qt.seq_idx[mrow]) * qt.max_blocks + place.pos / qt.page];
    }
    wait_vm<0>();
    if constexpr (!ROWS) {
        // The KS wavefronts of a group of columns share its rows of tiles out and hand each other their parts where the ring was, 16 bytes a lane.
        f32x4* parts = reinterpret_cast<f32x4*>(lds_raw);
        auto part_at = [&](int of, int i, int j) { return ((of * CG + cg) * (S::JOIN_ROWS * WNT) + i % S::JOIN_ROWS * WNT + j) * 64 + lane; };
#pragma unroll
        for (int first = 0; first < MT; first += S::JOIN_ROWS) {
            __syncthreads();                                    // (the ring, or the rows before, have been read)
#pragma unroll
            for (int i = first; i < MT && i < first + S::JOIN_ROWS; ++i)
                if (i % KS != part)
#pragma unroll
                    for (int j = 0; j < WNT; ++j) parts[part_at(part, i, j)] = acc[i][j];
            __syncthreads();
#pragma unroll
            for (int i = first; i < MT && i < first + S::JOIN_ROWS; ++i) {
                if (i % KS != part) continue;
#pragma unroll
                for (int o = 1; o < KS; ++o) {
                    const int of = (part + o) % KS;
#pragma unroll
                    for (int j = 0; j < WNT; ++j) {
                        const f32x4 p = parts[part_at(of, i, j)];
                        acc[i][j][0] += p[0]; acc[i][j][1] += p[1]; acc[i][j][2] += p[2]; acc[i][j][3] += p[3];
                    }
                }
            }
        }
    }
    // this wavefront's rows of tiles: place i of acc is row tile_of(i) of the tile, if it ends up here
    auto tile_of = [&](int i) { return ROWS ? i * RG + part : i; };
    auto ends_here = [&](int i) { return ROWS ? mine(i) : i % KS == part; };
    if constexpr (MODE == kRopeCache) {
        // the tile lies in LDS in 32 bits, with its rows' places, for the epilogue that all kernels share
        constexpr int SS = BN + 4;
        float* stage = reinterpret_cast<float*>(lds_raw);
        int* row_pos = reinterpret_cast<int*>(lds_raw + static_cast<size_t>(BM) * SS * 4);
        int* row_page = row_pos + BM;
        __syncthreads();
        if (tid < BM) {
            row_pos[tid] = place.pos;
            row_page[tid] = place.page;
        }
#pragma unroll
        for (int i = 0; i < MTW; ++i)
            if (ends_here(i))
#pragma unroll
                for (int j = 0; j < WNT; ++j) *reinterpret_cast<f32x4*>(stage + (tile_of(i) * 16 + r) * SS + cg * (16 * WNT) + j * 16 + q * 4) = acc[i][j];
        __syncthreads();
        store_staged<BM, BN, 64 * NW, MODE, false>(stage, row_pos, row_page, out, M, N, m0, n0, tid, qt, 0, gx, static_cast<size_t>(N));
        return;
    }
#pragma unroll
    for (int i = 0; i < MTW; ++i) {
        const int m = m0 + tile_of(i) * 16 + r;
        if (!ends_here(i) || m >= M) continue;
        if constexpr (is_gated(MODE)) {
            typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
#pragma unroll
            for (int j = 0; j < WNT; j += 2) {
                if (nw + j * 16 >= N) continue;
                bf16x4 o, bg = {}, bu = {};
                if (MODE == kGatedExtraBF16 && gx.bias != nullptr) {
                    bg = *reinterpret_cast<const bf16x4*>(gx.bias + nw + j * 16);
                    bu = *reinterpret_cast<const bf16x4*>(gx.bias + nw + j * 16 + 16);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = static_cast<__bf16>(gated_value<MODE>(acc[i][j][e], acc[i][j + 1][e], gx, static_cast<float>(bg[e]), static_cast<float>(bu[e])));
                *reinterpret_cast<bf16x4*>(static_cast<bf16*>(out) + static_cast<size_t>(m) * (N / 2) + (n0 + cg * (16 * WNT) + j * 16) / 2 + q * 4) = o;
            }
        } else if constexpr (is_stored_bf16(MODE)) {
            typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
#pragma unroll
            for (int j = 0; j < WNT; ++j) {
                if (nw + j * 16 >= N) continue;
                bf16x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = static_cast<__bf16>(stored_value<MODE>(acc[i][j][e]));
                *reinterpret_cast<bf16x4*>(static_cast<bf16*>(out) + static_cast<size_t>(m) * N + nw + j * 16) = o;
            }
        } else {
            float* o = static_cast<float*>(out) + (static_cast<size_t>(MODE == kStoreF32 ? split : 0) * M + m) * N;   // (a part of its own)
#pragma unroll
            for (int j = 0; j < WNT; ++j) {
                const int n = nw + j * 16;
                if (n >= N) continue;
                f32x4 v = acc[i][j];
                if constexpr (MODE == kAddF32) {
                    const f32x4 h = had[ROWS ? i : i / KS][j];
                    v[0] += h[0]; v[1] += h[1]; v[2] += h[2]; v[3] += h[3];
                }
                *reinterpret_cast<f32x4*>(o + n) = v;
            }
        }
    }
}

template <typename T, int MT, int CG, int KS, int WT, bool HALF, int MODE>
static int launch_panel(const T* A, const T* W, void* out, int M, int N, int K, int ksplit, const QkvTarget& qt,
                        const GateExtra& gx, hipStream_t stream) {
    using S = PanelSizes<T, MT, CG, KS, WT, HALF>;
    if constexpr ((MODE == kRopeCache && !S::TURNS) || (is_gated(MODE) && WT % 2 != 0)) {
        return kErrUnsupported;
    } else {
        static OncePerDevice told;
        constexpr int LDS = MODE == kRopeCache && S::TURNED > S::LDS ? S::TURNED : S::LDS;
        const int status = allow_lds(told, reinterpret_cast<const void*>(&gemm_panel_kernel<T, MT, CG, KS, WT, HALF, MODE>), LDS);
        if (status != 0) return status;
        const int tiles_m = (M + S::BM - 1) / S::BM, tiles_n = (N + S::BN - 1) / S::BN;
        hipLaunchKernelGGL((gemm_panel_kernel<T, MT, CG, KS, WT, HALF, MODE>), dim3(tiles_m * tiles_n * ksplit), dim3(64 * S::NW), LDS, stream, A,
                           W, out, M, N, K, tiles_m, tiles_n, ksplit, qt, gx);
        return launch_status();
    }
}

template <int MODE, typename T>
static int launch_panel_mode(int mt, int bn, const T* A, const T* W, void* out, int M, int N, int K, int ksplit, const QkvTarget& qt,
                             const GateExtra& gx, hipStream_t stream) {
#define LLME_PANEL(MT, BN) \
    if (mt == MT && bn == BN) return launch_panel<T, MT, BN / 32, 256 / BN, 2, false, MODE>(A, W, out, M, N, K, ksplit, qt, gx, stream);
    LLME_PANEL(2, 64)
    LLME_PANEL(3, 64)
    LLME_PANEL(4, 64)
    LLME_PANEL(5, 64)
    LLME_PANEL(6, 64)
    LLME_PANEL(3, 128)
    LLME_PANEL(4, 128)
    LLME_PANEL(5, 128)
    LLME_PANEL(6, 128)
    LLME_PANEL(7, 128)
    LLME_PANEL(8, 128)
    LLME_PANEL(9, 128)
    LLME_PANEL(10, 128)
    LLME_PANEL(11, 128)
    LLME_PANEL(12, 128)
#undef LLME_PANEL
    // bfloat16 only: three or four tiles of columns a wavefront (48 columns are no pairs of gate and up); those that HALF is for in slabs of 32 k
    if constexpr (sizeof(T) == 2) {
#define LLME_PANEL(MT, BN, HALF) \
    if (mt == MT && bn == BN) return launch_panel<T, MT, 4, 2, BN / 64, HALF, MODE>(A, W, out, M, N, K, ksplit, qt, gx, stream);
        LLME_PANEL(6, 192, false)
        LLME_PANEL(8, 192, false)
        LLME_PANEL(10, 192, true)
        LLME_PANEL(12, 192, true)
        LLME_PANEL(8, 256, true)
        LLME_PANEL(12, 256, true)
#undef LLME_PANEL
    }
    return kErrUnsupported;
}

int gemm_panel(int mt, int bn, int mode, const bf16* A, const bf16* W, void* out, int M, int N, int K, int ksplit, const QkvTarget& qt,
               const GateExtra& gx, hipStream_t stream) {
    if (M <= 0 || N <= 0 || N % 16 != 0 || K <= 0 || K % 32 != 0 || K >= (1 << 22) || ksplit < 1) return kErrUnsupported;
    if (is_gated(mode) && N % 32 != 0) return kErrUnsupported;
    switch (mode) {
        case kStoreF32: return launch_panel_mode<kStoreF32>(mt, bn, A, W, out, M, N, K, ksplit, qt, gx, stream);
        case kAddF32: return launch_panel_mode<kAddF32>(mt, bn, A, W, out, M, N, K, 1, qt, gx, stream);
        case kGatedBF16: return launch_panel_mode<kGatedBF16>(mt, bn, A, W, out, M, N, K, 1, qt, gx, stream);
        case kGatedExtraBF16: return launch_panel_mode<kGatedExtraBF16>(mt, bn, A, W, out, M, N, K, 1, qt, gx, stream);
        case kSquaredReluBF16: return launch_panel_mode<kSquaredReluBF16>(mt, bn, A, W, out, M, N, K, 1, qt, gx, stream);
        case kRopeCache: return bn % qt.hd ? kErrUnsupported : launch_panel_mode<kRopeCache>(mt, bn, A, W, out, M, N, K, 1, qt, gx, stream);
        default: return kErrUnsupported;
    }
}

// 32-bit operands, W row-major; K and N multiples of 4, all pointers 16-byte aligned.
int gemm_panel_f32(int mt, int bn, int mode, const float* A, const float* W, float* out, int M, int N, int K, int ksplit, hipStream_t stream) {
    if (M <= 0 || N <= 0 || N % 4 != 0 || K <= 0 || K % 4 != 0 || K >= (1 << 22) || ksplit < 1) return kErrUnsupported;
    if (mode == kAddF32) return launch_panel_mode<kAddF32>(mt, bn, A, W, out, M, N, K, 1, QkvTarget{}, GateExtra{}, stream);
    return launch_panel_mode<kStoreF32>(mt, bn, A, W, out, M, N, K, ksplit, QkvTarget{}, GateExtra{}, stream);
}

// Tiles of 192 and 256 columns are there for the rounds that they save: a product takes whole rounds of one tile a compute unit, and
// what fills one and a half rounds of 128 x 128 is one round of 128 x 192 (16 x 16 of them cover 2,048 x 3,072). A turn of 128 x 192 x 64 takes
// 0.63 us, of 128 x 128 0.46 (0.26 of it the matrix pipes at the 2.0 GHz that the chip holds under them, 0.31 the loads alone). Of 160 x 192, 192 x 192 and
// both tiles of 256 columns LDS holds three slabs of 64 k at most, too few: 192 x 192 x 64 took 1.15 us. HALF slabs of 32 k make their ring six places (192 x 256: five) for a
// barrier every 32 k: 0.95 us. A's chunks are then 16 rows x 32 k: four lanes a row are 64 bytes side by side, which is what the loads'
// path wants, and a row's four pieces are permuted by 0 2 3 1 of its number's bits 2 and 3, so that the 16 lanes that LDS serves at a time
// (0-3, 12-15, 20-23, 24-27 and so on) meet no bank twice. Measured (us, weights from memory, the best before / with these; one round unless said):
// rotating q/k/v of the 1B sizes (3,072 x 2,048) at 2,048 rows 37.6 / 28.6, 2,600: 39.3 / 34.5, 2,995: 46.8 / 38.4; stored 6,160 x 2,048 at 1,200 rows
// 44.1 / 33.9; added 3,072 x 3,072 at 2,048 rows 49.4 / 41.4, 2,995: 70.3 / 58.1; added 3,072 x 8,192 at 2,048 rows 114 / 96; in parts at 1,000 rows 67 / 50;
// gated 16,384 x 2,048 at 430 rows 39.0 / 34.0, in three rounds at 2,300 rows 150 / 136. Against two wavefronts a compute unit's pipe with 256 x 256 of
// these (HALF): 99 us where gemm_mfma.hip's loop of that tile takes 83.

// The tile and the cut over k, by an estimate fitted to 700 timings of 20 to 4,096 rows at the 1B, 3B and 8B sizes, when these tiles
// shared out k (9 % off on average). With rows shared out, weights from memory and added sums among them, it is 4 to 13 % short, and the
// tile that it chooses takes 0.8 % longer than the best on average over 200 sizes, 9 % at worst: rounds of workgroups over the chip x (3.2 us + 2.9 for the end of a tile
// of 128 x 128, in proportion + the slabs' bytes at 98 a ns, less on a full chip and in large tiles, whose products take the time),
// joined by their 2.5th powers with W's way from memory (1.2 us + 5.6 TB/s); parts cost their way out and back in the kernel that joins
// them, 0.3 us a MB.
// HALF slabs: 0.93 (k = 2,048) to 1.09 (14,336) of it, 1.03 times that in more rounds than one (the chip's clock falls in long products).
// Products that are not cut: tiles of 192 and 256 columns take 3 to 6 % longer than that against the narrower ones, 160 and 192 x 192 in more rounds
// than one up to 20 % (a fit to 650 pairs of 130 to 4,096 rows at the same sizes). Without it sizes that two tiles of one area cover in as many rounds,
// or a wide one in a round less, went to the slower: added 1,779 x 3,072 x 8,192 in 128 x 192 93.0 us, in 192 x 128 85.2; stored 2,641 x 6,160 x 3,072 in
// two rounds of 192 x 192 117, in three of 192 x 128 108, 3,397 rows in three of 160 x 192 153, in four of 176 x 128 135; gated 540 x 16,384 x 3,072 in one
// of 192 x 256 67.8, in two of 144 x 128 62.7.
// wide: 32-bit operands, whose products take the time (a compute unit makes 500 a ns).
// ks_only: the number of parts (0: up to 8, of at least 256 k); heads: tiles hold whole heads of this many columns; pairs: a wavefront holds
// whole pairs of gate and up (32 columns each, which the 48 of a tile of 192 are not).
PanelPlan panel_plan(int M, int N, int K, int ks_only, int heads, bool wide, bool pairs) {
    // The last plans made by this thread, in sets of four that replace their oldest: a layer's products ask for the same few again and
    // again, and steps with prompt rows wait for the host, which an estimate of all tiles takes 1.5 us, of all cuts too 6. (Sizes of
    // models are multiples of large powers of two: the set comes from the high bits of products with odd numbers.)
    struct Made {
        int M = 0, N = 0, K = 0, other = 0;
        PanelPlan plan{};
    };
    struct Set {
        Made made[4];
        unsigned oldest = 0;
    };
    static thread_local Set memo[16];
    const int other = ks_only * 4096 + heads * 4 + (pairs ? 2 : 0) + (wide ? 1 : 0);
    unsigned mixed = 0;
    for (const int v : {M, N, K, other}) mixed = (mixed ^ static_cast<unsigned>(v)) * 2654435761u, mixed ^= mixed >> 15;
    Set& set = memo[mixed >> 28];
    for (const Made& m : set.made)
        if (m.M == M && m.N == N && m.K == K && m.other == other) return m.plan;
    // rows / 16, columns, and how much longer than estimated a tile takes, against those of 64 and 128 columns, in hundredths
    static const int shapes[][3] = {{2, 64, 0}, {3, 64, 0}, {4, 64, 0}, {5, 64, 0}, {6, 64, 0}, {3, 128, 0}, {4, 128, 0}, {5, 128, 0}, {6, 128, 0},
                                    {7, 128, 0}, {8, 128, 0}, {9, 128, 0}, {10, 128, 0}, {11, 128, 0}, {12, 128, 0},
                                    {6, 192, 4}, {8, 192, 3}, {10, 192, 6}, {12, 192, 6}, {8, 256, 3}, {12, 256, 4}};
    const int cus = compute_units();
    PanelPlan best{0, 0, 0, 0, 0.f};
    for (const auto& s : shapes) {
        const int bm = 16 * s[0], bn = s[1];
        const bool half = bn == 256 || (bn == 192 && s[0] >= 10);
        if ((heads > 0 && bn % heads != 0) || (bn > 128 && wide) || (bn == 192 && pairs) || (heads > 0 && s[0] == 12 && bn == 256)) continue;
        const long tiles = static_cast<long>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        for (int ks = ks_only > 0 ? ks_only : 1; ks <= (ks_only > 0 ? ks_only : 8); ++ks) {
            if (ks > 1 && ks_only == 0 && K / ks < 256) break;
            const long wgs = tiles * ks, rounds = (wgs + cus - 1) / cus;
            const float full = wgs < cus ? static_cast<float>(wgs) / cus : 1.f, area = static_cast<float>(bm) * bn;
            const float size = wide ? 4.f : 2.f, bytes = size * 1e-3f * K / ks * (bm + bn), rate = 98.f / (1.f + 0.54f * full * area / 24576.f);
            const float multiplied = wide ? 2e-3f * K / ks * area / 500.f : 0.f;
            const float of_half = half ? (0.903f + 1.3e-5f * K / ks) * (rounds > 1 ? 1.03f : 1.f) : 1.f;
            const float chip = of_half * rounds * (3.2f + 2.9f * area / 16384.f + (multiplied > bytes / rate ? multiplied : bytes / rate));
            const float memory = 1.2f + size * 1e-6f * N * K / 5.6f;
            float us = powf(powf(chip, 2.5f) + powf(memory, 2.5f), 0.4f);
            if (ks_only == 1) us *= half && bn == 192 && rounds > 1 ? 1.2f : 1.f + 0.01f * s[2];
            if (ks > 1) us += 0.3f * 4e-6f * ks * M * N;
            if (best.mt == 0 || us < best.us) best = PanelPlan{s[0], bn, ks, static_cast<int>(rounds), us};
        }
    }
    set.made[set.oldest++ % 4] = Made{M, N, K, other, best};
    return best;
}

}  // namespace llme

using namespace llme;

// A sum over k that another kernel adds up (llme_parts_norm): how many parts of a [M, K] w [N, K] (bfloat16 and blocked, or wide: 32-bit and row-major) are worth it (0: none, the
// product adds into its output itself). A product that adds its parts with atomics pays about 1 us a MB for them; up to 64 bfloat16
// rows that is less than the longer norm costs, and both wait for W (down-proj of the 1B sizes with its weights from memory, us, atomics /
// parts, and the norm 0.7 to 1.7 longer: 20 rows 10.1 / 10.2, 64 rows 12.1 / 11.3, with rows shared out 70 rows 13.0 / 10.0, 96 rows
// 14.3 / 10.7).
extern "C" int llme_gemm_parts_plan(int M, int N, int K, int wide) {
    if (M <= (wide ? 16 : 64) || M > 1024 || N % (wide ? 4 : 16) != 0 || K % (wide ? 4 : 32) != 0 || K >= (1 << 22)) return 0;
    const PanelPlan p = panel_plan(M, N, K, 0, 0, wide != 0);
    return p.ksplit > 1 ? p.ksplit : 0;
}

// parts [ksplit, M, N] float32: part i is the sum over the i-th share of k (whole slabs of the tile's; a share may be empty: zeros).
// tile: 0 (chosen), or 1000 x rows + columns (tests and measurements).
extern "C" int llme_gemm_parts(const void* a, const void* w, float* parts, int M, int N, int K, int ksplit, int tile, int wide,
                               hipStream_t stream) {
    if (ksplit < 1 || tile < 0 || tile / 1000 % 16 != 0) return kErrBadArgument;
    if (M <= 0 || N <= 0) return 0;
    int mt = tile / 16000, bn = tile % 1000;
    if (tile == 0) {
        const PanelPlan p = panel_plan(M, N, K, ksplit, 0, wide != 0);
        mt = p.mt;
        bn = p.bn;
    }
    if (wide) return gemm_panel_f32(mt, bn, kStoreF32, static_cast<const float*>(a), static_cast<const float*>(w), parts, M, N, K, ksplit, stream);
    return gemm_panel(mt, bn, kStoreF32, static_cast<const bf16*>(a), static_cast<const bf16*>(w), parts, M, N, K, ksplit, QkvTarget{},
                      GateExtra{}, stream);
}

LLME_LOAD_ENTRY(gemm_panel)
