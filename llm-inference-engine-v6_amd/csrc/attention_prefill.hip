// Prefill attention over bfloat16 cache pages with K and V shared through LDS.
// Formula as in the plain-precision kernel (src/kernels.cpp:413-474); tile arithmetic as in
// attention_tiles.h. What differs from the kernel that loads straight into registers is where
// the operands come from: a workgroup's four wavefronts need the same keys (heads of one kv
// head over the same rows, or neighbouring rows of one head), so the workgroup fetches every
// 64-key stretch of K and V once, straight into LDS, and each wavefront reads its operands from there.
//
// Work item = (request, span of rows, group of HPW query heads of one kv head): wavefront w
// takes head w % HPW of the group and the row group w / HPW of the span, each row group being
// QT tiles of 16 rows. HPW is the largest of 4, 2, 1 that divides the heads per kv head.
// Stretches run from the first key the span's first row sees to the last row's own key.
//
// What bounds it: a wavefront's 32 rows x 64 keys are 32 exponentials a lane (16 cycles each), as many multiply-adds and maxima, half as many
// conversions (about 800 cycles), 36 matrix instructions of 16 cycles with heads of 64 and 68 with heads of 128 (576, 1,088), and 16 or
// 32 KB read from LDS (128 bytes a cycle for the whole unit: 128, 256). One after the other, with a wait of LDS's latency at every
// operand, that was 1,900 and 4,100 cycles. So a turn multiplies the NEXT stretch's scores while it makes this stretch's weights, reads
// every operand a step before it is multiplied, loads straight into LDS a stretch ahead (K two: its scores are a turn ahead), meets once, and has
// the matrix cores add up the weights (a column of ones: 4 instructions for 64 of the vector units'). Two wavefronts for a
// tile, each with half the keys, which steps of few items used to take, are no faster now (45 to 1,024 tokens: 1 to 4 % slower, 256 rows behind
// 8,192: 50 / 40).
// Measured on one card, us, one thing after the other / so, 32 query and 8 kv heads: heads of 64, 45 tokens 4.74 / 4.85, 512 9.6 / 9.4, 1,024 17.0 / 15.0,
// 2,048 39.3 / 30.8, 4,096 109 / 88, 8,192 390 / 321 (857 TFLOP/s); heads of 128, 1,024 29.0 / 20.6, 2,048 58.9 / 49.2, prompts of 2,000, 3,691 and 2,500
// together 282 / 208 (940 TFLOP/s); 256 rows behind 8,192, heads of 64, in 8 runs of keys 51 / 40, behind 1,024 beside 17 decoded requests 20.1 / 19.9.
// (Cards differ: 2,048 tokens with heads of 64 took 30.2 to 36.7, 8,192 305 to 337.)
//
// Takes head sizes 64 and 128 and pages that are multiples of 16; other sizes go to the kernel
// without LDS.
//
// Few rows over a long context (a portion of a prompt far into it) are few work items that each
// walk many keys, and in a prompt of a few thousand tokens the items of the last rows take twice
// the average while the chip has room left. Then an item's keys are cut into up to `nsplit` runs of
// `run` stretches, one work item each, which leave their rows' maxima, sums and unscaled outputs
// in 32-bit scratch indexed by batch row; a second kernel joins them, as it joins the splits of
// the decode kernel. Items with few keys have one run and write their output themselves.
#include "attention_tiles.h"

#include <type_traits>

namespace llme {

constexpr int KB = 64;                     // keys per stretch

// Two buffers of K and two of V, a stretch each: in K a half is [16 keys][HD], in V [HD][16 keys]. Behind them zeros, 16 bytes every 512, which
// are read in the place of the values of a block that none of a wavefront's rows sees (a weight of zero alone would let an infinity through).
template <int HD>
struct StageLayout {
    static constexpr int HALF = 16 * HD * 2;           // bytes
    static constexpr int OPERAND = KB / 16 * HALF;
    static constexpr int ZEROS = 4 * OPERAND;
    static constexpr int BYTES = ZEROS + HD / 16 * 512;
};

// The place of a 16-byte piece in row `key` of K's buffer (key within its 32-key block): pieces are permuted by bits of the
// row's number such that the 16 lanes that LDS serves at a time (0-3, 12-15, 20-23, 24-27 and so on), which read rows 8 (r / 4) + r % 4 at
// neighbouring pieces (see block_scores), meet no bank twice.
template <int HD>
__device__ __forceinline__ unsigned k_turn(int key) {
    return HD == 128 ? ((key >> 3) & 3) << 2 | (key & 3) : ((key >> 3) & 3) << 1 | ((key >> 1) & 1);
}

// One work item: span `bx` (counted over the requests with two or more tokens, the last spans of
// a request first) for head group `by`, run `z` of its keys (SPLIT; else all keys).
template <int HD, int QT, int HPW, bool SPLIT>
__device__ __forceinline__ void prefill_item(int bx, int by, int z, int nsplit, int run, float* __restrict__ part_o,
                                             float* __restrict__ part_ml, unsigned char* lds, const bf16* __restrict__ q,
                                             const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
                                             bf16* __restrict__ out, const int* __restrict__ q_start,
                                             const int* __restrict__ ctx_len, const int* __restrict__ block_table,
                                             int max_blocks, int n_seq, int n_q, int n_kv, int page, float scale,
                                             int window) {
    constexpr int DC = HD / 32, DT = HD / 16, ROWS = 16 * QT, RG = 4 / HPW, SPAN = RG * ROWS;
    using L = StageLayout<HD>;

    // which request and which of its spans this workgroup has
    int s = 0, first = 0, n_span = 0, acc = 0;
    bool found = false;
    for (int i = 0; i < n_seq; ++i) {
        const int a = q_start[i], n = q_start[i + 1] - a;
        const int nt = (n >= 2) ? (n + SPAN - 1) / SPAN : 0;
        if (!found && bx < acc + nt) {
            s = i;
            first = (nt - 1 - (bx - acc)) * SPAN;          // the last spans see the most keys and start first
            n_span = n - first < SPAN ? n - first : SPAN;
            first += a;                                    // as a batch row
            found = true;
        }
        acc += nt;
    }
    if (!found) return;                                    // the whole workgroup
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));                          // (what is made of it is made per item, and not kept in registers from one to the next)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, r = lane & 15, g4 = lane >> 4;
    const int G = n_q / n_kv;
    const int head = by * HPW + wave % HPW;                // HPW divides G: one kv head per workgroup
    const int kvh = (by * HPW) / G;
    const int rg = wave / HPW;
    const int pos_span = ctx_len[s] + (first - q_start[s]); // position of the span's first row

    // this wavefront's rows
    const int first_w = first + rg * ROWS;
    int n_rows = n_span - rg * ROWS;
    n_rows = n_rows < 0 ? 0 : (n_rows > ROWS ? ROWS : n_rows);
    const int pos0 = pos_span + rg * ROWS;
    bf16x8 qf[QT][DC];
    float m[QT];                                           // of row r
    f32x4 l[QT], o[QT][DT];                                // of rows 4 g4 + e
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int rr = qt * 16 + r;
        const bool ok = rr < n_rows;
        load_q<HD>(q + (static_cast<size_t>(ok ? first_w + rr : first) * n_q + head) * HD, ok, qf[qt]);
        m[qt] = kNoMax;
        l[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int my_end = n_rows > 0 ? pos0 + n_rows : 0;            // this wavefront's rows see keys < my_end
    const int my_lo = (window > 0 && pos0 - window + 1 > 0) ? pos0 - window + 1 : 0;
    // stretches that begin at free_lo or behind and end before free_hi are seen whole by every row
    const int free_lo = (window > 0 && pos0 + ROWS - window > 0) ? pos0 + ROWS - window : 0;
    const int free_hi = n_rows > 0 ? pos0 + 1 : 0;

    // the workgroup's keys
    int key_end = pos_span + n_span;
    const int key_lo = (window > 0 && pos_span - window + 1 > 0) ? pos_span - window + 1 : 0;
    int k_begin = key_lo & ~(KB - 1);
    int runs = 1;
    if (SPLIT) {
        runs = key_runs(k_begin, key_end, run, nsplit);
        if (z >= runs) return;                             // (the whole workgroup: no such run)
        k_begin += z * run * KB;
        if (z < runs - 1) key_end = k_begin + run * KB;    // (the last run takes the rest)
    }
    my_end = my_end < key_end ? my_end : key_end;
    const PagedKV kv{k_cache, v_cache, block_table + static_cast<size_t>(s) * max_blocks, page, n_kv, kvh, HD,
                     page_magic_of(page), static_cast<unsigned>(n_kv) * page * HD, static_cast<unsigned>(kvh) * page * HD};
    const float scale_log2 = scale * kLog2e;
    const int n_stretch = (key_end - k_begin + KB - 1) / KB;

    // ---- loads: half `wave` of every stretch is this wavefront's, its K and its V in NL pieces of 1 KB each ----
    constexpr int NL = HD / 32, K_ROWS = 1024 / (2 * HD);               // keys in 1 KB of K
    // a half without a key in [key_lo, key_end) is not to be read (its page may not be there): of K the nearest one that has is, whose
    // scores are replaced, and V's places become zeros (an offset that is nowhere within the descriptor)
    const int first_half = key_lo & ~15, last_half = (key_end - 1) & ~15;
    constexpr unsigned kOutside = 0x40000000u;
    auto half_at = [&](int j) {
        const int h0 = k_begin + j * KB + 16 * wave;
        return h0 > last_half ? last_half : h0 < first_half ? first_half : h0;
    };
    // the page ids of this wavefront's half in 64 stretches, one a lane
    auto look_up = [&](int j) { return kv.table[page_of(kv, half_at(j + lane)).block]; };
    unsigned k_off[2];                                      // of a lane in 1 KB of K: one of two, by its place in the half
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int key = 16 * (wave & 1) + (HD == 128 ? 8 * u : K_ROWS * u) + lane / (64 / K_ROWS), slot = lane % (64 / K_ROWS);
        k_off[u] = static_cast<unsigned>(lane / (64 / K_ROWS)) * (HD * 2) + (slot ^ k_turn<HD>(key)) * 16;
    }
    const unsigned v_off = static_cast<unsigned>(lane >> 1) * (kv.page * 2) + (lane & 1) * 16;
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)lds));
    auto descriptor = [](const bf16* p, unsigned bytes) {
        const unsigned long long at = reinterpret_cast<unsigned long long>(p);
        return u32x4{static_cast<unsigned>(at), static_cast<unsigned>(at >> 32) & 0xFFFFu, bytes, 0x00020000u};
    };
    struct Half {
        int page, offset;
        bool inside;
    };
    auto ask_k = [&](const Half& h, int buffer) {
        const u32x4 rsrc = descriptor(kv.k + static_cast<size_t>(h.page) * kv.page_stride + kv.head_off + static_cast<size_t>(h.offset) * HD, L::HALF);
#pragma unroll
        for (int i = 0; i < NL; ++i)
            load_1kb_to_lds(rsrc, lds_base + buffer * L::OPERAND + wave * L::HALF + i * 1024, k_off[HD == 128 ? i >> 1 : i], i * 1024);
    };
    auto ask_v = [&](const Half& h, int buffer) {
        const u32x4 rsrc = descriptor(kv.v + static_cast<size_t>(h.page) * kv.page_stride + kv.head_off + h.offset, static_cast<unsigned>(HD - 1) * kv.page * 2 + 32);
#pragma unroll
        for (int i = 0; i < NL; ++i)
            load_1kb_to_lds(rsrc, lds_base + (2 + buffer) * L::OPERAND + wave * L::HALF + i * 1024, h.inside ? v_off : kOutside,
                            h.inside ? i * 32 * kv.page * 2 : 0);
    };
    int ids = look_up(0);
    auto half_of = [&](int j) {
        return Half{__builtin_amdgcn_readlane(ids, j & 63), __builtin_amdgcn_readfirstlane(page_of(kv, half_at(j)).offset),
                    half_at(j) == k_begin + j * KB + 16 * wave};
    };
    // what everybody asked for is there, and everybody is done with what it read
    auto meet = [&] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- products ----
    // (what only the rare branches of a turn make of the lane's number is made there and not kept in registers throughout)
    auto rarely = [](int x) {
        asm volatile("" : "+v"(x));
        return x;
    };
    constexpr int NB = KB / 32;                             // 32-key blocks of a stretch
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i) ones[i] = static_cast<__bf16>(1.f);
    const unsigned char* k_lane = lds + (8 * (r >> 2) + (r & 3)) * (2 * HD);
    const unsigned k_piece = (g4 ^ k_turn<HD>(8 * (r >> 2) + (r & 3))) * 16;
    const unsigned char* v_lane = lds + 2 * L::OPERAND + (g4 >> 1) * L::HALF + r * 32 + (g4 & 1) * 16;
    // Scores of row i of K's operand of half hf: key 8 (i / 4) + 4 hf + i % 4, so that a lane, whose results are rows 4 g4 + e, gets the
    // eight keys 8 g4 .. of the block, which are 16 bytes of V's rows.
    auto read_k = [&](int buffer, int b, int hf, bf16x8 (&kf)[DC]) {
#pragma unroll
        for (int c = 0; c < DC; ++c)
            kf[c] = *reinterpret_cast<const bf16x8*>(k_lane + buffer * L::OPERAND + b * 2 * L::HALF + hf * (4 * 2 * HD) + (k_piece ^ (c * 64)));
    };
    auto scores_of = [&](const bf16x8 (&kf)[DC], f32x4 (&to)[QT]) {
#pragma unroll
        for (int c = 0; c < DC; ++c)
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
                to[qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[c], qf[qt][c], c == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : to[qt], 0, 0, 0);
    };
    auto all_scores = [&](int buffer, f32x4 (&to)[NB][2][QT]) {
#pragma unroll
        for (int g = 0; g < 2 * NB; ++g) {
            bf16x8 kf[DC];
            read_k(buffer, g >> 1, g & 1, kf);
            scores_of(kf, to[g >> 1][g & 1]);
        }
    };
    auto weights_of = [&](const f32x4& sc, int qt, int hf, bf16x8& pf) {
#pragma unroll
        for (int e = 0; e < 4; ++e) pf[hf * 4 + e] = static_cast<__bf16>(fast_exp2(fmaf(sc[e], scale_log2, -m[qt])));
    };
    Half h_v = half_of(0), h_k = half_of(1);                // of the V and the K that are asked for next
    ask_k(h_v, 0);
    ask_v(h_v, 0);
    if (n_stretch > 1) ask_k(h_k, 1);
    h_v = h_k;
    f32x4 sa[NB][2][QT], sb[NB][2][QT];
    meet();
    all_scores(0, sa);

    // One stretch: its weights and values, and the next one's scores. cur: its scores; buffer: of its V (the next K lies in the other).
    auto turn = [&](int j, auto which, f32x4 (&cur)[NB][2][QT], f32x4 (&next)[NB][2][QT]) {
        constexpr int BUFFER = decltype(which)::value;
        meet();
        bf16x8 kf[2][DC];
        read_k(BUFFER ^ 1, 0, 0, kf[0]);                    // (on its way while the loads are asked for and the maxima made)
        __builtin_amdgcn_sched_barrier(0);
        const int t0 = k_begin + j * KB;
        if (j + 2 < n_stretch) {
            if (((j + 2) & 63) == 0) {
                ids = look_up(j + 2);
                asm volatile("" ::"v"(ids));               // (waited for here, and not wherever it is read)
            }
            h_k = half_of(j + 2);
            ask_k(h_k, BUFFER);
        }
        if (j + 1 < n_stretch) ask_v(h_v, BUFFER ^ 1);
        h_v = h_k;
        if (t0 >= my_end) return;                           // (no row sees any of it, nor of what follows)
        if (t0 + KB <= my_lo) {                        // (no row sees any of it yet)
            all_scores(BUFFER ^ 1, next);
            return;
        }
        if (t0 < free_lo || t0 + KB > free_hi) {
            const int l_ = rarely(lane), r_ = l_ & 15, g_ = l_ >> 4;
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                const int row = qt * 16 + r_;
                const int last = (row < n_rows ? pos0 + row : -1) - t0 - g_ * 8, first_seen = window > 0 ? pos0 + row - window + 1 - t0 - g_ * 8 : -KB;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int t = 32 * b + hf * 4 + e;
                            cur[b][hf][qt][e] = (t <= last && t >= first_seen) ? cur[b][hf][qt][e] : -INFINITY;
                        }
            }
        }
        float mx[QT];
        bool moves = false;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            mx[qt] = cur[0][0][qt][0];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                    for (int e = 0; e < 4; ++e) mx[qt] = fmaxf(mx[qt], cur[b][hf][qt][e]);
            moves |= fmaf(mx[qt], scale_log2, -m[qt]) > kLazy;
        }
        if (__any(moves)) {                                 // some row's maximum moves (see block_weights): rescale what is summed
            const int l_ = rarely(lane);
            auto from = [](float x, int at) { return __int_as_float(__builtin_amdgcn_ds_bpermute(at * 4, __float_as_int(x))); };
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                float mr = fmaxf(mx[qt], from(mx[qt], l_ ^ 16));
                mr = fmaxf(mr, from(mr, l_ ^ 32));
                const float ms = mr * scale_log2;
                const float m_new = (ms > m[qt] + kLazy) ? ms : m[qt];
                const float alpha = fast_exp2(m[qt] - m_new);
                m[qt] = m_new;
#pragma unroll
                for (int e = 0; e < 4; ++e) {               // factor of row 4 g4 + e
                    const float ar = from(alpha, (l_ >> 4) * 4 + e);
                    l[qt][e] *= ar;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) o[qt][dt][e] *= ar;
                }
            }
        }
        const unsigned char* v_at[2] = {v_lane + BUFFER * L::OPERAND, v_lane + BUFFER * L::OPERAND + 2 * L::HALF};
        if (t0 + 32 <= my_lo) v_at[0] = lds + L::ZEROS;
        if (t0 + 32 >= my_end) v_at[1] = lds + L::ZEROS;
        bf16x8 pf[NB][QT];
        // No branch from here on: the next scores' products and these weights' exponentials go side by side. The compiler puts a read of
        // LDS where it is used and waits for it there, so the order is given: every step reads what the next one multiplies. (Behind
        // the last stretch the products are of whatever LDS holds, and nobody's.)
        constexpr int NV = 4, STEPS = NB * DT / NV;     // values: NV tiles of columns a step
        bf16x8 vf[2][NV];
        auto read_values = [&](int step, bf16x8 (&to)[NV]) {
#pragma unroll
            for (int i = 0; i < NV; ++i) to[i] = *reinterpret_cast<const bf16x8*>(v_at[step * NV / DT] + (step * NV + i) % DT * 512);
        };
#pragma unroll
        for (int g = 0; g < 2 * NB; ++g) {
            if (g + 1 < 2 * NB) read_k(BUFFER ^ 1, (g + 1) >> 1, (g + 1) & 1, kf[(g + 1) & 1]);
            else read_values(0, vf[0]);
            scores_of(kf[g & 1], next[g >> 1][g & 1]);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) weights_of(cur[g >> 1][g & 1][qt], qt, g & 1, pf[g >> 1][qt]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int u = 0; u < STEPS; ++u) {
            if (u + 1 < STEPS) read_values(u + 1, vf[(u + 1) & 1]);
            const int b = u * NV / DT;
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    f32x4& to = o[qt][(u * NV + i) % DT];
                    to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[b][qt], vf[u & 1][i], to, 0, 0, 0);
                }
            if (u * NV % DT == 0)
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) l[qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[b][qt], ones, l[qt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int j = 0; j < n_stretch; j += 2) {                // (one behind the last only meets the others)
        turn(j, std::integral_constant<int, 0>{}, sa, sb);
        turn(j + 1, std::integral_constant<int, 1>{}, sb, sa);
    }

#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        if (SPLIT && runs > 1) {
            // this run's part of row `row`, head `head`: the maximum from the lanes of the row's first quarter, the sum from a lane that
            // has it, outputs unscaled (the join divides)
            if (g4 == 0 && qt * 16 + r < n_rows)
                part_ml[((static_cast<size_t>(first_w + qt * 16 + r) * n_q + head) * nsplit + z) * 2] = m[qt];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = qt * 16 + g4 * 4 + e;
                if (row >= n_rows) continue;
                const size_t pidx = (static_cast<size_t>(first_w + row) * n_q + head) * nsplit + z;
                if (r == 0) part_ml[pidx * 2 + 1] = l[qt][e];
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) part_o[pidx * HD + dt * 16 + r] = o[qt][dt][e];
            }
            continue;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = qt * 16 + g4 * 4 + e;
            if (row >= n_rows) continue;
            const float inv = 1.0f / l[qt][e];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                out[(static_cast<size_t>(first_w + row) * n_q + head) * HD + dt * 16 + r] =
                    static_cast<bf16>(o[qt][dt][e] * inv);
        }
    }
}

// With many items per workgroup, the workgroups take work items from a counter, heaviest first, until none is left: spans differ
// in the keys they see by the length of the context, and a grid with one workgroup per item
// leaves most of the chip idle while the few longest finish. queue[0] counts the items taken,
// queue[1] the workgroups that have left; both are zero before and after the kernel (the last
// workgroup to leave clears them), so the same two integers serve every launch on a stream.
// (Registers: 128 with heads of 64, whole keys and one tile of rows a wavefront, for the four workgroups a unit that LDS holds (three are as
// fast: 2,048 tokens 30.6 us, 30.4 with four). Otherwise up to 256, for the two that LDS holds of heads of 128. None of it may lie in scratch memory: with prefill_item inlined
// twice, once for the fixed order and once for the counter, and with what it makes of the thread's number hoisted in front of the loop, 12 registers did,
// and short items fetched them in front of their keys: 256 rows behind 1,024 beside 17 decoded requests 20.5 us a launch, 19.8 without.)
template <int HD, int QT, bool SPLIT>
constexpr int kWavesASimd = HD == 64 && QT == 1 && !SPLIT ? 4 : 2;
template <int HD, int QT, int HPW, bool SPLIT>
__global__ __launch_bounds__(256, (kWavesASimd<HD, QT, SPLIT>)) void attention_prefill_shared_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
    bf16* __restrict__ out, const int* __restrict__ q_start, const int* __restrict__ ctx_len,
    const int* __restrict__ block_table, int max_blocks, int n_seq, int n_q, int n_kv, int page, float scale,
    int window, int spans, int* __restrict__ queue, int nsplit, int run, float* __restrict__ part_o,
    float* __restrict__ part_ml, DecodeBeside beside) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    __shared__ int next_item;
    unsigned char* lds = lds_raw;
    if (static_cast<int>(blockIdx.x) < beside.blocks) {
        // one of the step's decode work items: the workgroup's four wavefronts, the stages' LDS
        static_assert(DEC_WAVES * 64 == 256 && decode_lds_floats(HD) * 4 <= StageLayout<HD>::BYTES, "the decode item's sums must fit into the stages");
        const int b = blockIdx.x, per_seq = beside.head_tiles * beside.nsplit;
        decode_item<HD, true>(q, k_cache, v_cache, out, beside.part_o, beside.part_ml, q_start, ctx_len, block_table,
                              max_blocks, n_q, n_kv, page, scale, window, beside.split_len, beside.nsplit, b / per_seq,
                              (b % per_seq) / beside.nsplit, b % beside.nsplit, reinterpret_cast<float*>(lds_raw));
        return;
    }
    if (threadIdx.x < HD / 16 * 4)                          // (an item meets before it reads them)
        *reinterpret_cast<unsigned*>(lds + StageLayout<HD>::ZEROS + threadIdx.x / 4 * 512 + threadIdx.x % 4 * 4) = 0;
    const int head_groups = n_q / HPW;
    const int n_items = spans * head_groups * (SPLIT ? nsplit : 1);
    // Few items per workgroup (no queue): a fixed order, to and fro over the workgroups (the items are
    // sorted, heaviest first: workgroup w of G takes w, 2 G - 1 - w, 2 G + w, ..), so that every
    // workgroup's items add up to about the same number of keys. The counter's answer is a trip
    // to memory per item, with two barriers around it, and costs more than its evening-out
    // wins until a workgroup has several items to take.
    const int G = static_cast<int>(gridDim.x) - beside.blocks, w = static_cast<int>(blockIdx.x) - beside.blocks;
    for (int round = 0;; ++round) {
        if (queue != nullptr || round > 0) __syncthreads();    // everybody is done with the last item's LDS
        int item = round * G + ((round & 1) ? G - 1 - w : w);
        if (queue != nullptr) {
            if (threadIdx.x == 0) next_item = atomicAdd(queue, 1);
            __syncthreads();
            item = __builtin_amdgcn_readfirstlane(next_item);
        }
        if (item >= n_items) break;                        // the counter, and the first item of a round, only grow: every workgroup gets here
        const int whole = SPLIT ? item / nsplit : item;     // (an item's runs are neighbours in either order)
        prefill_item<HD, QT, HPW, SPLIT>(whole / head_groups, whole % head_groups, SPLIT ? item % nsplit : 0, nsplit,
                                             run, part_o, part_ml, lds, q, k_cache, v_cache, out, q_start, ctx_len,
                                             block_table, max_blocks, n_seq, n_q, n_kv, page, scale, window);
    }
    if (queue == nullptr) return;
    if (threadIdx.x == 0) {
        // whoever leaves last has seen every other workgroup take its final number: nobody touches
        // the counter any more
        if (atomicAdd(queue + 1, 1) == static_cast<int>(gridDim.x) - beside.blocks - 1) {
            atomicExch(queue, 0);
            atomicExch(queue + 1, 0);
        }
    }
}

static int heads_per_workgroup(int n_q, int n_kv) {
    const int G = n_q / n_kv;
    return G % 4 == 0 ? 4 : (G % 2 == 0 ? 2 : 1);
}

// Rows per work item: 32 per row group (measured: 64 are no faster at any length, and leave
// fewer items to spread over the chip), times the row groups of a workgroup. The caller may halve
// them (16 per row group) where a step has few items: an item's time is set by its walk over the
// keys, a stretch after the other, and a stretch of 16 rows is shorter than one of 32. Measured on
// whole prompts (us, 32 / 16 rows; 32 query and 8 kv heads): heads of 64, 256 tokens 8.5 / 6.7, 1,024
// 19.5 / 15.3, 2,048 35.8 / 31.1, 2,500 42.4 / 41.4, 2,700 45.1 / 46.6, 3,072 52.4 / 58.2; heads of 128, 512 tokens 15.4 /
// 11.5, 1,000 25.1 / 19.7, 1,600 38.2 / 33.2, 1,800 43.0 / 40.8, 2,048 48.9 / 49.0; 24 query heads, 2,000 tokens 44.9 / 38.4, 2,400
// 54.4 / 51.1, 3,000 69 / 80: half the rows win until the items of 32 rows number two and a half a compute unit with heads
// of 64 and, at least, seven quarters with heads of 128.
int prefill_shared_rows(int hd, int n_q, int n_kv) {
    if ((hd != 64 && hd != 128) || n_kv <= 0 || n_q % n_kv != 0) return 0;
    return 32 * (4 / heads_per_workgroup(n_q, n_kv));
}

template <int HD, int QT, int HPW, bool SPLIT>
static int launch_shared(const bf16* q, const bf16* kc, const bf16* vc, bf16* out, const int* q_start,
                         const int* ctx_len, const int* table, int max_blocks, int n_seq, int n_q, int n_kv, int page,
                         float scale, int window, int items, int* queue, int nsplit, int run, float* part_o,
                         float* part_ml, const DecodeBeside& beside, hipStream_t stream) {
    constexpr int LDS = StageLayout<HD>::BYTES;
    auto kernel = attention_prefill_shared_kernel<HD, QT, HPW, SPLIT>;
    static OncePerDevice told;                         // per instantiation
    const int status = allow_lds(told, reinterpret_cast<const void*>(kernel), LDS);
    if (status != 0) return status;
    static int resident = 0;                           // workgroups the chip holds at a time
    if (resident == 0) {
        int dev = 0, cus = 0, per_cu = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e == hipSuccess)
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), 256,
                                                             LDS);
        if (e != hipSuccess) return static_cast<int>(e);
        resident = cus * (per_cu > 0 ? per_cu : 1);
    }
    const int n_items = items * (n_q / HPW) * (SPLIT ? nsplit : 1);
    // (measured with 32 query and 8 kv heads, us, fixed order / counter; 512 workgroups are resident with items of 32 rows. Up to two rounds the
    // fixed order wins by up to 17 % and loses 5 % at most: heads of 64, 4,096 tokens, 1,024 items, 87.4 / 93.2, three prompts of 1,000 28.8 / 34.9, four of
    // 700 behind 2,048 88.3 / 84.1; heads of 128, 2,048 tokens 48.2 / 54.1, 4,096 134 / 139. Between two and three it is 4 to 11 % faster where requests
    // are equal (5,000 tokens 121 / 126, three prompts of 1,500 49.0 / 55.1), but 7 to 31 % slower where a long one is not the first or long ones meet
    // (900, 1,300, 3,000 and 700 tokens 84.0 / 78.4, 3,000 and 3,100 122.7 / 103.6, 2,000, 3,691 and 2,500 195 / 134, with heads of 128 278 / 203): the heaviest
    // items of every request are first in that request alone. From three rounds on the counter is no slower (8,192 tokens 312 / 310))
    int* counter = n_items <= 2 * resident ? nullptr : queue;
    hipLaunchKernelGGL(kernel, dim3(beside.blocks + (n_items < resident ? n_items : resident)), dim3(256), LDS, stream,
                       q, kc, vc, out, q_start, ctx_len, table, max_blocks, n_seq, n_q, n_kv, page, scale, window, items,
                       counter, nsplit, run, part_o, part_ml, beside);
    return launch_status();
}

int launch_prefill_shared(const bf16* q, const bf16* kc, const bf16* vc, bf16* out, const int* q_start,
                          const int* ctx_len, const int* table, int max_blocks, int n_seq, int n_q, int n_kv, int hd,
                          int page, float scale, int window, int items, int rows_per_item, int* queue, int nsplit,
                          int run, float* part_o, float* part_ml, const DecodeBeside& beside,
                          hipStream_t stream) {
    if (queue == nullptr) return kErrBadArgument;
    if (nsplit < 1 || (nsplit > 1 && (run < 1 || part_o == nullptr || part_ml == nullptr))) return kErrBadArgument;
    const int hpw = heads_per_workgroup(n_q, n_kv);
    const int rows = rows_per_item / (4 / hpw);            // per row group
#define LLME_SHARED_ARGS q, kc, vc, out, q_start, ctx_len, table, max_blocks, n_seq, n_q, n_kv, page, scale, window, \
                         items, queue, nsplit, run, part_o, part_ml, beside, stream
#define LLME_SHARED(HD, QT, HPW)                                                       \
    if (hd == HD && rows == 16 * QT && hpw == HPW) {                                   \
        if (nsplit > 1)                                                                \
            return launch_shared<HD, QT, HPW, true>(LLME_SHARED_ARGS);                 \
        return launch_shared<HD, QT, HPW, false>(LLME_SHARED_ARGS);                    \
    }
    LLME_SHARED(64, 2, 4) LLME_SHARED(64, 2, 2) LLME_SHARED(64, 2, 1)
    LLME_SHARED(128, 2, 4) LLME_SHARED(128, 2, 2) LLME_SHARED(128, 2, 1)
    LLME_SHARED(64, 1, 4) LLME_SHARED(64, 1, 2) LLME_SHARED(64, 1, 1)
    LLME_SHARED(128, 1, 4) LLME_SHARED(128, 1, 2) LLME_SHARED(128, 1, 1)
#undef LLME_SHARED
#undef LLME_SHARED_ARGS
    return kErrUnsupported;
}

}  // namespace llme

LLME_LOAD_ENTRY(attention_prefill)
