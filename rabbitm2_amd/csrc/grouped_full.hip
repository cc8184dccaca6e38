// The expert FFN of many tokens at full f32 activation precision: the grouped form for f32 weights, and
// for bf16 weights of dims that the tiles of prefill.hip do not divide. (Those would otherwise run one
// GEMV per (token, slot) pair, reading an expert's weights once per pair instead of once per call.)
//
// Reference semantics: rabbit2/src/rabbit2.c:531-542 for every token: h = silu(W1 xb) * (W3 xb),
// tmp = W2 h, moe += w_k * tmp in selection order, x += moe; blobs w1[H][D] | w3[H][D] | w2[D][H] (:173).
//
// The lists, their order and the combine are prefill.hip's; the two GEMMs are grouped_full_kernel's.
#include <math.h>

#include <type_traits>

#include "rbt2_internal.h"

namespace rbt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kFullWaves = 4, kFullAhead = 3;  // waves per block; k-steps of weights in flight ahead
constexpr int kFullWin = 128;                  // bytes of a weight row per k-step
constexpr int kPastWeights = 0x70000000;       // an offset past any weight matrix (full_supported)
constexpr int kBufStream = 2;                  // buffer loads of data read once: non-temporal

struct FullArgs {
    const uint8_t *experts;
    uint64_t stride, w_off, w3_off;
    int N, Kd;             // output columns, reduction length
    const float *act;      // activation rows, act_stride floats apart, zeros from Kd to the next multiple of 4
    int act_stride, gather;
    const int32_t *perm;
    int topk;
    const int32_t *counts, *offsets, *m_off, *choice;  // choice: the dispatch's plan (bit 1: column-major slots)
    int E;
    float *out;            // output rows in list order, out_stride floats apart
    int out_stride;
    // dense form: T rows through up to three weight matrices [seg_rows][Kd], out[s][t][seg_rows[s]] (added to,
    // with resid)
    const uint8_t *seg_w[3];
    float *seg_out[3];
    int seg_rows[3];
    int T, resid;
};

// x = hi + mid + lo exactly, each part a bf16 (its upper 16 bits): 8 + 8 + 8 bits of the significand by
// truncation. A non-finite x is its own hi part (a NaN made quiet, so that truncation keeps it one).
__device__ __forceinline__ void split3(float x, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    const uint32_t u = __float_as_uint(x);
    const bool fin = (u & 0x7F800000u) != 0x7F800000u;
    hi = x != x ? (u | 0x00400000u) & 0xFFFF0000u : u & 0xFFFF0000u;
    const float r1 = fin ? x - __uint_as_float(hi) : 0.0f;
    mid = __float_as_uint(r1) & 0xFFFF0000u;
    lo = __float_as_uint(r1 - __uint_as_float(mid)) & 0xFFFF0000u;
}
__device__ __forceinline__ uint32_t pack_hi16(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xFFFF0000u); }

// One tile: 16 RG list rows x 16 columns of W1 and of W3 per wave (MATS = 2: h = silu(W1 a) * (W3 a), 64
// columns per block) or 32 columns of W2 (MATS = 1: y = W2 a, 128 columns per block).
//
// Weights go from HBM into registers in the operands' order (blob_operands: whole 128-byte lines of the
// row-major blobs), kFullAhead k-steps of 128 bytes per row ahead, each weight byte once per tile. The f32
// activation rows are loaded four steps ahead (buffer loads: rows past the list and columns past the row
// read as zeros without a request) and pass through a two-stage LDS ring that all waves read. Products:
//   bf16 weights: the activation as three bf16 parts that carry all 24 bits (split on the way into LDS),
//     three v_mfma_f32_16x16x32_bf16 per 32 columns; every product is exact in the f32 accumulator;
//   f32 weights: v_mfma_f32_16x16x4_f32.
// The sums are no further from 64 bits than the GEMVs' lanes and trees: bf16, a step's products are summed
// from zero (the small parts first), eight steps' sums are added up, and those to the running sums; every
// other step multiplies the negated activations and is subtracted, because the bf16 products' sums are not
// rounded to nearest: their errors lean one way, and what the errors of many rows have in common does not
// average out behind the kernel as their values do (a 400-token prompt, whose attention averages 400 value
// rows: logits 3.4-3.8e-7 from 64 bits without this, 2.4-2.6e-7 with it, 2.5-2.7e-7 token by token). f32:
// 16 columns' products are summed from zero and added to the running sums, which carry their rounding
// errors along. The tile order and the rotation of the k-steps by weight tile are
// prefill.hip's (the row tiles of a weight tile run together on one XCD and stay in step).
// Bound: short lists by the weight stream (dim 2048, 64 experts, top-8, hidden 1024, f32: 12 tokens, about
// 51 experts, 166 + 86 us, 5.2 TB/s; 200 tokens, two row groups per tile, 297 + 153 us against 3936 + 1939
// us of per-pair GEMVs, of which the compensated sums take 58 + 26); long ones by the wave's own chain of
// LDS reads and products (bf16, dim 1600, 40 experts of 150 rows, hidden 800: 207 + 116 us, 440 TFLOP/s
// issued). Four waves per block, two blocks per CU: with eight-wave blocks (one per CU) every wave waits at
// each step's barrier, 22 + 27 against 18 + 17 us at dim 1000, hidden 330, 50 tokens; activations one step
// ahead instead of four: 26 + 31 us; tiles of 128 rows and eight waves: 307 against 217 us on the 150-row
// lists (spills).
// GR: bytes per weight load, from the rows' alignment (16, 4 or 2); the last k-step of a row may be partial.
template <int DT, int MATS, int RG, int GR, bool DENSE = false, int KS = 1>
__global__ __launch_bounds__(64 * kFullWaves * KS, 2) void grouped_full_kernel(const FullArgs a) {
    constexpr int ESZ = DT == RBT_DT_BF16 ? 2 : 4, KW = kFullWin / ESZ;  // columns per k-step
    constexpr int ROWS = 16 * RG, NT = 64 * kFullWaves, NCOL = (MATS == 2 ? 16 : 32) * kFullWaves;
    constexpr int PARTS = DT == RBT_DT_BF16 ? 3 : 1;
    constexpr int ABYTES = ROWS * kFullWin, STAGE = PARTS * ABYTES;  // LDS bytes of a part, of a k-step
    constexpr int UNITS = ROWS * 8, AU = (UNITS + NT - 1) / NT;     // activation units of KW / 8 columns
    constexpr int UL = KW / 32;                                      // 16-byte loads per unit
    constexpr int SLOTS = kFullAhead + 1;  // register sets of weights
    constexpr uint32_t kNegate = 0x80008000u;  // the sign bits of two bf16
    constexpr int AS = AU * UL > 2 ? 2 : SLOTS;  // register sets of activations (two where a set is large)
    __shared__ __align__(1024) uint8_t rings[KS * 2 * STAGE];
    const int kg = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);  // this wave's part of the k-steps
    const int tid = threadIdx.x - kg * NT, lane = tid & 63, W = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *ring = rings + kg * 2 * STAGE;
    int ntiles_n, total, e = 0, jt, il, row0, rows, n0, N = a.N, seg = 0;
    if constexpr (DENSE) {
        ntiles_n = 0;
#pragma unroll
        for (int s = 0; s < 3; ++s) ntiles_n += (a.seg_rows[s] + NCOL - 1) / NCOL;
        total = ntiles_n * ((a.T + ROWS - 1) / ROWS);
    } else {
        ntiles_n = (a.N + NCOL - 1) / NCOL;
        total = a.m_off[a.E] * ntiles_n;
    }
    const int range = (total + 7) >> 3;
    const int slot = (int)(blockIdx.x >> 3), tau = (int)(blockIdx.x & 7) * range + slot;
    if (slot >= range || tau >= total) return;
    if constexpr (DENSE) {
        const int mt = (a.T + ROWS - 1) / ROWS;
        jt = tau / mt;
        il = tau - jt * mt;
        row0 = il * ROWS;
        rows = min(ROWS, a.T - row0);
        int j = jt;
        while (seg < 2 && j >= (a.seg_rows[seg] + NCOL - 1) / NCOL) {
            j -= (a.seg_rows[seg] + NCOL - 1) / NCOL;
            ++seg;
        }
        n0 = j * NCOL;
        N = a.seg_rows[seg];
    } else {
        tile_of(tau, a.m_off, a.E, a.m_off[a.E], ntiles_n, (__builtin_amdgcn_readfirstlane(*a.choice) >> 1) & 1, &e, &jt, &il);
        row0 = a.offsets[e] + il * ROWS;
        rows = __builtin_amdgcn_readfirstlane(min(ROWS, a.counts[e] - il * ROWS));
        n0 = jt * NCOL;
    }
    const int rowb = a.Kd * ESZ;  // bytes per weight row
    const int nch = (rowb + kFullWin - 1) / kFullWin;
    const int rot = (e + jt * max(1, nch / ntiles_n)) % nch;
    const int nst = nch / KS, first = (rot + kg * nst) % nch;  // k-steps of this wave (nch a multiple of KS)
    auto cidx = [&](int c) { return c + first < nch ? c + first : c + first - nch; };

    // weight rows of this lane: column group g, half s2 (rows 8 s2 .. 8 s2 + 7 of the group's 16), as buffer loads
    // from the tile's first row on: rows past the matrix, columns past the row and steps past the last get an
    // offset past the buffer's end, which reads as zeros without a request
    __amdgpu_buffer_rsrc_t rw[2];
    uint32_t wrow[2][2];
    const int woff = 16 * blob_chunk(lane);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const uint8_t *base = DENSE ? a.seg_w[seg] : a.experts + (size_t)e * a.stride + (MATS == 2 && g ? a.w3_off : a.w_off);
        rw[g] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base) + (size_t)n0 * (size_t)rowb, 0,
                                                  (int)((uint32_t)(N - n0) * (uint32_t)rowb), kBufConfig);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
            wrow[g][s2] = (uint32_t)((MATS == 2 ? 16 * W : 32 * W + 16 * g) + 8 * s2 + (lane & 7)) * (uint32_t)rowb;
    }
    // activation units of this thread: row u / 8, granule u % 8 of the step's KW columns
    const size_t base_row = !DENSE && a.gather ? 0 : (size_t)row0;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.act) + base_row * (size_t)a.act_stride, 0, kWrBufRecords, kBufConfig);
    uint32_t aoff[AU], adst[AU];
    int acol[AU];
#pragma unroll
    for (int i = 0; i < AU; ++i) {
        const int u = tid + NT * i, r = u >> 3, g = u & 7;
        const int lr = row0 + (r < rows ? r : 0);
        const size_t arow = !DENSE && a.gather ? (size_t)(a.perm[lr] / a.topk) : (size_t)lr;
        acol[i] = (KW / 8) * g;
        aoff[i] = r < rows ? (uint32_t)((arow - base_row) * a.act_stride + acol[i]) * 4u : (uint32_t)kWrBufRecords;
        adst[i] = (uint32_t)(r * kFullWin + 16 * (g ^ ((r >> 1) & 7)));
    }

    u32x4 aset[AS][AU][UL];
    u32x4 wv[SLOTS][2][2];
    auto load_a = [&](u32x4 (&av)[AU][UL], int c) {
        const int k0 = c < nst ? KW * cidx(c) : a.Kd;  // steps past the last: zeros, without a request
#pragma unroll
        for (int i = 0; i < AU; ++i)
#pragma unroll
            for (int j = 0; j < UL; ++j) {
                uint32_t off = aoff[i] + (uint32_t)(k0 + 4 * j) * 4u;
                if (k0 + acol[i] + 4 * j >= a.Kd) off = (uint32_t)kWrBufRecords;  // past the row: zeros
                av[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0);
            }
    };
    auto store_a = [&](const u32x4 (&av)[AU][UL], int buf, uint32_t flip) {
        uint8_t *st = ring + buf * STAGE;
#pragma unroll
        for (int i = 0; i < AU; ++i) {
            if (UNITS % NT != 0 && tid + NT * i >= UNITS) continue;
            if constexpr (PARTS == 1) {
                *reinterpret_cast<u32x4 *>(st + adst[i]) = av[i][0];
            } else {
                u32x4 p[3];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t x0[3], x1[3];
                    split3(__uint_as_float(av[i][j >> 1][2 * (j & 1)]), x0[0], x0[1], x0[2]);
                    split3(__uint_as_float(av[i][j >> 1][2 * (j & 1) + 1]), x1[0], x1[1], x1[2]);
#pragma unroll
                    for (int q = 0; q < 3; ++q) p[q][j] = pack_hi16(x0[q], x1[q]) ^ flip;
                }
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4 *>(st + q * ABYTES + adst[i]) = p[q];
            }
        }
    };
    auto load_w = [&](u32x4 (&dst)[2][2], int c) {
        const int off = c < nst ? cidx(c) * kFullWin + woff : rowb;
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                auto at = [&](int o) { return (int)(o < rowb ? wrow[g][s2] + (uint32_t)o : (uint32_t)kPastWeights); };
                if constexpr (GR == 16) {
                    dst[g][s2] = __builtin_amdgcn_raw_buffer_load_b128(rw[g], at(off), 0, kBufStream);
                } else if constexpr (GR == 4) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        dst[g][s2][j] = __builtin_amdgcn_raw_buffer_load_b32(rw[g], at(off + 4 * j), 0, kBufStream);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint16_t w0 = __builtin_amdgcn_raw_buffer_load_b16(rw[g], at(off + 4 * j), 0, kBufStream);
                        const uint16_t w1 = __builtin_amdgcn_raw_buffer_load_b16(rw[g], at(off + 4 * j + 2), 0, kBufStream);
                        dst[g][s2][j] = (uint32_t)w0 | ((uint32_t)w1 << 16);
                    }
                }
            }
    };

    // bf16: mid holds the sums of the last steps, acc of everything before them; f32: the sums, and what
    // their adds rounded away
    f32x4 acc[RG][2], mid[RG][2];
#pragma unroll
    for (int q = 0; q < RG; ++q) acc[q][0] = acc[q][1] = mid[q][0] = mid[q][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto flush = [&]() {
#pragma unroll
        for (int q = 0; q < RG; ++q)
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                acc[q][g] += mid[q][g];
                mid[q][g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
    };

    // k-step c, its operands in slot J = c % SLOTS. Loads return in issue order and a wait covers every older
    // load, so a step issues activations (AS steps ahead, stored to LDS one step ahead) before weights
    // (kFullAhead steps ahead): the LDS store waits for activations issued AS - 1 steps ago and not for
    // the weights behind them. Every load is issued in every step, past the last one too (no branches, so the
    // waits stay exact, and one copy of the steps: the code of a second, branching set for the last steps
    // was fetched anew by every block).
    auto step = [&](auto jc, int c) {
        constexpr int J = decltype(jc)::value;
        store_a(aset[(J + 1) % AS], (c + 1) & 1, J & 1 ? 0u : kNegate);  // the buffer that step c - 1 read
        load_a(aset[J % AS], c + AS);
        load_w(wv[(J + kFullAhead) % SLOTS], c + kFullAhead);
        const uint8_t *st = ring + (c & 1) * STAGE;
        blob_operands(wv[J][0][0], wv[J][0][1]);
        blob_operands(wv[J][1][0], wv[J][1][1]);
#pragma unroll
        for (int q = 0; q < RG; ++q) {
            if (16 * q < rows) {  // wave-uniform: the row group holds list entries
                const int r = 16 * q + (lane & 15);
                f32x4 t[2] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
                const uint8_t *ap[2];
#pragma unroll
                for (int s2 = 0; s2 < 2; ++s2) ap[s2] = st + r * kFullWin + 16 * ((4 * s2 + (lane >> 4)) ^ ((r >> 1) & 7));
                if constexpr (DT == RBT_DT_BF16) {
#pragma unroll
                    for (int p = PARTS - 1; p >= 0; --p)  // the small parts first
#pragma unroll
                        for (int s2 = 0; s2 < 2; ++s2) {
                            const bf16x8 x = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(ap[s2] + p * ABYTES));
#pragma unroll
                            for (int g = 0; g < 2; ++g)
                                t[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(bf16x8, wv[J][g][s2]),
                                                                               t[g], 0, 0, 0);
                        }
                } else {
#pragma unroll
                    for (int s2 = 0; s2 < 2; ++s2) {
                        const u32x4 x = *reinterpret_cast<const u32x4 *>(ap[s2]);
                        t[0] = t[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int g = 0; g < 2; ++g)
                                t[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(x[i]),
                                                                            __uint_as_float(wv[J][g][s2][i]), t[g], 0, 0, 0);
#pragma unroll
                        for (int g = 0; g < 2; ++g) {
#pragma clang fp reassociate(off)
                            const f32x4 was = acc[q][g];
                            acc[q][g] = was + t[g];
                            mid[q][g] += t[g] - (acc[q][g] - was);  // what the sum rounded away
                        }
                    }
                }
                if constexpr (DT == RBT_DT_BF16) {
                    mid[q][0] = J & 1 ? mid[q][0] - t[0] : mid[q][0] + t[0];
                    mid[q][1] = J & 1 ? mid[q][1] - t[1] : mid[q][1] + t[1];
                }
            }
        }
        __syncthreads();
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    static_assert(SLOTS == 4 && kFullAhead == 3, "one step call per slot below");
    // prologue, in the steady state's order
#pragma unroll
    for (int p = 0; p < SLOTS; ++p) {
        if (p < AS) load_a(aset[p % AS], p);
        if (p < kFullAhead) load_w(wv[p], p);
    }
    store_a(aset[0], 0, 0u);
    __syncthreads();
    for (int c = 0;; c += SLOTS) {
        step(I0{}, c);
        if (c + 1 >= nst) break;
        step(I1{}, c + 1);
        if (c + 2 >= nst) break;
        step(I2{}, c + 2);
        if (c + 3 >= nst) break;
        step(I3{}, c + 3);
        if (DT == RBT_DT_BF16 && (c & SLOTS)) flush();
        if (c + SLOTS >= nst) break;
    }
    flush();

    if constexpr (KS > 1) {  // the parts' sums meet in the first part's waves, through the (idle) rings
        static_assert(KS == 2 && 2 * STAGE * KS >= kFullWaves * RG * 2 * 64 * 16, "two parts, exchange in the rings");
        f32x4 *xch = reinterpret_cast<f32x4 *>(rings);  // [wave][q][g][lane]
        if (kg == 1) {
#pragma unroll
            for (int q = 0; q < RG; ++q)
#pragma unroll
                for (int g = 0; g < 2; ++g) xch[((W * RG + q) * 2 + g) * 64 + lane] = acc[q][g];
        }
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int q = 0; q < RG; ++q)
#pragma unroll
            for (int g = 0; g < 2; ++g) acc[q][g] += xch[((W * RG + q) * 2 + g) * 64 + lane];
    }
    // acc[q][g] lane holds column (lane % 16) of group g for list rows 16 q + 4 (lane / 16) + i
    auto row_of = [&](int r) { return DENSE ? a.seg_out[seg] + (size_t)(row0 + r) * N : a.out + (size_t)(row0 + r) * a.out_stride; };
    // A sum that is NaN is taken again below, product by product, as the GEMVs and the engine add: the lower parts
    // of an activation can be 0 where it is not (0 times an infinite weight), and where a sum overflows, what its
    // add rounded away is inf - inf.
    uint32_t nan = 0;  // this lane's (bit 8 q + 4 g + i)
    float z = 0.0f;
#pragma unroll
    for (int q = 0; q < RG; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) z += 0.0f * acc[q][0][i] + 0.0f * acc[q][1][i];
    if (__builtin_expect(__any(z != 0.0f), 0)) {
#pragma unroll
        for (int q = 0; q < RG; ++q)
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (acc[q][g][i] != acc[q][g][i]) {
                        nan |= 1u << (8 * q + 4 * g + i);
                        acc[q][g][i] = 0.0f;
                    }
    }
#pragma unroll
    for (int q = 0; q < RG; ++q) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * q + 4 * (lane >> 4) + i;
            if (r >= rows) continue;
            float *orow = row_of(r);
            if constexpr (MATS == 2) {
                const int n = n0 + 16 * W + (lane & 15);
                const float g = acc[q][0][i], u = acc[q][1][i];
                // silu(g) * u, rabbit2.c:535-537; the columns that pad the row are zeros
                if (n < a.out_stride) orow[n] = n < a.N ? (g / (1.0f + expf(-g))) * u : 0.0f;
            } else {
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const int n = n0 + 32 * W + 16 * g + (lane & 15);
                    const float y = acc[q][g][i];
                    if (n < N) orow[n] = DENSE && a.resid ? orow[n] + y : y;
                }
            }
        }
    }
    if (__builtin_expect(!__any(nan != 0), 1)) return;
    // its (only) argument is read anew here: kept in registers through the steps for this, it cost the down product
    // of dim 1000, hidden 330, 50 tokens 0.8 of 16.5 us
    const __attribute__((address_space(4))) FullArgs *ap =
        (const __attribute__((address_space(4))) FullArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ap));
    if (MATS == 2) nan = (nan | nan >> 4) & 0x0F0F0F0Fu;  // one output of both sums
    for (; nan; nan &= nan - 1) {
        const int at = __builtin_ctz(nan), g = (at >> 2) & 1, r = 16 * (at >> 3) + 4 * (lane >> 4) + (at & 3);
        const int n = n0 + (MATS == 2 ? 16 * W : 32 * W + 16 * g) + (lane & 15);
        if (r >= rows || n >= N) continue;
        const float *x = ap->act + (!DENSE && ap->gather ? (size_t)(ap->perm[row0 + r] / ap->topk) : (size_t)(row0 + r)) * ap->act_stride;
        const uint8_t *w = (DENSE ? ap->seg_w[seg] : ap->experts + (size_t)e * ap->stride + ap->w_off) + (size_t)n * ap->Kd * ESZ;
        float y = 0.0f, u = 0.0f;
        for (int k = 0; k < ap->Kd && (y == y || u == u); ++k) {
            y += rbt::load_w<DT>(w, k) * x[k];
            if constexpr (MATS == 2) u += rbt::load_w<DT>(w + (ap->w3_off - ap->w_off), k) * x[k];
            else u = y;
        }
        float *o = row_of(r) + n;
        if constexpr (MATS == 2)
            *o = (y / (1.0f + expf(-y))) * u;
        else
            *o = DENSE && ap->resid ? *o + y : y;
    }
}

// Bytes per weight load that the rows of Kd elements from `base` on (rows and experts `step` apart) allow.
int load_granule(uint64_t base, uint64_t stride, int Kd, int esz) {
    const uint64_t bits = base | stride | (uint64_t)Kd * esz;
    return bits % 16 == 0 ? 16 : bits % 4 == 0 ? 4 : bits % 2 == 0 && esz == 2 ? 2 : 0;
}

template <int MATS, bool DENSE = false, int KS = 1>
hipError_t launch_full(const Launch &L, const FullArgs &a, int dtype, int rg, int max_mtiles) {
    constexpr int NCOL = (MATS == 2 ? 16 : 32) * kFullWaves;
    int ntiles_n = (a.N + NCOL - 1) / NCOL;
    uint64_t base = reinterpret_cast<uintptr_t>(a.experts) | a.w_off | a.w3_off;
    if (DENSE) {
        ntiles_n = 0;
        base = 0;
        for (int s = 0; s < 3; ++s) {
            ntiles_n += (a.seg_rows[s] + NCOL - 1) / NCOL;
            if (a.seg_rows[s]) base |= reinterpret_cast<uintptr_t>(a.seg_w[s]);
        }
    }
    const long long tiles = (long long)max_mtiles * ntiles_n, blocks = (tiles + 7) / 8 * 8;
    const int gr = load_granule(base, a.stride, a.Kd, dtype == RBT_DT_BF16 ? 2 : 4);
    if (blocks > 0x7FFFFFFFll || gr == 0) return hipErrorInvalidValue;
    const dim3 g((unsigned)blocks), b(64 * kFullWaves * KS);
#define FULL_CASE(DT, RG, GR) \
    if (dtype == DT && rg == RG && gr == GR) return launch(L, grouped_full_kernel<DT, MATS, RG, GR, DENSE, KS>, g, b, 0, a);
#define FULL_TILES(DT, GR) \
    FULL_CASE(DT, 2, GR)   \
    if constexpr (KS == 1) { FULL_CASE(DT, 4, GR) }
    FULL_TILES(RBT_DT_BF16, 16)
    FULL_TILES(RBT_DT_BF16, 4)
    FULL_TILES(RBT_DT_BF16, 2)
    FULL_TILES(RBT_DT_F32, 16)
    FULL_TILES(RBT_DT_F32, 4)
#undef FULL_TILES
#undef FULL_CASE
    return hipErrorInvalidValue;
}

// Mean list rows up to which tiles have 32 rows: half the LDS and 162 instead of 212 registers, and a list
// that passes 32 rows re-reads its weights from L2 (f32 200 tokens, 25 rows on average: 250 us either way;
// with +2 on eight experts' logits 304 against 384 us).
constexpr int kFullShortLists = 40;
constexpr int kDenseTallTiles = 256;  // dense form: 64-row tiles from which they are taken

}  // namespace

bool full_supported(int dtype, int T, int E, int K, int D, int H, const void *experts, uint64_t stride,
                    const float *xb) {
    const int esz = dtype == RBT_DT_BF16 ? 2 : 4;
    const uint64_t base = reinterpret_cast<uintptr_t>(experts);
    return T >= 1 && T <= 65535 && E <= kDispatchMaxE && (long long)T * K <= (1 << 24) && D % 4 == 0 &&
           (reinterpret_cast<uintptr_t>(xb) & 15u) == 0 && load_granule(base, stride, D, esz) != 0 &&
           load_granule(base, stride, H, esz) != 0 &&
           // 32-bit buffer offsets: the gathered rows of xb, a tile's rows of h, and a weight matrix
           (uint64_t)T * D * 4 < (uint64_t)kWrBufRecords && 128ull * full_h_stride(H) * 4 < (uint64_t)kWrBufRecords &&
           (uint64_t)D * H * esz < (uint64_t)kPastWeights / 2;
}

// The grouped form reads each selected expert once, the per-pair GEMVs once per pair; it has two more
// launches and longer kernels (~25 us at the smallest sizes). So it pays from a number of saved bytes on:
// pairs minus experts expected to be selected, times an expert's bytes. Measured, GEMVs / grouped, us:
//   f32, dim 2048, 64 experts, top-8, hidden 1024: 8 tokens (550 MB saved) 191 / 205, 11 (970 MB) 245 / 265,
//     200 5763 / 426
//   bf16, dim 1600, 40 experts, top-6, hidden 800: 2 tokens (12 MB) 46 / 60, 8 (150 MB) 110 / 79, 1000
//     11045 / 364
//   bf16, dim 1000, 20 experts, top-3, hidden 330: 11 tokens (32 MB) 40 / 57, 50 (260 MB) 98 / 61
// The shapes of the specialised GEMVs (experts_decode.hip) stream twice as fast and need more, and
// more again where their gate/up reads an expert once too and only W2 is read per pair.
bool full_pays(bool fast_gemv, int dtype, int T, int E, int K, int D, int H) {
    const double p = (double)T * K, sel = E * (1.0 - pow(1.0 - (double)K / E, (double)T));
    return (p - sel) * 3.0 * H * D * (dtype == RBT_DT_BF16 ? 2 : 4) >= (!fast_gemv ? 100e6 : gateup_reads_once(dtype, T, E, K, D, H) ? 1000e6 : 450e6);
}

size_t full_workspace_bytes(int T, int E, int K, int D) {
    const size_t P = (size_t)T * K;
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    return up(4 * (size_t)E) + 3 * up(4 * (size_t)(E + 1)) + up(8) + 2 * up(4 * P) + up(4 * P * (size_t)D);
}

bool dense_full_supported(int dtype, int T, int Kd, int rows, const float *x) {
    // row stride and alignment of x as the buffer loads need them; the model's tensors are 64-byte aligned
    return T >= 1 && T <= 65535 && Kd % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0 &&
           load_granule(0, 0, Kd, dtype == RBT_DT_BF16 ? 2 : 4) != 0 && 128ull * Kd * 4 < (uint64_t)kWrBufRecords &&
           (uint64_t)rows * Kd * (dtype == RBT_DT_BF16 ? 2 : 4) < (uint64_t)kPastWeights / 2;
}

hipError_t launch_dense_full(const Launch &L, int dtype, const float *x, int T, int Kd, const void *const W[3],
                             float *const out[3], const int rows[3], float *resid) {
    FullArgs a{};
    a.Kd = Kd;
    a.act = x;
    a.act_stride = Kd;
    a.T = T;
    a.resid = resid != nullptr;
    int tiles64 = 0;
    for (int s = 0; s < 3; ++s) {
        a.seg_w[s] = static_cast<const uint8_t *>(W[s]);
        a.seg_out[s] = resid ? resid : out[s];
        a.seg_rows[s] = rows[s];
        tiles64 += (rows[s] + 32 * kFullWaves - 1) / (32 * kFullWaves) * ((T + 63) / 64);
    }
    // Few tiles leave CUs idle, and a CU moves ~27 GB/s whatever its tile: short tiles then, with the k-steps in
    // two parts (dim 2048, us: wo of 400 rows 34 -> 29, of 24 rows 34 -> 29; q/k/v of 400 rows in 64-row tiles
    // 68 against 80)
    const int rg = tiles64 >= kDenseTallTiles ? 4 : 2, nch = (Kd * (dtype == RBT_DT_BF16 ? 2 : 4) + kFullWin - 1) / kFullWin;
    if (rg == 2 && nch % 2 == 0) return launch_full<1, true, 2>(L, a, dtype, 2, (T + 31) / 32);
    return launch_full<1, true>(L, a, dtype, rg, (T + 16 * rg - 1) / (16 * rg));
}

hipError_t launch_grouped_full(const Launch &Ld, const Launch &Lg, const Launch &Lw, const Launch &Lc, int dtype,
                               const void *experts, uint64_t stride, const float *xb, int T, int E, int K, int D, int H,
                               const int32_t *routing, const float *weights, float *hbuf, void *ws, float *x_inout,
                               float *moe_out, GroupedCall *call_out) {
    if (T <= 0 || K <= 0) return hipErrorInvalidValue;
    const int P = T * K;
    uint8_t *w = static_cast<uint8_t *>(ws);
    auto carve = [&](size_t bytes) {
        uint8_t *p = w;
        w += (bytes + 255) / 256 * 256;
        return p;
    };
    int32_t *counts = reinterpret_cast<int32_t *>(carve(4 * (size_t)E));
    int32_t *offsets = reinterpret_cast<int32_t *>(carve(4 * (size_t)(E + 1)));
    int32_t *m_off = reinterpret_cast<int32_t *>(carve(4 * (size_t)(E + 1)));
    int32_t *m_off128 = reinterpret_cast<int32_t *>(carve(4 * (size_t)(E + 1)));  // written by the dispatch, not used
    int32_t *choice = reinterpret_cast<int32_t *>(carve(8));
    int32_t *perm = reinterpret_cast<int32_t *>(carve(4 * (size_t)P));
    int32_t *pos_of = reinterpret_cast<int32_t *>(carve(4 * (size_t)P));
    float *y = reinterpret_cast<float *>(carve(4 * (size_t)P * D));
    const int rg = P <= kFullShortLists * E ? 2 : 4;
    if (call_out) *call_out = GroupedCall{counts, 16 * rg, nullptr};
    hipError_t e = launch_dispatch(Ld, routing, P, E, counts, offsets, perm, pos_of, m_off, 16 * rg, m_off128,
                                   choice, 2, PlanShape{}, reinterpret_cast<int32_t *>(y));
    if (e != hipSuccess) return e;
    const int max_mtiles = (P + 16 * rg - 1) / (16 * rg) + E;  // >= sum over experts of ceil(count / (16 rg))
    const uint64_t mat = (uint64_t)H * D * (dtype == RBT_DT_BF16 ? 2 : 4);
    const int hs = full_h_stride(H);
    const uint8_t *ex = static_cast<const uint8_t *>(experts);
    FullArgs a{ex, stride, 0, mat, H, D, xb, D, 1, perm, K, counts, offsets, m_off, choice, E, hbuf, hs, {}, {}, {}, 0, 0};
    e = launch_full<2>(Lg, a, dtype, rg, max_mtiles);
    if (e != hipSuccess) return e;
    a = FullArgs{ex, stride, 2 * mat, 0, D, H, hbuf, hs, 0, perm, K, counts, offsets, m_off, choice, E, y, D, {}, {}, {}, 0, 0};
    e = launch_full<1>(Lw, a, dtype, rg, max_mtiles);
    if (e != hipSuccess) return e;
    return launch_combine(Lc, y, pos_of, weights, T, K, D, x_inout, moe_out);
}

}  // namespace rbt
