// FP32 GEMMs on the BF16 matrix units: every operand element is split into three BF16 terms on its way
// into LDS (split_bf16x3: 24 significand bits), and a product takes the six term products down to
// 2^-16 of the whole, accumulated in FP32. The FP32 units reach 157 TFLOP/s; six BF16 products per
// FP32 product 417 at the nominal BF16 rate and 204 at the rate that a large BF16 product reaches on
// this card (1223).
//
// Design (per k-tile of 32):
//   * global -> registers with 128-bit buffer loads (k-contiguous operands: 4 k of a row; mn-contiguous
//     ones: 2 or 4 k-rows x 4 columns, so that the split, which packs pairs of k, transposes on the
//     way). A descriptor ends at the operand's last element and its range check, dword by dword,
//     supplies the zeros past it; the loads need no more than an element's alignment. So every size
//     and leading dimension runs the same loop (a 1000 x 300 x 701 layer forward and backward: 53 us
//     with the FP32-unit kernels, whose loads go element by element there, 41 here);
//   * split, then three LDS planes [rows][32 k] of 64-byte rows; a lane's fragment of one term is one
//     128-bit LDS read;
//   * v_mfma_f32_16x16x32_bf16 blocks (the 32x32x16 form measured 2-6% slower in these tiles);
//   * one LDS stage and two barriers per k-tile (gemm_f32_block), so that several blocks share a CU;
//   * an accumulator that is not finite is computed again on the FP32 units, since the terms of an
//     infinity (or of a value that rounds up to 2^112: the terms are scaled) are NaN.
#include <cstdio>
#include <string>

#include "gemm_tiles.hpp"

namespace it {
namespace {

// One operand's k-tile: global -> registers -> LDS terms, and LDS -> MFMA fragments.
//   KCONTIG: global element (r, k) at base[r * ld + k] (A not transposed, or B transposed).
//   otherwise: global element (r, k) at base[k * ld + r].
template <bool KCONTIG_, int ROWS, int THREADS>
struct F32Operand {
    static constexpr bool KCONTIG = KCONTIG_;
    static constexpr int NT = THREADS;
    static constexpr int VEC = 4, BK = ET<float>::BK;
    static constexpr int PLANE = ROWS * 64;  // bytes of one term's plane
    static constexpr int STAGE_BYTES = 3 * PLANE;
    // k-rows of an mn-contiguous unit: 2 where 4 would leave threads without a unit.
    static constexpr int KQ = (BK / 4) * (ROWS / VEC) < THREADS ? 2 : 4;
    static constexpr int KGROUPS = BK / KQ;
    static constexpr int LOADS = KCONTIG ? 1 : KQ;
    static constexpr int ITEMS = KCONTIG ? ROWS * BK / VEC : KGROUPS * (ROWS / VEC);
    static constexpr int ITERS = (ITEMS + THREADS - 1) / THREADS;

    u32x4 reg[ITERS][LOADS];

    // mn-contiguous units: (k-group of KQ rows, 4 columns), the k-groups fastest.
    __device__ __forceinline__ static void unit(int item, int &kg, int &rc) {
        kg = item % KGROUPS;
        rc = item / KGROUPS;
    }

    // Byte of k position kb / 2 (kb: byte in the 64-byte row) of `row` in a plane. Rows swap places
    // within groups of 4 by the group's number, and a row's 16-byte chunks by its place: measured, a
    // fragment's 128-bit reads (16 rows, 4 chunks) then go at 203 bytes per clock and CU, as linear
    // ones do (122 without the chunk swap), and every write pattern (8 bytes of consecutive rows or
    // of rows 4 apart, 4 bytes of rows 4 apart) at its linear rate (65, 50).
    __device__ __forceinline__ static int off(int row, int kb) {
        const int q = (row & ~3) | ((row ^ (row >> 2)) & 3);
        return q * 64 + ((((kb >> 4) ^ (q >> 1)) & 3) << 4) + (kb & 15);
    }

    // Zeros the elements of a k-contiguous tile at k positions from `left` on (its row's next
    // elements, or the next row's).
    __device__ __forceinline__ void mask(int64_t left, int tid) {
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int kc = (tid + it * THREADS) % (BK / VEC);
#pragma unroll
            for (int e = 0; e < 4; ++e) reg[it][0][e] = kc * VEC + e < left ? reg[it][0][e] : 0u;
        }
    }

    // Softmax cross-entropy gradient of FP32 logits (the A operand of dL/dh = G.E or dL/dE = G^T.h): the
    // loaded logits x become (exp(x - max) / sum - onehot) * scale before the split, the exponential
    // as 2^((x - max) log2 e). Tokens are rows of a k-contiguous tile, whose {max, scale / sum, target}
    // wait in LDS, and k-rows of an mn-contiguous one, whose statistics come with the tile's loads.
    struct Xent {
        const f32x4 *row;  // k-contiguous: per tile row {max, scale / sum, target's bits, -}
        int64_t c0;        // the tile's first class
        int left;          // k-contiguous: classes from there on (elements past them are zeros)
        float scale;
    };
    float2 xs[KCONTIG ? 1 : ITERS][LOADS];
    uint32_t xt[KCONTIG ? 1 : ITERS][LOADS];

    __device__ __forceinline__ void load_xent(const float2 *st, const uint32_t *tg, float scale, int64_t k0,
                                              int64_t klim, int tid) {
        static_assert(!KCONTIG, "a k-contiguous tile's tokens are its rows");
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            int kg, rc;
            unit(tid + it * THREADS, kg, rc);
#pragma unroll
            for (int q = 0; q < LOADS; ++q) {
                const int64_t tok = k0 + kg * KQ + q;
                const bool ok = tok < klim;  // tokens past the end: zeros
                const float2 s = st[ok ? tok : klim - 1];
                const uint32_t t = tg[ok ? tok : klim - 1];
                xs[it][q] = {ok ? s.x : INFINITY, ok ? s.y * scale : 0.f};
                xt[it][q] = ok ? t : 0xffffffffu;
            }
        }
    }

    __device__ __forceinline__ static uint32_t xent(uint32_t x, float mx, float ps, bool target, float scale) {
        constexpr float LOG2E = 1.4426950408889634f;
        const float g = __builtin_amdgcn_exp2f((__uint_as_float(x) - mx) * LOG2E) * ps - (target ? scale : 0.f);
        return __float_as_uint(g);
    }

    // Splits and writes part `part` of `parts` of the tile (the caller interleaves them with MFMAs).
    template <bool XF = false>
    __device__ __forceinline__ void store(char *lds, int tid, int part, int parts, const Xent &x = Xent{}) const {
        constexpr int PIECES = KCONTIG ? ITERS : 4 * ITERS;
        auto mine = [&](int piece) { return piece * parts / PIECES == part; };
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int item = tid + it * THREADS;
            if (ITEMS % THREADS != 0 && item >= ITEMS) continue;
            if constexpr (KCONTIG) {
                if (!mine(it)) continue;
                const int rr = item / (BK / VEC), kc = item % (BK / VEC);
                u32x4 v = reg[it][0];
                if constexpr (XF) {
                    const f32x4 t = x.row[rr];
                    const int c = kc * VEC, tc = (int)(__float_as_uint(t[2]) - (uint32_t)x.c0);  // target's k in the tile
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = c + e < x.left ? xent(v[e], t[0], t[1], tc == c + e, x.scale) : 0u;
                }
                const Bf16x3 a = split_bf16x3(v[0], v[1]), b = split_bf16x3(v[2], v[3]);
                char *d = lds + off(rr, kc * 8);
#pragma unroll
                for (int p = 0; p < 3; ++p) *(u32x2 *)(d + p * PLANE) = u32x2{a.t[p], b.t[p]};
            } else {
                int kg, rc;
                unit(item, kg, rc);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (!mine(it * 4 + j)) continue;
                    char *d = lds + off(rc * 4 + j, kg * KQ * 2);
                    uint32_t v[LOADS];
#pragma unroll
                    for (int q = 0; q < LOADS; ++q) {
                        v[q] = reg[it][q][j];
                        if constexpr (XF)
                            v[q] = xent(v[q], xs[it][q].x, xs[it][q].y, xt[it][q] == (uint32_t)(x.c0 + rc * VEC + j), x.scale);
                    }
                    const Bf16x3 a = split_bf16x3(v[0], v[1]);
                    if constexpr (KQ == 4) {
                        const Bf16x3 b = split_bf16x3(v[2], v[3]);
#pragma unroll
                        for (int p = 0; p < 3; ++p) *(u32x2 *)(d + p * PLANE) = u32x2{a.t[p], b.t[p]};
                    } else {
#pragma unroll
                        for (int p = 0; p < 3; ++p) *(uint32_t *)(d + p * PLANE) = a.t[p];
                    }
                }
            }
        }
    }

    // Term p of the v_mfma_f32_16x16x32_bf16 fragment of the 16 rows from `row` (a multiple of 16):
    // lane l holds row l % 16 at k 8 (l / 16) .. +7.
    __device__ __forceinline__ static u32x4 frag(const char *lds, int row, int p, int lane) {
        return *(const u32x4 *)(lds + p * PLANE + row * 64 + off(lane & 15, (lane >> 4) * 16));
    }
};

// The loads of an operand tile O: a descriptor from the tile's first element to the operand's last,
// each item's byte offset, formed once per block, and the k-tile's as the load's scalar offset, so a
// load costs no vector instruction besides itself. Past the end the range check returns zeros: rows
// past M or N of a k-contiguous operand, k past K of an mn-contiguous one. An mn-contiguous operand's
// columns past M (or N) read the next row's elements; they reach only outputs that are not stored.
template <class O>
struct TileLoad {
    __amdgpu_buffer_rsrc_t rs;
    uint32_t voff[O::ITERS][O::LOADS];
    uint32_t kstride;

    // base: the operand of this batch item, rows x K; r0: the tile's first row.
    __device__ __forceinline__ void init(const float *base, int64_t ld, int64_t rows, int64_t K, int64_t r0, int tid) {
        const int64_t skip = O::KCONTIG ? r0 * ld : r0;
        const int64_t left = (O::KCONTIG ? (rows - 1) * ld + K : (K - 1) * ld + rows) - skip;
        const int n = left > 0x1fffffff ? 0x7fffffff : (int)(left * 4);
        rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base + skip), (short)0, n, 0x00020000);
        kstride = O::KCONTIG ? 4u : (uint32_t)(ld * 4);
#pragma unroll
        for (int it = 0; it < O::ITERS; ++it) {
            const int item = tid + it * O::NT;
            if constexpr (O::KCONTIG) {
                const int rr = item / (O::BK / O::VEC), kc = item % (O::BK / O::VEC);
                voff[it][0] = (uint32_t)((rr * ld + kc * O::VEC) * 4);
            } else {
                int kg, rc;
                O::unit(item, kg, rc);
#pragma unroll
                for (int q = 0; q < O::LOADS; ++q)
                    voff[it][q] = (uint32_t)(((kg * O::KQ + q) * ld + rc * O::VEC) * 4);
            }
        }
    }

    __device__ __forceinline__ void load(O &o, int64_t k0, int tid) const {
        const uint32_t koff = (uint32_t)k0 * kstride;
#pragma unroll
        for (int it = 0; it < O::ITERS; ++it) {
            const int item = tid + it * O::NT;
            if (O::ITEMS % O::NT != 0 && item >= O::ITEMS) continue;
#pragma unroll
            for (int q = 0; q < O::LOADS; ++q)
                o.reg[it][q] =
                    __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[it][q], koff, 0));
        }
    }
};

// Byte offsets from a tile's start within 31 bits: a k-contiguous operand's rows, or an mn-contiguous
// one's k range (with the k-tile past its end that a block reads ahead).
bool spans_fit(const GemmArgs &a, bool ta, bool tb) {
    auto fits = [&](bool kcontig, int64_t ld) { return (kcontig ? 256 * ld + a.K : (a.K + 64) * ld) * 4 < (1ll << 31); };
    return fits(!ta, a.lda) && fits(tb, a.ldb);
}

// The tile shapes: BM x BN output tiles of WM x WN waves, times KG groups of them, each with its own
// LDS stage, that take every KG-th k-tile (group 0 adds the others' sums and finishes the tile).
template <int BM_, int BN_, int WM_, int WN_, int KG_ = 1>
struct Shape {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, KG = KG_;
    static constexpr int THREADS = WM * WN * 64;  // of one k group
    static constexpr bool WIDE = BM * BN / (WM * WN) >= 64 * 64;
    // Waves per SIMD the registers are held to.
    static constexpr int WAVES = WIDE ? 2 : KG > 1 ? 4 : 3;
    static constexpr int SMEM = 3 * 64 * (BM + BN);
};
using S128 = Shape<128, 128, 2, 2>;      // 64 x 64 per wave, two blocks per CU
using S256 = Shape<256, 128, 4, 2>;      // the same per wave, one block per CU
using S64 = Shape<64, 64, 2, 2>;         // 32 x 32 per wave, three blocks per CU
using S6432 = Shape<64, 32, 2, 2, 2>;    // 32 x 16 per wave, two blocks of eight waves per CU

// One block: output tile `tile` (in map_tile order) of batch-and-split index z, with `smem0` of KG *
// S::SMEM bytes.
// DUAL: the B tile's rows 0..BN/2-1 are gate-weight rows and BN/2..BN-1 the same up-weight rows.
// FIX (64 x 64 tiles of batch-1 products): with split K, each split's partial tile goes to p.partial
// at device scope and the tile's last block to arrive at `arrive` (a zero counter, left at zero)
// adds the splits in split order and runs the epilogue, so no separate reduction launch follows.
// XF: A is the softmax cross-entropy gradient of the logits it holds (F32Operand::Xent).
template <class S, bool TA, bool TB, bool DUAL, bool FIX = false, bool XF = false>
__device__ __forceinline__ void gemm_f32_block(const GemmArgs &p, int tile, int64_t z, char *smem0,
                                               int *arrive = nullptr) {
    constexpr int BM = S::BM, BN = S::BN, WM = S::WM, WN = S::WN, KG = S::KG, THREADS = S::THREADS;
    constexpr int BK = ET<float>::BK;
    constexpr int WTM = BM / WM, WTN = BN / WN, FM = WTM / 16, FN = WTN / 16;
    static_assert(KG == 1 || (BM == 64 && !DUAL && !FIX && !XF), "k groups: plain products");
    static_assert(!XF || (!TB && !DUAL && !FIX), "cross-entropy operand: one product, B not transposed");
    // Tiles of 64 rows store straight from transposed accumulators; larger ones stage the epilogue
    // through LDS, whose full-line stores suit outputs of hundreds of megabytes; SwiGLU pairs waves
    // in LDS.
    constexpr bool XPOSE = !DUAL && BM == 64;
    using OA = F32Operand<!TA, BM, THREADS>;
    using OB = F32Operand<TB, BN, THREADS>;
    using OBL = F32Operand<TB, DUAL ? BN / 2 : BN, THREADS>;  // as loaded (DUAL: the gate or up half)
    static_assert(!DUAL || (!TA && TB && WTN == BN / 2), "SwiGLU is Y = X.W^T, a wave's columns all gate or all up");
    constexpr int SA = OA::STAGE_BYTES;

    const int tid = threadIdx.x % THREADS, lane = tid & 63, wave = tid >> 6;
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / THREADS);
    const int wm = wave / WN, wn = wave % WN;
    char *const smem = KG == 1 ? smem0 : smem0 + kg * S::SMEM;
    int tm, tn;
    map_tile(tile, p.tiles_m, p.tiles_n, tm, tn);
    const int64_t b = z % p.batch, split = z / p.batch;
    const int64_t bo = b / p.batch_inner, bi = b % p.batch_inner;
    const float *A = (const float *)p.A + bo * p.sA_out + bi * p.sA_in;
    const float *B = (const float *)p.B + bo * p.sB_out + bi * p.sB_in;
    const float *B2 = DUAL ? (const float *)p.B2 + bo * p.sB_out + bi * p.sB_in : nullptr;
    const int64_t coff = bo * p.sC_out + bi * p.sC_in;
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * (DUAL ? BN / 2 : BN);

    if (p.causal != CAUSAL_NONE && n0 > m0 + BM - 1 + p.causal_offset) {
        // Entire tile is above the diagonal: no products needed.
        if (p.causal == CAUSAL_WRITE) {
            for (int e = threadIdx.x; e < BM * BN; e += THREADS * KG) {
                const int64_t row = m0 + e / BN, col = n0 + e % BN;
                if (row < p.M && col < p.N) store_out(p.C, coff + row * p.ldc + col, -INFINITY, p.out_bf16);
            }
        }
        return;
    }

    int64_t kb = split * p.k_per_split;
    int64_t ke = min(p.K, kb + p.k_per_split);
    if (p.kmode == KMODE_LOWER) ke = min(ke, m0 + BM);
    if (p.kmode == KMODE_UPPER) kb = max(kb, (m0 / BK) * BK);
    const int ntiles = ke > kb ? (int)((ke - kb + BK - 1) / BK) : 0;

    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = zero;

    // Register staging sets: PF of them, so that a k-tile's loads go out PF tiles before its split.
    // The 64 x 64 tile has room for two, which a block alone on its CU needs (measured [4096, 256,
    // 16384]: 544 -> 302 us unsplit).
    constexpr int PF = S::WIDE || KG > 1 ? 1 : 2;
    OA oa[PF];
    OBL ob[PF];
    std::conditional_t<DUAL, OBL, char> ob2[PF];
    TileLoad<OA> ra;
    TileLoad<OBL> rb, rb2;
    ra.init(A, p.lda, p.M, p.K, m0, tid);
    rb.init(B, p.ldb, p.N, p.K, n0, tid);
    if constexpr (DUAL) rb2.init(B2, p.ldb, p.N, p.K, n0, tid);
    __shared__ f32x4 xrow[XF && !TA ? BM : 1];
    if constexpr (XF && !TA) {
        for (int r = tid; r < BM; r += THREADS) {
            const int64_t tok = min(m0 + r, p.M - 1);
            const float2 st = p.xent_stats[tok];
            xrow[r] = f32x4{st.x, st.y * p.xent_scale, __uint_as_float(p.xent_tgt[tok]), 0.f};
        }
        __syncthreads();
    }
    auto gload = [&](int set, int64_t k0) {
#pragma unroll
        for (int q = 0; q < PF; ++q)
            if (q == set) {
                ra.load(oa[q], k0, tid);
                if constexpr (XF && TA) oa[q].load_xent(p.xent_stats, p.xent_tgt, p.xent_scale, k0, ke, tid);
                rb.load(ob[q], k0, tid);
                if constexpr (DUAL) rb2.load(ob2[q], k0, tid);
            }
    };
    // Part `part` of `parts` of a register set's split and LDS writes; k0: its k-tile. A k-contiguous
    // operand's elements past K (the next row's) are zeroed, in both operands: one that is not finite
    // would cost the wave its second computation.
    auto gstore = [&](int set, int64_t k0, int part, int parts) {
#pragma unroll
        for (int q = 0; q < PF; ++q)
            if (q == set) {
                if (part == 0 && k0 + BK > ke) {
                    if constexpr (!TA && !XF) oa[q].mask(ke - k0, tid);
                    if constexpr (TB) ob[q].mask(ke - k0, tid);
                    if constexpr (DUAL) ob2[q].mask(ke - k0, tid);
                }
                if constexpr (XF)
                    oa[q].template store<true>(smem, tid, part, parts, {xrow, TA ? m0 : k0, (int)min(ke - k0, (int64_t)BK), p.xent_scale});
                else
                    oa[q].store(smem, tid, part, parts);
                ob[q].store(smem + SA, tid, part, parts);
                if constexpr (DUAL) ob2[q].store(smem + SA + OBL::STAGE_BYTES, tid, part, parts);
            }
    };
    // XPOSE: B as the MFMA's row operand, the block comes out transposed.
    auto mul = [&](f32x4 &c, const u32x4 &a, const u32x4 &bb) {
        const bf16x8 av = __builtin_bit_cast(bf16x8, a), bv = __builtin_bit_cast(bf16x8, bb);
        c = XPOSE ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv, av, c, 0, 0, 0)
                  : __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, c, 0, 0, 0);
    };

    if (ntiles > 0) {
        // One LDS stage, two barriers per k-tile: a wave takes all its fragments of tile t into
        // registers, and once every wave has, tile t+1 is split and written over it between the
        // MFMAs of tile t, and the loads of tile t+1+PF go out. The last tile is read again at the
        // end, into a stage nobody reads.
        //
        // The matrix unit rounds its sum once per 8 products, and not evenly: sums drift down by
        // about 1e-8 of their size per 1000 roundings. So only the leading term product goes into
        // the running sums; the five small ones, 2^-8 of it and less, have sums of their own
        // (LOWSUM: for the whole k range; otherwise for one k-tile and strip of 16 rows at a time,
        // which takes fewer registers). Measured against 64 bits, N(0, 1) data: K = 256 9.0e-8, K =
        // 4096 2.2e-7 (the FP32 units, summing in k order: 2.9e-7 and 1.1e-6; all six products in
        // one sum: 2.3e-7 and 5.0e-7, with that drift).
        constexpr int QA[5] = {2, 0, 1, 1, 0}, QB[5] = {0, 2, 1, 0, 1};
        constexpr bool LOWSUM = !S::WIDE;
        f32x4 low[LOWSUM ? FM : 1][FN];
#pragma unroll
        for (int i = 0; i < (LOWSUM ? FM : 1); ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) low[i][j] = zero;
        const int last = ntiles - 1, nt = (ntiles + KG - 1) / KG;
        auto kt = [&](int t) { return kb + (int64_t)min(t * KG + kg, last) * BK; };
        u32x4 fa[3][FM], fb[3][FN];
        auto ktile = [&](int t, int set) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int i = 0; i < FM; ++i) fa[q][i] = OA::frag(smem, wm * WTM + i * 16, q, lane);
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    if constexpr (DUAL)
                        fb[q][j] = OBL::frag(smem + SA + wn * OBL::STAGE_BYTES, j * 16, q, lane);
                    else
                        fb[q][j] = OB::frag(smem + SA, wn * WTN + j * 16, q, lane);
                }
            }
            __syncthreads();
            const bool live = KG == 1 || t * KG + kg < ntiles;
            // Per 16-row strip of the wave's tile: a share of tile t+1's split and LDS writes, then
            // the strip's products; the 64 x 64 tile the other way round, so that the split's vector
            // instructions issue while its products are under way ([768, 256, 4096] of a transposed A
            // 25.4 -> 25.0 us, [4096, 768, 256] 18.8 -> 18.6; the other tiles measured slower so).
            constexpr bool FEED_LAST = !S::WIDE && KG == 1;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                f32x4 (&lo)[FN] = low[LOWSUM ? i : 0];
                auto feed = [&]() __attribute__((always_inline)) {
                    gstore(set, kt(t + 1), i, FM);
                    if (i == FM - 1) gload(set, kt(t + 1 + PF));
                };
                if constexpr (!FEED_LAST) feed();
                if (KG > 1 && !live) continue;
                if constexpr (!LOWSUM) {
#pragma unroll
                    for (int j = 0; j < FN; ++j) lo[j] = zero;
                }
#pragma unroll
                for (int q = 0; q < 5; ++q)
#pragma unroll
                    for (int j = 0; j < FN; ++j) mul(lo[j], fa[QA[q]][i], fb[QB[q]][j]);
#pragma unroll
                for (int j = 0; j < FN; ++j) mul(acc[i][j], fa[0][i], fb[0][j]);
                if constexpr (!LOWSUM) {
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] += lo[j];
                }
                if constexpr (FEED_LAST) feed();
                // Strips in order: left alone, the scheduler gathers all splits first and spills. The
                // wide tiles' split runs between their MFMAs: 4096^3 679 -> 653 us (X.W^T); the 64 x 64
                // tile measured 1% slower so.
                if constexpr (S::WIDE) {
#pragma unroll
                    for (int g = 0; g < 6 * FN; ++g) {
                        __builtin_amdgcn_sched_group_barrier(sg::VALU, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(sg::MFMA, 1, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
#pragma unroll
        for (int q = 0; q < PF; ++q) gload(q, kt(q));
        gstore(0, kt(0), 0, 1);
        gload(0, kt(PF));
        // Tile t+1's registers are set (t + 1) % PF: whole groups of PF tiles in a branch-free body,
        // then the remaining tiles.
        int t = 0;
        for (; t + PF <= nt; t += PF) {
#pragma unroll
            for (int q = 0; q < PF; ++q) ktile(t + q, (q + 1) % PF);
        }
#pragma unroll
        for (int q = 0; q + 1 < PF; ++q)
            if (t + q < nt) ktile(t + q, (q + 1) % PF);
        if constexpr (LOWSUM) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] += low[i][j];
        }
    }
    if constexpr (KG > 1) {
        // The other groups hand their sums over through LDS and are done.
        constexpr int REGION = THREADS * FM * FN * 16;
        static_assert((KG - 1) * REGION <= KG * S::SMEM, "the groups' sums fit in the stages");
        __syncthreads();
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    *(f32x4 *)(smem0 + (kg - 1) * REGION + ((i * FN + j) * THREADS + tid) * 16) = acc[i][j];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int g = 0; g < KG - 1; ++g)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] += *(const f32x4 *)(smem0 + g * REGION + ((i * FN + j) * THREADS + tid) * 16);
    }

    // The sums are of scaled terms (BF16X3_SCALE for each operand). An element that is not finite (acc * 0
    // is NaN) may owe that to the split or to the scale: this wave then takes its products again on the
    // FP32 units, straight from memory.
    // Lane l of a 16x16 block holds rows (XPOSE: columns) 4 (l / 16) + r, r = 0..3, and column (row)
    // l % 16.
    float nf = 0.f;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // (columns past M or N may hold anything)
                const int mn = (lane >> 4) * 4 + r;
                const int64_t row = m0 + wm * WTM + i * 16 + (XPOSE ? (lane & 15) : mn);
                const int64_t col = (DUAL ? n0 : n0 + wn * WTN) + j * 16 + (XPOSE ? mn : (lane & 15));
                nf = row < p.M && col < p.N ? fmaf(acc[i][j][r], 0.f, nf) : nf;
            }
    if (__any(nf != nf)) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = zero;
        // Steps of 16 k: lane group g takes k 4g..4g+3 of both operands, one per MFMA, as the FP32 units'
        // tiles do; two steps of loads go out together (XF: one, for its registers). Elements from ke on
        // are zeros.
        constexpr int H = XF ? 1 : 2;
        const bool up = DUAL && __builtin_amdgcn_readfirstlane(wn) != 0;  // this wave's B rows are up-weight rows
        const int kq = (lane >> 4) * 4;
        auto quad = [&](const __amdgpu_buffer_rsrc_t &rs, bool kcontig, int64_t ld, int row, int64_t k) {
            u32x4 v;
            if (kcontig)
                v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)((row * ld + k) * 4), 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (!kcontig) v[e] = __builtin_amdgcn_raw_buffer_load_b32(rs, (uint32_t)(((k + e) * ld + row) * 4), 0, 0);
                v[e] = k + e < ke ? v[e] : 0u;
            }
            return __builtin_bit_cast(f32x4, v);
        };
#pragma unroll 1
        for (int64_t k0 = kb; k0 < ke; k0 += 16 * H) {
            f32x4 av[H][FM], bv[H][FN];
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const int64_t k = k0 + 16 * h + kq;
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    const int rl = wm * WTM + i * 16 + (lane & 15);
                    av[h][i] = quad(ra.rs, !TA, p.lda, rl, k);
                    if constexpr (XF) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int64_t tok = TA ? k + e : m0 + rl, cls = TA ? m0 + rl : k + e;
                            const bool ok = k + e < ke && m0 + rl < p.M;
                            const float2 st = ok ? p.xent_stats[tok] : float2{0.f, 0.f};
                            const bool target = ok && p.xent_tgt[tok] == (uint32_t)cls;
                            const uint32_t g = OA::xent(__float_as_uint(av[h][i][e]), st.x, st.y * p.xent_scale, target, p.xent_scale);
                            av[h][i][e] = ok ? __uint_as_float(g) : 0.f;
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    if constexpr (DUAL)
                        bv[h][j] = up ? quad(rb2.rs, TB, p.ldb, j * 16 + (lane & 15), k)
                                      : quad(rb.rs, TB, p.ldb, j * 16 + (lane & 15), k);
                    else
                        bv[h][j] = quad(rb.rs, TB, p.ldb, wn * WTN + j * 16 + (lane & 15), k);
                }
            }
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
                            acc[i][j] = XPOSE ? __builtin_amdgcn_mfma_f32_16x16x4f32(bv[h][j][e], av[h][i][e], acc[i][j], 0, 0, 0)
                                              : __builtin_amdgcn_mfma_f32_16x16x4f32(av[h][i][e], bv[h][j][e], acc[i][j], 0, 0, 0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] *= 1.f / (BF16X3_SCALE * BF16X3_SCALE);
    }

    if constexpr (XPOSE) {
        // Lane l of block (i, j) has output row i*16 + l%16 and its consecutive columns j*16 +
        // 4*(l/16) .. +3.
        auto each = [&](auto &&f) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    f(acc[i][j], wm * WTM + i * 16 + (lane & 15), wn * WTN + j * 16 + (lane >> 4) * 4);
        };
        if constexpr (FIX) {
            if (p.splits > 1) {
                // Partial tile of split z at device scope (written through this XCD's L2), then the
                // arrival count: the tile's last block reads every split's partial at device scope
                // (missing its own L2), adds them in split order from zero, as the separate
                // reduction does, and finishes the tile. Offsets are 32-bit (splits * M * N * 4 <
                // 2^31, checked by the host).
                const __amdgpu_buffer_rsrc_t prt = __builtin_amdgcn_make_buffer_rsrc(
                    p.partial, (short)0, (int)(p.splits * p.M * p.N * 4), 0x00020000);
                each([&](const f32x4 &v, int rl, int cl) __attribute__((always_inline)) {
                    const int64_t row = m0 + rl, col = n0 + cl;
                    if (row < p.M && col < p.N)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), prt,
                                                               (uint32_t)(((z * p.M + row) * p.N + col) * 4), 0,
                                                               CP_DEVICE_SCOPE);
                });
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's partials reached device scope
                __syncthreads();
                __shared__ int last_in;
                if (tid == 0) {
                    const int old = __hip_atomic_fetch_add(arrive, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    last_in = old == p.splits - 1;
                    if (last_in) __hip_atomic_store(arrive, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                __syncthreads();
                if (!last_in) return;
                each([&](const f32x4 &v, int rl, int cl) __attribute__((always_inline)) {
                    const int64_t row = m0 + rl, col = n0 + cl;
                    if (row >= p.M || col >= p.N) return;
                    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
                    for (int sp = 0; sp < p.splits; ++sp)
                        sum += sp == z ? v
                                       : __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                       prt, (uint32_t)(((sp * p.M + row) * p.N + col) * 4),
                                                                       0, CP_DEVICE_SCOPE));
                    finish4<true, true>(p, sum, row, col, coff, 0);
                });
                return;
            }
        }
        each([&](const f32x4 &v, int rl, int cl) __attribute__((always_inline)) {
            finish4<true>(p, v, m0 + rl, n0 + cl, coff, z);
        });
    } else {
        // Epilogue through LDS: each wave stages half of its columns at a time with static register
        // indices, then finishes them row-major with 4-column vectors (DUAL: the gate and up waves of
        // a row half finish their slice together).
        constexpr int EC = WTN / 2, EP = EC * 4 + 16, SLAB = WTM * EP;
        static_assert(KG == 1 && WM * WN * SLAB <= S::SMEM, "epilogue staging fits in the stage");
        __syncthreads();
        char *wl = smem + wave * SLAB;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int jj = 0; jj < FN / 2; ++jj)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        *(float *)(wl + (i * 16 + (lane >> 4) * 4 + r) * EP + (jj * 16 + (lane & 15)) * 4) =
                            acc[i][h * (FN / 2) + jj][r];
            __syncthreads();
            if constexpr (DUAL) {
                static_assert(WN == 2, "one gate and one up wave per row half");
                const char *gl = smem + (wm * 2) * SLAB, *ul = gl + SLAB;
                const int pt = wn * 64 + lane;
                for (int it = 0; it < (WTM * EC + 511) / 512; ++it) {
                    const int e = (it * 128 + pt) * 4;
                    if (WTM * EC % 512 != 0 && e >= WTM * EC) break;
                    const int rl = e / EC, cl = e % EC;
                    finish_swiglu4<true>(p, *(const f32x4 *)(gl + rl * EP + cl * 4),
                                                     *(const f32x4 *)(ul + rl * EP + cl * 4), m0 + wm * WTM + rl,
                                                     n0 + h * EC + cl, coff);
                }
            } else {
                for (int it = 0; it < WTM * EC / 256; ++it) {
                    const int e = (it * 64 + lane) * 4;
                    const int rl = e / EC, cl = e % EC;
                    const f32x4 v = *(const f32x4 *)(wl + rl * EP + cl * 4);
                    finish4<true>(p, v, m0 + wm * WTM + rl, n0 + wn * WTN + h * EC + cl, coff, z);
                }
            }
            __syncthreads();
        }
    }
}

template <class S, bool TA, bool TB, bool DUAL, bool XF = false>
__global__ __launch_bounds__(S::THREADS * S::KG, S::WAVES) void gemm_f32_terms(const GemmArgs p) {
    __shared__ __attribute__((aligned(16))) char smem[S::KG * S::SMEM];
    gemm_f32_block<S, TA, TB, DUAL, false, XF>(p, blockIdx.x, blockIdx.y, smem);
}

// A group of GEMMs: 64 x 64 tiles, batch 1, one split count for the group. Split-K partial sums go to
// each problem's own region, and each tile's last block to arrive adds its splits and finishes it.
template <bool TA, bool TB>
__global__ __launch_bounds__(S64::THREADS, S64::WAVES) void gemm_f32_terms_group(const GemmGroupArgs grp) {
    __shared__ __attribute__((aligned(16))) char smem[S64::SMEM];
    int gi, split, tile;
    if (!group_block(grp, gi, split, tile)) return;
    const GemmArgs p = grp.g[gi];  // a copy: through the reference the whole argument went to scratch
    gemm_f32_block<S64, TA, TB, false, true>(p, tile, split, smem, grp.arrive + grp.cstart[gi] + tile);
}

template <class S, bool TA, bool TB, bool DUAL, bool XF = false>
void go(const GemmArgs &a, dim3 grid, hipStream_t s) {
    hipLaunchKernelGGL((gemm_f32_terms<S, TA, TB, DUAL, XF>), grid, dim3(S::THREADS * S::KG), 0, s, a);
}

// bm x bn: the output tile (SwiGLU: half as wide as its B tile).
template <bool TA, bool TB>
void launch_plain(int bm, int bn, const GemmArgs &a, dim3 grid, hipStream_t s) {
    if constexpr (!TA)
        if (bm == 256) return go<S256, TA, TB, false>(a, grid, s);
    if (bm == 128) return go<S128, TA, TB, false>(a, grid, s);
    if (bn == 32) return go<S6432, TA, TB, false>(a, grid, s);
    go<S64, TA, TB, false>(a, grid, s);
}

// The tiles as the planner prices them, in microseconds: a k-tile of a block that shares its CU (its
// share of the CU's time) and of one that has it alone, a round's launch, prologue and epilogue, and what a
// transposed A costs a k-tile (64-byte pieces of its rows, which the 64 x 32 tile waits for). Fitted on
// every tile and split count of 132 shapes, warm: the TINY step's, ragged ones, squares, layers of up to
// 8192 rows, and random ones of 17 to 8192 rows and up to 16384 columns and 11008 k. The picks take 1.4%
// longer than the fastest measured plans; the former constants, with powers of two as split counts, took
// 5% and up to 1.4x ([701, 300, 1000] of a transposed A 19.7 us on 64 x 32 tiles, 14.8 on 64 x 64 with four
// splits).
struct Tile {
    int bm, bn, occ;  // occ: blocks a CU runs at once
    double shared, alone, round, ta;
};
constexpr Tile T256{256, 128, 1, 1.97, 1.97, 14.4, 1.0}, T128{128, 128, 2, 1.05, 1.42, 12.3, 1.0},
    T64{64, 64, 3, 0.55, 0.715, 2.8, 1.0}, T6432{64, 32, 2, 0.314, 0.332, 2.95, 1.51},
    TGROUP{64, 64, 3, 0.50, 0.60, 3.0, 1.0};  // a group's 64 x 64 blocks, fitted on eleven groups
// The SwiGLU form's epilogue weighs more on the wide tile's few blocks: [4096, 688, 256] takes 26.9 us on
// 64 x 64 and 28.3 on 128 x 128, [8192, 688, 256] 46.4 and 42.1, [8192, 2816, 1024] 586 and 464. Over 35
// shapes the picks take 0.2% longer than the faster tile.
constexpr Tile T128_DUAL{128, 128, 2, 1.05, 1.42, 14.5, 1.0};
// Split-K partial sums out and back, and the reduction's launch: 4 us, where device times alone gave 1.6, because
// small products wait on the host, which a second launch keeps longer (a 112 x 96 x 514 layer, called from
// Python, 32.5 us unsplit and 36.8 split). A group adds in the kernel.
constexpr double PARTIAL_BW = 5.4e12, REDUCE = 4e-6, GROUP_BW = 3.1e12, GROUP_SUM = 1.6e-6;
constexpr int SPLITS[] = {1, 2, 3, 4, 5, 6, 8, 12, 16, 24, 32};

struct Plan {
    int bm, bn, splits;
    int64_t k_per_split;
};

// One launch of `blocks` blocks of ksteps k-tiles, in seconds: whole rounds of the blocks that a CU runs at
// once, and a last one that costs what the blocks it gives a CU take alone ([3333, 3333, 2222] on 128 x 128
// tiles: 512 blocks and 217 more, 300 us, against 338 for two nearly full rounds of 256 x 128; the TINY
// layer's group: five splits, 980 blocks, 65.5 us, four, 784 in one round and 16 more, 75.6).
double launch_time(const Tile &t, bool ta, int64_t blocks, int64_t ksteps, int64_t cus) {
    const int64_t full = blocks / (t.occ * cus), rest = cdiv(blocks % (t.occ * cus), cus);
    const double ktiles = (ta ? t.ta : 1.0) * ksteps;
    return 1e-6 * (full * (t.round + ktiles * std::max(t.occ * t.shared, t.alone)) +
                   (rest ? t.round + ktiles * std::max(rest * t.shared, t.alone) : 0.0));
}

// Picks the tile and the split count, lowest price first. Near ties (3%) keep the earlier
// plan, except that between two unsplit plans the one with more blocks wins (more loads in flight per
// k-step); the 64 x 32 tile has to win outright.
Plan choose_plan(const GemmArgs &a, int64_t cus, bool ta, double *est) {
    constexpr int bk = ET<float>::BK;
    const bool plain = !a.dual && a.causal == CAUSAL_NONE && a.kmode == KMODE_FULL;
    const int64_t kall = std::max<int64_t>(1, cdiv(a.K, bk)) * bk;
    Plan best{64, a.dual ? 32 : 64, 1, kall};
    double best_t = 1e30;
    int64_t best_blocks = 0;
    for (const Tile &tile : {T256, a.dual ? T128_DUAL : T128, T64, T6432}) {
        if (tile.bm != tile.bn && (!plain || a.xent_stats)) continue;
        if (tile.bm == 256 && (ta || a.swiglu_bwd || a.rope_table)) continue;
        const int bn = a.dual ? tile.bn / 2 : tile.bn;
        const int64_t tiles = cdiv(a.M, tile.bm) * cdiv(a.N, bn) * a.batch;
        for (const int s : SPLITS) {
            if (s > 1 && (!plain || a.no_split)) break;
            const int64_t kps = s == 1 ? kall : cdiv(cdiv(a.K, s), bk) * bk;
            if (s > 1 && kps < 4 * bk) break;
            const int64_t splits = s > 1 ? cdiv(a.K, kps) : 1, blocks = tiles * splits;
            double t = launch_time(tile, ta, blocks, kps / bk, cus);
            if (splits > 1) t += 2.0 * splits * a.M * a.N * a.batch * 4.0 / PARTIAL_BW + REDUCE;
            const bool better = t < best_t * 0.97;
            const bool tie_more_blocks = t < best_t * 1.03 && splits == 1 && best.splits == 1 &&
                                         blocks > best_blocks && tile.bn != 32;
            if (better || tie_more_blocks) {
                best_t = better ? t : std::min(t, best_t);
                best = Plan{tile.bm, bn, (int)splits, kps};
                best_blocks = blocks;
            }
        }
    }
    if (est) *est = best_t;
    return best;
}

int64_t cus_of(const it_context *ctx) { return ctx->num_cus > 0 ? ctx->num_cus : 256; }

// 4-column vectors of an FP32 output need an element's alignment only.
void any_alignment(GemmArgs &a) { a.c_vec_ok = a.c_vec_ok || !a.out_bf16; }

}  // namespace

bool f32_terms_applicable(const GemmArgs &a, bool ta, bool tb) {
    // A few rows wait on latency, not on the matrix units: M = 1, N = 768, K = 256 takes 0.7 us more here
    // than on the FP32 units' 64 x 32 tile, which loads two k-tiles ahead.
    // (X.W^T there goes to gemv_nt where its rows are whole 16-byte chunks.)
    // More rows stay here for their precision also where the FP32 units are faster, which they are in
    // products of few k-tiles (a k-tile's split sits between its load and its products): K = 256 FP32
    // units 2.9e-7 from 64 bits and 9.9 us against 0.9e-7 and 11.6 ([4096, 256, 256], X.W), 512^3 9.6
    // against 11.9. Over 127 of choose_plan's shapes the terms are 1.20x as fast, from 0.65x ([192, 176, 160]
    // of a transposed A) to 3.0x; callers that would rather have the time ask for the units (IT_EPI_F32_UNITS).
    return a.M > 16 && !a.f32_units && !a.a_kscale && spans_fit(a, ta, tb);
}

it_status launch_gemm_f32(it_context *ctx, bool ta, bool tb, GemmArgs a, const char *tag) {
    Plan plan = choose_plan(a, cus_of(ctx), ta, nullptr);
#ifdef IT_TUNING
    // Planner sweeps only (a tuning build): IT_PLAN="tile,splits[,width]" forces the plan.
    if (const char *env = std::getenv("IT_PLAN")) {
        int bm = 0, sp = 0, bn = 0;
        const int n = std::sscanf(env, "%d,%d,%d", &bm, &sp, &bn);
        if (n >= 2) plan = Plan{bm, a.dual ? bm / 2 : n == 3 ? bn : bm, sp, cdiv(cdiv(a.K, sp), 32) * 32};
    }
#endif
    auto apply = [&](const Plan &pl) {
        plan = pl;
        a.tiles_m = (int)cdiv(a.M, pl.bm);
        a.tiles_n = (int)cdiv(a.N, pl.bn);
        a.k_per_split = pl.k_per_split;
        a.splits = (int)std::max<int64_t>(1, cdiv(a.K, pl.k_per_split));
    };
    apply(plan);
    any_alignment(a);
    if (a.splits > 1) {
        void *ws = nullptr;
        if (ensure_scratch(ctx, (size_t)a.splits * a.batch * a.M * a.N * sizeof(float), &ws) != IT_OK) {
            clear_error();
            a.no_split = 1;  // no scratch (a capture may not allocate): the best plan without
            apply(choose_plan(a, cus_of(ctx), ta, nullptr));
        }
        a.partial = (float *)ws;
    }
    const int64_t gx = (int64_t)a.tiles_m * a.tiles_n, gy = a.batch * a.splits;
    if (gx > 0x7fffffff || gy > 65535)
        return fail(IT_ERR_DIMS, "it_gemm: grid too large (tiles " + std::to_string(gx) + ", batch*splits " +
                                     std::to_string(gy) + ")");
    const dim3 grid((unsigned)gx, (unsigned)gy);
    std::string key;
    hipEvent_t ev = nullptr;
    if (ctx->profiling) {
        char buf[192];
        std::snprintf(buf, sizeof(buf), "gemm_f32_%c%c_%dx%d%s%s|%s[%lld,%lld,%lld]x%lld s%d", ta ? 'T' : 'N',
                      tb ? 'T' : 'N', plan.bm, a.dual ? plan.bm : plan.bn, a.dual ? "_swiglu" : a.xent_stats ? "_xent" : "",
                      a.causal || a.kmode ? "_causal" : "", tag ? tag : "", (long long)a.M, (long long)a.N,
                      (long long)a.K, (long long)a.batch, a.splits);
        key = buf;
        profile_begin(ctx, key, &ev);
    }
    hipStream_t s = ctx->stream;
    if (a.dual) {  // X.W^T (checked by the caller)
        if (plan.bm == 128) go<S128, false, true, true>(a, grid, s);
        else go<S64, false, true, true>(a, grid, s);
    } else if (a.xent_stats) {  // B not transposed (checked by the caller)
        if (plan.bm == 128) ta ? go<S128, true, false, false, true>(a, grid, s) : go<S128, false, false, false, true>(a, grid, s);
        else ta ? go<S64, true, false, false, true>(a, grid, s) : go<S64, false, false, false, true>(a, grid, s);
    } else if (!ta && !tb) {
        launch_plain<false, false>(plan.bm, plan.bn, a, grid, s);
    } else if (!ta && tb) {
        launch_plain<false, true>(plan.bm, plan.bn, a, grid, s);
    } else if (ta && !tb) {
        launch_plain<true, false>(plan.bm, plan.bn, a, grid, s);
    } else {
        launch_plain<true, true>(plan.bm, plan.bn, a, grid, s);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail_hip(e, "gemm_f32_terms launch");
    if (a.splits > 1) {
        const it_status st = launch_splitk_reduce(s, a);
        if (st != IT_OK) return st;
    }
    if (ctx->profiling) profile_end(ctx, key, ev);
    return IT_OK;
}

// One gemm_f32_terms_group launch (64 x 64 tiles, one split count for the group; each tile's last split
// block adds the partial sums) where the planner prices it below the separate plans.
bool launch_gemm_f32_group(it_context *ctx, bool ta, bool tb, const GemmArgs *args, int count, const char *tag,
                           it_status *status) {
    constexpr int bk = ET<float>::BK;
    const int64_t cus = cus_of(ctx);
    if (count < 2) return false;
    double separate = 0.0;
    for (int i = 0; i < count; ++i) {
        const GemmArgs &a = args[i];
        if (a.batch != 1 || a.dual || a.causal != CAUSAL_NONE || a.kmode != KMODE_FULL || a.swiglu_bwd || a.xent_stats ||
            a.K <= 0 || a.N % 4 != 0 || a.no_split)
            return false;
        double t = 0.0;
        choose_plan(a, cus, ta, &t);
        separate += t;
    }
    // The model of the group at one split count s. The XCD schedule takes at most count * s + 7
    // chunks (a chunk per GEMM and split, plus one more where an XCD's share ends inside one), so s
    // stays where that fits the table.
    double best_t = 1e30;
    int best_s = 0;
    for (int s = 1; s <= 32 && count * s + 7 <= GROUP_CHUNKS; ++s) {
        int64_t blocks = 0, ksteps = 0;
        double traffic = 0.0;
        bool ok = true;
        for (int i = 0; i < count && ok; ++i) {
            const GemmArgs &a = args[i];
            const int64_t kps = cdiv(cdiv(a.K, s), bk) * bk;
            ok = s == 1 || kps >= 4 * bk;
            const int64_t splits = s > 1 ? cdiv(a.K, kps) : 1;
            blocks += cdiv(a.M, 64) * cdiv(a.N, 64) * splits;
            ksteps = std::max(ksteps, cdiv(kps, bk));
            if (splits > 1) traffic += 2.0 * splits * a.M * a.N * 4.0;
        }
        if (!ok) break;
        double t = launch_time(TGROUP, ta, blocks, ksteps, cus);
        if (traffic > 0.0) t += traffic / GROUP_BW + GROUP_SUM;  // the tiles' last blocks add the partial sums
        if (t < best_t) {
            best_t = t;
            best_s = s;
        }
    }
#ifdef IT_TUNING
    // Planner sweeps only (a tuning build): IT_GROUP_SPLITS forces the group's split count.
    if (const char *env = std::getenv("IT_GROUP_SPLITS")) {
        best_s = std::max(1, std::min(32, std::atoi(env)));
        best_t = 0.0;
    }
#endif
    if (!best_s || best_t >= 0.97 * separate) return false;
    GemmGroupArgs grp{};
    grp.count = count;
    int64_t scratch = 0, tiles = 0;
    bool split_any = false;
    for (int i = 0; i < count; ++i) {
        GemmArgs &a = grp.g[i];
        a = args[i];
        const int64_t kps = cdiv(cdiv(a.K, best_s), bk) * bk;
        a.splits = best_s > 1 ? (int)cdiv(a.K, kps) : 1;
        a.k_per_split = best_s > 1 ? kps : cdiv(a.K, bk) * bk;
        a.tiles_m = (int)cdiv(a.M, 64);
        a.tiles_n = (int)cdiv(a.N, 64);
        any_alignment(a);
        grp.cstart[i] = (int)tiles;
        tiles += (int64_t)a.tiles_m * a.tiles_n;
        if (a.splits > 1) {
            // the in-kernel sum addresses a problem's partials with 32-bit byte offsets
            if ((int64_t)a.splits * a.M * a.N * 4 >= (1ll << 31)) return false;
            split_any = true;
            scratch += (int64_t)a.splits * a.M * a.N;
        }
    }
    if (tiles > COUNTERS) return false;
    grp.cstart[count] = (int)tiles;
    const int grid_blocks = xcd_schedule(grp);
    if (!grid_blocks) return false;
    if (split_any) {
        void *ws = nullptr;
        if (ensure_counters(ctx, &grp.arrive) != IT_OK ||
            ensure_scratch(ctx, (size_t)scratch * sizeof(float), &ws) != IT_OK) {
            clear_error();
            return false;  // no scratch (a capture may not allocate): separate products
        }
        float *part = (float *)ws;
        for (int i = 0; i < count; ++i)
            if (grp.g[i].splits > 1) {
                grp.g[i].partial = part;
                part += (int64_t)grp.g[i].splits * grp.g[i].M * grp.g[i].N;
            }
    }
    std::string key;
    hipEvent_t ev = nullptr;
    if (ctx->profiling) {
        key = std::string("gemm_f32_") + (ta ? 'T' : 'N') + (tb ? 'T' : 'N') + "_64x64_group|" + (tag ? tag : "");
        for (int i = 0; i < count; ++i)
            key += (i ? "+[" : "[") + std::to_string(args[i].M) + "," + std::to_string(args[i].N) + "," +
                   std::to_string(args[i].K) + "]";
        key += "x1 s" + std::to_string(best_s);
        profile_begin(ctx, key, &ev);
    }
    const dim3 grid((unsigned)grid_blocks), block(S64::THREADS);
    if (!ta && tb) hipLaunchKernelGGL((gemm_f32_terms_group<false, true>), grid, block, 0, ctx->stream, grp);
    else if (!ta && !tb) hipLaunchKernelGGL((gemm_f32_terms_group<false, false>), grid, block, 0, ctx->stream, grp);
    else if (ta && !tb) hipLaunchKernelGGL((gemm_f32_terms_group<true, false>), grid, block, 0, ctx->stream, grp);
    else hipLaunchKernelGGL((gemm_f32_terms_group<true, true>), grid, block, 0, ctx->stream, grp);
    const hipError_t e = hipGetLastError();
    *status = e == hipSuccess ? IT_OK : fail_hip(e, "gemm group launch");
    if (ctx->profiling && *status == IT_OK) profile_end(ctx, key, ev);
    return true;
}

}  // namespace it
