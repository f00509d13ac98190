// Linear-layer GEMMs on bf16 operands (the bf16 precision of the training
// step): forward y = x W^T (matmul_nt_v2.comp), dx = dy W
// (linear_backward_dx_batched.comp) and dW = dy^T x
// (linear_backward_dw_batched.comp), on the gemm16 kernel.
//
// Tile plan (measured on MI355X with DMA staging, T = 2048-token step shapes):
//   * >= 512 tiles of 256 x 256       -> 256 x 256, 8 waves (vocab-sized GEMMs)
//   * >= 512 tiles of 128 x 128       -> 128 x 128, 8 waves of 64 x 32
//   * K >= 16384 and >= 256 tiles of 128 x 128 -> 256 x 256 split-K 3 ways
//   * K >= 4096 and >= 256 tiles of 128 x 128  -> 128 x 128, 8 waves
//   * K >= 16384 and < 256 such tiles -> 256 x 256 split-K 8 ways (head dh)
//   * <= 96 tiles of 128 x 64, or < 256 with K <= 1024 -> plan_few
//   * < 384 tiles of 128 x 64, K >= 2048 -> 128 x 64 split-K 2 ways
//   * otherwise                       -> 128 x 64
// Operands that break the kernel's layout rules (16-byte alignment, ld and
// the contiguous extent multiples of 8, < 2 GiB) take the generic MFMA GEMM.
#include <math.h>

#include <algorithm>

#include "gemm16.hpp"
#include "ops.hpp"
#include "qkv8.hpp"

namespace vkh {

namespace {

using TBig = Tile16<256, 256, 2, 4>;
using T128 = Tile16<128, 128, 2, 2>;
using T128x64 = Tile16<128, 64, 2, 2>;
using T128w8 = Tile16<128, 128, 2, 4>;  // 8 waves of 64 x 32
// The in-block split-K block (two 4-wave groups, one block per CU whatever its
// LDS) with three slab buffers per group (144 KB): two slabs in flight per
// group for these latency-bound N = 1024 shapes.  Alone: o / down forward
// 20.0 / 27.8 -> 18.4 / 24.5 us, gate/up and q/k/v dx 50.3 / 34.7 -> 48.4 / 33.6
// us; the bf16 step 19.33-19.34 -> 19.31-19.32 ms.  (In fp32 mode, whose slabs
// are half as deep, it made the fp32 step slower: 77.3 against 76.65 ms.)
using T128x64s3 = Tile16<128, 64, 2, 2, 3>;
// Few-tile products (plan_few): smaller tiles, split over K.
using T64 = Tile16<64, 64, 2, 2>;
using T32x64 = Tile16<32, 64, 1, 4>;  // K-major A only (a bf16 MN tile is 64 rows or 128 n)
using T32 = Tile16<32, 32, 2, 2, 3>;  // fp32, whose products of few tiles are bound by the
                                      // matrix cores of the CUs they reach
// (Three slab buffers were measured slower for these tiles: the larger LDS
// footprint drops a block per CU.  Staging the slabs through VGPRs two slabs
// ahead, which doubles the time a load has to arrive without more LDS, was
// measured equal on every per-layer shape alone and in the step: slab
// latency is not what bounds these GEMMs.)

constexpr bool kUseKs2 = true;

enum class Pick { Big, T128, T128x64, T128w8, T128x64ks2, T64, T32x64, T64ks2, T32x64ks2, T32, T32ks2 };
struct Plan {
    Pick tile;
    int splits;
    bool column_order = false;  // tiles in plain column order (no row groups)
};

size_t ws_for(const Plan &p, const GemmShape &s) {
    if (p.splits <= 1) return 0;
    switch (p.tile) {
    case Pick::Big: return gemm16_ws_bytes<TBig>(s, p.splits);
    case Pick::T128: return gemm16_ws_bytes<T128>(s, p.splits);
    case Pick::T128w8: return gemm16_ws_bytes<T128w8>(s, p.splits);
    case Pick::T64: return gemm16_ws_bytes<T64>(s, p.splits);
    case Pick::T32x64: return gemm16_ws_bytes<T32x64>(s, p.splits);
    case Pick::T32: return gemm16_ws_bytes<T32>(s, p.splits);
    default: return gemm16_ws_bytes<T128x64>(s, p.splits);
    }
}

// Products of few tiles (short sequences, small models): most CUs would idle on
// 128-row tiles, and a block's K loop is a serial chain of slabs (0.29 us each in
// bf16, 0.36 in fp32, where the matrix cores are the slower part).  The tile and
// the split over K come from a model of the launch: its fixed cost, the slower of
// the slab chain, the CU's matrix time when blocks share it, operand traffic and
// output traffic, and the reduce launch of a split.  Fitted by least squares on the
// logarithm to timings of 16-512 rows over widths 256-32000 in the three layouts; of
// the 5668 in profiles/gemm_few_tiles.csv it is off by 12 % (fp32) and 17 % (bf16) rms
// with no bias, and the pick is 4 % above the best of a product's on average.  Against
// the 128 x 64 tiles before it: fp32 16 x 1024 x 3072 107 -> 9.7 us, 128 x 512 x 512
// 22 -> 7.3, 512 x 1024 x 1024 39 -> 16; bf16 16 x 1024 x 3072 18.8 -> 7.3 us,
// 128 x 1024 x 1024 10.6 -> 6.5, 512 x 768 x 32000 95 -> 55.
// fp32 also has the in-block split (two wave groups on the halves of K, no reduce
// launch).  `base` is the plan of the large tiles, whose number of partial sums over K
// is the least that the pick may have: fewer, longer chains would round worse (one
// chain where base had two was 1.4 times as far from 64 bits at K = 1957).  With
// ws.keep_sums the pick has base's very sums (a 2-layer 256-wide fp32 step of 128
// tokens 980 -> 620 us with the same bits), with ws.min_chains at least that many.
Plan plan_few(const GemmShape &s, const GemmWs &ws, bool f32, bool mn_a, const Plan &base) {
    struct Fit { double launch, slab0, slab1, mfma, l2, red, part, hbm; };
    constexpr Fit kB{3.8, 0.088, 0.199, 0.225, 21.2, 2.5, 6.6, 5.2},
        kF{4.5, 0.314, 0.047, 0.574, 10.7, 2.0, 6.5, 4.4};
    const Fit &f = f32 ? kF : kB;
    const double es = f32 ? 4 : 2;
    const double hbm = (es * s.K * ((double)s.M + s.N) + 4.0 * s.M * s.N) / (f.hbm * 1e6);
    const int nk = (s.K + (f32 ? 31 : 63)) / (f32 ? 32 : 64);
    const int min_slabs = f32 ? 1 : 8;  // of a split: 512 of K in bf16, as in plan()
    const bool halves = base.tile == Pick::T128x64ks2;
    const int chains = std::max(1, std::min(nk, std::max(halves ? 2 : base.splits, ws.min_chains)));
    const size_t ws_bytes = ws.p ? ws.bytes : 0;
    // the halves in bf16 and products without scratch: in one block
    if (!f32 && halves && ws.keep_sums) return base;
    Plan best{chains > 1 ? Pick::T128x64ks2 : Pick::T128x64, 1};
    double tb = 1e30;
    auto tile = [&](Pick pick, Pick ks2, int bm, int bn) {
        const double tiles = (double)ceil_div(s.M, bm) * ceil_div(s.N, bn);
        if (f32 && (chains <= 2 || !ws_bytes)) {  // both groups of a block share its CU's matrix cores
            const double slabs = (nk + 1) / 2, share = ceil(tiles / 256) * 2 * f.mfma * bm * bn / 4096;
            const double t = std::max(slabs * std::max(f.slab0 + f.slab1 * (bm + bn) / 128, share),
                                      tiles * nk * (bm + bn) * 128 / (f.l2 * 1e6));
            if (f.launch + 0.7 + std::max(t, hbm) < tb) {
                tb = f.launch + 0.7 + std::max(t, hbm);
                best = Plan{ks2, 1};
            }
            if (ws.keep_sums && halves) return;
        }
        for (int sp = chains; sp <= 32; sp *= 2) {
            const Plan p{pick, sp};
            if (sp > chains && (ws.keep_sums || nk / sp < min_slabs)) break;
            if (ws_for(p, s) > ws_bytes) break;
            const double slabs = (nk + sp - 1) / sp, blocks = tiles * sp;
            const double share = ceil(blocks / 256) * f.mfma * bm * bn / 4096;
            double t = std::max(slabs * std::max(f.slab0 + f.slab1 * (bm + bn) / 128, share),
                                blocks * slabs * (bm + bn) * 128 / (f.l2 * 1e6));
            t = f.launch + std::max(t, hbm);
            if (sp > 1) t += f.red + blocks * bm * bn * 8 / (f.part * 1e6);
            if (t < tb) tb = t, best = p;
        }
    };
    tile(Pick::T128x64, Pick::T128x64ks2, 128, 64);
    tile(Pick::T64, Pick::T64ks2, 64, 64);
    // In bf16 up to one 32 x 64 tile per CU: beyond, several of them on a CU are bound by
    // their operand traffic, which the model does not see (128 x 8200 over K = 1016, 516
    // tiles: 21.7 us against 14.4 on 64 x 64 and 14.6 on 128 x 64; of 260 drawn products
    // the most that one lost to 128 x 64 was 24 %, and 7 % with this line).
    if (f32 || (!mn_a && (long)ceil_div(s.M, 32) * ceil_div(s.N, 64) <= 256))
        tile(Pick::T32x64, Pick::T32x64ks2, 32, 64);
    if (f32) tile(Pick::T32, Pick::T32ks2, 32, 32);
    return best;
}

// The plan of the large tiles.
Plan plan_large(const GemmShape &s, size_t ws_bytes) {
    auto tiles = [&](int bm, int bn) { return (long)ceil_div(s.M, bm) * (long)ceil_div(s.N, bn); };
    if (tiles(256, 256) >= 512) return {Pick::Big, 1};
    const long t128 = tiles(128, 128), t64 = tiles(128, 64);
    if (t128 >= 512) return {Pick::T128w8, 1};
    const int nk = (s.K + 63) / 64;
    Plan p{Pick::T128x64, 1};
    if (s.K >= 16384 && t128 >= 256)
        // a long contraction onto at least a chip-wide wave of 128 x 128 tiles
        // (Qwen3-4B gate/up dx, K = 19456): 256 x 256 split 3 ways, 199 us
        // against 236 (128 x 128, 8 waves) and 361 (128 x 64)
        p = Plan{Pick::Big, 3};
    else if (s.K >= 4096 && t128 >= 256)
        // Qwen3-4B o / down forward and q/k/v dx (N = 2560, K = 4096..9728):
        // 128 x 128 on 8 waves, 50 / 113 / 79 us against 56 / 167 / 104 (128 x 64);
        // in column order (the LoRA step: 66.7 against 68.1 ms with row groups)
        p = Plan{Pick::T128w8, 1, true};
    else if (s.K >= 16384 && t128 < 256)
        // the head's dh at config 3 (M = 2048, N = 1024, K = 151936: 32 tiles of
        // 256 x 256): split 8 ways, 256 blocks; in the step 18.78-18.79 against
        // 18.91 ms for 128 x 128 split 4 (Big split 16: 18.93-18.96; 128 x 128
        // split 8: 19.06-19.10)
        p = Plan{Pick::Big, 8};
    else if (t64 < 384 && s.K >= 2048)
        // two wave groups in one block: alone, faster than split-K + reduce up
        // to K = 4096 and slower at 6144, but in the two-stream step faster
        // for every such shape (22.2 vs 22.5 ms with split-K kept at 6144 and
        // for the weight gradients, 22.8 ms with split-K everywhere)
        p = kUseKs2 ? Plan{Pick::T128x64ks2, 1} : Plan{Pick::T128x64, 2};
    while (p.splits > 1 && (nk / p.splits < 8 || ws_for(p, s) > ws_bytes)) --p.splits;
    return p;
}

// mn_a: the A operand is MN-major (the weight gradients).
Plan plan(const GemmShape &s, const GemmWs &ws, bool mn_a = false) {
    auto tiles = [&](int bm, int bn) { return (long)ceil_div(s.M, bm) * (long)ceil_div(s.N, bn); };
    // few tiles: up to 96 of 128 x 64, and up to 255 where K is short (beyond, the
    // two-group 128 x 64 blocks are as fast: 256 x 4096 x 4096 26.5 against 32.5 us)
    const long t64 = tiles(128, 64);
    if (t64 <= 96 || (t64 < 256 && s.K <= 1024))
        return plan_few(s, ws, false, mn_a, plan_large(s, ~size_t(0)));
    return plan_large(s, ws.p ? ws.bytes : 0);
}

// Whether the fused-epilogue forward kernels (8-wave 128 x 128 tiles only) take
// the product: where plan() picks that tile, or, for a launch paired with one
// of the same shape on a second stream (the forward's two half batches), where
// M is whole tiles and the pair together fills a chip-wide round (the config-3
// step's q|k|v and gate/up halves: 256 + 256 and 384 + 384 tiles; the forward
// as two concurrent half batches measured 18.58-18.59 against 18.85 ms).
bool fused_tile_ok(const GemmShape &s, bool paired) {
    const Plan p = plan(s, GemmWs{nullptr, 0});
    if (p.tile == Pick::T128w8 && p.splits == 1) return true;
    return paired && s.M % 128 == 0 && 2L * (s.M / 128) * ceil_div(s.N, 128) >= 512;
}

template <Lay LA, Lay LB, class Epi>
hipError_t run16(const Op16 &a, const Op16 &b, const GemmShape &s, const Epi &e, const GemmWs &ws,
                 hipStream_t st) {
    const Plan p = plan(s, ws, LA == Lay::MN);
    const SplitK sk{p.splits, (f32x4 *)ws.p};
    const int g = p.column_order ? 0 : tile_group_rows<LA, LB>();
    switch (p.tile) {
    case Pick::Big: return launch_gemm16<TBig, LA, LB>(a, b, s, e, sk, g, st);
    case Pick::T128: return launch_gemm16<T128, LA, LB>(a, b, s, e, sk, g, st);
    case Pick::T128w8: return launch_gemm16<T128w8, LA, LB>(a, b, s, e, sk, g, st);
    case Pick::T128x64ks2: return launch_gemm16_ks2<T128x64s3, LA, LB>(a, b, s, e, g, st);
    case Pick::T64: return launch_gemm16<T64, LA, LB>(a, b, s, e, sk, g, st);
    case Pick::T32x64:
        if constexpr (LA == Lay::K) return launch_gemm16<T32x64, LA, LB>(a, b, s, e, sk, g, st);
        else return hipErrorInvalidValue;
    default: return launch_gemm16<T128x64, LA, LB>(a, b, s, e, sk, g, st);
    }
}

// ── fp32 operands (the reference-precision step) ───────────────────────
// The same kernels with F32 set: slabs of 32 fp32 values (128-byte tile rows,
// the bf16 slab's layout), four v_mfma_f32_16x16x4_f32 per 16-byte fragment.
// At a sixteenth of the bf16 matrix rate the slab DMA has ample time to land,
// so the plan only has to spread whole rounds of tiles over the 256 CUs.
// Measured per shape alone at the config-3 step's 12 layer GEMMs (T = 2048):
//   * 128 x 128 on 8 waves where its tile count fills rounds at least as
//     evenly as 128 x 64 (q/k/v and gate/up forward, o dx, q/k/v dW: 130-196 us
//     against 143-210 on 128 x 64 and 210-290 on 4-wave 128 x 128 or 256 x 256);
//   * 128 x 64 where that evens the rounds (384 tiles of 128 x 128 = 768 of
//     128 x 64: down dx 107 against 134 us, gate/up dW 209 against 259);
//   * fewer than 512 tiles of 128 x 64 (the N = 1024 outputs and dW of o /
//     down): 128 x 64 with the K range split over the two wave groups of one
//     block.  Alone, split-K over two launches plus the reduce is faster
//     (q/k/v dx 149, gate/up dx 213, down dW 119 us against 174, 254, 154),
//     but in the two-stream step the in-block form is (76.3-77.0 against
//     76.5-77.1 ms in four alternating pairs; plain 128 x 64: 77.3-77.4): the
//     reduce launches' 4.2 ms of partial traffic per step is gone.
// Fewer than 256 tiles of 128 x 64, or fewer than 512 with a K of at most 1024:
// plan_few (there the in-block split leaves CUs idle or its second group without
// work: 2560-wide products of 512 rows 95 -> 64 us, 3072 x 1024 dW of 16 rows 15 -> 8).
Plan plan32(const GemmShape &s, const GemmWs &ws, bool mn_a = false) {
    auto tiles = [&](int bm, int bn) { return (long)ceil_div(s.M, bm) * (long)ceil_div(s.N, bn); };
    auto fill = [](long t) { return (double)t / (256.0 * (double)((t + 255) / 256)); };
    const long t128 = tiles(128, 128), t64 = tiles(128, 64);
    Plan p{Pick::T128x64, 1};
    if (t128 >= 256 && fill(t128) >= fill(t64)) p = Plan{Pick::T128w8, 1};
    else if (t64 < 512) p = Plan{Pick::T128x64ks2, 1};
    if ((p.tile == Pick::T128x64ks2 && (t64 < 256 || s.K <= 1024)) || ws.min_chains > 2)
        return plan_few(s, ws, true, mn_a, p);
    return p;
}

template <Lay LA, Lay LB, class Epi>
hipError_t run32(const Op16 &a, const Op16 &b, const GemmShape &s, const Epi &e, const GemmWs &ws,
                 hipStream_t st) {
    const Plan p = plan32(s, ws, LA == Lay::MN);
    const SplitK sk{p.splits, (f32x4 *)ws.p};
    const int g = p.column_order ? 0 : tile_group_rows<LA, LB>();
    switch (p.tile) {
    case Pick::Big: return launch_gemm16<TBig, LA, LB, Epi, true>(a, b, s, e, sk, g, st);
    case Pick::T128: return launch_gemm16<T128, LA, LB, Epi, true>(a, b, s, e, sk, g, st);
    case Pick::T128w8: return launch_gemm16<T128w8, LA, LB, Epi, true>(a, b, s, e, sk, g, st);
    case Pick::T128x64ks2: return launch_gemm16_ks2<T128x64, LA, LB, Epi, true>(a, b, s, e, g, st);
    case Pick::T64: return launch_gemm16<T64, LA, LB, Epi, true>(a, b, s, e, sk, g, st);
    case Pick::T32x64: return launch_gemm16<T32x64, LA, LB, Epi, true>(a, b, s, e, sk, g, st);
    case Pick::T64ks2: return launch_gemm16_ks2<T64, LA, LB, Epi, true>(a, b, s, e, g, st);
    case Pick::T32x64ks2: return launch_gemm16_ks2<T32x64, LA, LB, Epi, true>(a, b, s, e, g, st);
    case Pick::T32: return launch_gemm16<T32, LA, LB, Epi, true>(a, b, s, e, sk, g, st);
    case Pick::T32ks2: return launch_gemm16_ks2<T32, LA, LB, Epi, true>(a, b, s, e, g, st);
    default: return launch_gemm16<T128x64, LA, LB, Epi, true>(a, b, s, e, sk, g, st);
    }
}

// fp32 operand view: 16-byte aligned, ld and the contiguous run multiples of 4
// floats (whole 16-byte chunks), under 2 GiB (32-bit buffer offsets).
bool make_op32(const float *p, long ld, long rows, long run, Op16 &o, bool padded = false) {
    if (padded) run = std::min(ld, (run + 3) / 4 * 4);
    if (((uintptr_t)p & 15u) || ld % 4 || run % 4 || rows <= 0) return false;
    const size_t bytes = ((size_t)(rows - 1) * ld + run) * 4;
    if (bytes >= (1ull << 31)) return false;
    o = Op16{reinterpret_cast<const bf16 *>(p), ld, (unsigned)bytes};
    return true;
}

Mat matf32(const float *p, long ld) { return Mat{p, ld, DType::F32}; }

// Operand of `rows` storage rows whose contiguous run is `run` elements.
bool make_op(const bf16 *p, long ld, long rows, long run, Op16 &o, bool padded = false) {
    if (padded) run = std::min(ld, (run + 7) / 8 * 8);
    if (((uintptr_t)p & 15u) || ld % 8 || run % 8 || rows <= 0) return false;
    const size_t bytes = ((size_t)(rows - 1) * ld + run) * 2;
    if (bytes >= (1ull << 31)) return false;
    o = Op16{p, ld, (unsigned)bytes};
    return true;
}

Mat matb(const bf16 *p, long ld) { return Mat{p, ld, DType::BF16}; }

// Rows per chunk when a [rows, ld] bf16 operand view reaches 2 GiB (the DMA
// path's 32-bit offsets): 0 if it fits whole, else a multiple of 64 rows.
int rows_per_2g_chunk(long rows, long ld, long run) {
    if (((rows - 1) * ld + run) * 2 < (1l << 31)) return 0;
    const long fit = ((1l << 31) - 1) / (2 * ld);  // rows whose view fits
    const long n = (rows + fit - 1) / fit;           // chunks
    return (int)(((rows + n - 1) / n + 63) / 64 * 64);
}

// ── LoRA term in the epilogue ──────────────────────────────────────────
// EpiLora<Base> adds rank-r LoRA products (train/lora.zig:99-251) to the tile
// before Base stores it:
//   C[t, col_s + c] = acc + alpha sum_i U_s[t, i] F_s(c, i)
// for every adapter s whose columns [col_s, col_s + ncols) hold c: the
// forward's y += aor inter B^T, or the backward's dx += aor (dy B) A summed
// over the adapters of one shared input.  The output is then written once,
// instead of stored by the GEMM, read back and stored again by a separate
// update pass.  The products run on v_mfma_f32_16x16x4_f32 in the
// accumulator layout: lane (g, c) supplies A[c][k] = alpha U_s[row0 + 16 i + c][k]
// and B[k][c] = F_s(col0 + 16 j + c - col_s, k) for the contraction index
// k = 16 kb + 4 g + e at step e, so the results land on acc[i][j] where Base
// reads them.  Base's own alpha must be 1 (the linear layers' products).
template <class Base>
struct EpiLora {
    static constexpr bool kSplits = Base::kSplits;
    Base base;
    LoraSegs sg;
    int r;
    float alpha;

    template <int TM, int TN>
    VKH_DEV void apply(const f32x4 (&acc_in)[TM][TN], const FragPos &fp, const GemmShape &s) const {
        f32x4 acc[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = acc_in[i][j];
        const int g = fp.lane / 16, c = fp.lane % 16;
        for (int si = 0; si < sg.n; ++si) {
            const LoraSeg &q = sg.s[si];
            // wave-uniform: none of the wave's columns in this adapter's range
            if (fp.col0 + 16 * TN <= q.col || fp.col0 >= q.col + q.ncols) continue;
            for (int kb = 0; kb < r; kb += 16) {
                const int k = kb + 4 * g;
                const bool kok = k < r;  // r is a multiple of 4
                f32x4 ua[TM];
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    const int row = fp.row0 + 16 * i + c;
                    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (kok && row < s.M) t = *reinterpret_cast<const float4 *>(q.u + (long)row * q.ldu + k);
                    ua[i] = f32x4{alpha * t.x, alpha * t.y, alpha * t.z, alpha * t.w};
                }
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const long cb = fp.col0 + 16 * j;  // wave-uniform
                    if (cb < q.col || cb >= q.col + q.ncols) continue;
                    const long cc = cb + c - q.col;
                    f32x4 fb = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (kok) {
                        if (q.fsc == 1) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) fb[e] = q.f[(long)(k + e) * q.fsi + cc];
                        } else {
                            const float4 t = *reinterpret_cast<const float4 *>(q.f + cc * q.fsc + k);
                            fb = f32x4{t.x, t.y, t.z, t.w};
                        }
                    }
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j] = mfma16x16x4(ua[i][e], fb[e], acc[i][j]);
                }
            }
        }
        base.template apply<TM, TN>(acc, fp, s);
    }
};

bool al16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

// The adapters' layout rules of EpiLora on an output of n_out columns:
// 16-column blocks, whole 16-byte U rows and factor reads, r <= 64.
bool lora_epi_ok(const LoraSegs &g, int r, int n_out) {
    if (r < 1 || r > 64 || r % 4 || g.n < 1 || g.n > 3) return false;
    for (int i = 0; i < g.n; ++i) {
        const LoraSeg &q = g.s[i];
        if (q.col < 0 || q.col % 16 || q.ncols <= 0 || q.ncols % 16 || q.col + q.ncols > n_out) return false;
        if (!q.u || !al16(q.u) || q.ldu % 4 || q.ldu < r || !q.f) return false;
        if (q.fsc != 1 && (!al16(q.f) || q.fsc % 4 || q.fsi != 1)) return false;
    }
    return true;
}

}  // namespace

bool g16_lora_ok(const bf16 *a, long lda, long arows, long arun, const bf16 *b, long ldb, long brows,
                 long brun, const LoraSegs &g, int r, int n_out) {
    Op16 oa, ob;
    return make_op(a, lda, arows, arun, oa) && make_op(b, ldb, brows, brun, ob) &&
           lora_epi_ok(g, r, n_out);
}

hipError_t g16_nt_lora(const bf16 *x, long ldx, const bf16 *w, long ldw, float *y, long ldy, int M,
                       int N, int K, const float *R, long ldr, const LoraSegs &g, int r,
                       float alpha, const GemmWs &ws, hipStream_t st) {
    Op16 a, b;
    if (!make_op(x, ldx, M, K, a) || !make_op(w, ldw, N, K, b) || !lora_epi_ok(g, r, N))
        return hipErrorInvalidValue;
    EpiLora<EpiStore> e{EpiStore{y, ldy, R, ldr, 1.f, 0.f}, g, r, alpha};
    return run16<Lay::K, Lay::K>(a, b, GemmShape{M, N, K}, e, ws, st);
}

hipError_t g16_nn_lora(const bf16 *dy, long lddy, const bf16 *w, long ldw, float *dx, long lddx,
                       int M, int N, int K, const LoraSegs &g, int r, float alpha, const GemmWs &ws,
                       hipStream_t st) {
    Op16 a, b;
    if (!make_op(dy, lddy, M, N, a) || !make_op(w, ldw, N, K, b) || !lora_epi_ok(g, r, K))
        return hipErrorInvalidValue;
    EpiLora<EpiStore> e{EpiStore{dx, lddx, nullptr, 0, 1.f, 0.f}, g, r, alpha};
    return run16<Lay::K, Lay::MN>(a, b, GemmShape{M, K, N}, e, ws, st);
}

hipError_t g16_nn_bf16_lora(const bf16 *dy, long lddy, const bf16 *w, long ldw, bf16 *dx,
                            long lddx, int M, int N, int K, const LoraSegs &g, int r, float alpha,
                            const GemmWs &ws, hipStream_t st) {
    Op16 a, b;
    if (!make_op(dy, lddy, M, N, a) || !make_op(w, ldw, N, K, b) || !lora_epi_ok(g, r, K))
        return hipErrorInvalidValue;
    EpiLora<EpiStoreBf16> e{EpiStoreBf16{dx, lddx, 1.f}, g, r, alpha};
    return run16<Lay::K, Lay::MN>(a, b, GemmShape{M, K, N}, e, ws, st);
}

hipError_t g16_nt(const bf16 *x, long ldx, const bf16 *w, long ldw, float *y, long ldy, int M,
                  int N, int K, const float *R, long ldr, float alpha, float beta,
                  const GemmWs &ws, hipStream_t st) {
    Op16 a, b;
    if (!make_op(x, ldx, M, K, a) || !make_op(w, ldw, N, K, b))
        return gemm_nt(Precision::BF16, matb(x, ldx), matb(w, ldw), y, ldy, M, N, K, R, ldr, alpha,
                       beta, st);
    EpiStore e{y, ldy, R, ldr, alpha, beta};
    return run16<Lay::K, Lay::K>(a, b, GemmShape{M, N, K}, e, ws, st);
}

// gu[M, 2F] = x[M, K] w_gu[2F, K]^T and gated[M, F] = bf16(swiglu1(gu[:, f], gu[:, F + f])) in
// one launch, where the plain plan for the [M, 2F] product is the 8-wave 128 x 128 tile
// (each block then takes 64 gate and the matching 64 up features); hipErrorNotSupported
// (nothing launched) elsewhere, and the caller runs g16_nt + swiglu_forward.  (The same
// epilogue on the 256 x 256 tile, 128 + 128 features per block and a 128 KB hand-over, was
// parity-green but measured config 4 at 59.93-60.07 against 59.68-59.73 ms and config 5
// unchanged, 584.1-584.6 against 584.0-585.0 ms.)
hipError_t g16_gate_up_swiglu(const bf16 *x, long ldx, const bf16 *w, long ldw, float *gu,
                              long ldgu, bf16 *gated, long ldg, int M, int F, int K, hipStream_t st,
                              bool paired) {
    if (M <= 0 || F <= 0 || F % 64) return hipErrorNotSupported;
    if (!fused_tile_ok(GemmShape{M, 2 * F, K}, paired)) return hipErrorNotSupported;
    Op16 a, b;
    if (!make_op(x, ldx, M, K, a) || !make_op(w, ldw, 2L * F, K, b)) return hipErrorNotSupported;
    const unsigned tiles = (unsigned)(ceil_div(M, T128w8::BM) * (F / (T128w8::BN / 2)));
    hipLaunchKernelGGL((gemm16_swiglu_kernel<T128w8>), dim3(tiles), dim3(T128w8::NT), 0, st, a, b, M,
                       F, K, gu, ldgu, gated, ldg, tile_group_rows<Lay::K, Lay::K>());
    return hipGetLastError();
}

namespace {

template <typename TO>
struct QkvEpi {
    QkvLayout L;
    const float *wq, *wk;  // q / k RMSNorm gains (qk_norm)
    TO *out;               // the attention operand [rows, (Hq + 2 Hkv) hd]
    long ld_out;
    const float2 *tab;     // RoPE cos / sin [seq_len][rotary_dim / 2]
};

// The q|k|v projection with the Q/K-RMSNorm + RoPE forward in its epilogue (head_dim
// 128, so a 128 x 128 tile is 128 rows of one head): the tile stores its fp32
// projection (the backward's pre-norm values), stages it in the idle slab buffers (16-float
// group u of row r at u ^ ((r >> 2) & 3), so the four row groups of a store land on
// different banks), and its waves then run the standalone pass's item code
// (qkv_fwd_item8, 16 lanes per row) on it and write the bf16 attention operand.
template <class Cfg, bool F32 = false, typename TO = bf16>
__global__ __launch_bounds__(Cfg::NT, 1) void gemm16_qkv_kernel(Op16 a, Op16 b, GemmShape s, float *C,
                                                               long ldc, QkvEpi<TO> q, int tgrp) {
    constexpr int BM = Cfg::BM, BN = Cfg::BN, NT = Cfg::NT, NW = NT / 64;
    constexpr int WM = BM / Cfg::WGM, WN = BN / Cfg::WGN;
    constexpr int TM = WM / 16, TN = WN / 16;
    constexpr int LPH = 16, G = 64 / LPH;  // lanes per row, rows per wave
    static_assert(BN == 128 && BM * BN * 4 <= Cfg::LDS && BM % (NW * G) == 0, "one head per tile");
    __shared__ __attribute__((aligned(16))) char smem[Cfg::LDS];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int wm = wave / Cfg::WGN, wn = wave % Cfg::WGN;
    const int nbm = (s.M + BM - 1) / BM, nbn = s.N / BN;
    const int nb = nbm * nbn;
    int bid = blockIdx.x;
    if (nb % 8 == 0) bid = (bid % 8) * (nb / 8) + bid / 8;
    int bm, bn;
    tile_rc(bid, nbm, nbn, tgrp, bm, bn);
    const int m0 = bm * BM, n0 = bn * BN;
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int KW = F32 ? 32 : 64;  // k per slab
    gemm16_tile_dma<Cfg, Lay::K, Lay::K, TM, TN, F32>(a, b, m0, n0, s.M, s.N, 0, (s.K + KW - 1) / KW,
                                                      s.K, acc, smem);
    float *lt = reinterpret_cast<float *>(smem);  // the slab loop ended with a barrier
    const int g = lane / 16, c = lane % 16;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int tr = wm * WM + 16 * i + 4 * g + r, tc = wn * WN + 16 * j + c;
                if (m0 + tr < s.M) C[(long)(m0 + tr) * ldc + n0 + tc] = acc[i][j][r];
                lt[tr * BN + (tc ^ (((tr >> 2) & 3) << 4))] = acc[i][j][r];
            }
    lds_barrier();
    const QkvLayout &L = q.L;
    const int h = bn, half = L.rotary_dim / 2, j8 = lane % LPH;
    const Rope8 rp = rope8(j8, half);
    const bool is_q = h < L.n_q_heads, qkh = h < L.n_q_heads + L.n_kv_heads;
    float gq[8], gk[8];
    if (L.qk_norm) {
        ld8(q.wq + 8 * j8, gq);
        ld8(q.wk + 8 * j8, gk);
    }
    for (int tr = wave * G + lane / LPH; tr < BM; tr += NW * G) {
        const int t = m0 + tr;
        const bool valid = t < s.M, qk = valid && qkh;
        float y[8];
        ld8(lt + tr * BN + ((8 * j8) ^ (((tr >> 2) & 3) << 4)), y);
        float2 cs[8];
        if (qk && rp.rot_lane) {
            const float4 *tp =
                reinterpret_cast<const float4 *>(q.tab + (long)(t % L.seq_len) * half + rp.col);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 v = tp[i];
                cs[2 * i] = make_float2(v.x, v.y);
                cs[2 * i + 1] = make_float2(v.z, v.w);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) cs[i] = make_float2(1.f, 0.f);
        }
        qkv_fwd_item8<LPH>(L, y, cs, qk, is_q, gq, gk, rp, lane, half);
        if (valid) st8(q.out + (long)t * q.ld_out + h * BN + 8 * j8, y);
    }
}

}  // namespace

// y[M, N] = x w^T (the fp32 q|k|v projection) and the bf16 attention operand out = RoPE(
// Q/K-RMSNorm(y)) (qkv_prepare_forward's values, bit for bit) in one launch, where head_dim
// is 128 and the product's plain plan is the 8-wave 128 x 128 tile; hipErrorNotSupported
// (nothing launched) elsewhere.
hipError_t g16_qkv_norm_rope(const bf16 *x, long ldx, const bf16 *w, long ldw, float *y, long ldy,
                             int M, int N, int K, const QkvLayout &L, const float *wq,
                             const float *wk, bf16 *out, long ld_out, const float2 *tab,
                             hipStream_t st, bool paired) {
    if (M <= 0 || L.head_dim != 128 || L.n_rows != M || L.seq_len <= 0 || L.rotary_dim % 16 ||
        L.rotary_dim > 128 || N != (L.n_q_heads + 2 * L.n_kv_heads) * 128)
        return hipErrorNotSupported;
    const GemmShape s{M, N, K};
    if (!fused_tile_ok(s, paired)) return hipErrorNotSupported;
    const Plan p = plan(s, GemmWs{nullptr, 0});  // its tile order where it is this tile
    if (((uintptr_t)out & 15u) || ld_out % 8 || (L.qk_norm && (((uintptr_t)wq | (uintptr_t)wk) & 15u)) ||
        (L.rotary_dim && ((uintptr_t)tab & 15u)))
        return hipErrorNotSupported;
    Op16 a, b;
    if (!make_op(x, ldx, M, K, a) || !make_op(w, ldw, N, K, b)) return hipErrorNotSupported;
    const int g = p.tile == Pick::T128w8 && p.column_order ? 0 : tile_group_rows<Lay::K, Lay::K>();
    const unsigned tiles = (unsigned)(ceil_div(M, T128w8::BM) * (N / T128w8::BN));
    hipLaunchKernelGGL((gemm16_qkv_kernel<T128w8>), dim3(tiles), dim3(T128w8::NT), 0, st, a, b, s, y,
                       ldy, QkvEpi<bf16>{L, wq, wk, out, ld_out, tab}, g);
    return hipGetLastError();
}

// The fp32 forms of the two fused projections (fp32 operands on the DMA-staged kernels'
// fp32 slab mode, fp32 outputs), where the fp32 plan is the 8-wave 128 x 128 tile.
hipError_t g32_qkv_norm_rope(const float *x, long ldx, const float *w, long ldw, float *y, long ldy,
                             int M, int N, int K, const QkvLayout &L, const float *wq,
                             const float *wk, float *out, long ld_out, const float2 *tab,
                             hipStream_t st) {
    if (M <= 0 || L.head_dim != 128 || L.n_rows != M || L.seq_len <= 0 || L.rotary_dim % 16 ||
        L.rotary_dim > 128 || N != (L.n_q_heads + 2 * L.n_kv_heads) * 128)
        return hipErrorNotSupported;
    const GemmShape s{M, N, K};
    const Plan p = plan32(s, GemmWs{nullptr, 0});
    if (p.tile != Pick::T128w8 || p.splits != 1) return hipErrorNotSupported;
    if (((uintptr_t)out & 15u) || ld_out % 4 || (L.qk_norm && (((uintptr_t)wq | (uintptr_t)wk) & 15u)) ||
        (L.rotary_dim && ((uintptr_t)tab & 15u)))
        return hipErrorNotSupported;
    Op16 a, b;
    if (!make_op32(x, ldx, M, K, a) || !make_op32(w, ldw, N, K, b)) return hipErrorNotSupported;
    const int g = p.column_order ? 0 : tile_group_rows<Lay::K, Lay::K>();
    const unsigned tiles = (unsigned)(ceil_div(M, T128w8::BM) * (N / T128w8::BN));
    hipLaunchKernelGGL((gemm16_qkv_kernel<T128w8, true, float>), dim3(tiles), dim3(T128w8::NT), 0, st,
                       a, b, s, y, ldy, QkvEpi<float>{L, wq, wk, out, ld_out, tab}, g);
    return hipGetLastError();
}

hipError_t g32_gate_up_swiglu(const float *x, long ldx, const float *w, long ldw, float *gu,
                              long ldgu, float *gated, long ldg, int M, int F, int K, hipStream_t st) {
    if (M <= 0 || F <= 0 || F % 64) return hipErrorNotSupported;
    const GemmShape s{M, 2 * F, K};
    const Plan p = plan32(s, GemmWs{nullptr, 0});
    if (p.tile != Pick::T128w8 || p.splits != 1) return hipErrorNotSupported;
    Op16 a, b;
    if (!make_op32(x, ldx, M, K, a) || !make_op32(w, ldw, 2L * F, K, b)) return hipErrorNotSupported;
    const unsigned tiles = (unsigned)(ceil_div(M, T128w8::BM) * (F / (T128w8::BN / 2)));
    hipLaunchKernelGGL((gemm16_swiglu_kernel<T128w8, true, float>), dim3(tiles), dim3(T128w8::NT), 0,
                       st, a, b, M, F, K, gu, ldgu, gated, ldg, p.column_order ? 0 : tile_group_rows<Lay::K, Lay::K>());
    return hipGetLastError();
}

hipError_t g16_nn(const bf16 *dy, long lddy, const bf16 *w, long ldw, float *dx, long lddx, int M,
                  int N, int K, float alpha, float beta, const GemmWs &ws, hipStream_t st, bool padded) {
    // an over-2 GiB dy (the head's dz at 8192 tokens): independent row chunks
    if (const int mc = M > 64 ? rows_per_2g_chunk(M, lddy, N) : 0) {
        for (int m0 = 0; m0 < M; m0 += mc) {
            const hipError_t e = g16_nn(dy + (long)m0 * lddy, lddy, w, ldw, dx + (long)m0 * lddx,
                                        lddx, std::min(mc, M - m0), N, K, alpha, beta, ws, st, padded);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    // C[m, k'] = sum_n dy[m, n] W[n, k']: A = dy (K-major over n), B(k', n) = W[n][k'] (MN)
    Op16 a, b;
    if (!make_op(dy, lddy, M, N, a, padded) || !make_op(w, ldw, N, K, b, padded))
        return gemm_nn(Precision::BF16, matb(dy, lddy), matb(w, ldw), dx, lddx, M, N, K, alpha,
                       beta, st);
    EpiStore e{dx, lddx, nullptr, 0, alpha, beta};
    return run16<Lay::K, Lay::MN>(a, b, GemmShape{M, K, N}, e, ws, st);
}

hipError_t g16_nn_bf16(const bf16 *dy, long lddy, const bf16 *w, long ldw, bf16 *dx, long lddx,
                       int M, int N, int K, const GemmWs &ws, hipStream_t st) {
    Op16 a, b;
    if (!make_op(dy, lddy, M, N, a) || !make_op(w, ldw, N, K, b)) return hipErrorInvalidValue;
    EpiStoreBf16 e{dx, lddx, 1.f};
    return run16<Lay::K, Lay::MN>(a, b, GemmShape{M, K, N}, e, ws, st);
}

hipError_t g16_tn(const bf16 *dy, long lddy, const bf16 *x, long ldx, float *dw, long lddw, int M,
                  int N, int K, float alpha, float beta, const GemmWs &ws, hipStream_t st, bool padded) {
    // an over-2 GiB dy (the head's dz at 8192 tokens): the contraction over m in
    // row chunks, each chunk after the first accumulating (beta = 1)
    const int ca = M > 64 ? rows_per_2g_chunk(M, lddy, N) : 0, cb = M > 64 ? rows_per_2g_chunk(M, ldx, K) : 0;
    if (const int mc = (ca && cb) ? std::min(ca, cb) : std::max(ca, cb)) {
        for (int m0 = 0; m0 < M; m0 += mc) {
            const hipError_t e = g16_tn(dy + (long)m0 * lddy, lddy, x + (long)m0 * ldx, ldx, dw, lddw,
                                        std::min(mc, M - m0), N, K, alpha, m0 ? 1.f : beta, ws, st,
                                        padded);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    // C[n, k'] = sum_m dy[m, n] x[m, k']: both operands MN-major over m
    Op16 a, b;
    if (!make_op(dy, lddy, M, N, a, padded) || !make_op(x, ldx, M, K, b, padded))
        return gemm_tn(Precision::BF16, matb(dy, lddy), matb(x, ldx), dw, lddw, M, N, K, alpha,
                       beta, st);
    EpiStore e{dw, lddw, nullptr, 0, alpha, beta};
    return run16<Lay::MN, Lay::MN>(a, b, GemmShape{N, K, M}, e, ws, st);
}

hipError_t g32_nt(const float *x, long ldx, const float *w, long ldw, float *y, long ldy, int M,
                  int N, int K, const float *R, long ldr, float alpha, float beta,
                  const GemmWs &ws, hipStream_t st) {
    Op16 a, b;
    if (!make_op32(x, ldx, M, K, a) || !make_op32(w, ldw, N, K, b))
        return gemm_nt(Precision::FP32, matf32(x, ldx), matf32(w, ldw), y, ldy, M, N, K, R, ldr,
                       alpha, beta, st);
    EpiStore e{y, ldy, R, ldr, alpha, beta};
    return run32<Lay::K, Lay::K>(a, b, GemmShape{M, N, K}, e, ws, st);
}

hipError_t g32_nn(const float *dy, long lddy, const float *w, long ldw, float *dx, long lddx, int M,
                  int N, int K, float alpha, float beta, const GemmWs &ws, hipStream_t st, bool padded) {
    Op16 a, b;
    if (!make_op32(dy, lddy, M, N, a, padded) || !make_op32(w, ldw, N, K, b, padded))
        return gemm_nn(Precision::FP32, matf32(dy, lddy), matf32(w, ldw), dx, lddx, M, N, K, alpha,
                       beta, st);
    EpiStore e{dx, lddx, nullptr, 0, alpha, beta};
    return run32<Lay::K, Lay::MN>(a, b, GemmShape{M, K, N}, e, ws, st);
}

hipError_t g32_tn(const float *dy, long lddy, const float *x, long ldx, float *dw, long lddw, int M,
                  int N, int K, float alpha, float beta, const GemmWs &ws, hipStream_t st, bool padded) {
    Op16 a, b;
    if (!make_op32(dy, lddy, M, N, a, padded) || !make_op32(x, ldx, M, K, b, padded))
        return gemm_tn(Precision::FP32, matf32(dy, lddy), matf32(x, ldx), dw, lddw, M, N, K, alpha,
                       beta, st);
    EpiStore e{dw, lddw, nullptr, 0, alpha, beta};
    return run32<Lay::MN, Lay::MN>(a, b, GemmShape{N, K, M}, e, ws, st);
}

// ── linear products of any operand form ────────────────────────────────
namespace {

// One operand's packed copy: dst[r][0 .. V chunks) = src[r][0 .. run), then zeros.
struct PackSeg {
    const void *src;
    void *dst;
    size_t n;         // 16-byte chunks of dst
    unsigned chunks;  // ... per row
    int run;
};

// Copies of one or two operands whose rows become whole 16-byte chunks of TD.
// One 16-byte store per thread; the source is read in vector loads at its
// element alignment (global loads need no more on gfx950).  Bound by HBM: a
// [151936, 1024] fp32 -> bf16 pack takes 190 us (933 MB, 4.9 TB/s).  Both
// operands go in one launch: a launch costs more than a small pack (64 x 256:
// 10.4 us for a product with two pack launches before it, 8.7 with one).
template <typename TS, typename TD>
__global__ __launch_bounds__(256) void pack_rows_k(PackSeg s0, PackSeg s1) {
    constexpr int V = 16 / sizeof(TD);
    typedef TD vec_t __attribute__((ext_vector_type(V)));
    const size_t stride = (size_t)gridDim.x * 256, n = s0.n + s1.n;
    for (size_t j = (size_t)blockIdx.x * 256 + threadIdx.x; j < n; j += stride) {
        const bool second = j >= s0.n;
        const PackSeg &s = second ? s1 : s0;
        const size_t i = second ? j - s0.n : j, r = i / s.chunks;
        const int c = (int)(i - r * s.chunks) * V;
        const TS *p = (const TS *)s.src + r * s.run + c;
        TS t[V];
        if (c + V <= s.run) {
            __builtin_memcpy(t, p, sizeof(t));
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e) t[e] = c + e < s.run ? p[e] : (TS)0.f;
        }
        vec_t v;
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = (TD)(float)t[e];
        reinterpret_cast<vec_t *>(s.dst)[i] = v;
    }
}

template <typename TS, typename TD>
hipError_t pack_rows(const PackSeg &s0, const PackSeg &s1, hipStream_t st) {
    const size_t n = s0.n + s1.n;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL((pack_rows_k<TS, TD>), dim3((unsigned)std::min<size_t>((n + 255) / 256, 65536)),
                       dim3(256), 0, st, s0, s1);
    return hipGetLastError();
}

int chunk_elems(LinForm f) { return f == LinForm::F32 ? 4 : 8; }
size_t packed_bytes(LinForm f, long rows, long run) {
    const size_t v = chunk_elems(f), b = (run + v - 1) / v * 16 * (size_t)rows;
    return (b + 255) / 256 * 256;
}
bool needs_pack(LinForm f, const void *p, long run) {
    return f == LinForm::MIXED || ((uintptr_t)p & 15u) || run % chunk_elems(f);
}

struct LinDims {
    long ra, ca, rb, cb;  // rows and contiguous run of the two operands
    GemmShape s;          // the product
};
LinDims lin_dims(LinOp op, int M, int N, int K) {
    if (op == LinOp::NT) return {M, K, N, K, {M, N, K}};
    if (op == LinOp::NN) return {M, N, N, K, {M, K, N}};
    return {M, N, M, K, {N, K, M}};
}
size_t lin_split_bytes(LinForm f, const GemmShape &s) {
    return f == LinForm::F32 ? g32_ws_bytes_for(s.M, s.N, s.K) : g16_ws_bytes_for(s.M, s.N, s.K);
}

}  // namespace

bool lin_packs(LinOp op, LinForm f, const void *a, const void *b, int M, int N, int K) {
    const LinDims d = lin_dims(op, M, N, K);
    return needs_pack(f, a, d.ca) || needs_pack(f, b, d.cb);
}

size_t lin_ws_bytes(LinOp op, LinForm f, const void *a, const void *b, int M, int N, int K) {
    const LinDims d = lin_dims(op, M, N, K);
    return (needs_pack(f, a, d.ca) ? packed_bytes(f, d.ra, d.ca) : 0) +
           (needs_pack(f, b, d.cb) ? packed_bytes(f, d.rb, d.cb) : 0) + lin_split_bytes(f, d.s);
}

// Packs the operands whose `rows` are not 0 (dense rows of `run` elements).
hipError_t lin_pack(LinForm f, const void *a, long ra, long ca, void *da, const void *b, long rb,
                    long cb, void *db, hipStream_t st) {
    const long v = chunk_elems(f);
    auto seg = [&](const void *p, long rows, long run, void *dst) {
        const unsigned ch = (unsigned)((run + v - 1) / v);
        return PackSeg{p, dst, (size_t)rows * ch, ch ? ch : 1, (int)run};
    };
    const PackSeg s0 = seg(a, ra, ca, da), s1 = seg(b, rb, cb, db);
    if (f == LinForm::MIXED) return pack_rows<float, bf16>(s0, s1, st);
    if (f == LinForm::F32) return pack_rows<float, float>(s0, s1, st);
    return pack_rows<bf16, bf16>(s0, s1, st);
}

bool lin_lora_ok(LinOp op, LinForm f, int M, int N, int K, const LoraSegs &g, int r) {
    const LinDims d = lin_dims(op, M, N, K);
    auto fits = [&](long rows, long run) { return packed_bytes(f, rows, run) < (1ull << 31); };
    return op != LinOp::TN && fits(d.ra, d.ca) && fits(d.rb, d.cb) && lora_epi_ok(g, r, d.s.N);
}

hipError_t lin_run(LinOp op, LinForm f, const void *a, const void *b, float *out, int M, int N, int K,
                   const GemmWs &ws, hipStream_t st, const LoraSegs *lora, int r, float alpha) {
    const LinDims d = lin_dims(op, M, N, K);
    const long v = chunk_elems(f);
    char *w = (char *)ws.p;
    long lda = d.ca, ldb = d.cb;
    const bool pa = needs_pack(f, a, d.ca), pb = needs_pack(f, b, d.cb);
    if (pa || pb) {
        void *da = w, *db = w + (pa ? packed_bytes(f, d.ra, d.ca) : 0);
        const hipError_t e = lin_pack(f, a, pa ? d.ra : 0, d.ca, da, b, pb ? d.rb : 0, d.cb, db, st);
        if (e != hipSuccess) return e;
        w = (char *)db + (pb ? packed_bytes(f, d.rb, d.cb) : 0);
        if (pa) a = da, lda = (d.ca + v - 1) / v * v;
        if (pb) b = db, ldb = (d.cb + v - 1) / v * v;
    }
    const GemmWs rest{w, ws.p ? ws.bytes - (size_t)(w - (char *)ws.p) : 0};
    // views of 2 GiB and more go through g16_* / g32_* (row chunks or the generic kernel)
    const int es = f == LinForm::F32 ? 4 : 2;
    const size_t ba = ((size_t)(d.ra - 1) * lda + (lda > d.ca ? lda : d.ca)) * es,
                 bb = ((size_t)(d.rb - 1) * ldb + (ldb > d.cb ? ldb : d.cb)) * es;
    if (ba < (1ull << 31) && bb < (1ull << 31)) {
        // both aligned now; the zeros past a packed row's run are part of its chunks
        const Op16 oa{(const bf16 *)a, lda, (unsigned)ba}, ob{(const bf16 *)b, ldb, (unsigned)bb};
        const EpiStore ep{out, d.s.N, nullptr, 0, 1.f, 0.f};
        if (lora) {
            const EpiLora<EpiStore> el{ep, *lora, r, alpha};
            if (f == LinForm::F32)
                return op == LinOp::NT ? run32<Lay::K, Lay::K>(oa, ob, d.s, el, rest, st)
                                       : run32<Lay::K, Lay::MN>(oa, ob, d.s, el, rest, st);
            return op == LinOp::NT ? run16<Lay::K, Lay::K>(oa, ob, d.s, el, rest, st)
                                   : run16<Lay::K, Lay::MN>(oa, ob, d.s, el, rest, st);
        }
        if (f == LinForm::F32) {
            if (op == LinOp::NT) return run32<Lay::K, Lay::K>(oa, ob, d.s, ep, rest, st);
            if (op == LinOp::NN) return run32<Lay::K, Lay::MN>(oa, ob, d.s, ep, rest, st);
            return run32<Lay::MN, Lay::MN>(oa, ob, d.s, ep, rest, st);
        }
        if (op == LinOp::NT) return run16<Lay::K, Lay::K>(oa, ob, d.s, ep, rest, st);
        if (op == LinOp::NN) return run16<Lay::K, Lay::MN>(oa, ob, d.s, ep, rest, st);
        return run16<Lay::MN, Lay::MN>(oa, ob, d.s, ep, rest, st);
    }
    if (lora) return hipErrorInvalidValue;  // lin_lora_ok does not hold
    if (f == LinForm::F32) {
        const float *x = (const float *)a, *y = (const float *)b;
        if (op == LinOp::NT) return g32_nt(x, lda, y, ldb, out, N, M, N, K, nullptr, 0, 1.f, 0.f, rest, st);
        if (op == LinOp::NN) return g32_nn(x, lda, y, ldb, out, K, M, N, K, 1.f, 0.f, rest, st);
        return g32_tn(x, lda, y, ldb, out, K, M, N, K, 1.f, 0.f, rest, st);
    }
    const bf16 *x = (const bf16 *)a, *y = (const bf16 *)b;
    if (op == LinOp::NT) return g16_nt(x, lda, y, ldb, out, N, M, N, K, nullptr, 0, 1.f, 0.f, rest, st);
    if (op == LinOp::NN) return g16_nn(x, lda, y, ldb, out, K, M, N, K, 1.f, 0.f, rest, st);
    return g16_tn(x, lda, y, ldb, out, K, M, N, K, 1.f, 0.f, rest, st);
}

size_t g32_ws_bytes_for(int M, int N, int K, int min_chains) {
    const GemmShape s{M, N, K};
    GemmWs any{(void *)1, ~size_t(0)};  // (planned for, not used)
    any.min_chains = min_chains;
    return std::max(ws_for(plan32(s, any), s), ws_for(plan32(s, any, true), s));
}

size_t g16_ws_bytes_for(int M, int N, int K, bool keep_sums) {
    const GemmShape s{M, N, K};
    GemmWs any{(void *)1, ~size_t(0)};
    any.keep_sums = keep_sums;
    return std::max(ws_for(plan(s, any), s), ws_for(plan(s, any, true), s));
}

}  // namespace vkh
