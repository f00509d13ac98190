// Cut cross-entropy over the vocabulary (reference: shaders/cce_forward.comp,
// cce_backward_dh.comp, cce_backward_dw.comp; oracle src/cpu/cce.zig:89-268).
//
// Forward: the logits z = h W^T are produced tile by tile by the MFMA GEMM
// and never stored; its epilogue reduces each wave's 64-column slice of a row
// to (max, sum exp(z - max), sum z) and captures the target logit.  A second
// kernel merges the slices per row (fp64) into lse and the per-row loss
// lse - (1 - eps) z_t - eps mean(z) + lambda_z lse^2, and a third averages.
//
// Backward: the logits are recomputed once by the GEMM whose epilogue writes
//   dz = ((1 + 2 lambda_z lse) exp(z - lse) - (1 - eps)[v == t] - eps / V) / N
// (bf16 in the bf16 precision, fp32 otherwise) to HBM, then two MFMA GEMMs
// form dh = dz W and dW = dz^T h.  The reference recomputes the logits twice
// with scalar dot products (per row for dh, per vocab row for dW,
// cce_backward_dh.comp:109-123, cce_backward_dw.comp:73-103); on a 288 GB
// part the [N, V] dz buffer (0.6 GB at N = 2048) is cheap and turns the
// backward into three dense GEMMs.
//
// With fp32 dz (the fp32 precision) the forward's epilogue can also store the
// fp32 logits into the dz buffer (z_out), and the backward then forms dz from
// them in place with one streaming pass (cce_dz_k, the dz epilogue's
// arithmetic element by element) instead of recomputing the logits GEMM: the
// same values bit for bit, 2.5 GB of traffic in place of a 0.64 TFLOP product.
#include <math.h>

#include "gemm16.hpp"
#include "ops.hpp"

namespace vkh {

namespace {

constexpr int WN = 64;  // columns per wave slice with the 128x128 tile
constexpr float LOG2E = 1.4426950408889634f;

struct CceWork {
    float *pm, *ps, *pz;  // [N][nparts]
    float *zt;            // [N]
    int nparts;
};

inline CceWork carve(float *work, const CceShape &s) {
    const int np = (s.V + WN - 1) / WN;
    const size_t part = (size_t)s.N * np;
    return CceWork{work, work + part, work + 2 * part, work + 3 * part, np};
}

struct EpiCceStats {
    static constexpr bool kSplits = false;
    CceWork w;
    const uint32_t *tgt;
    int V;
    float *zo = nullptr;  // when set: the logits themselves, rows of ldz
    long ldz = 0;

    template <int TM, int TN>
    VKH_DEV void apply(const f32x4 (&acc)[TM][TN], const FragPos &fp, const GemmShape &s) const {
        static_assert(TN * 16 == WN, "wave slice width");
        const int part = fp.col0 / WN;
        // the last tile's second slice can lie wholly past V: it owns no partial
        if (part >= w.nparts) return;
        // slices wholly inside the vocabulary (all but the last) skip the
        // per-column range checks
        if (fp.col0 + WN <= V) rows<TM, TN, true>(acc, fp, s, part);
        else rows<TM, TN, false>(acc, fp, s, part);
    }

    template <int TM, int TN, bool FULL>
    VKH_DEV void rows(const f32x4 (&acc)[TM][TN], const FragPos &fp, const GemmShape &s,
                      int part) const {
        const int c16 = fp.lane % 16, g = fp.lane / 16;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = fp.row0 + 16 * i + 4 * g + r;
                const bool rok = row < s.M;
                // the target column relative to this lane's first column: the
                // lane of fragment j holds it when tc == 16 j
                const int tc = rok ? (int)tgt[row] - fp.col0 - c16 : -1;
                float mx = -INFINITY, zs = 0.f;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if (FULL || fp.col0 + 16 * j + c16 < V) {
                        const float z = acc[i][j][r];
                        mx = fmaxf(mx, z);
                        zs += z;
                        if (tc == 16 * j) w.zt[row] = z;
                        if (zo && rok) zo[(size_t)row * ldz + fp.col0 + 16 * j + c16] = z;
                    }
                }
                mx = row16_max(mx);
                const float mxl = mx * LOG2E;
                float se = 0.f;
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    if (FULL || fp.col0 + 16 * j + c16 < V)
                        se += __builtin_amdgcn_exp2f(fmaf(acc[i][j][r], LOG2E, -mxl));
                se = row16_sum(se);
                zs = row16_sum(zs);
                if (rok && c16 == 0) {
                    const size_t idx = (size_t)row * w.nparts + part;
                    w.pm[idx] = mx;
                    w.ps[idx] = se;
                    w.pz[idx] = zs;
                }
            }
    }
};

// dz of one row: the coefficients of dz = sf exp(z - lse) - off - [v == t] tsc
// (the 1 / N folded in), and one element of it.  The dz epilogue and cce_dz_k
// both compute through these, so their results agree bit for bit.
struct DzRow {
    float lL2, sf;
};
VKH_DEV DzRow dz_row(float l, float zl2, float inv_n) { return DzRow{l * LOG2E, (1.0f + zl2 * l) * inv_n}; }
VKH_DEV float dz_elem(float z, const DzRow &r, float off, float tsc, bool is_t) {
    const float p = __builtin_amdgcn_exp2f(fmaf(z, LOG2E, -r.lL2));
    float d = fmaf(r.sf, p, -off);
    if (is_t) d -= tsc;
    return d;
}

template <typename TZ>
struct EpiCceDz {
    static constexpr bool kSplits = false;
    TZ *dz;
    const uint32_t *tgt;
    const float *lse;
    int V;
    long ldz;  // zeros go to columns [V, ldz)
    float inv_n, t_scale, eps_over_v, zl2;

    template <int TM, int TN>
    VKH_DEV void apply(const f32x4 (&acc)[TM][TN], const FragPos &fp, const GemmShape &s) const {
        if (fp.col0 + 16 * TN <= V) rows<TM, TN, true>(acc, fp, s);
        else rows<TM, TN, false>(acc, fp, s);
    }

    // dz = (sf p - eps / V - [v == t] (1 - eps)) / N with p = exp(z - lse),
    // sf = 1 + 2 lambda_z lse; the 1 / N folded into the coefficients
    template <int TM, int TN, bool FULL>
    VKH_DEV void rows(const f32x4 (&acc)[TM][TN], const FragPos &fp, const GemmShape &s) const {
        const int c16 = fp.lane % 16, g = fp.lane / 16;
        const float off = eps_over_v * inv_n, tsc = t_scale * inv_n;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = fp.row0 + 16 * i + 4 * g + r;
                if (row >= s.M) continue;
                const DzRow dr = dz_row(lse[row], zl2, inv_n);
                const int tc = (int)tgt[row] - fp.col0 - c16;
                TZ *out = dz + (size_t)row * ldz + fp.col0 + c16;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if (!FULL && fp.col0 + 16 * j + c16 >= V) {
                        if (fp.col0 + 16 * j + c16 < ldz) out[16 * j] = (TZ)0.f;
                        continue;
                    }
                    out[16 * j] = (TZ)dz_elem(acc[i][j][r], dr, off, tsc, tc == 16 * j);
                }
            }
    }
};

// dz from the stored fp32 logits z, rows of ldz (z and dz may be the same buffer: each
// element is read and then written by one thread).  Block (x, row): 4 columns
// per thread with 16-byte rows (ldz % 4 == 0 and 16-byte aligned), else 1.
template <typename TZ, int VEC>
__global__ __launch_bounds__(256) void cce_dz_k(const float *z, TZ *dz, const uint32_t *tgt,
                                                const float *lse, int V, long ldz, float inv_n,
                                                float t_scale, float eps_over_v, float zl2) {
    const int row = blockIdx.y;
    const int c0 = (blockIdx.x * 256 + threadIdx.x) * VEC;
    if (c0 >= ldz) return;
    const DzRow dr = dz_row(lse[row], zl2, inv_n);
    const float off = eps_over_v * inv_n, tsc = t_scale * inv_n;
    const int t = (int)tgt[row];
    const size_t i = (size_t)row * ldz + c0;
    if constexpr (VEC == 4) {
        const float4 zv = *reinterpret_cast<const float4 *>(z + i);
        float d0 = dz_elem(zv.x, dr, off, tsc, t == c0), d1 = dz_elem(zv.y, dr, off, tsc, t == c0 + 1),
              d2 = dz_elem(zv.z, dr, off, tsc, t == c0 + 2), d3 = dz_elem(zv.w, dr, off, tsc, t == c0 + 3);
        if (c0 + 4 > V) {  // the zeros of a padded row (its stored logits end at V)
            if (c0 >= V) d0 = 0.f;
            if (c0 + 1 >= V) d1 = 0.f;
            if (c0 + 2 >= V) d2 = 0.f;
            d3 = 0.f;
        }
        if constexpr (sizeof(TZ) == 4) {
            *reinterpret_cast<float4 *>(dz + i) = make_float4(d0, d1, d2, d3);
        } else {
            dz[i] = (TZ)d0; dz[i + 1] = (TZ)d1; dz[i + 2] = (TZ)d2; dz[i + 3] = (TZ)d3;
        }
    } else {
        dz[i] = c0 < V ? (TZ)dz_elem(z[i], dr, off, tsc, t == c0) : (TZ)0.f;
    }
}

__global__ void cce_merge_k(CceShape s, CceWork w, float *lse, float *loss_row) {
    const int lane = threadIdx.x % 64;
    const int row = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
    if (row >= s.N) return;
    const float *pm = w.pm + (size_t)row * w.nparts;
    const float *ps = w.ps + (size_t)row * w.nparts;
    const float *pz = w.pz + (size_t)row * w.nparts;
    float M = -INFINITY;
    for (int i = lane; i < w.nparts; i += 64) M = fmaxf(M, pm[i]);
    M = wave_max(M);
    double S = 0, Z = 0;
    for (int i = lane; i < w.nparts; i += 64) {
        S += (double)ps[i] * exp((double)pm[i] - (double)M);
        Z += (double)pz[i];
    }
    S = wave_sum(S);
    Z = wave_sum(Z);
    if (lane == 0) {
        const float l = (float)(log(S) + (double)M);
        lse[row] = l;
        const double eps = s.label_smoothing;
        const double ce = (double)l - (double)(1.0f - s.label_smoothing) * (double)w.zt[row] -
                          eps * (Z / (double)s.V);
        const double zp = (double)s.z_loss_scale * (double)l * (double)l;
        if (loss_row) loss_row[row] = (float)(ce + zp);
        w.pm[(size_t)row * w.nparts] = (float)(ce + zp);  // reuse slot 0 for the mean
    }
}

__global__ void cce_mean_k(CceShape s, CceWork w, float *loss_mean) {
    __shared__ double sh[4];
    double acc = 0;
    for (int r = threadIdx.x; r < s.N; r += blockDim.x) acc += (double)w.pm[(size_t)r * w.nparts];
    acc = wave_sum(acc);
    if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = acc;
    __syncthreads();
    if (threadIdx.x == 0) loss_mean[0] = (float)((sh[0] + sh[1] + sh[2] + sh[3]) / (double)s.N);
}

// The logits GEMM's tile (wave slices of 64 columns in each, as the epilogues need):
// the one with the least rounds x tile area over its rate relative to 256 x 256.
// fp32 is bound by the matrix cores, so the small tiles lose little and fill the
// chip better (127 x 32003 x 768 took 197 us on 126 blocks of 256 x 256; 502 of
// 64 x 128 share its matrix work over all CUs); bf16 needs the large ones wherever they
// fill it.  The rates are read off the heads of profiles/head_logits_tiles.csv, on which
// the pick is 2 % above the best tile on average and 11 % at most.
template <bool F32, class Epi>
hipError_t logits_tiles(const Op16 &a, const Op16 &b, const GemmShape &sh, const Epi &epi, hipStream_t st) {
    const SplitK one{1, nullptr};
    constexpr int g = tile_group_rows<Lay::K, Lay::K>();
    auto cost = [&](int bm, int bn, double rate) {
        const double tiles = (double)ceil_div(sh.M, bm) * ceil_div(sh.N, bn);
        return ceil(tiles / 256) * bm * bn / rate;
    };
    const double c0 = cost(256, 256, 1.0), c1 = cost(128, 256, F32 ? 0.98 : 0.8),
                 c2 = cost(128, 128, F32 ? 0.96 : 0.65), c3 = cost(64, 128, F32 ? 0.9 : 0.45);
    if (c0 <= c1 && c0 <= c2 && c0 <= c3)
        return launch_gemm16<Tile16<256, 256, 2, 4>, Lay::K, Lay::K, Epi, F32>(a, b, sh, epi, one, g, st);
    if (c1 <= c2 && c1 <= c3)
        return launch_gemm16<Tile16<128, 256, 2, 4>, Lay::K, Lay::K, Epi, F32>(a, b, sh, epi, one, g, st);
    if (c2 <= c3)
        return launch_gemm16<Tile16<128, 128, 2, 2>, Lay::K, Lay::K, Epi, F32>(a, b, sh, epi, one, g, st);
    return launch_gemm16<Tile16<64, 128, 2, 2>, Lay::K, Lay::K, Epi, F32>(a, b, sh, epi, one, g, st);
}

// fp32 operands; the generic MFMA GEMM where they do not fit the DMA-staged rules.
template <class Epi>
hipError_t logits32(const CceShape &s, const float *h, const float *w, const Epi &epi, hipStream_t st) {
    const long ld = s.hs();
    GemmShape sh{s.N, s.V, s.D};
    const size_t hb = (size_t)s.N * ld * 4, wb = (size_t)s.V * ld * 4;
    if (ld % 4 == 0 && ((uintptr_t)h & 15u) == 0 && ((uintptr_t)w & 15u) == 0 && hb < (1ull << 31) &&
        wb < (1ull << 31))
        return logits_tiles<true>(Op16{(const bf16 *)h, ld, (unsigned)hb},
                                  Op16{(const bf16 *)w, ld, (unsigned)wb}, sh, epi, st);
    GemmOperand a{h, ld, vec_ok(h, ld, 4, Lay::K)};
    GemmOperand b{w, ld, vec_ok(w, ld, 4, Lay::K)};
    return launch_gemm<TileCfg<128, 128, 32>, false, float, Lay::K, float, Lay::K>(a, b, sh, epi, st);
}

// bf16 operands, the same way.
template <class Epi>
hipError_t logits16(const CceShape &s, const bf16 *h, const bf16 *w, const Epi &epi,
                    hipStream_t st) {
    const long ld = s.hs();
    GemmShape sh{s.N, s.V, s.D};
    const size_t hb = (size_t)s.N * ld * 2, wb = (size_t)s.V * ld * 2;
    if (ld % 8 == 0 && ((uintptr_t)h & 15u) == 0 && ((uintptr_t)w & 15u) == 0 && hb < (1ull << 31) &&
        wb < (1ull << 31))
        return logits_tiles<false>(Op16{h, ld, (unsigned)hb}, Op16{w, ld, (unsigned)wb}, sh, epi, st);
    GemmOperand a{h, ld, vec_ok(h, ld, 2, Lay::K)};
    GemmOperand b{w, ld, vec_ok(w, ld, 2, Lay::K)};
    return launch_gemm<TileCfg<128, 128, 64>, true, bf16, Lay::K, bf16, Lay::K>(a, b, sh, epi, st);
}

template <typename TZ>
hipError_t dz_from_logits(const CceShape &s, const float *z, const EpiCceDz<TZ> &e, hipStream_t st) {
    const long ld = s.zs();
    const bool v4 = ld % 4 == 0 && ((uintptr_t)z & 15u) == 0 && ((uintptr_t)e.dz & 15u) == 0;
    const dim3 grid((unsigned)ceil_div(ld, 256 * (v4 ? 4 : 1)), (unsigned)s.N);
    if (v4)
        hipLaunchKernelGGL((cce_dz_k<TZ, 4>), grid, dim3(256), 0, st, z, e.dz, e.tgt, e.lse, s.V, ld,
                           e.inv_n, e.t_scale, e.eps_over_v, e.zl2);
    else
        hipLaunchKernelGGL((cce_dz_k<TZ, 1>), grid, dim3(256), 0, st, z, e.dz, e.tgt, e.lse, s.V, ld,
                           e.inv_n, e.t_scale, e.eps_over_v, e.zl2);
    return hipGetLastError();
}

template <typename TZ>
EpiCceDz<TZ> dz_epi(const CceShape &s, TZ *dz, const uint32_t *tgt, const float *lse) {
    return EpiCceDz<TZ>{dz, tgt, lse, s.V, s.zs(), 1.0f / (float)s.N, 1.0f - s.label_smoothing,
                        s.label_smoothing / (float)s.V, 2.0f * s.z_loss_scale};
}

hipError_t merge(const CceShape &s, const CceWork &cw, float *lse, float *loss_row, float *loss_mean,
                 hipStream_t st) {
    hipLaunchKernelGGL(cce_merge_k, dim3(ceil_div(s.N, 4)), dim3(256), 0, st, s, cw, lse, loss_row);
    if (loss_mean) hipLaunchKernelGGL(cce_mean_k, dim3(1), dim3(256), 0, st, s, cw, loss_mean);
    return hipGetLastError();
}

}  // namespace

size_t cce_work_floats(const CceShape &s) {
    const size_t np = (s.V + WN - 1) / WN;
    return 3 * (size_t)s.N * np + s.N;
}

hipError_t cce_forward(const CceShape &s, const float *h, const float *w, const uint32_t *tgt,
                       float *lse, float *loss_row, float *loss_mean, float *work, hipStream_t st,
                       float *z_out) {
    if (s.N <= 0) return hipSuccess;
    const CceWork cw = carve(work, s);
    const hipError_t err = logits32(s, h, w, EpiCceStats{cw, tgt, s.V, z_out, s.zs()}, st);
    return err != hipSuccess ? err : merge(s, cw, lse, loss_row, loss_mean, st);
}

hipError_t cce_backward(const CceShape &s, const float *h, const float *w, const uint32_t *tgt,
                        const float *lse, float *dz, float *dh, float *dw, float dw_beta,
                        const GemmWs &ws, hipStream_t st, const float *z) {
    if (s.N <= 0) return hipSuccess;
    const EpiCceDz<float> e = dz_epi(s, dz, tgt, lse);
    hipError_t err = z ? dz_from_logits(s, z, e, st) : logits32(s, h, w, e, st);
    if (err != hipSuccess) return err;
    // dW[V, D] = dz^T h ;  dh[N, D] = dz W
    const bool pad = s.ldh || s.ldz;
    if (dw) {
        err = g32_tn(dz, s.zs(), h, s.hs(), dw, s.D, s.N, s.V, s.D, 1.f, dw_beta, ws, st, pad);
        if (err != hipSuccess) return err;
    }
    if (dh) err = g32_nn(dz, s.zs(), w, s.hs(), dh, s.D, s.N, s.V, s.D, 1.f, 0.f, ws, st, pad);
    return err;
}

hipError_t cce_forward16(const CceShape &s, const bf16 *h, const bf16 *w, const uint32_t *tgt,
                         float *lse, float *loss_row, float *loss_mean, float *work,
                         hipStream_t st, float *z_out) {
    if (s.N <= 0) return hipSuccess;
    const CceWork cw = carve(work, s);
    const hipError_t err = logits16(s, h, w, EpiCceStats{cw, tgt, s.V, z_out, s.zs()}, st);
    return err != hipSuccess ? err : merge(s, cw, lse, loss_row, loss_mean, st);
}

hipError_t cce_backward16(const CceShape &s, const bf16 *h, const bf16 *w, const uint32_t *tgt,
                          const float *lse, bf16 *dz, float *dh, float *dw, float dw_beta,
                          const GemmWs &ws, hipStream_t st, const float *z) {
    if (s.N <= 0) return hipSuccess;
    const EpiCceDz<bf16> e = dz_epi(s, dz, tgt, lse);
    hipError_t err = z ? dz_from_logits(s, z, e, st) : logits16(s, h, w, e, st);
    if (err != hipSuccess) return err;
    const bool pad = s.ldh || s.ldz;
    if (dw) {
        err = g16_tn(dz, s.zs(), h, s.hs(), dw, s.D, s.N, s.V, s.D, 1.f, dw_beta, ws, st, pad);
        if (err != hipSuccess) return err;
    }
    if (dh) err = g16_nn(dz, s.zs(), w, s.hs(), dh, s.D, s.N, s.V, s.D, 1.f, 0.f, ws, st, pad);
    return err;
}

}  // namespace vkh
