// Backward with shared coefficients, bf16, n <= 8, rows of at most 4096 channels: with one H for all samples nothing of dx
// depends on a batch-wide result, so one pass over dy and x forms everything:
//
//   dM = dy x^T    W1 = dy diag(w) x^T    XX = x x^T   (per sample, on the matrix cores)    reference stream_ops.cuh:852-927
//   dx[j,c] = sum_i M[i,j] dy[i,c] + Hpre[j] da[c]                                        reference stream_ops.cuh:761-850, :646-663
//   da = df w / q - a s1 / (C q^3),  df = Hpost . dy, a = Hpre . x, s1 = Hpost^T W1 Hpre  reference rmsnorm.cuh:255-294
//   dw = sum over samples of df a / q;  dM, dHpre, dHpost summed over samples (the Sinkhorn backward runs once, on the sums)
//
// A workgroup walks samples b, b + G, ... and holds one at a time in registers (a lane: 8 consecutive channels of one
// stream, four neighbouring lanes: the four streams of a group, as bwd_resident.hip), the next one on its way to registers
// of its own.  The batch sums of dw and of the coefficient gradients are kept in float64 by the lanes that form them and leave
// as one row per workgroup.
// What bounds it: bytes (dy and x in, dx out).  With one sample per workgroup every sample leaves a row of C floats for dw, at
// n = 4 a fourteenth of the launch's traffic, and the batch-sum launch reads them back: n=4 B=8192 C=2560 126 + 37 us, here 104
// (4.8 TB/s) + 8; n=8 B=4000 C=2560 146 + 32, here 151 + 8.  (bwd_static_preferred() has more.)
#include "coef_bwd_small.h"
#include "lds_stage.h"
#include "tuning.h"

#include <algorithm>

namespace mhc {

struct BwdStaticArgs {
    BwdReduceArgs r;       // inputs
    void *dx, *df;         // [B, n, C]; [B, C] or nullptr (only with r.f_inject)
    double *u, *red;       // one row per workgroup: [G][C] sums of df a / q, [G][D + 3] raw dM | dHpre | dHpost
};

template <int SEL> __device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), SEL * 0x55, 0xF, 0xF, true));
}
__device__ __forceinline__ float quad_sum(float v) {
    v += dpp_mov<kDppQuadXor1>(v);
    v += dpp_mov<kDppQuadXor2>(v);
    return v;
}

// the next sample's words fit beside the others, and fewer workgroups are no loss
template <int NP, int TW, int ITEMS> constexpr bool static_next() { return NP == 4 && (ITEMS >= 4 || TW == 8); }
template <int NP, int ITEMS> constexpr bool static_lean() { return NP == 8 && ITEMS >= 3; }

// TW waves of ITEMS chunks of 128 channels.  NEXT: the next sample is requested while this one is worked on.
// RAG: rows of any length (C % 8 != 0): the last chunk of a row is loaded from C - 8 on and shifted down.
template <int NP, int WMODE, int TW, int ITEMS, bool NEXT, bool RAG>
__global__ __launch_bounds__(64 * TW, 2) void bwd_static_kernel(BwdStaticArgs sa) {
    using SK = SkSmall<NP>;
    using CB = CoefBwdSmall<NP, false, true, true>;
    constexpr int NB = NP / 4, K = 3 * NP * NP;
    constexpr bool inject = WMODE == kGramInject;
    const BwdReduceArgs &a = sa.r;
    __shared__ float slot_s[K * TW * 4];  // one slot per 16-lane row
    __shared__ float tot_s[K + 1];        // the sums, then s1
    __shared__ float xch_s[CB::kXch];
    // LEAN: the weights (fp32) and the sums of dw live in LDS ([chunk][2 x 4 floats | 2 x 4 doubles by lane]), not in registers
    constexpr bool LEAN = static_lean<NP, ITEMS>() && !inject;
    extern __shared__ __align__(16) double lean_s[];  // [TW ITEMS 128] sums, then [TW ITEMS 128] floats of w
    float *const w_s = reinterpret_cast<float *>(lean_s + TW * ITEMS * 128);
    const int n = a.n, C = a.C, G = gridDim.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blk = lane >> 2, i = lane & 3;

    CB cb;
    if (tid < SK::kGroup) cb.prefetch(a, blockIdx.x, tid);
    float hohp = 0.f;  // the threads that will hold the sums of W1: their factor of s1
    if (!inject && tid >= NP * NP && tid < 2 * NP * NP) {
        const int e = tid - NP * NP, r = e / NP, c = e % NP;
        hohp = r < n && c < n ? a.Hpost[r] * a.Hpre[c] : 0.f;
    }
    bool in[ITEMS], sv[NB];
    int cc[ITEMS], shift[ITEMS];
    size_t rowoff[NB];
    float hpre[NB], hpost[NB], Mc[NB][NB][4];  // Mc[I][J][ii] = M[source stream 4J + ii][target stream 4I + i]
#pragma unroll
    for (int I = 0; I < NB; I++) {
        sv[I] = 4 * I + i < n;  // streams >= n: masked, they alias stream 0
        rowoff[I] = (size_t)(sv[I] ? 4 * I + i : 0) * C;
        hpre[I] = sv[I] ? a.Hpre[4 * I + i] : 0.f;
        hpost[I] = sv[I] ? a.Hpost[4 * I + i] : 0.f;
#pragma unroll
        for (int J = 0; J < NB; J++)
#pragma unroll
            for (int ii = 0; ii < 4; ii++) Mc[I][J][ii] = sv[I] && 4 * J + ii < n ? a.M[(4 * J + ii) * n + 4 * I + i] : 0.f;
    }
    RawVec<bf16_t, 8> wb[LEAN ? 1 : ITEMS];
    RawVec<float, 8> wf[LEAN ? 1 : ITEMS];
    double usum[LEAN ? 1 : ITEMS][2];  // channels 2 i, 2 i + 1 of the chunk (the four lanes of a quad form the same eight summands)
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int c = (wave + TW * it) * 128 + blk * 8;
        in[it] = c < C;
        cc[it] = in[it] ? (RAG ? min(c, C - 8) : c) : 0;
        shift[it] = RAG && in[it] && c + 8 > C ? c + 8 - C : 0;
        const int k = LEAN ? 0 : it;
        usum[k][0] = usum[k][1] = 0.0;
        if constexpr (!inject) {
            if constexpr (WMODE == kGramWBf16) {
                if constexpr (RAG) { wb[k].load_any(static_cast<const bf16_t *>(a.w) + cc[it]); wb[k].drop(shift[it]); }
                else wb[k].load(static_cast<const bf16_t *>(a.w) + cc[it]);
            } else {
                if constexpr (RAG) { wf[k].load_any(static_cast<const float *>(a.w) + cc[it]); wf[k].drop(shift[it]); }
                else wf[k].load(static_cast<const float *>(a.w) + cc[it]);
            }
            if constexpr (LEAN) {  // (the quad's four lanes hold the same eight: lane i leaves two of them)
                float wv[8];
                if constexpr (WMODE == kGramWBf16) wb[0].get(wv);
                else wf[0].get(wv);
                const int c = (wave + TW * it) * 128 + blk * 8 + 2 * i;
                w_s[c] = i == 0 ? wv[0] : i == 1 ? wv[2] : i == 2 ? wv[4] : wv[6];
                w_s[c + 1] = i == 0 ? wv[1] : i == 1 ? wv[3] : i == 2 ? wv[5] : wv[7];
                lean_s[c] = lean_s[c + 1] = 0.0;
            }
        }
    }

    if constexpr (LEAN) __syncthreads();

    struct Tile { uint4 g[ITEMS][NB], x[ITEMS][NB], f[ITEMS]; float q; };
    auto fetch = [&](Tile &t, int b) {  // raw words: they are masked where they are taken
        const bf16_t *gb = static_cast<const bf16_t *>(a.dy) + (size_t)b * n * C, *xb = static_cast<const bf16_t *>(a.x) + (size_t)b * n * C;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
#pragma unroll
            for (int I = 0; I < NB; I++) {
                t.g[it][I] = ldg16<RAG>(gb + rowoff[I] + cc[it]);
                t.x[it][I] = ldg16<RAG>(xb + rowoff[I] + cc[it]);
            }
            if constexpr (inject) t.f[it] = ldg16<RAG>(static_cast<const bf16_t *>(a.f_inject) + (size_t)b * C + cc[it]);
        }
        if constexpr (!inject) t.q = a.q[b];
    };
    auto take = [&](uint4 v, int it, bool ok) {
        if constexpr (RAG) v = drop8(v, shift[it]);
        return masked16(v, in[it] && ok);
    };
    double dm64 = 0.0, dpre64 = 0.0, dpost64 = 0.0;  // this lane's coefficient gradients (first SK::kGroup lanes)

    Tile cur, nxt;
    if constexpr (NEXT) fetch(cur, blockIdx.x);
    for (int b = blockIdx.x; b < a.B; b += G) {
        if constexpr (!NEXT) fetch(cur, b);
        // (made opaque once per sample: addresses and the weights as floats, formed ahead of the loop, would hold registers)
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            asm volatile("" : "+v"(cc[it]));
            if constexpr (WMODE == kGramWBf16 && !LEAN) {
#pragma unroll
                for (int k = 0; k < 4; k++) asm volatile("" : "+v"(wb[it].w[k]));
            }
        }
        uint4 gr[ITEMS][NB], xr[ITEMS][NB], fr[ITEMS];
        const float qraw = inject ? 1.f : cur.q;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
#pragma unroll
            for (int I = 0; I < NB; I++) { gr[it][I] = take(cur.g[it][I], it, sv[I]); xr[it][I] = take(cur.x[it][I], it, sv[I]); }
            if constexpr (inject) fr[it] = take(cur.f[it], it, i == 0);
        }
        if constexpr (NEXT) {
            __builtin_amdgcn_sched_barrier(0);
            if (b + G < a.B) fetch(nxt, b + G);
            else nxt = Tile{};  // (not the old words: they would stay in registers)
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- Gram sums ----------------------------------------------------------------------------------
        f32x4_t acc[3][NB][NB];
#pragma unroll
        for (int m = 0; m < 3; m++)
#pragma unroll
            for (int I = 0; I < NB; I++)
#pragma unroll
                for (int J = 0; J < NB; J++) acc[m][I][J] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            if constexpr (NP == 8) __builtin_amdgcn_sched_barrier(0);
            bf16x4_t g0[NB], g1[NB], x0[NB], x1[NB];  // first / second group of four channels
#pragma unroll
            for (int I = 0; I < NB; I++) {
                g0[I] = bf16x4_of(gr[it][I].x, gr[it][I].y); g1[I] = bf16x4_of(gr[it][I].z, gr[it][I].w);
                x0[I] = bf16x4_of(xr[it][I].x, xr[it][I].y); x1[I] = bf16x4_of(xr[it][I].z, xr[it][I].w);
            }
#pragma unroll
            for (int I = 0; I < NB; I++)
#pragma unroll
                for (int J = 0; J < NB; J++) {
                    acc[0][I][J] = mfma4(g0[I], x0[J], acc[0][I][J]);
                    acc[0][I][J] = mfma4(g1[I], x1[J], acc[0][I][J]);
                }
            if constexpr (inject) {
                const bf16x4_t f0 = bf16x4_of(fr[it].x, fr[it].y), f1 = bf16x4_of(fr[it].z, fr[it].w);
#pragma unroll
                for (int I = 0; I < NB; I++) {
                    acc[1][I][0] = mfma4(g0[I], f0, acc[1][I][0]);
                    acc[1][I][0] = mfma4(g1[I], f1, acc[1][I][0]);
                }
            } else {
                float wv[8];
                if constexpr (LEAN) lds_floats<8>(w_s + (wave + TW * it) * 128 + blk * 8, wv);
                else if constexpr (WMODE == kGramWBf16) wb[it].get(wv);
                else wf[it].get(wv);
#pragma unroll
                for (int I = 0; I < NB; I++) {
                    // dy * w as a bf16 pair (rounded value + remainder): dHpre is a difference of two sums built on W1, a
                    // single rounding of the products is not enough for it.  The product with a bf16 weight has 16 bits, which
                    // the pair holds exactly; with an fp32 weight ragged rows take the rest of its 24 bits too.
                    const uint32_t gw[4] = {gr[it][I].x, gr[it][I].y, gr[it][I].z, gr[it][I].w};
                    constexpr bool REST = RAG && WMODE == kGramWF32;
                    uint32_t hw[4], lw[4], rw[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float p0 = bf16lo_to_f32(gw[k]) * wv[2 * k], p1 = bf16hi_to_f32(gw[k]) * wv[2 * k + 1];
                        hw[k] = pack_bf16x2(p0, p1);
                        const float q0 = p0 - bf16lo_to_f32(hw[k]), q1 = p1 - bf16hi_to_f32(hw[k]);
                        lw[k] = pack_bf16x2(q0, q1);
                        if constexpr (REST) rw[k] = pack_bf16x2(q0 - bf16lo_to_f32(lw[k]), q1 - bf16hi_to_f32(lw[k]));
                    }
#pragma unroll
                    for (int J = 0; J < NB; J++) {
                        acc[1][I][J] = mfma4(bf16x4_of(hw[0], hw[1]), x0[J], acc[1][I][J]);
                        acc[1][I][J] = mfma4(bf16x4_of(hw[2], hw[3]), x1[J], acc[1][I][J]);
                        acc[1][I][J] = mfma4(bf16x4_of(lw[0], lw[1]), x0[J], acc[1][I][J]);
                        acc[1][I][J] = mfma4(bf16x4_of(lw[2], lw[3]), x1[J], acc[1][I][J]);
                        if constexpr (REST) {
                            acc[1][I][J] = mfma4(bf16x4_of(rw[0], rw[1]), x0[J], acc[1][I][J]);
                            acc[1][I][J] = mfma4(bf16x4_of(rw[2], rw[3]), x1[J], acc[1][I][J]);
                        }
                        acc[2][I][J] = mfma4(x0[I], x0[J], acc[2][I][J]);
                        acc[2][I][J] = mfma4(x1[I], x1[J], acc[2][I][J]);
                    }
                }
            }
        }
        // Lane (block, j) holds column j of its block's products, register = row.  Sum over the four blocks of a 16-lane row
        // with DPP, one LDS slot per row; K threads finish the sums.
        const int slot = tid >> 4;
#pragma unroll
        for (int m = 0; m < 3; m++)
#pragma unroll
            for (int I = 0; I < NB; I++)
#pragma unroll
                for (int J = 0; J < NB; J++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        float v = acc[m][I][J][r];
                        v += dpp_mov<kDppRowRor4>(v);
                        v += dpp_mov<kDppRowRor8>(v);
                        if ((tid & 15) < 4) slot_s[(m * NP * NP + (4 * I + r) * NP + 4 * J + (tid & 3)) * (TW * 4) + slot] = v;
                    }
        stage_barrier();  // (the loads and stores of global memory stay under way)
#pragma unroll
        for (int k0 = 0; k0 < K; k0 += 64 * TW) {
            const int k = k0 + tid;
            if (k < K) {
                float v = 0.f;
#pragma unroll
                for (int sl = 0; sl < TW * 4; sl++) v += slot_s[k * (TW * 4) + sl];
                tot_s[k] = v;
                if (!inject && k0 == 0 && tid >= NP * NP && tid < 2 * NP * NP) {
                    float t = hohp * v;
                    if constexpr (NP == 4) t = row16_allreduce(t);
                    else t = wave_allreduce_sum(t);
                    if (tid == NP * NP) tot_s[K] = t;
                }
            }
        }
        stage_barrier();
        if (tid < SK::kGroup) {
            float tpost, tA1, tA2, s1;
            cb.qinv = inject ? 0.f : fast_rcp(qraw);
            cb.fetch_sums(tot_s, 1);
            cb.gram_vectors(n, tid, xch_s, tpost, tA1, tA2, s1);
            dm64 += (double)cb.dMe;
            dpre64 += (double)cb.dhpre_of(tA1, tA2, s1);
            dpost64 += (double)tpost;
        }
        // ---- dx, the summands of dw, df -------------------------------------------------------------------
        float qinv = 0.f, k2 = 0.f;
        if constexpr (!inject) {
            qinv = 1.0f / qraw;
            k2 = tot_s[K] * qinv * qinv * qinv / (float)C;
        }
        // eight results of a row in two halves, stored together
        auto put_half = [](bf16_t *p, uint32_t (&w)[4], const float (&v)[4], int h, int left) {
            w[2 * h] = pack_bf16x2(v[0], v[1]);
            w[2 * h + 1] = pack_bf16x2(v[2], v[3]);
            if (h == 0) return;
            if constexpr (!RAG) {
                st16<true>(p, w[0], w[1], w[2], w[3]);
            } else if (left >= 8) {
                st16_any<true>(p, w[0], w[1], w[2], w[3]);
            } else {  // left: elements up to the row's end
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (e < left) p[e] = (bf16_t)(w[e / 2] >> (16 * (e & 1)));
            }
        };
        bf16_t *const dxb = static_cast<bf16_t *>(sa.dx) + (size_t)b * n * C;
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const int c = RAG ? (wave + TW * it) * 128 + blk * 8 : cc[it];
            if constexpr (NP == 8) __builtin_amdgcn_sched_barrier(0);  // one item after the other: registers
            if (!in[it]) continue;  // quads are inside or outside together: the DPP exchanges stay within a quad
            uint32_t ow[NB][4], dfw[4];
            // four channels at a time: registers
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float gv[NB][4], xv[NB][4];
#pragma unroll
                for (int I = 0; I < NB; I++) {
                    const uint32_t gw[2] = {h ? gr[it][I].z : gr[it][I].x, h ? gr[it][I].w : gr[it][I].y};
                    const uint32_t xw[2] = {h ? xr[it][I].z : xr[it][I].x, h ? xr[it][I].w : xr[it][I].y};
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        gv[I][2 * k] = bf16lo_to_f32(gw[k]); gv[I][2 * k + 1] = bf16hi_to_f32(gw[k]);
                        xv[I][2 * k] = bf16lo_to_f32(xw[k]); xv[I][2 * k + 1] = bf16hi_to_f32(xw[k]);
                    }
                }
                float dfv[4], da[4];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    float pd = 0.f;
#pragma unroll
                    for (int I = 0; I < NB; I++) pd += hpost[I] * gv[I][v];
                    dfv[v] = quad_sum(pd);
                }
                if constexpr (inject) {
#pragma unroll
                    for (int v = 0; v < 4; v++) da[v] = 0.f;
                    if (sa.df && i == 0) put_half(static_cast<bf16_t *>(sa.df) + (size_t)b * C + c, dfw, dfv, h, C - c);
                } else {
                    float uv[4], w4[4];
                    if constexpr (LEAN) lds_floats<4>(w_s + (wave + TW * it) * 128 + blk * 8 + 4 * h, w4);
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        float wv;
                        if constexpr (LEAN) wv = w4[v];
                        else if constexpr (WMODE == kGramWBf16) wv = v & 1 ? bf16hi_to_f32(wb[it].w[2 * h + v / 2]) : bf16lo_to_f32(wb[it].w[2 * h + v / 2]);
                        else wv = __uint_as_float(wf[it].w[4 * h + v]);
                        float pa = 0.f;
#pragma unroll
                        for (int I = 0; I < NB; I++) pa += hpre[I] * xv[I][v];
                        const float av = quad_sum(pa);
                        da[v] = dfv[v] * wv * qinv - av * k2;
                        uv[v] = dfv[v] * av * qinv;
                    }
                    if ((i >> 1) == h) {
                        double *const us = LEAN ? lean_s + (wave + TW * it) * 128 + blk * 8 + 2 * i : usum[LEAN ? 0 : it];
                        us[0] += (double)(i & 1 ? uv[2] : uv[0]);
                        us[1] += (double)(i & 1 ? uv[3] : uv[1]);
                    }
                }
#pragma unroll
                for (int I = 0; I < NB; I++) {
                    float out[4];
#pragma unroll
                    for (int v = 0; v < 4; v++) out[v] = hpre[I] * da[v];
#pragma unroll
                    for (int J = 0; J < NB; J++)
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            out[v] += Mc[I][J][0] * quad_lane<0>(gv[J][v]);
                            out[v] += Mc[I][J][1] * quad_lane<1>(gv[J][v]);
                            out[v] += Mc[I][J][2] * quad_lane<2>(gv[J][v]);
                            out[v] += Mc[I][J][3] * quad_lane<3>(gv[J][v]);
                        }
                    if (sv[I]) put_half(dxb + (size_t)(4 * I + i) * C + c, ow[I], out, h, C - c);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NEXT) cur = nxt;
    }

    // ---- one row of sums per workgroup ---------------------------------------------------------------------
    if constexpr (!inject) {
#pragma unroll
        for (int it = 0; it < ITEMS; it++) {
            const int c = (wave + TW * it) * 128 + blk * 8 + 2 * i;
#pragma unroll
            for (int v = 0; v < 2; v++)
                if (c + v < C) sa.u[(size_t)blockIdx.x * C + c + v] = LEAN ? lean_s[c + v] : usum[LEAN ? 0 : it][v];
        }
    }
    if (tid < SK::kGroup) {
        const size_t at = (size_t)blockIdx.x * (n * n + 2 * n + 3);  // rows padded like dt
        if (cb.mv) sa.red[at + cb.r0 * n + cb.c0] = dm64;
        if (tid < n) {
            sa.red[at + n * n + tid] = dpre64;
            sa.red[at + n * n + n + tid] = dpost64;
        }
    }
}

static int static_waves(int n, int C) {
    if (n <= 4) return C <= 256 ? 2 : (C <= 2560 ? 4 : 8);
    return C <= 1024 ? 4 : 8;
}
// Workgroups that fit the chip at once (waves per SIMD by registers), then as few as keep the number of rounds.
int bwd_static_rows(int B, int n, int C) {
    const int tw = static_waves(n, C), items = (C + 128 * tw - 1) / (128 * tw), nb = n <= 4 ? 1 : 2;
    const int per_simd = nb == 1 ? (tw == 2 ? 3 : items <= 2 ? 4 : items == 3 && tw == 4 ? 3 : 2) : (items == 1 ? 3 : 2);
    const int slots = 256 * 4 * per_simd / tw;
    int rounds = std::max(2, (B + slots - 1) / slots);
    if (const int hook = tuning_get(kTuneStaticSpg); hook > 1) rounds = hook;  // experiment hook
    return (B + rounds - 1) / rounds;
}
// Where this pays against one sample per workgroup (bwd_resident.hip), which needs fewer registers, so that more of a chip's
// loads are under way, and hands over a row per sample instead of per workgroup (us, that + its batch sums | this + its):
//   n=4 C=256:  B=3072 10.0 + 10.2 | 11.2 + 10.0, 4096 11.4 + 11.7 | 12.7 + 8.8;  C=512: 2048 11.1 + 9.0 | 11.8 + 8.8, 3072 14.0 + 10.3 |
//               14.0 + 8.9;  C=1280: 3072 25.4 + 10.6 | 25.1 + 6.8;  C=2048: 3072 33.1 + 10.6 | 37.0 + 7.9, 4096 41.6 + 12.0 | 45.1 + 8.2;
//               C=2560: 3072 42.1 + 10.9 | 44.8 + 8.1, 4096 58.4 + 13.3 | 56.3 + 8.0
//   (there seven waves, here eight:)  n=4 C=3072: B=512 14.1 + 7.0 | 13.8 + 5.1, 2048 43.0 + 9.4 | 37.4 + 5.1;  C=4096: 512 19.1 + 7.3 |
//               16.2 + 5.4, 4096 120.7 + 19.7 | 85.9 + 5.8
//   n=8 C=512:  B=1536 16.6 + 12.4 | 16.3 + 12.5, 2048 19.4 + 15.0 | 20.6 + 10.4;  C=768: 2048 28.2 + 14.7 | 28.4 + 8.7;  C=2048: 2048 54.2 +
//               14.8 | 59.0 + 7.4, 3072 81.3 + 19.2 | 84.8 + 7.7;  C=2560: 2048 69.2 + 15.6 | 77.2 + 7.8, 3072 109.5 + 22.5 | 109.9 + 7.9;
//               C=4096: 512 34.6 + 6.4 | 32.1 + 7.7, 1024 69.0 + 10.2 | 57.0 + 7.7
//   n=6 C=1280 (ten chunks on eight waves): B=4096 71.6 + 15.6 | 87.3 + 8.0;  n=5 C=256: B=4096 27.4 + 12.4 | 33.4 + 8.7
// Ragged rows are held in more chunks than they have (launch_static_items) and shifted down sample by sample; whole backward, one
// sample per workgroup | this:
//   n=4 C=333:  B=4150 31.2 | 36.9, 7000 47.1 | 48.9;  n=2 C=333: 4150 28.1 | 28.6, 7000 41.7 | 36.3;  n=4 C=777: 4150 45.9 | 45.6
//   n=4 C=1283: 3080 55.1 | 86.1, 7000 110.7 | 161.8;  C=1789: 4150 97.6 | 100.9, 6000 137.9 | 127.6;  C=2555: 4150 113.0 | 116.4, 6000
//               160.7 | 152.6;  C=2811: 520 41.0 | 31.2;  n=8 C=777: 2060 54.6 | 52.2;  C=2045: 3080 158.7 | 143.1;  C=2051: 3080 163.9 |
//               177.8, 4000 202.5 | 218.5;  C=2555: 4000 232.1 | 244.9;  C=3069: 3080 293.6 | 215.9
bool bwd_static_preferred(int B, int n, int C) {
    if (const int hook = tuning_get(kTuneStaticSpg); hook > 0) return hook > 1 && B > 1;
    if (C % 8 != 0) {
        if (n <= 4 && C > 256 && C <= 512 && B < (n <= 2 ? 5000 : 9000)) return false;
        if (n <= 4 && C > 1024 && C <= 2560) return C > 1536 && B >= 6000;
        if (n > 4 && C > 2048 && C <= 2560) return false;
    }
    if (n <= 4) return B >= (C > 2560 ? 512 : (C > 256 && C <= 1536 ? 3072 : 4096));
    if (C > 3072) return B >= 768;
    if (C > 1536) return B >= 3072;
    return C >= 512 && C <= 1024 && B >= 2048;
}

template <int NP, int WMODE, int TW, bool RAG>
static hipError_t launch_static_items(const BwdStaticArgs &sa, int rows, hipStream_t stream) {
    int items = (sa.r.C + 128 * TW - 1) / (128 * TW);
    if (RAG && items == 1 && TW != 2) items = 2;  // fewer instantiations
    if (RAG && items > 2 && items < 5 && TW == 4) items = 5;
#define MHC_STATIC_ITEMS(N)                                                                                           \
    case N:                                                                                                           \
        if constexpr ((TW == 2 ? N == 1 : TW == 4 ? N <= (NP == 4 ? 5 : 2) : N >= (NP == 4 ? 3 : 2) && N <= 4) &&        \
                      !(RAG && TW == 4 && (N == 1 || N == 3 || N == 4))) {                                            \
            const size_t smem = static_lean<NP, N>() && WMODE != kGramInject ? (size_t)TW * N * 128 * 12 : 0;         \
            if (hipError_t e = allow_dynamic_lds<&bwd_static_kernel<NP, WMODE, TW, N, static_next<NP, TW, N>(), RAG>>(smem); e != hipSuccess) return e; \
            bwd_static_kernel<NP, WMODE, TW, N, static_next<NP, TW, N>(), RAG><<<rows, 64 * TW, smem, stream>>>(sa);            \
            return hipGetLastError();                                                                                 \
        }                                                                                                             \
        return hipErrorInvalidValue
    switch (items) {
        MHC_STATIC_ITEMS(1);
        MHC_STATIC_ITEMS(2);
        MHC_STATIC_ITEMS(3);
        MHC_STATIC_ITEMS(4);
        MHC_STATIC_ITEMS(5);
        default: return hipErrorInvalidValue;
    }
#undef MHC_STATIC_ITEMS
}

template <int NP, int WMODE>
static hipError_t launch_static_waves(const BwdStaticArgs &sa, int rows, hipStream_t stream) {
    const bool rag = sa.r.C % 8 != 0;
#define MHC_STATIC_WAVES(TW) return rag ? launch_static_items<NP, WMODE, TW, true>(sa, rows, stream) : launch_static_items<NP, WMODE, TW, false>(sa, rows, stream)
    switch (static_waves(sa.r.n, sa.r.C)) {
        case 2:
            if constexpr (NP == 4) MHC_STATIC_WAVES(2);
            else return hipErrorInvalidValue;
        case 4: MHC_STATIC_WAVES(4);
        default: MHC_STATIC_WAVES(8);
    }
#undef MHC_STATIC_WAVES
}

hipError_t launch_bwd_static(const void *dy, const void *x, const void *w, int w_dtype, const void *f_inject, const float *Hpre,
                             const float *Hpost, const float *M, const float *q, void *dx, void *df, void *u, void *red, int B, int n,
                             int C, hipStream_t stream) {
    BwdStaticArgs sa{{dy, x, w, f_inject, Hpre, Hpost, M, q, nullptr, nullptr, nullptr, nullptr, nullptr, BwdCoefOut{}, 0,
                      w_dtype == kBF16, B, n, C, 0, padded_D(n), 0.f, nullptr, 1},
                     dx, df, static_cast<double *>(u), static_cast<double *>(red)};
    const int rows = bwd_static_rows(B, n, C);
#define MHC_STATIC(NP)                                                                       \
    return f_inject ? launch_static_waves<NP, kGramInject>(sa, rows, stream)                 \
                    : (w_dtype == kBF16 ? launch_static_waves<NP, kGramWBf16>(sa, rows, stream) \
                                        : launch_static_waves<NP, kGramWF32>(sa, rows, stream))
    if (n <= 4) MHC_STATIC(4);
    MHC_STATIC(8);
#undef MHC_STATIC
}

}  // namespace mhc
