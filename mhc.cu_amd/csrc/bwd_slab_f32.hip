// Backward of the fp32 tier, n <= 4, behind the channel sums and the coefficient backward: everything that
// still needs x and dy, in one pass over them.
//
//   dx[b,j,c]  = sum_i M[i,j] dy[b,i,c] + Hpre[j] da[b,c] - cx x[b,j,c] + sum_d dP[b,d] phi[d,jC+c]
//   dphi[d,jC+c] = sum_b dP[b,d] x[b,j,c]          dw[c] = sum_b df[b,c] a[b,c] / q_b
//   (reference stream_ops.cuh:646-663, :761-850, rmsnorm.cuh:255-294, ops.py:332-351)
//
// Bound by bytes: x and dy in, dx out (157 MB at B=2560 n=4 C=1280).  The three launches it replaces (dP phi
// into dx, the dx kernel, dphi) moved 367 MB and took 84 us there; this one takes 39 us (4.0 TB/s, 1.2 us of it for the
// float64 sums and for adding dP phi in one piece) and leaves the finalize launch fewer rows (10 -> 4 us).
//
// A workgroup owns 32 channels of all streams and a range of samples that its four waves share out in tiles of
// 16.  The products run on v_mfma_f32_16x16x4_f32 (IEEE fp32): the tile is 16 samples x 16 channels, a lane holds
// the two channels 2 l, 2 l + 1 (l = lane & 15; one per product column tile) of the four samples 4 g .. 4 g + 3
// (g = lane / 16), which is at once
//   * the layout of an accumulator (dx: rows = samples), so the mixing is lane-local arithmetic on the
//     accumulator of dP phi, and
//   * the layout of the right-hand operand of dphi (contraction over samples: product i takes sample 4 g + i),
// so x and dy go from memory into registers in 128-byte pieces and nothing but the samples' coefficients and dP
// passes through LDS (wave-private, no barrier).  D <= 24 rows of phi are 6 products of depth 4 (row 6 g + s in
// product s) and stay in LDS.  dphi stays in registers for the whole range of samples and is added up over
// the four waves at the end; with the batch split S ways the copies are summed by the finalize launch.  The sums over
// samples of dw and dt are float64 from the first sample on (batch_sums.h).
// 206 (n = 3) and 249 (n = 4) registers: two workgroups per CU, which hide each other's loads.
#include "launchers.h"
#include "mhc_common.h"

namespace mhc {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

constexpr int kSfCh = 32;       // channels per workgroup
constexpr int kSfTile = 16;     // samples per wave and step
constexpr int kSfCo = 28;       // LDS floats per sample: M row-major in rows of 4 | Hpre | Hpost | 1/q, k2, cx
constexpr int kSfDp = 36;       // LDS pitch of a dP row (32 floats)
constexpr int kSfWave = kSfTile * (kSfCo + kSfDp);

constexpr int sf_phi_pitch(int n) { return (n * 32 + 16) / 32 * 32 + 16; }

struct SlabF32Args {
    const float *dy, *x, *w_f32; const bf16_t *w_bf16;
    const float *phi, *Hpre, *Hpost, *M, *q, *s1, *cx, *dP, *dt;
    float *dx, *df, *dphi;
    double *dw_part, *dt_part;
    int B, C, D, slabs, per_split, per_wave;  // samples
};

// INJECT: the kernel-level view (df is an output, no RMSNorm backward)
template <int N, bool INJECT>
__global__ __launch_bounds__(256, 2) void bwd_slab_f32_kernel(SlabF32Args a) {
    extern __shared__ __align__(16) float lds[];
    constexpr int DP = 32, nDp = 6;
    constexpr int PP = sf_phi_pitch(N);  // six rows apart = 32 banks apart: the lane groups of a product read without conflict
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l = lane & 15, g = lane >> 4;
    const int C = a.C, B = a.B, D = a.D, nC = N * C;
    const int s0 = blockIdx.y * a.per_split, s1 = min(B, s0 + a.per_split);
    if ((int)blockIdx.x == a.slabs) {
        // one more workgroup per split: the column sums of dt over the split (float64)
        double *red = reinterpret_cast<double *>(lds);
        const int col = tid & 31, rg = tid >> 5;
        double acc = 0.0;
        if (col < D + 3)
            for (int b = s0 + rg; b < s1; b += 8) acc += (double)a.dt[(size_t)b * (D + 3) + col];
        red[rg * 32 + col] = acc;
        __syncthreads();
        if (tid < D + 3) {
            double v = 0.0;
#pragma unroll
            for (int i = 0; i < 8; i++) v += red[i * 32 + tid];
            a.dt_part[(size_t)blockIdx.y * (D + 3) + tid] = v;
        }
        return;
    }
    const int c = blockIdx.x * kSfCh + 2 * l;
    const bool cok = c < C;  // C is even: a lane's two channels are both inside or both outside
    const int cl = cok ? c : 0;
    float *co = lds + wave * kSfWave, *dp = co + kSfTile * kSfCo;

    // phi: the slab of 24 rows in LDS; product s contracts rows 6 g + s, rows >= D meet zeros of dP
    float *phi_s = lds + 4 * kSfWave;
    for (int e = tid; e < 4 * nDp * N * 16; e += 256) {
        const int d = e / (N * 16), j = e / 16 % N, k = blockIdx.x * kSfCh + 2 * (e % 16);
        *reinterpret_cast<float2 *>(phi_s + d * PP + j * 32 + 2 * (e % 16)) =
            *reinterpret_cast<const float2 *>(a.phi + (size_t)(d < D ? d : 0) * nC + (size_t)j * C + (k < C ? k : 0));
    }
    __syncthreads();
    float w[2] = {0.f, 0.f};
    if (!INJECT) {
#pragma unroll
        for (int v = 0; v < 2; v++) w[v] = a.w_bf16 ? bf16_to_f32(a.w_bf16[cl + v]) : a.w_f32[cl + v];
    }
    f32x4_t dphi[N][2][2];  // [stream][row tile of 16][channel of the pair]
#pragma unroll
    for (int j = 0; j < N; j++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int v = 0; v < 2; v++) dphi[j][t][v] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    double usum[2] = {0.0, 0.0};

    const uint32_t off0 = 4u * (uint32_t)cl, row_bytes = 4u * (uint32_t)nC;  // 15 rows of at most 4 * 32768 floats
    const int w0 = s0 + __builtin_amdgcn_readfirstlane(wave) * a.per_wave, w1 = min(s1, w0 + a.per_wave);
    for (int b0 = w0; b0 < w1; b0 += kSfTile) {
        // the tile's coefficients: lane = (sample lane / 4, row lane % 4), samples beyond the range are zeros
        {
            const int bs = lane >> 2, r = lane & 3, b = b0 + bs;
            const bool ok = b < w1;
            const int bc = ok ? b : w0;
            const int rc = r < N ? r : 0;
            float m[N];
#pragma unroll
            for (int k = 0; k < N; k++) m[k] = a.M[(size_t)bc * N * N + rc * N + k];
            const float hp = a.Hpre[(size_t)bc * N + rc], ho = a.Hpost[(size_t)bc * N + rc];
            const float qv = INJECT ? 1.f : a.q[bc], sv = INJECT ? 0.f : a.s1[bc], xv = a.cx[bc];
            const float4 p0 = reinterpret_cast<const float4 *>(a.dP + (size_t)bc * DP)[2 * r];
            const float4 p1 = reinterpret_cast<const float4 *>(a.dP + (size_t)bc * DP)[2 * r + 1];
            const bool rok = ok && r < N;
#pragma unroll
            for (int k = 0; k < 4; k++) co[bs * kSfCo + 4 * r + k] = rok && k < N ? m[k < N ? k : 0] : 0.f;
            co[bs * kSfCo + 16 + r] = rok ? hp : 0.f;
            co[bs * kSfCo + 20 + r] = rok ? ho : 0.f;
            const float qi = INJECT || !ok ? 0.f : 1.0f / qv;
            if (r == 0) co[bs * kSfCo + 24] = qi;
            if (r == 1) co[bs * kSfCo + 25] = ok ? sv * qi * qi * qi / (float)C : 0.f;
            if (r == 2) co[bs * kSfCo + 26] = ok ? xv : 0.f;
            float *pr = dp + bs * kSfDp + 8 * r;
            pr[0] = ok ? p0.x : 0.f; pr[1] = ok ? p0.y : 0.f; pr[2] = ok ? p0.z : 0.f; pr[3] = ok ? p0.w : 0.f;
            pr[4] = ok ? p1.x : 0.f; pr[5] = ok ? p1.y : 0.f; pr[6] = ok ? p1.z : 0.f; pr[7] = ok ? p1.w : 0.f;
        }
        float2 xv[N][4], gv[N][4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // uniform base + 32-bit byte offset of the lane: one register per sample instead of two per access
            const uint32_t o = off0 + (b0 + 4 * g + i < w1 ? 4 * g + i : 0) * row_bytes;
#pragma unroll
            for (int j = 0; j < N; j++) {
                gv[j][i] = *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(a.dy + (size_t)b0 * nC + (size_t)j * C) + o);
                xv[j][i] = *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(a.x + (size_t)b0 * nC + (size_t)j * C) + o);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // (a wave's LDS accesses complete in order; the fence keeps the compiler from reordering them)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        auto ld4 = [](float *d, const float *s) {
            const float4 t = *reinterpret_cast<const float4 *>(s);
            d[0] = t.x; d[1] = t.y; d[2] = t.z; d[3] = t.w;
        };
        if (INJECT && a.df) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float hpost[4];
                ld4(hpost, co + (4 * g + i) * kSfCo + 20);
                float2 d = make_float2(0.f, 0.f);
#pragma unroll
                for (int j = 0; j < N; j++) { d.x += hpost[j] * gv[j][i].x; d.y += hpost[j] * gv[j][i].y; }
                if (cok && b0 + 4 * g + i < w1)
                    *reinterpret_cast<float2 *>(reinterpret_cast<char *>(a.df + (size_t)b0 * C) + off0 + (4 * g + i) * 4u * (uint32_t)C) = d;
            }
        }
        // mixing part of dx, lane-local
        f32x4_t out[N][2];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float *cb = co + (4 * g + i) * kSfCo;
            float m[4 * N], hpre[4], hpost[4], k3[4];
#pragma unroll
            for (int k = 0; k < N; k++) ld4(m + 4 * k, cb + 4 * k);
            if (!INJECT) { ld4(hpre, cb + 16); ld4(hpost, cb + 20); }
            ld4(k3, cb + 24);
#pragma unroll
            for (int v = 0; v < 2; v++) {
                float da = 0.f;
                if constexpr (!INJECT) {
                    float s_a = 0.f, s_df = 0.f;
#pragma unroll
                    for (int j = 0; j < N; j++) {
                        s_a += hpre[j] * (v ? xv[j][i].y : xv[j][i].x);
                        s_df += hpost[j] * (v ? gv[j][i].y : gv[j][i].x);
                    }
                    da = s_df * w[v] * k3[0] - s_a * k3[1];
                    usum[v] += (double)(s_df * s_a * k3[0]);
                }
#pragma unroll
                for (int j = 0; j < N; j++) {
                    float o = (INJECT ? 0.f : hpre[j] * da) - k3[2] * (v ? xv[j][i].y : xv[j][i].x);
#pragma unroll
                    for (int k = 0; k < N; k++) o += m[4 * k + j] * (v ? gv[k][i].y : gv[k][i].x);
                    out[j][v][i] = o;
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // one sample's coefficients at a time: registers
        }
        // + dP phi: product s, left operand lane (sample l, rows 6 g + s of dP).  Summed up by itself and added once: in the
        // accumulator of the mixing part each of the 24 steps would be rounded at the size of dx (error of dx 1.5e-7
        // instead of 9e-8).
        float av[nDp];
#pragma unroll
        for (int s = 0; s < nDp; s++) av[s] = dp[l * kSfDp + nDp * g + s];
#pragma unroll
        for (int j = 0; j < N; j++) {
            f32x4_t t[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int s = 0; s < nDp; s++) {
                const float2 ph = *reinterpret_cast<const float2 *>(phi_s + (nDp * g + s) * PP + j * 32 + 2 * l);
                t[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], ph.x, t[0], 0, 0, 0);
                t[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], ph.y, t[1], 0, 0, 0);
            }
            out[j][0] += t[0];
            out[j][1] += t[1];
            __builtin_amdgcn_sched_barrier(0);
        }
        // dphi: product i contracts samples 4 g + i, left operand lane (row l of the tile of 16, same samples)
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const float av = dp[(4 * g + i) * kSfDp + 16 * t + l];
#pragma unroll
                for (int j = 0; j < N; j++) {
                    dphi[j][t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, xv[j][i].x, dphi[j][t][0], 0, 0, 0);
                    dphi[j][t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, xv[j][i].y, dphi[j][t][1], 0, 0, 0);
                }
            }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (cok && b0 + 4 * g + i < w1) {
                const uint32_t o = off0 + (4 * g + i) * row_bytes;
#pragma unroll
                for (int j = 0; j < N; j++)
                    *reinterpret_cast<float2 *>(reinterpret_cast<char *>(a.dx + (size_t)b0 * nC + (size_t)j * C) + o) =
                        make_float2(out[j][0][i], out[j][1][i]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the next tile's coefficients overwrite these
        __builtin_amdgcn_wave_barrier();
    }
    // sums over the four waves: dphi, then dw
    __syncthreads();
    constexpr int R = N * 4;  // accumulator quads per lane
#pragma unroll
    for (int j = 0; j < N; j++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int v = 0; v < 2; v++)
                *reinterpret_cast<f32x4_t *>(lds + ((size_t)(wave * R + (j * 2 + t) * 2 + v) * 64 + lane) * 4) = dphi[j][t][v];
    double *us = reinterpret_cast<double *>(lds + (size_t)4 * R * 64 * 4);  // [4 waves][32]
    if (!INJECT) {
#pragma unroll
        for (int v = 0; v < 2; v++) {
            usum[v] += __shfl_xor(usum[v], 16, kWave);
            usum[v] += __shfl_xor(usum[v], 32, kWave);
        }
        if (g == 0) { us[wave * 32 + 2 * l] = usum[0]; us[wave * 32 + 2 * l + 1] = usum[1]; }
    }
    __syncthreads();
    float *o = a.dphi + (size_t)blockIdx.y * D * nC;
    // wave k takes the quads k, k + 4, ... pairwise: quads (j, t) are 2 (j t) and 2 (j t) + 1 = the two channels
    for (int p = wave; p < N * 2; p += 4) {
        const int j = p >> 1, t = p & 1;
        f32x4_t s[2];
#pragma unroll
        for (int v = 0; v < 2; v++) {
            s[v] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 4; k++) s[v] += *reinterpret_cast<const f32x4_t *>(lds + ((size_t)(k * R + p * 2 + v) * 64 + lane) * 4);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int d = 16 * t + 4 * g + i;
            if (d < D && cok) *reinterpret_cast<float2 *>(o + (size_t)d * nC + (size_t)j * C + c) = make_float2(s[0][i], s[1][i]);
        }
    }
    if (!INJECT && tid < 32 && blockIdx.x * kSfCh + tid < C)
        a.dw_part[(size_t)blockIdx.y * C + blockIdx.x * kSfCh + tid] = (us[tid] + us[32 + tid]) + (us[64 + tid] + us[96 + tid]);
}

bool bwd_slab_f32_supported(int x_dtype, int phi_dtype, int n, int C) {
    return x_dtype == kF32 && phi_dtype == kF32 && n <= 4 && C % 2 == 0;
}

// Samples are dealt out in tiles of 16 to 4 S waves per slab: as many splits as two resident workgroups per CU
// allow, then no more than the number of tiles of the longest wave needs.
static int slab_f32_tiles(int B, int C, int *splits) {
    const int slabs = (C + kSfCh - 1) / kSfCh, tiles = (B + kSfTile - 1) / kSfTile;
    int smax = 512 / slabs;
    if (smax > 16) smax = 16;  // the finalize launch sums sixteen copies per round
    if (smax < 1) smax = 1;
    const int per_wave = (tiles + 4 * smax - 1) / (4 * smax);
    *splits = (tiles + 4 * per_wave - 1) / (4 * per_wave);
    return per_wave;
}

int bwd_slab_f32_splits(int B, int C) {
    int s;
    slab_f32_tiles(B, C, &s);
    return s;
}

hipError_t launch_bwd_slab_f32(const float *dy, const float *x, const void *w, int w_dtype, const void *f_inject,
                               const float *phi, const float *Hpre, const float *Hpost, const float *M, const float *q,
                               const BwdCoefOut &co, float *dx, float *df, float *dphi, double *dw_part, double *dt_part,
                               int B, int n, int C, hipStream_t stream) {
    int S;
    const int tiles = slab_f32_tiles(B, C, &S);
    SlabF32Args a;
    a.dy = dy; a.x = x;
    a.w_f32 = w_dtype == kBF16 ? nullptr : static_cast<const float *>(w);
    a.w_bf16 = w_dtype == kBF16 ? static_cast<const bf16_t *>(w) : nullptr;
    a.phi = phi; a.Hpre = Hpre; a.Hpost = Hpost; a.M = M; a.q = q; a.s1 = co.s1; a.cx = co.cx; a.dP = co.dP; a.dt = co.dt;
    a.dx = dx; a.df = df; a.dphi = dphi; a.dw_part = dw_part; a.dt_part = dt_part;
    a.B = B; a.C = C; a.D = n * n + 2 * n;
    a.slabs = (C + kSfCh - 1) / kSfCh;
    a.per_wave = tiles * kSfTile;
    a.per_split = 4 * a.per_wave;
    const dim3 grid(a.slabs + 1, S);
    const size_t sum = sizeof(float) * ((size_t)4 * n * 4 * 64 * 4 + 256), tile = sizeof(float) * (4 * kSfWave + 24 * sf_phi_pitch(n));
    const size_t smem = sum > tile ? sum : tile;
#define MHC_SLAB_F32(N)                                                                                    \
    do {                                                                                                   \
        if (hipError_t e = f_inject ? allow_dynamic_lds<&bwd_slab_f32_kernel<N, true>>(smem)               \
                                    : allow_dynamic_lds<&bwd_slab_f32_kernel<N, false>>(smem);             \
            e != hipSuccess)                                                                               \
            return e;                                                                                      \
        if (f_inject) bwd_slab_f32_kernel<N, true><<<grid, 256, smem, stream>>>(a);                        \
        else bwd_slab_f32_kernel<N, false><<<grid, 256, smem, stream>>>(a);                                \
    } while (0)
    switch (n) {
        case 1: MHC_SLAB_F32(1); break;
        case 2: MHC_SLAB_F32(2); break;
        case 3: MHC_SLAB_F32(3); break;
        case 4: MHC_SLAB_F32(4); break;
        default: return hipErrorInvalidValue;
    }
#undef MHC_SLAB_F32
    return hipGetLastError();
}

}  // namespace mhc
