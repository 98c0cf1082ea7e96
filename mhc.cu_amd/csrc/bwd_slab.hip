// Backward, second launch for n <= 4 in the bf16 tier: everything that needs dP, in ONE pass over
// dy and x.  A workgroup owns a slab of channels (all n streams) and walks the samples of its batch
// split in tiles:
//
//   dx[b,j,c]  = sum_i M_b[i,j] dy[b,i,c] + Hpre_b[j] da[b,c] - cx_b x[b,j,c] + sum_d dP[b,d] phi[d, jC+c]
//   df[b,c]    (kernel-level view)                                   reference stream_ops.cuh:761-850,
//   dphi[d,k] += sum_b dP[b,d] x_flat[b,k]                           :646-663, ops.py:332-351
//   dw[c]     += sum_b df[b,c] a[b,c] / q_b                          reference rmsnorm.cuh:282-294
//   dbias / dalpha partial sums of dt over the split's samples       reference ops.py:319-325
//
// The two projection products run on the matrix cores: their contraction index (b for dphi, d for the
// dx term) is not the contiguous one in memory, so the x tile and the phi slab are staged row-major in LDS
// and read back transposed; dP arrives from the reduce kernel as bf16 [B, DP] and as a transposed hi/lo
// pair [2][DP][BP].  x and dy are read once from HBM, dx is written once; no atomics.
//
// Two kernels: bwd_slab_stage_kernel for bf16 dy (and for fp32 storage of both), bwd_slab_f32dy_kernel for fp32 dy beside bf16 x.
#include "launchers.h"

#include <algorithm>

#include "lds_stage.h"
#include "phase_profiler.h"
#include "tuning.h"

namespace mhc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

constexpr int kSlabCW = 64;                 // channels per slab
constexpr int kSlabNS = 4;                  // streams (padded)
constexpr int kSlabKW = kSlabNS * kSlabCW;  // x_flat columns per slab tile row
constexpr int kSlabLDX = kSlabKW + 8;       // LDS pitch of the bf16 tiles (elements)
constexpr int kSlabLDF = kSlabKW + 4;       // LDS pitch of the fp32 projection-term tile

struct BwdSlabArgs {
    const void *dy;          // [B, n, C]
    const bf16_t *x;         // [B, n, C]
    const void *w;           // [C]
    const void *f_inject;    // bf16 [B, C] or nullptr
    const bf16_t *phi;       // [D, nC]
    const float *Hpre, *Hpost, *M, *q, *s1, *cx;  // per sample
    const bf16_t *dPb;       // dP, fragment-major (frag_dpb, DP = 32)
    const bf16_t *dPT;       // dP^T hi/lo planes, fragment-major (frag_dpt), plane stride 32 * BP
    const float *dt;         // [B, D+3]
    void *dx;                // [B, n, C], in the type of x's storage
    bf16_t *df;              // [B, C] or nullptr
    float *dphi_part;        // [S][D][nC]
    double *dw_part;         // [S][C]
    double *dt_part;         // [S][D+3]
    int w_bf16, B, BP, n, C, tiles;  // tiles of the batch (32 samples, bf16 dy: 16), see the kernels for a split's
};

__device__ __forceinline__ bf16x8_t slab_frag_t(const bf16_t *tile, int k0, int col0, int lane) {
    // lane (n = lane & 31, kg = lane >> 5) gets tile[k0 + kg*8 + i][col0 + n], i = 0..7
    return __builtin_bit_cast(bf16x8_t, lds_frag_tr(tile, kSlabLDX, k0, col0, lane));
}

__device__ __forceinline__ void unpack8(const uint4 &r, float (&v)[8]) {
    v[0] = bf16lo_to_f32(r.x); v[1] = bf16hi_to_f32(r.x);
    v[2] = bf16lo_to_f32(r.y); v[3] = bf16hi_to_f32(r.y);
    v[4] = bf16lo_to_f32(r.z); v[5] = bf16hi_to_f32(r.z);
    v[6] = bf16lo_to_f32(r.w); v[7] = bf16hi_to_f32(r.w);
}

// Eight consecutive values of dy kept as loaded until they are used.
struct Raw8 {
    float4 r0, r1;
    __device__ __forceinline__ void load(const float *p) {
        r0 = reinterpret_cast<const float4 *>(p)[0];
        r1 = reinterpret_cast<const float4 *>(p)[1];
    }
    __device__ __forceinline__ void get(float (&v)[8]) const {
        v[0] = r0.x; v[1] = r0.y; v[2] = r0.z; v[3] = r0.w; v[4] = r1.x; v[5] = r1.y; v[6] = r1.z; v[7] = r1.w;
    }
};

// fp32 dy.  Tiles of 32 samples; the projection term of dx goes from the accumulators through LDS to the thread that
// owns (sample, 8 channels) of all streams, which finishes dx on the VALU and stores 16 bytes per stream.  Two barriers
// per tile.
__global__ __launch_bounds__(256, 2) void bwd_slab_f32dy_kernel(BwdSlabArgs a) {
    extern __shared__ float smem_f[];
    float *dxf_s = smem_f;                                                  // [32][LDF] fp32
    bf16_t *x_s = reinterpret_cast<bf16_t *>(dxf_s + 32 * kSlabLDF);         // [32][LDX] bf16
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = a.n, C = a.C, nC = n * C, D = n * n + 2 * n;
    const int pwg = blockIdx.y * gridDim.x + blockIdx.x;
    (void)pwg;
    MHC_PHASE_ZERO(kPhaseBwdSlab, pwg);
    MHC_PHASE_BEGIN(pclk);
    const int c0 = blockIdx.x * kSlabCW;
    // whole tiles per split, the counts of two splits differing by at most one: any split count up to the
    // tile count can be used, so the grid can be sized to the chip instead of to a divisor of the batch
    const unsigned nsplit = gridDim.y;
    const int b_begin = (int)((uint64_t)blockIdx.y * (unsigned)a.tiles / nsplit) * 32;
    const int b_end = min(a.B, (int)((uint64_t)(blockIdx.y + 1) * (unsigned)a.tiles / nsplit) * 32);
    const bool inject = a.f_inject != nullptr;
    const int row = lane & 31, kg = lane >> 5;
    // VALU ownership: sample bl of the tile, channels c0 + ch*8 .. +8 of every stream
    const int bl = tid >> 3, ch = tid & 7;
    const int cth = c0 + ch * 8;
    const bool cok = cth < C;  // C % 8 == 0: a chunk is entirely inside or outside

    // ---- software pipeline: the loads of tile t+1 are issued before the VALU phase of tile t ----
    // raw tile data of this thread (sample slot bl, 8 channels, all streams) and the MFMA operands
    // that come straight from global memory (dP^T hi/lo rows d, dP rows b)
    struct TileRegs {
        uint4 xr[kSlabNS];
        Raw8 gr[kSlabNS];
    };
    // Loads carry no predicate (a predicate would be applied right behind the load and make the
    // prefetch wait): slots beyond the batch, streams >= n and channel chunks >= C alias valid
    // data instead.  Aliased values are finite whenever the real inputs are and only ever meet
    // zero coefficients (dP^T is zero beyond B, H and M are zero beyond n) or land in rows and
    // columns that are never stored.
    auto load_tile = [&](int sb, TileRegs &t) {
        const int b = sb + bl;
        const bool bok = b < b_end && cok;
        const size_t base = bok ? (size_t)b * nC + cth : 0;
        const bf16_t *xb = a.x + base;
        const float *gb = static_cast<const float *>(a.dy) + base;
#pragma unroll
        for (int j = 0; j < kSlabNS; j++) {
            const size_t so = j < n ? (size_t)j * C : 0;
            t.xr[j] = *reinterpret_cast<const uint4 *>(xb + so);
            t.gr[j].load(gb + so);
        }
    };
    // ---- phi slab -> LDS (as [32 d][KW]) -> this wave's transposed fragments ----------------
    // wave w owns N-tiles t = 2w, 2w+1; tile t covers stream t/2, channels c0 + (t%2)*32 .. +32
    // The slab is requested first and the first tile right behind it, so that the tile's round
    // trip runs under the staging of the slab.
    bf16_t *phi_s = reinterpret_cast<bf16_t *>(dxf_s);  // staged in the (not yet used) fp32 tile
    constexpr int kPhiIters = 32 * (kSlabKW / 8) / 256;
    static_assert(32 * (kSlabKW / 8) % 256 == 0, "phi slab staging assumes whole rounds of 256 threads");
    uint4 phir[kPhiIters];
#pragma unroll
    for (int i = 0; i < kPhiIters; i++) {
        const int e = tid + i * 256;
        const int d = e / (kSlabKW / 8), chunk = e % (kSlabKW / 8);
        const int j = chunk / (kSlabCW / 8), c = c0 + (chunk % (kSlabCW / 8)) * 8;
        const bool ok = d < D && j < n && c < C;
        phir[i] = load16_masked(
            reinterpret_cast<const uint4 *>(a.phi + (ok ? (size_t)d * nC + (size_t)j * C + c : 0)), ok);
    }
    TileRegs cur, nxt;
    if (b_begin < b_end) load_tile(b_begin, cur);
#pragma unroll
    for (int i = 0; i < kPhiIters; i++) {
        const int e = tid + i * 256;
        const int d = e / (kSlabKW / 8), chunk = e % (kSlabKW / 8);
        *reinterpret_cast<uint4 *>(phi_s + (size_t)d * kSlabLDX + chunk * 8) = phir[i];
    }
    __syncthreads();
    bf16x8_t phif[2][2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) phif[t][ks] = slab_frag_t(phi_s, ks * 16, (2 * wave + t) * 32, lane);
    __syncthreads();  // fragments are in registers; the region becomes dxf_s

    f32x16_t acc[2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[t][i] = 0.f;
    float usum[8];
#pragma unroll
    for (int v = 0; v < 8; v++) usum[v] = 0.f;
    double dtsum = 0.0;  // slab 0 only: thread (col = tid & 31, row group = tid >> 5)

    float wv[8];
#pragma unroll
    for (int v = 0; v < 8; v++)
        wv[v] = (cok && !inject) ? (a.w_bf16 ? bf16_to_f32(static_cast<const bf16_t *>(a.w)[cth + v])
                                              : static_cast<const float *>(a.w)[cth + v]) : 0.f;


    MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 0, pclk);
    // One tile: `cur` holds its data (requested a whole tile earlier); the next tile's loads go to
    // `nxt` right behind this tile's small operand loads and have the three phases to arrive.  The
    // loop alternates the two register sets instead of copying one into the other (a copy waits for
    // the loads it copies).
    auto process_tile = [&](int sb, TileRegs &cur, TileRegs &nxt) {
        const int b = sb + bl;
        const bool bok = b < b_end && cok;
        // MFMA operands that come straight from global memory: dP^T hi/lo (rows d) and dP (rows b);
        // issued first, they arrive while the x tile is written and the barrier is crossed
        uint4 ah[2], al[2], ap2[2];
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const bf16_t *ap = a.dPT + frag_base(0, a.BP >> 4, (sb >> 4) + ks) + lane * 8;
            // splits are whole 32-sample tiles and BP is padded to 32 (dP^T zero beyond B), so every
            // fragment of the tile is inside the buffers; dP rows beyond B only feed unused rows
            ah[ks] = *reinterpret_cast<const uint4 *>(ap);
            al[ks] = *reinterpret_cast<const uint4 *>(ap + (size_t)32 * a.BP);
            ap2[ks] = *reinterpret_cast<const uint4 *>(a.dPb + frag_base(sb >> 5, 2, ks) + lane * 8);
        }
        // this thread's sample coefficients for phase C: asked for here so that they arrive behind
        // the barriers and the matrix-core phase (slots beyond the split alias sample 0, streams
        // >= n alias stream 0; both are discarded below)
        float hpre[kSlabNS], hpost[kSlabNS], Mr[kSlabNS][kSlabNS], cxv, qv = 1.f, s1v = 0.f;
        {
            const size_t bc = b < b_end ? b : 0;
#pragma unroll
            for (int i = 0; i < kSlabNS; i++) {
                hpre[i] = a.Hpre[bc * n + (i < n ? i : 0)];
                hpost[i] = a.Hpost[bc * n + (i < n ? i : 0)];
#pragma unroll
                for (int j = 0; j < kSlabNS; j++) Mr[i][j] = a.M[bc * n * n + ((i < n && j < n) ? i * n + j : 0)];
            }
            cxv = a.cx[bc];
            if (!inject) { qv = a.q[bc]; s1v = a.s1[bc]; }
        }
        if (sb + 32 < b_end) load_tile(sb + 32, nxt);
        // x tile -> LDS
#pragma unroll
        for (int j = 0; j < kSlabNS; j++)
            *reinterpret_cast<uint4 *>(x_s + (size_t)bl * kSlabLDX + j * kSlabCW + ch * 8) = cur.xr[j];
        // dt column sums (slab 0): 32 columns x 8 row groups, 4 samples of the tile each
        if (blockIdx.x == 0) {
            const int col = tid & 31, rg = tid >> 5;
            if (col < D + 3) {
#pragma unroll
                for (int rr = 0; rr < 4; rr++) {
                    const int bb = sb + rg * 4 + rr;
                    if (bb < b_end) dtsum += a.dt[(size_t)bb * (D + 3) + col];
                }
            }
        }
        __syncthreads();
        MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 1, pclk);

        // ---- phase B: matrix cores ----------------------------------------------------------------
        {
            // dphi += dP^T(hi + lo) x ; projection term of dx: dP phi
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int col0 = (2 * wave + t) * 32;
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    const bf16x8_t xf = slab_frag_t(x_s, ks * 16, col0, lane);
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, ah[ks]), xf, acc[t], 0, 0, 0);
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, al[ks]), xf, acc[t], 0, 0, 0);
                }
                f32x16_t o;
#pragma unroll
                for (int i = 0; i < 16; i++) o[i] = 0.f;
#pragma unroll
                for (int ks = 0; ks < 2; ks++)
                    o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, ap2[ks]), phif[t][ks], o, 0, 0, 0);
                // accumulator layout: column = lane & 31, register i -> row 8*(i/4) + 4*(lane/32) + i%4
#pragma unroll
                for (int i = 0; i < 16; i++)
                    dxf_s[(size_t)(8 * (i >> 2) + 4 * kg + (i & 3)) * kSlabLDF + col0 + row] = o[i];
            }
        }
        __syncthreads();
        MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 2, pclk);

        // ---- phase C: finish dx ------------------------------------------------------------------
        if (bok) {
            float qinv = 0.f, k2 = 0.f;
#pragma unroll
            for (int i = 0; i < kSlabNS; i++) {
                if (i >= n) { hpre[i] = 0.f; hpost[i] = 0.f; }
#pragma unroll
                for (int j = 0; j < kSlabNS; j++)
                    if (i >= n || j >= n) Mr[i][j] = 0.f;
            }
            if (!inject) {
                qinv = 1.0f / qv;
                k2 = s1v * qinv * qinv * qinv / (float)C;
            }
            float dfv[8];
            uint32_t dxw[kSlabNS][2];  // packed dx of the first half, stored with the second (16 bytes per stream)
            // two halves of four channels keep the live unpacked values small
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float xv[kSlabNS][4], gv[kSlabNS][4];
#pragma unroll
                for (int j = 0; j < kSlabNS; j++) {
                    float t8[8];
                    unpack8(cur.xr[j], t8);
#pragma unroll
                    for (int v = 0; v < 4; v++) xv[j][v] = t8[4 * h + v];
                    cur.gr[j].get(t8);
#pragma unroll
                    for (int v = 0; v < 4; v++) gv[j][v] = t8[4 * h + v];
                }
                float da[4];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    float s_a = 0.f, s_df = 0.f;
#pragma unroll
                    for (int i = 0; i < kSlabNS; i++) { s_a += hpre[i] * xv[i][v]; s_df += hpost[i] * gv[i][v]; }
                    dfv[4 * h + v] = s_df;
                    da[v] = inject ? 0.f : s_df * wv[4 * h + v] * qinv - s_a * k2;
                    usum[4 * h + v] += s_df * s_a * qinv;
                }
#pragma unroll
                for (int j = 0; j < kSlabNS; j++) {
                    if (j < n) {
                        const float4 p0 = *reinterpret_cast<const float4 *>(dxf_s + (size_t)bl * kSlabLDF + j * kSlabCW + ch * 8 + 4 * h);
                        float out[4] = {p0.x, p0.y, p0.z, p0.w};
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            float sacc = out[v] + hpre[j] * da[v] - cxv * xv[j][v];
#pragma unroll
                            for (int i = 0; i < kSlabNS; i++) sacc += Mr[i][j] * gv[i][v];
                            out[v] = sacc;
                        }
                        if (h == 0) {
                            dxw[j][0] = pack_bf16x2(out[0], out[1]);
                            dxw[j][1] = pack_bf16x2(out[2], out[3]);
                        } else {
                            st16<true>(static_cast<bf16_t *>(a.dx) + (size_t)b * nC + (size_t)j * C + cth, dxw[j][0], dxw[j][1],
                                       pack_bf16x2(out[0], out[1]), pack_bf16x2(out[2], out[3]));
                        }
                    }
                }
            }
            if (inject && a.df) store_vec<bf16_t, 8>(a.df + (size_t)b * C + cth, dfv);
        }
        // no barrier needed here: the next tile's x_s writes come after barrier 2 of this tile (all
        // fragment reads done) and its dxf_s writes come after its own barrier 1 (all phase C done)
        MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 3, pclk);
    };
    for (int sb = b_begin; sb < b_end; sb += 64) {
        process_tile(sb, cur, nxt);
        if (sb + 32 < b_end) process_tile(sb + 32, nxt, cur);
    }

    // ---- outputs of the split -----------------------------------------------------------------------
    float *dphi_out = a.dphi_part + (size_t)blockIdx.y * D * nC;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int tile = 2 * wave + t, j = tile >> 1;
        const int c = c0 + (tile & 1) * 32 + row;
        if (j < n && c < C) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int d = 8 * (i >> 2) + 4 * kg + (i & 3);
                if (d < D) dphi_out[(size_t)d * nC + (size_t)j * C + c] = acc[t][i];
            }
        }
    }
    MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 4, pclk);
    __syncthreads();  // everyone is done with dxf_s; reuse it for the two small reductions
    if (!inject) {
        // dw summands: sum over the 32 sample slots that share a channel chunk
        float *red = dxf_s;  // [32][64 + 1]
#pragma unroll
        for (int v = 0; v < 8; v++) red[bl * 65 + ch * 8 + v] = usum[v];
        __syncthreads();
        if (tid < 64) {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < 32; r++) s += red[r * 65 + tid];
            if (c0 + tid < C) a.dw_part[(size_t)blockIdx.y * C + c0 + tid] = s;
        }
        __syncthreads();
    }
    if (blockIdx.x == 0) {
        double *red = reinterpret_cast<double *>(dxf_s);  // [8][32]
        red[tid] = dtsum;
        __syncthreads();
        if (tid < D + 3 && tid < 32) {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < 8; r++) s += red[r * 32 + tid];
            a.dt_part[(size_t)blockIdx.y * (D + 3) + tid] = s;
        }
    }
    MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 5, pclk);
}


// ---------------------------------------------------------------------------------------------
// The same pass for bf16 dy.
//
// What bounds it is bytes - x and dy once in, dx once out - and how they are asked for.  Plain copies of two arrays into a
// third in this access pattern reach 5.7 TB/s with 256-byte pieces of a row and some 130 KB per CU on their way, 4.8 with
// 128-byte pieces, and the kernel above, used for both types before, reached 3.9: two tiles in 248 registers, phases
// that run one after the other between barriers while the memory waits.  Here
//   - every operand goes from global memory straight into LDS (global_load_lds, no registers in between), 16 samples
//     at a time, x three and dy two tiles ahead (95 KB);
//   - dP phi is formed transposed (phi^T as the A operand, dP as B, 16x16x32): a lane of the accumulators
//     then holds four consecutive channels of ONE sample for every stream, which is what the mixing needs,
//     so the projection term never leaves the registers;
//   - dx replaces dy in LDS and leaves one tile later, row by row in 256-byte pieces: written as the lanes hold it, in
//     pieces of 64 bytes, the stores alone cost 20 us at B=8192 C=2560;
//   - the waves are of two kinds.  Loaders (a wave per 32 channels) request the tiles and do nothing else: one that
//     also accumulated dphi held the barrier up (109 us).  Mixers (a wave per 16 channels) accumulate dphi, form dx and
//     store it.
// A period is one tile: one barrier, and nothing else between the waves.  CW channels per workgroup, one workgroup per CU.
// Measured, n=4 B=8192 C=2560: 130 -> 94 us (503 MB, 5.3 TB/s); backward in graphs of ten, with the former kernel and channel
// sums -> now: B=8192 C=2560 209 -> 164 us, B=1280 C=2560 42.4 -> 36.9, B=2048 C=1280 41.0 -> 33.1, n=3 B=5000 C=1920 86.7 ->
// 68.4, n=2 B=3000 C=1024 37.6 -> 28.8.
// Tried and slower at B=8192 C=2560 (backward): tiles of 32 samples in two stages with eight waves of one kind 193 us; dy
// in the mixers' registers, dx stored from them, 214 us.
//
// LDS: a ring of x [N][16][CW] with the tile's dP^T hi, lo and dP in operand order (1 KiB each) and its samples'
// coefficients, dense arrays copied as they are; a ring of dy, then dx, [N][16][CW].  The 16-byte chunks of a
// row are permuted (slab_swizzle) so that neither the transposed reads (dphi) nor the row reads (dx) meet in a bank.
// ---------------------------------------------------------------------------------------------

// F32: float32 storage.  The channel sums have left x and dy in bf16 where dx will be (mix_bwd_reduce.hip): the 256 bytes of 64
// channels hold 128 of x, then 128 of dy, and this kernel's slab of 64 reads such a piece and later puts 64 values of dx in its
// place.  x and dy are then one tile, three tiles ahead, a row of 16 chunks like those of a slab of 128; dx, twice as wide as dy, leaves
// through two places of its own.  Backward in graphs of ten, resident path -> channel sums and this: n=4 B=4369 C=1280 142 -> 113 us,
// 2000 2560 133 -> 90, n=3 3000 3136 199 -> 124, n=2 4369 2560 185 -> 105.
template <int N, int CW, bool F32> struct SlabStage {
    static_assert(!F32 || CW == f32_piece_channels(N), "a slab reads whole pieces");
    static constexpr int TB = 16, kLoaders = CW / 32, kMixers = CW / 16, kThreads = 64 * (kLoaders + kMixers);  // 6 CW
    static constexpr int kXAhead = 3, kGAhead = F32 ? 0 : 2;  // tiles requested ahead
    static constexpr int kXRing = kXAhead + 1, kGRing = kGAhead + 2;
    static constexpr int kRowBytes = CW * (F32 ? 4 : 2), kChunks = kRowBytes / 16, kRows = 1024 / kRowBytes;  // of a tile's row; rows per KiB
    static constexpr int kTile = N * TB * kRowBytes;      // bytes of x or dy, or of both; of dx
    static constexpr int kP = kTile, kCoef = kP + 3 * 1024;
    // coefficient blocks of 64 floats: M | Hpre | Hpost | cx | q | s1 | dt (slab 0 only)
    static constexpr int kSegM = (TB * N * N + 63) / 64, kSegs = kSegM + 5, kSegDt = (TB * (N * N + 2 * N + 3) + 63) / 64;
    static constexpr int kXBytes = kCoef + (kSegs + kSegDt) * 256;
    // a loader's share of the dP and coefficient blocks (the last ones twice where they do not come out even, so that
    // every loader has the same number of instructions in flight)
    static constexpr int kShare = (3 + kSegs + kLoaders - 1) / kLoaders, kShareDt = (3 + kSegs + kSegDt + kLoaders - 1) / kLoaders;
    static constexpr int kG = kXRing * kXBytes;           // the dy / dx ring
    static constexpr int kW = kG + kGRing * kTile;        // the slab's w in fp32
    static constexpr int kLds = kW + CW * 4;
    static constexpr int kPhi = 32 * N * CW * 2;          // prologue: the phi slab, in the part of the dy ring not yet requested
    static constexpr int kRing = kChunks * 8;             // what slab_swizzle() goes by
    static_assert(kPhi <= (kGRing - kGAhead) * kTile && kLds <= 160 * 1024, "the rings fit the LDS of a CU");
};

template <int N, int CW, bool INJECT, bool F32>
__global__ __launch_bounds__(CW * 6, 3) void bwd_slab_stage_kernel(BwdSlabArgs a) {
    static_assert(!(INJECT && F32), "an injected f takes the other kernels");
    using ST = SlabStage<N, CW, F32>;
    constexpr int kChunks = ST::kChunks, kRows = ST::kRows, kRowBytes = ST::kRowBytes;
    constexpr int D = N * N + 2 * N, TB = ST::TB;
    extern __shared__ float smem_f[];
    char *const smem = reinterpret_cast<char *>(smem_f);
    const uint32_t smem_at = lds_address(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int C = a.C, nC = N * C;
    const int slab = blockIdx.x, c0 = slab * CW;
    const unsigned nsplit = gridDim.y;
    // tiles y, y + S, ..: all splits go through the batch together and begin where the channel sums, which go through it from its end,
    // have just read x and dy: the memory-side cache (256 MB) still holds that part.  Backward us, splits of consecutive tiles | this: n=4 C=2560
    // B=8192 162.3 | 156.4 (the order of either kernel alone: 161.0, 168.1), 3000 63.3 | 62.6;  C=1920 4096 63.8 | 62.9;  C=1280 8192 84.1 | 84.7
    // (forward + backward 121.9 | 121.9);  n=3 C=1024 8192 60.0 | 58.4;  n=2 C=2560 8192 91.5 | 90.3;  n=1 C=4096 6000 80.5 | 80.0
    const int b_begin = blockIdx.y * TB, b_step = nsplit * TB, b_end = a.B;
    const int T = (a.tiles - 1 - (int)blockIdx.y) / (int)nsplit + 1;
    const int pwg = blockIdx.y * gridDim.x + blockIdx.x;
    (void)pwg;
    MHC_PHASE_ZERO(kPhaseBwdSlab, pwg);
    MHC_PHASE_BEGIN(pclk);
    const bool loader = wave >= ST::kMixers;
    const int lw = wave - ST::kMixers;  // loader index

    // One KiB of a tile of x, dy or dx is kRows sample rows of one stream: where lane's 16 bytes belong, for the rows from row0
    const auto lane_row = [&](int row0) { return row0 + lane / kChunks; };
    const auto lane_chunk = [&](int row) { return (lane % kChunks) ^ slab_swizzle<ST::kRing>(row); };
    const auto lane_col = [&](int row) { return c0 + lane_chunk(row) * (F32 ? 4 : 8); };  // of x or dy; F32: of dx

    // ---- loads of a tile (loaders); loader l brings rows l kRows .. of every stream --------------------
    // slots beyond the batch alias its last sample, columns beyond C the last ones: they only meet zero columns of
    // dP^T or land in rows and columns that are not stored
    // (F32: C is a multiple of 64; a loader brings every kLoaders-th group of rows)
    const int ld_row = lane_row(lw * kRows), ld_col = min(lane_col(ld_row), C - 8);
    constexpr int kLoads = F32 ? N * TB / kRows / ST::kLoaders : N;  // instructions per loader for a tile of x, or of both
    auto load_tile = [&](const void *src, int t, uint32_t dst) {
        const int sb = b_begin + t * b_step;
        if constexpr (F32) {
            const char *base = static_cast<const char *>(src) + ((size_t)sb * nC + c0) * 4;
#pragma unroll
            for (int j = 0; j < N; j++)
#pragma unroll
                for (int i = 0; i < TB / kRows / ST::kLoaders; i++) {
                    const int row0 = (lw + i * ST::kLoaders) * kRows, row = lane_row(row0);
                    load_to_lds<16>(base + (size_t)j * C * 4, (uint32_t)min(row, b_end - sb - 1) * nC * 4 + lane_chunk(row) * 16,
                                    dst + (j * TB + row0) * kRowBytes);
                }
        } else {
            const bf16_t *base = static_cast<const bf16_t *>(src) + (size_t)sb * nC;
            const uint32_t off = (uint32_t)(min(ld_row, b_end - sb - 1) * nC + ld_col) * 2;
#pragma unroll
            for (int j = 0; j < N; j++) load_to_lds<16>(base + (size_t)j * C, off, dst + (j * TB + lw * kRows) * kRowBytes);
        }
    };
    auto load_dy = [&](int t) {
        if constexpr (!F32) load_tile(a.dy, t, smem_at + ST::kG + t % ST::kGRing * ST::kTile);
    };
    // The dP operands and the blocks of 64 coefficients of a tile are dealt out to the loaders: what this one brings is
    // settled once, so that a tile costs it no more than the instructions.
    struct Block {
        const char *src;          // for the first sample of the batch
        uint32_t step, at, dst;   // bytes per sample; this lane's bytes behind the tile's first; place behind the tile's x
        int words;                // coefficients: floats per sample; 0: a KiB of dP operands
    };
    const int blocks = 3 + ST::kSegs + (slab == 0 ? ST::kSegDt : 0);
    auto block_of = [&](int k) {
        k = min(k, blocks - 1);
        if (k < 2) return Block{reinterpret_cast<const char *>(a.dPT + (size_t)k * 32 * a.BP), 64u, lane * 16u, ST::kP + k * 1024u, 0};
        // dP: [d / 8][16 samples][8] out of the fragments of 32 samples
        if (k == 2) return Block{reinterpret_cast<const char *>(a.dPb), 64u, (lane >> 5) * 1024u + ((lane >> 4) & 1) * 512u + (lane & 15) * 16u, ST::kP + 2048u, 0};
        const int s = k - 3;
        const float *src;
        int words = 1, i = lane;
        if (s < ST::kSegM) { src = a.M; words = N * N; i += s * 64; }
        else if (s == ST::kSegM) { src = a.Hpre; words = N; }
        else if (s == ST::kSegM + 1) { src = a.Hpost; words = N; }
        else if (s == ST::kSegM + 2 || (INJECT && s < ST::kSegs)) src = a.cx;
        else if (s == ST::kSegM + 3) src = a.q;
        else if (s == ST::kSegM + 4) src = a.s1;
        else { src = a.dt; words = D + 3; i += (s - ST::kSegs) * 64; }
        return Block{reinterpret_cast<const char *>(src), words * 4u, i * 4u, ST::kCoef + s * 256u, words};
    };
    Block mine[ST::kShareDt];
#pragma unroll
    for (int i = 0; i < ST::kShareDt; i++) mine[i] = block_of(lw + i * ST::kLoaders);
    auto load_x = [&](int t) {
        const uint32_t st = smem_at + t % ST::kXRing * ST::kXBytes;
        const int sb = b_begin + t * b_step, left = min(b_end - sb, TB);
        load_tile(F32 ? a.dx : static_cast<const void *>(a.x), t, st);
#pragma unroll
        for (int i = 0; i < ST::kShareDt; i++) {
            const Block &m = mine[i];
            if (i >= ST::kShare && slab != 0) break;
            if (m.words == 0) {  // (the second half of a 32-sample fragment of dP lies 256 bytes behind the first)
                const bool half = m.dst == ST::kP + 2048u && (sb & 16);
                load_to_lds<16>(m.src + (size_t)(half ? sb - 16 : sb) * m.step + (half ? 256 : 0), m.at, st + m.dst);
            } else {
                load_to_lds<4>(m.src + (size_t)sb * m.step, min(m.at, left * m.step - 4), st + m.dst);
            }
        }
    };

    // ---- prologue: the loaders request the first tiles; phi slab -> LDS, row-major [32 d][N][CW] -> the mixers' transposed
    // fragments.  The mixers alone bring phi and w, and the two barriers do not wait for global memory: a loader that also
    // brought a part of phi waited for all its first tiles before it could hand that part on (the compiler does not count the
    // requests), and no tile was requested meanwhile.  Backward in graphs of ten, n=4 B=1280 C=2560: 37.5 -> 36.5 us, n=2 B=3000
    // C=1024 29.4 -> 28.5.
    if (loader) {
        // in the order in which the loop below counts them: what period p - 1 would have requested before what period p would
        load_x(0);
        if (T > 1) load_x(1);
        load_dy(0);
        if (T > 2) load_x(2);
        if (T > 1) load_dy(1);
    }
    char *const phi_s = smem + ST::kG + ST::kGAhead * ST::kTile;
    if (!loader) {
        constexpr int kThreads = 64 * ST::kMixers, kPc = CW / 8, kPhiIters = N * 32 * kPc / kThreads;
        static_assert(kPhiIters * kThreads == N * 32 * kPc, "whole chunks of phi for every mixer");
        uint4 phir[kPhiIters];
#pragma unroll
        for (int i = 0; i < kPhiIters; i++) {
            const int e = tid + i * kThreads;
            const int d = e / (N * kPc), j = e / kPc % N, c = c0 + e % kPc * 8;
            const bool ok = d < D && c < C;
            phir[i] = load16_masked(reinterpret_cast<const uint4 *>(a.phi + (ok ? (size_t)d * nC + (size_t)j * C + c : 0)), ok);
        }
        if (tid < CW)
            reinterpret_cast<float *>(smem + ST::kW)[tid] =
                (c0 + tid < C && !INJECT) ? (a.w_bf16 ? bf16_to_f32(static_cast<const bf16_t *>(a.w)[c0 + tid])
                                                      : static_cast<const float *>(a.w)[c0 + tid]) : 0.f;
#pragma unroll
        for (int i = 0; i < kPhiIters; i++) *reinterpret_cast<uint4 *>(phi_s + (tid + i * kThreads) * 16) = phir[i];
    }
    stage_barrier();

    double usum[4] = {0.0, 0.0, 0.0, 0.0};  // mixers: float32 terms, a sample each (the walk may be hundreds of tiles long)
    double dtsum = 0.0;                     // loaders of slab 0: column tid & 31, row group
    // mixer lane (l16, kq): the four channels from c0 + cl of sample l16
    const int l16 = lane & 15, kq = lane >> 4, cl = 16 * wave + 4 * kq;

    if (loader) {
        // ---- requests the tiles --------------------------------------------------------------------------
        stage_barrier();  // the mixers hold their fragments of phi
        for (int p = 0; p < T; p++) {
            // Tile p has landed, for everybody behind the barrier: its dy is the last of it, requested in period p - 2, and
            // behind that are the x of tile p + 2 and the dy of tile p + 1 (period p - 1).  Towards the end there are fewer.
            // (F32: behind it are the tiles p + 1 and p + 2)
            if constexpr (F32) {
                if (p + 1 >= T) wait_vmem<0>();
                else if (p + 2 >= T) { if (slab == 0) wait_vmem<kLoads + ST::kShareDt>(); else wait_vmem<kLoads + ST::kShare>(); }
                else if (slab == 0) wait_vmem<2 * (kLoads + ST::kShareDt)>();
                else wait_vmem<2 * (kLoads + ST::kShare)>();
            } else {
                if (p + 2 >= T) wait_vmem<0>();
                else if (slab == 0) wait_vmem<2 * N + ST::kShareDt>();
                else wait_vmem<2 * N + ST::kShare>();
            }
            stage_barrier();
            // everybody is done with x of tile p - 1 and with dx of tile p - 2, whose places these take
            if (p + ST::kXAhead < T) load_x(p + ST::kXAhead);
            if (p + ST::kGAhead < T) load_dy(p + ST::kGAhead);
            if (slab == 0) {  // dt column sums: 32 columns x 2 kLoaders row groups
                const char *st = smem + p % ST::kXRing * ST::kXBytes;
                const int col = tid & 31, rg = (tid >> 5) - 2 * ST::kMixers, left = b_end - (b_begin + p * b_step);
                const float *dts = reinterpret_cast<const float *>(st + ST::kCoef) + ST::kSegs * 64;
                if (col < D + 3) {
#pragma unroll
                    for (int rr = 0; rr < TB / (2 * ST::kLoaders); rr++) {
                        const int bb = rg * (TB / (2 * ST::kLoaders)) + rr;
                        if (bb < left) dtsum += dts[bb * (D + 3) + col];
                    }
                }
            }
        }
        stage_barrier();  // the mixers' last dx
    } else {
        // ---- dphi and dx of a tile, stores dx of the one before -------------------------------------------
        bf16x8_t phif[N];  // A operand: rows = this wave's 16 channels of a stream, contraction over d
        {
            const int q = lane & 3, jj = (lane >> 2) & 3;
#pragma unroll
            for (int j = 0; j < N; j++) {
                const char *p = phi_s + ((kq * 8 + jj) * N + j) * CW * 2 + (16 * wave + 4 * q) * 2;
                typedef __attribute__((address_space(3))) lds_tr_v4i16 *lds_ptr;
                const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p));
                const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 4 * N * CW * 2)));
                phif[j] = __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
            }
        }
        const float4 w4 = *reinterpret_cast<const float4 *>(smem + ST::kW + cl * 4);
        const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
        const float inv_c = 1.0f / (float)C;
        stage_barrier();  // the loaders may fill the places that hold phi
        // this lane's 8 bytes of its sample's row of x, of dy (F32: 8 chunks behind), and what it writes of dx
        const auto row_place = [&](int chunk) { return l16 * kRowBytes + ((chunk ^ slab_swizzle<ST::kRing>(l16)) * 16); };
        const int row_at = row_place(cl >> 3) + (kq & 1) * 8, row_dy = F32 ? row_place(8 + (cl >> 3)) + (kq & 1) * 8 : row_at;
        // a tile of dx leaves in pieces of one KiB, kOut for every mixer
        constexpr int kPieces = N * TB / kRows, kOut = (kPieces + ST::kMixers - 1) / ST::kMixers;
        auto store_dx = [&](int t) {
            const int sb = b_begin + t * b_step;
            const char *g = smem + ST::kG + t % ST::kGRing * ST::kTile;
#pragma unroll
            for (int i = 0; i < kOut; i++) {
                const int at = wave + i * ST::kMixers, piece = min(at, kPieces - 1), j = piece / (TB / kRows), row = lane_row(piece % (TB / kRows) * kRows);
                const int c = lane_col(row);
                const uint4 v = *reinterpret_cast<const uint4 *>(g + piece * 1024 + lane * 16);
                if (at < kPieces && sb + row < b_end && c < C) {  // C % 8 == 0: eight channels are inside or outside
                    if constexpr (F32) st16<true>(static_cast<float *>(a.dx) + (size_t)sb * nC + (uint32_t)(row * nC + j * C + c), v.x, v.y, v.z, v.w);
                    else st16<true>(static_cast<bf16_t *>(a.dx) + (size_t)sb * nC + (uint32_t)(row * nC + j * C + c), v.x, v.y, v.z, v.w);
                }
            }
        };
        // dphi: 32-column tiles wave, wave + kMixers (stream, 32-channel group)
        constexpr int kCols = N * CW / 32, kAcc = (kCols + ST::kMixers - 1) / ST::kMixers;
        f32x16_t acc[kAcc];
#pragma unroll
        for (int k = 0; k < kAcc; k++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[k][i] = 0.f;
        // transposed reads of x: this lane's row (lo; hi: + 4) and its 8 bytes of a 32-channel group
        const int tr_q = lane & 3, tr_row = (lane >> 5) * 8 + ((lane >> 2) & 3), tr_c = ((lane >> 4) & 1) * 2 + (tr_q >> 1);
        for (int t = 0; t < T; t++) {
            const char *st = smem + t % ST::kXRing * ST::kXBytes;
            char *const gs = smem + ST::kG + t % ST::kGRing * ST::kTile;
            const int sb = b_begin + t * b_step;
            const float *co = reinterpret_cast<const float *>(st + ST::kCoef);
            MHC_PHASE_ADD(kPhaseBwdSlab, pwg, t > 0 ? 2 : 0, pclk);
            stage_barrier();
            MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 1, pclk);
            if (t > 0) store_dx(t - 1);
            const bf16x8_t ah = *reinterpret_cast<const bf16x8_t *>(st + ST::kP + lane * 16);
            // what the mixing needs, requested ahead of the products, under which it arrives (n=4 B=1605 C=1728, whole backward:
            // 40.0 -> 39.1 us)
            float Mr[N][N], hpre[N], hpost[N];
            uint2 xr[N], gr[N];
            lds_floats<N>(co + ST::kSegM * 64 + l16 * N, hpre);
            lds_floats<N>(co + (ST::kSegM + 1) * 64 + l16 * N, hpost);
            lds_floats<N * N>(co + l16 * N * N, &Mr[0][0]);
#pragma unroll
            for (int j = 0; j < N; j++) {
                xr[j] = *reinterpret_cast<const uint2 *>(st + j * TB * kRowBytes + row_at);
                gr[j] = *reinterpret_cast<const uint2 *>((F32 ? st : gs) + j * TB * kRowBytes + row_dy);
            }
            __builtin_amdgcn_sched_barrier(0);
            const bf16x8_t al = *reinterpret_cast<const bf16x8_t *>(st + ST::kP + 1024 + lane * 16);
#pragma unroll
            for (int k = 0; k < kAcc; k++) {
                const int tile = wave + k * ST::kMixers, c = (tile % (CW / 32)) * 4 + tr_c;
                if (kCols % ST::kMixers != 0 && tile >= kCols) break;
                typedef __attribute__((address_space(3))) lds_tr_v4i16 *lds_ptr;
                const char *xs = st + (tile / (CW / 32) * TB + tr_row) * kRowBytes + (tr_q & 1) * 8;
                const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(xs + (c ^ slab_swizzle<ST::kRing>(tr_row)) * 16)));
                const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_ptr)(xs + 4 * kRowBytes + (c ^ slab_swizzle<ST::kRing>(tr_row + 4)) * 16)));
                const bf16x8_t xf = __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
                acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, xf, acc[k], 0, 0, 0);
                acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, xf, acc[k], 0, 0, 0);
            }
            // projection term: columns = samples, rows = this lane's channels
            const bf16x8_t pf = *reinterpret_cast<const bf16x8_t *>(st + ST::kP + 2048 + lane * 16);
            f32x4_t o[N];
#pragma unroll
            for (int j = 0; j < N; j++)
                o[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(phif[j], pf, f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            const float *sc = co + (ST::kSegM + 2) * 64 + l16;
            const float cxv = sc[0];
            float qinv = 0.f, k2 = 0.f;
            const bool real = sb + l16 < b_end;  // a slot beyond the batch adds nothing to usum, whatever its sample holds
            if constexpr (!INJECT) {
                qinv = 1.0f / sc[64];
                k2 = sc[128] * qinv * qinv * qinv * inv_c;
            }
            float dfv[4];
            uint32_t out[N][F32 ? 4 : 2];
#pragma unroll
            for (int p = 0; p < 2; p++) {  // channel pairs
                float r[N][2];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int c = 2 * p + e;
                    float xv[N], gv[N];
#pragma unroll
                    for (int j = 0; j < N; j++) {
                        const uint32_t xw = p ? xr[j].y : xr[j].x, gw = p ? gr[j].y : gr[j].x;
                        xv[j] = e ? bf16hi_to_f32(xw) : bf16lo_to_f32(xw);
                        gv[j] = e ? bf16hi_to_f32(gw) : bf16lo_to_f32(gw);
                    }
                    float s_a = 0.f, s_df = 0.f;
#pragma unroll
                    for (int j = 0; j < N; j++) { s_a += hpre[j] * xv[j]; s_df += hpost[j] * gv[j]; }
                    dfv[c] = s_df;
                    const float dq = s_df * qinv;
                    const float da = INJECT ? 0.f : dq * wv[c] - s_a * k2;
                    if constexpr (!INJECT) usum[c] += (double)(real ? dq * s_a : 0.f);
#pragma unroll
                    for (int j = 0; j < N; j++) {
                        float v = o[j][c] + hpre[j] * da - cxv * xv[j];
#pragma unroll
                        for (int i = 0; i < N; i++) v += Mr[i][j] * gv[i];
                        r[j][e] = v;
                    }
                }
#pragma unroll
                for (int j = 0; j < N; j++) {
                    if constexpr (F32) {
                        out[j][2 * p] = __float_as_uint(r[j][0]);
                        out[j][2 * p + 1] = __float_as_uint(r[j][1]);
                    } else {
                        out[j][p] = pack_bf16x2(r[j][0], r[j][1]);
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < N; j++) {
                if constexpr (F32) *reinterpret_cast<uint4 *>(gs + j * TB * kRowBytes + row_place(cl >> 2)) = make_uint4(out[j][0], out[j][1], out[j][2], out[j][3]);
                else *reinterpret_cast<uint2 *>(gs + j * TB * kRowBytes + row_at) = make_uint2(out[j][0], out[j][1]);
            }
            if (INJECT && a.df && sb + l16 < b_end && c0 + cl < C)
                store_vec<bf16_t, 4>(a.df + (size_t)sb * C + (uint32_t)(l16 * C + c0 + cl), dfv);
        }
        MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 2, pclk);
        stage_barrier();
        store_dx(T - 1);
        float *dphi_out = a.dphi_part + (size_t)blockIdx.y * D * nC;
#pragma unroll
        for (int k = 0; k < kAcc; k++) {
            const int tile = wave + k * ST::kMixers, c = c0 + tile % (CW / 32) * 32 + (lane & 31);
            if (tile < kCols && c < C) {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int d = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                    if (d < D) dphi_out[(size_t)d * nC + (size_t)(tile / (CW / 32)) * C + c] = acc[k][i];
                }
            }
        }
    }

    // ---- small outputs of the split -------------------------------------------------------------------
    MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 3, pclk);
    __syncthreads();  // everyone is done with the rings; reuse them for the two small reductions
    if constexpr (!INJECT) {
        double *red = reinterpret_cast<double *>(smem);  // [16][CW + 1]
        if (!loader) {
#pragma unroll
            for (int v = 0; v < 4; v++) red[l16 * (CW + 1) + cl + v] = usum[v];
        }
        __syncthreads();
        if (tid < CW) {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < 16; r++) s += red[r * (CW + 1) + tid];
            if (c0 + tid < C) a.dw_part[(size_t)blockIdx.y * C + c0 + tid] = s;
        }
        __syncthreads();
    }
    if (slab == 0) {
        double *red = reinterpret_cast<double *>(smem);  // [2 kLoaders][32]
        if (loader) red[tid - 64 * ST::kMixers] = dtsum;
        __syncthreads();
        if (tid < 32 && tid < D + 3) {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < 2 * ST::kLoaders; r++) s += red[r * 32 + tid];
            a.dt_part[(size_t)blockIdx.y * (D + 3) + tid] = s;
        }
    }
    MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 4, pclk);
}

bool bwd_slab_supported(int x_dtype, int y_dtype, int phi_dtype, int n, int C) {
    (void)y_dtype;
    return x_dtype == kBF16 && phi_dtype == kBF16 && n <= 4 && C % 8 == 0;
}

// Channels per workgroup of the bf16 kernel.  A CU carries one workgroup of either width, so the narrow one leaves half as
// many partial sums of dphi behind (C / 64 slabs in half as many splits) but has half the waves to hide its latencies
// and loads half as wide pieces of a row.  Backward, 64 | 128 channels (us, the better split count of each):
//   n=4  B=800 C=1280 23.1 | 25.8   1024 x 1024 22.2 | 25.6   2048 x 512 24.8 | 27.3   6000 x 256 34.5 | 37.8
//        1024 x 2048 28.3 | 29.9   2048 x 1280 33.1 | 35.2   4096 x 640 36.0 | 37.9   8192 x 320 39.8 | 43.1
//        8192 x 768 64.9 | 67.3   8192 x 1024 70.8 | 73.0   8192 x 1280 84.9 | 86.7   5000 x 1920 79.9 | 80.7
//        1280 x 2560 37.1 | 37.0   1000 x 3712 43.5 | 42.6   4000 x 2560 80.4 | 79.2   8192 x 2560 185 | 164
//   n=3  1500 x 1920 31.6 | 29.5   n=2  4000 x 1024 34.4 | 32.1   1000 x 2560 29.6 | 27.2
// The lines: n = 4 up to 1280 channels, or below 12 M activation elements.
static int slab_width(int B, int n, int C, bool f32 = false) {
    if (f32) return f32_piece_channels(n);
    if (const int forced = tuning_get(kTuneSlabWidth)) return forced == 1 ? 64 : 128;
    return n == 4 && (C <= 1280 || (long long)B * n * C < 12'000'000) ? 64 : 128;
}

int bwd_slab_batch_splits(int B, int n, int C, int y_dtype) {
    const bool staged = y_dtype != kF32;
    const int width = staged ? slab_width(B, n, C, y_dtype == kF32AsBF16) : kSlabCW, slabs = (C + width - 1) / width;
    const int tiles = (B - 1) / (staged ? 16 : 32) + 1;
    if (const int forced = tuning_get(kTuneSlabSplits); forced > 0) {  // experiment hook
        return forced < tiles ? forced : tiles;
    }
    // All workgroups resident at once: one per CU (bf16 dy) or two (fp32 dy).  One split more than that costs a second
    // round (B=1280 C=2560, 12 splits of 20 slabs 37.1 us, 20 splits 44.8), fewer leave CUs idle (8 splits 39.4).
    int S = std::max(1, (staged ? 256 : 512) / slabs);
    if (S > tiles) S = tiles;
    // Short rows: the splits that cost least, a tile being some 0.65 us of a walk and a copy of the partial dphi 0.09 us of the
    // finalize launch, which adds up hundreds of copies of few columns one after the other.  Backward us, as many splits as fit
    // (one to three tiles each) | four tiles each: n=2 B=3300 C=64 39.0 | 28.2, n=4 B=6200 C=64 39.5 | 32.6 (six: 31.3), n=1 B=2000 C=256
    // 26.7 | 21.3, n=3 B=1000 C=384 26.5 | 23.8, n=3 B=1300 C=384 29.0 | 24.5, n=4 B=100 C=64 21.8 | 25.4, n=2 B=650 C=1280 22.2 | 21.9.
    // Longer rows have few splits: n=2 B=450 C=1920 (two tiles each) 22.0 | 23.4, n=1 B=240 C=3200 17.4 | 18.5.
    if (staged && slabs <= 10) {
        const auto us = [&](int s) { return 0.65 * ((tiles + s - 1) / s) + 0.09 * s; };
        int best = S;
        for (int s = 1; s < S; s++)
            if (us(s) < us(best)) best = s;
        S = best;
    }
    if (!staged) {
        // the dphi partial copies (written here, read once by the finalize launch) stay below 16 MB or
        // 0.4 of the activation bytes this kernel moves, whichever is larger
        const int D = n * n + 2 * n;
        const double part = 2.0 * 4.0 * D * n * C;  // bytes written + read per split
        double budget = 0.4 * (3.0 * 2.0 * B * n * C);
        if (budget < 16e6) budget = 16e6;
        if (S > (int)(budget / part)) S = std::max(1, (int)(budget / part));
    }
    // the longest split decides: the fewest splits that keep its tile count
    const int tps = (tiles + S - 1) / S;
    return (tiles + tps - 1) / tps;  // <= tiles: every split has at least one tile
}

hipError_t launch_bwd_slab(const void *dy, int y_dtype, const void *x, const void *w, int w_dtype,
                           const void *f_inject, const void *phi, const float *Hpre,
                           const float *Hpost, const float *M, const float *q, const float *s1,
                           const float *cx, const void *dPb, const void *dPT, int BP, const float *dt,
                           void *dx, void *df, float *dphi_part, double *dw_part, double *dt_part, int S,
                           int B, int n, int C, hipStream_t stream) {
    const int tiles = y_dtype != kF32 ? (B - 1) / 16 + 1 : (B + 31) / 32;
    if (S < 1 || S > tiles) return hipErrorInvalidValue;
    BwdSlabArgs a{dy, static_cast<const bf16_t *>(x), w, f_inject, static_cast<const bf16_t *>(phi),
                  Hpre, Hpost, M, q, s1, cx, static_cast<const bf16_t *>(dPb),
                  static_cast<const bf16_t *>(dPT), dt, dx,
                  static_cast<bf16_t *>(df), dphi_part, dw_part, dt_part, w_dtype == kBF16, B, BP, n, C, tiles};
    if (y_dtype != kF32) {
        const bool f32 = y_dtype == kF32AsBF16;
        if (f32 && (f_inject || C % 64 != 0)) return hipErrorInvalidValue;
        const int cw = slab_width(B, n, C, f32);
        dim3 grid((C + cw - 1) / cw, S);
#define MHC_SLAB(N, CW, INJ, F32)                                                                                  \
    do {                                                                                                          \
        constexpr size_t lds = SlabStage<N, CW, F32>::kLds;                                                          \
        if (hipError_t e = allow_dynamic_lds<&bwd_slab_stage_kernel<N, CW, INJ, F32>>(lds); e != hipSuccess) return e; \
        bwd_slab_stage_kernel<N, CW, INJ, F32><<<grid, SlabStage<N, CW, F32>::kThreads, lds, stream>>>(a);                                     \
    } while (0)
#define MHC_SLAB_N(N)                                                                       \
    do {                                                                                    \
        if (f32) MHC_SLAB(N, 64, false, true);                                              \
        else if (cw == 64) { if (f_inject) MHC_SLAB(N, 64, true, false); else MHC_SLAB(N, 64, false, false); } \
        else { if (f_inject) MHC_SLAB(N, 128, true, false); else MHC_SLAB(N, 128, false, false); }        \
    } while (0)
        switch (n) {
            case 1: MHC_SLAB_N(1); break;
            case 2: MHC_SLAB_N(2); break;
            case 3: MHC_SLAB_N(3); break;
            default: MHC_SLAB_N(4); break;
        }
#undef MHC_SLAB_N
#undef MHC_SLAB
        return hipGetLastError();
    }
    const size_t smem = sizeof(float) * 32 * kSlabLDF + sizeof(bf16_t) * 32 * kSlabLDX;
    dim3 grid((C + kSlabCW - 1) / kSlabCW, S);
    bwd_slab_f32dy_kernel<<<grid, 256, smem, stream>>>(a);
    return hipGetLastError();
}

}  // namespace mhc
