// Projection of the dynamic-H path: raw dot products x_flat[b,:] . phi[d,:] for all D = n^2+2n
// rows of phi, plus sum(x_flat^2), as split-K partial sums.  The coefficient kernel finishes
// the reduction, divides by the RMS and applies alpha / bias / activations.
//
// Replaces compute_rms (reference src/csrc/kernels/fused_rmsnorm_matmul.cuh:119-153) and the
// cuBLASLt projection GEMM (src/python/bindings.cu:34-81, :436-443) with one pass over x.
//
// Three kernels:
//   proj_fwd_mfma_kernel    n <= 10; x and phi both bf16 (any C for n <= 8): v_mfma_f32_32x32x16_bf16 tiles
//                           (32 samples x 32 projection rows), or both fp32 (n <= 8):
//                           v_mfma_f32_32x32x2_f32, IEEE products; operands fetched row-contiguously
//                           through a wave-private LDS tile.
//   proj_fwd_wide_kernel    bf16, wider phi.
//   proj_fwd_generic_kernel any dtype / any C: fp32 FMA.
#include "launchers.h"

#include <type_traits>
#include "mhc_common.h"
#include "phase_profiler.h"
#include "phi_src.h"
#include "tuning.h"

namespace mhc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

// n <= 8 (the narrow kernel): rows of any length from one 64-element chunk on; beyond, whole 16-byte pieces
static inline bool use_mfma(int x_dtype, int phi_dtype, int n, int C) {
    return (x_dtype == kBF16 || x_dtype == kF32AsBF16) && phi_dtype == kBF16 && (C % 8 == 0 || (n <= 8 && n * C >= 64));
}

// --------------------------------------------------------------------------------------------
// generic path
// --------------------------------------------------------------------------------------------
constexpr int kGenDB = 16;  // projection rows per workgroup

template <typename TX, typename TP>
__global__ __launch_bounds__(256) void proj_fwd_generic_kernel(const TX *__restrict__ x,
                                                               const TP *__restrict__ phi,
                                                               float *__restrict__ Ppart,
                                                               float *__restrict__ ssqpart, int B,
                                                               int D, int DP, int nC) {
    __shared__ float red[4][kGenDB + 1];
    const int b = blockIdx.x, d0 = blockIdx.y * kGenDB, tid = threadIdx.x;
    const TX *xb = x + (size_t)b * nC;
    float acc[kGenDB], ssq = 0.f;
#pragma unroll
    for (int j = 0; j < kGenDB; j++) acc[j] = 0.f;
    for (int k = tid; k < nC; k += 256) {
        const float xv = to_f32<TX>(xb[k]);
        ssq += xv * xv;
#pragma unroll
        for (int j = 0; j < kGenDB; j++)
            if (d0 + j < D) acc[j] += xv * to_f32<TP>(phi[(size_t)(d0 + j) * nC + k]);
    }
#pragma unroll
    for (int j = 0; j < kGenDB; j++) acc[j] = wave_allreduce_sum(acc[j]);
    ssq = wave_allreduce_sum(ssq);
    if ((tid & 63) == 0) {
#pragma unroll
        for (int j = 0; j < kGenDB; j++) red[tid >> 6][j] = acc[j];
        red[tid >> 6][kGenDB] = ssq;
    }
    __syncthreads();
    if (tid <= kGenDB) {
        const float v = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
        if (tid < kGenDB) {
            if (d0 + tid < D) Ppart[(size_t)b * DP + d0 + tid] = v;
        } else if (blockIdx.y == 0) {
            ssqpart[b] = v;
        }
    }
}

// --------------------------------------------------------------------------------------------
// MFMA path.  Workgroup = 4 waves on the same 32-sample tile, each wave on its own K sub-slab;
// the four partial tiles are summed through LDS, so one partial per workgroup reaches memory.
// grid.x = sample_tiles * round_up(KS, 8), grid.y = groups of NT projection tiles.  Workgroup ids
// go round robin over the 8 XCDs, each with its own L2: the K slab is chosen by id % 8 (plus 8 per
// full set of sample tiles), so that all sample tiles of a slab run on one XCD and the slab of phi
// is fetched from memory once instead of once per XCD.  Ids whose slab is beyond KS do nothing.
// --------------------------------------------------------------------------------------------
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
constexpr int kNarrowPitch = 72;  // LDS row of a 64-element chunk: 128 data bytes + 16 pad (bf16 elements)

// XF32: x is stored as fp32 and rounded to bf16 (nearest even) on its way into the LDS tile; everything
// behind the tile, the sum of squares included, sees the rounded values.
// EXACT: the fp32 tier.  x and phi stay fp32 and are multiplied as they are; a 16-byte piece of a row is then
// four elements instead of eight and a chunk 32 instead of 64, everything else (LDS tile, pieces per lane,
// accumulators) is the same.  With 32 samples per tile and D padded to 32 instead of 128 x 128 tiles the fp32
// projection of B=2560 n=4 C=1280 went from 58 to 20 us.
// RAG: rows of any length (nC no multiple of the pieces): the last piece is read from nC - EL on and shifted down.
// NW: waves per workgroup, four, or eight where four would leave a wave several chunks to walk one after the other
// on a chip that is not full (narrow_waves below).
template <int NT, bool XF32 = false, bool PF32 = false, bool EXACT = false, bool RAG = false, int NW = 4>
__global__ __launch_bounds__(64 * NW, kMfmaMinWaves) void proj_fwd_mfma_kernel(const void *__restrict__ x_,
                                                            const void *__restrict__ phi_,
                                                            float *__restrict__ Ppart,
                                                            float *__restrict__ ssqpart, int B,
                                                            int D, int DP, int nC, int tiles_s, int KS,
                                                            int sub /* K per wave, whole chunks */,
                                                            PhiSrc src /* PF32 */) {
    extern __shared__ __align__(16) float lds[];  // per wave [(1 + NT) * 32][pitch] bf16; later [4][NT*16 + 1][64] fp32
    static_assert(!(EXACT && XF32), "XF32 rounds");
    using TXS = typename std::conditional<XF32 || EXACT, float, bf16_t>::type;  // storage type of x
    using TPS = typename std::conditional<PF32 || EXACT, float, bf16_t>::type;  // storage type of phi
    using TC = typename std::conditional<EXACT, float, bf16_t>::type;           // compute type
    constexpr int EL = 16 / sizeof(TC), CH = 8 * EL;  // elements of a 16-byte piece, of a chunk (8 pieces)
    const TXS *__restrict__ x = static_cast<const TXS *>(x_);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // Work item = (K slab, sample tile), tiles fastest.  Workgroup ids go round the 8 XCDs and XCD j takes the
    // contiguous items [j * per_xcd, (j + 1) * per_xcd): every XCD gets the same number, and a slab of phi is
    // fetched into one L2 (two where it straddles a border).  (One slab per XCD left XCDs without work whenever
    // KS was not a multiple of 8: half of the chip at B=8192, KS=4.)
    const int items = tiles_s * KS, per_xcd = (items + 7) >> 3;
    const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= items) return;  // the whole workgroup, before any barrier
    const int st = item % tiles_s, ks = item / tiles_s;
    const int pwg = blockIdx.y * gridDim.x + blockIdx.x;
    (void)pwg;
    MHC_PHASE_ZERO(kPhaseProjFwd, pwg);
    MHC_PHASE_BEGIN(pclk);
    const int row = lane & 31, kh = lane >> 5;
    const int b = st * 32 + row;
    const int dbase = blockIdx.y * NT * 32;
    const int kbeg = (ks * NW + wave) * sub;
    const int kend = min(kbeg + sub, nC);
    const bool bvalid = b < B;

    // Global loads are row-contiguous (8 lanes per 128-byte row piece, rows lr + 8 j): the operand
    // layout of the matrix cores has every lane on a different row, which the memory pipeline
    // serves at a quarter of this rate.  The chunk goes through a wave-private LDS tile and comes
    // back as fragments; no barrier is involved (a wave's LDS accesses complete in order).
    constexpr int PITCH = kNarrowPitch * 2;  // bytes
    char *cb = reinterpret_cast<char *>(lds) + (size_t)wave * (1 + NT) * 32 * PITCH;
    const int lr = lane >> 3, seg = lane & 7;
    // rows as 32-bit byte offsets from a uniform base (32 rows of x, all of phi: far below 4 GB), except where the
    // rows of phi lie in three matrices: eight registers less, which is one more wave per SIMD
    const char *xbase = reinterpret_cast<const char *>(x + (size_t)st * 32 * nC);
    uint32_t xoff[4], poff[NT][4];
    const float *prow[2];
    bool pval[NT][4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int bs = st * 32 + lr + 8 * j;
        xoff[j] = (bs < B ? (uint32_t)(lr + 8 * j) * nC : 0u) * (uint32_t)sizeof(TXS);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int d = dbase + t * 32 + lr + 8 * j;
            pval[t][j] = d < D;
            // the caller's matrices: 16 rows hold all of pre and post (n <= 8), every later one is a row of res
            if constexpr (PF32) {
                if (t == 0 && j < 2) prow[j] = phi_src_row(src, pval[t][j] ? d : 0, nC);
                else poff[t][j] = (uint32_t)(pval[t][j] ? d - 2 * src.n : 0) * (uint32_t)nC * (uint32_t)sizeof(TPS);
            } else poff[t][j] = (uint32_t)(pval[t][j] ? d : 0) * (uint32_t)nC * (uint32_t)sizeof(TPS);
        }
    }
    constexpr int XW = EL * sizeof(TXS) / 4;  // words of a lane's piece of x as loaded
    constexpr int PW = EL * sizeof(TPS) / 4;
    uint32_t xq[4][XW], pq[NT][4][PW];  // scalar words: whole-uint4 array elements can end up in scratch
    auto xat = [&](int j, int k) { return reinterpret_cast<const TXS *>(xbase + (xoff[j] + (uint32_t)k * (uint32_t)sizeof(TXS))); };
    auto pat = [&](int t, int j, int k) {
        if (PF32 && t == 0 && j < 2) return reinterpret_cast<const TPS *>(prow[j < 2 ? j : 0] + k);
        const char *base = PF32 ? reinterpret_cast<const char *>(src.phi[2]) : static_cast<const char *>(phi_);
        return reinterpret_cast<const TPS *>(base + (poff[t][j] + (uint32_t)k * (uint32_t)sizeof(TPS)));
    };
    auto load8 = [&](const auto *p, auto &q) {
        const uint4 v = ldg16<RAG>(p);
        q[0] = v.x; q[1] = v.y; q[2] = v.z; q[3] = v.w;
        if constexpr (sizeof(q) == 32) {
            const uint4 v2 = ldg16<RAG>(reinterpret_cast<const char *>(p) + 16);
            q[4] = v2.x; q[5] = v2.y; q[6] = v2.z; q[7] = v2.w;
        }
    };
    // the K tail: pieces behind kend are zero
    auto mask8 = [&](auto &q, bool ok, int s) {
        constexpr int kW = sizeof(q) / 4;
        if constexpr (RAG) drop_elems<kW * 4 / EL>(q, s);
#pragma unroll
        for (int i = 0; i < kW; i++) q[i] = ok ? q[i] : 0u;
    };
    // Rows beyond B (x) or D (phi) alias row 0: what they produce is finite and is either not stored
    // (samples >= B) or zeroed at the store (projection rows >= D), so only the K tail of the last
    // slab needs a mask - a uniform test per chunk instead of four selects per load (the kernel is
    // bound by VALU issue, not by memory, with four waves per SIMD).
    auto fetch = [&](int k0) {
        const int k = k0 + seg * EL;
        if (k0 + CH <= kend) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                load8(xat(j, k), xq[j]);
#pragma unroll
                for (int t = 0; t < NT; t++) load8(pat(t, j, k), pq[t][j]);
            }
            return;
        }
        const bool kv = k < kend;  // k is a multiple of EL, and so is kend unless it is a ragged nC
        const int off = kv ? (RAG ? min(k, nC - EL) : k) : 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            load8(xat(j, off), xq[j]);
#pragma unroll
            for (int t = 0; t < NT; t++) load8(pat(t, j, off), pq[t][j]);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            mask8(xq[j], kv, k - off);
#pragma unroll
            for (int t = 0; t < NT; t++) mask8(pq[t][j], kv, k - off);
        }
    };
    auto as_tile = [&](const auto &q) {
        if constexpr (sizeof(q) == 32)
            return make_uint4(pack_bf16x2(__uint_as_float(q[0]), __uint_as_float(q[1])),
                              pack_bf16x2(__uint_as_float(q[2]), __uint_as_float(q[3])),
                              pack_bf16x2(__uint_as_float(q[4]), __uint_as_float(q[5])),
                              pack_bf16x2(__uint_as_float(q[6]), __uint_as_float(q[7])));
        else
            return make_uint4(q[0], q[1], q[2], q[3]);
    };
    auto park = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            *reinterpret_cast<uint4 *>(cb + (size_t)(lr + 8 * j) * PITCH + seg * 16) = as_tile(xq[j]);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const uint4 p = as_tile(pq[t][j]);
                *reinterpret_cast<uint4 *>(cb + (size_t)(32 + t * 32 + lr + 8 * j) * PITCH + seg * 16) = p;
                if constexpr (PF32) {
                    const int k = k0 + seg * EL;
                    if (st == 0 && pval[t][j] && k < kend) {
                        TC *po = static_cast<TC *>(src.phi_out) + (size_t)(dbase + t * 32 + lr + 8 * j) * nC + k;
                        if constexpr (!RAG) {
                            *reinterpret_cast<uint4 *>(po) = p;
                        } else if (k + EL <= nC) {
                            st16_any<false>(po, p.x, p.y, p.z, p.w);
                        } else {  // the last piece of a ragged row
                            const uint32_t w4[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
                            for (int e = 0; e < EL; e++)
                                if (k + e < nC) po[e] = __builtin_bit_cast(TC, (typename std::conditional<EXACT, uint32_t, uint16_t>::type)(EXACT ? w4[e * 4 / EL] : w4[e / 2] >> (16 * (e & 1))));
                        }
                    }
                }
            }
        }
    };

    f32x16_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[t][i] = 0.f;
    float ssq = 0.f;

    const int nch = kbeg < kend ? (kend - kbeg + CH - 1) / CH : 0;
    int kc = kbeg + (nch ? st % nch : 0) * CH;  // first chunk
    if (nch) fetch(kc);
    if constexpr (PF32)
        if (item == 0 && blockIdx.y == 0) gather_small(src, threadIdx.x, 64 * NW, D);
    MHC_PHASE_ADD(kPhaseProjFwd, pwg, 0, pclk);
    for (int it = 0; it < nch; it++) {
        park(kc);
        kc = kc + CH < kend ? kc + CH : kbeg;
        // (a wave's LDS accesses complete in order; the fence keeps the compiler from moving the
        // fragment reads above the writes of its own tile)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        MHC_PHASE_ADD(kPhaseProjFwd, pwg, 1, pclk);
        if (it + 1 < nch) fetch(kc);  // in flight while this chunk is multiplied
#pragma unroll
        for (int u = 0; u < 4; u++) {
            // fragment of k-step u: lane (row, kh) holds the 16 bytes at u*32 + kh*16 of its row
            const uint4 av = *reinterpret_cast<const uint4 *>(cb + (size_t)row * PITCH + u * 32 + kh * 16);
            const uint32_t w4[4] = {av.x, av.y, av.z, av.w};
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const uint4 bv = *reinterpret_cast<const uint4 *>(cb + (size_t)(32 + t * 32 + row) * PITCH + u * 32 + kh * 16);
                if constexpr (EXACT) {
                    // four products of depth 2: product i contracts element i of both lane halves' pieces
                    const uint32_t b4[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(w4[i]), __uint_as_float(b4[i]), acc[t], 0, 0, 0);
                } else {
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, av), __builtin_bit_cast(bf16x8_t, bv),
                                                                    acc[t], 0, 0, 0);
                }
            }
            if (blockIdx.y == 0) {  // sum of squares; bf16: v_dot2c_f32_bf16, two elements per instruction
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (EXACT) {
                        ssq = fmaf(__uint_as_float(w4[i]), __uint_as_float(w4[i]), ssq);
                    } else {
                        const bf16x2_t pr = __builtin_bit_cast(bf16x2_t, w4[i]);
                        ssq = __builtin_amdgcn_fdot2_f32_bf16(pr, pr, ssq, false);
                    }
                }
            }
        }
        MHC_PHASE_ADD(kPhaseProjFwd, pwg, 2, pclk);
    }
    __syncthreads();  // every wave is done with its chunk tile: the memory becomes the cross-wave buffer
    ssq = xor32_add(ssq);  // both K halves of the row

    // cross-wave sum: every wave parks its tiles in LDS, then wave w adds and writes its 16 / NW accumulator
    // registers of every tile, wave 0 also x^2
    constexpr int R = NT * 16 + 1;
    {
        float *dst = lds + (size_t)wave * R * 64;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) dst[(t * 16 + i) * 64 + lane] = acc[t][i];
        dst[(R - 1) * 64 + lane] = ssq;
    }
    __syncthreads();
    // accumulator layout of the 32x32 tile: lane -> column (lane & 31),
    // register i -> row 8 * (i / 4) + 4 * (lane / 32) + (i % 4)
    float *out = Ppart + (size_t)ks * B * DP;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int d = dbase + t * 32 + row;
#pragma unroll
        for (int q = 0; q < 16 / NW; q++) {
            const int i = 16 / NW * wave + q;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) v += lds[((size_t)w * R + t * 16 + i) * 64 + lane];
            const int bs = st * 32 + 8 * (i >> 2) + 4 * kh + (i & 3);
            if (bs < B && d < DP) out[(size_t)bs * DP + d] = d < D ? v : 0.f;  // padded rows stay zero
        }
    }
    if (wave == 0 && blockIdx.y == 0 && kh == 0 && bvalid) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) v += lds[((size_t)w * R + R - 1) * 64 + lane];
        ssqpart[(size_t)ks * B + b] = v;
    }
    MHC_PHASE_ADD(kPhaseProjFwd, pwg, 3, pclk);
}

// --------------------------------------------------------------------------------------------
// MFMA path for wide projections (phi is the big operand, n > 8).
//
// Loads where every lane addresses a different row (the MFMA operand layout) are served at a
// fraction of the L1 rate, so here both operands are fetched with row-contiguous loads (8 lanes
// per 128-byte line), parked in LDS and read back in MFMA layout.
//   workgroup tile: 128 samples x (NT * 64) projection rows, K chunks of 64 elements
//   NWM x NWN waves: a wave owns 128 / NWM samples x NT*32 rows.  Eight waves (4 x 2, one 32 x 32
//   accumulator tile each at NT = 1) are 12 % faster than four with two tiles each (sixteen waves on
//   a 128 x 128 tile gain another 3 % at D = 1088 with exactly 24 K slabs and lose with any other
//   count; not taken): the kernel is
//   bound by its own pipeline (global loads, LDS parking, LDS reads and MFMAs take turns behind one
//   barrier per chunk), and two waves per SIMD let one wave's MFMAs run under the other's LDS reads.
//   P chunks of global loads are in flight per thread (register FIFO) ahead of the chunk being
//   multiplied; LDS is double-buffered, one barrier per chunk.
// Workgroups that read the same K slab sit on the same XCD (workgroup id modulo 8 selects the
// XCD, every XCD takes the same number of consecutive work items): the slab of x is pulled into that
// L2 once and the other row groups hit it there.
// grid.x = groups * sample_groups * KS rounded up to a multiple of 8
// --------------------------------------------------------------------------------------------
constexpr int kWideLd = 72;  // LDS row stride in bf16 elements: 128 data bytes + 16 pad

// PF32: phi comes from the caller's fp32 matrices, see PhiSrc
template <int NT, int P, int NWM = 2, int NWN = 2, bool PF32 = false>
__global__ __launch_bounds__(64 * NWM * NWN) void proj_fwd_wide_kernel(const bf16_t *__restrict__ x,
                                                            const bf16_t *__restrict__ phi,
                                                            float *__restrict__ Ppart,
                                                            float *__restrict__ ssqpart, int B,
                                                            int D, int DP, int nC, int groups,
                                                            int sgroups, int KS,
                                                            int cpk /* chunks per K slab */, PhiSrc src) {
    static_assert(P % 2 == 0, "buffer parity is tied to the FIFO slot");
    constexpr int R = NT * 32 * NWN;   // projection rows per workgroup
    constexpr int NTHR = 64 * NWM * NWN;     // NWM x NWN waves: a wave owns 128 / NWM samples x NT*32 rows
    constexpr int MT = 4 / NWM;              // 32-sample tiles per wave
    constexpr int XJ = 128 * 8 / NTHR;       // 16-byte segments of the x tile per thread
    constexpr int PJ = R * 8 / NTHR;         // same for the phi tile
    constexpr int RSTEP = NTHR / 8;          // rows covered by one round of the workgroup's loads
    extern __shared__ __align__(16) bf16_t lds_w[];  // [2][128 + R][kWideLd]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 31, kh = lane >> 5;
    const int wm = wave / NWN, wn = wave % NWN;
    // work item = (K slab, sample group, row group), rows fastest.  Workgroup ids go round the 8 XCDs,
    // so XCD j takes the contiguous items [j * per_xcd, (j + 1) * per_xcd): the same number on every
    // XCD, and the items that share a slab of x sit on one XCD (two where a slab straddles the border).
    const int items = groups * sgroups * KS, per_xcd = (items + 7) >> 3;
    const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || item >= items) return;  // whole workgroup, before any barrier
    const int group = item % groups;
    const int sg = (item / groups) % sgroups;
    const int ks = item / (groups * sgroups);
    const int nch_all = (nC + 63) / 64;
    const int cbeg = ks * cpk, cend = min(cbeg + cpk, nch_all);
    const bool want_ssq = group == 0;

    // global -> register stage: thread owns segment `seg` of rows lrow + 32 j
    const int lrow = tid >> 3, seg = tid & 7;
    const uint4 *xg[XJ], *pg[PJ];
    bool xv[XJ], pv[PJ];
#pragma unroll
    for (int j = 0; j < XJ; j++) {
        const int b = sg * 128 + lrow + RSTEP * j;
        xv[j] = b < B;
        xg[j] = reinterpret_cast<const uint4 *>(x + (size_t)(xv[j] ? b : 0) * nC) + seg;
    }
#pragma unroll
    for (int j = 0; j < PJ; j++) {
        const int d = group * R + lrow + RSTEP * j;
        pv[j] = d < D;
        if constexpr (PF32) pg[j] = reinterpret_cast<const uint4 *>(phi_src_row(src, pv[j] ? d : 0, nC)) + 2 * seg;
        else pg[j] = reinterpret_cast<const uint4 *>(phi + (size_t)(pv[j] ? d : 0) * nC) + seg;
    }
    // No per-lane predicate on the loads: rows beyond B / D alias row 0 (their products are never
    // stored) and nC % 64 == 0, so a loaded value is not touched until it is parked in LDS and
    // the loads of all P slots stay in flight.
    constexpr int PS = PF32 ? 2 : 1;            // 16-byte pieces per segment of phi
    uint4 rg[P][XJ + PJ * PS];  // per slot: XJ segments of x, then PJ of phi
    auto issue = [&](int slot_, int c) {
#pragma unroll
        for (int j = 0; j < PJ; j++)
#pragma unroll
            for (int h = 0; h < PS; h++) rg[slot_][XJ + j * PS + h] = pg[j][c * 8 * PS + h];
#pragma unroll
        for (int j = 0; j < XJ; j++) rg[slot_][j] = xg[j][c * 8];
    };

    f32x16_t acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[m][t][i] = 0.f;
    float ssq[XJ];
#pragma unroll
    for (int j = 0; j < XJ; j++) ssq[j] = 0.f;

    // park slot j in LDS buffer j & 1, then multiply that buffer; with prefetch, `next` is the
    // chunk whose loads refill the slot
    auto step = [&](int j, int cur, int next, auto prefetch) {
        bf16_t *xs = lds_w + (size_t)(j & 1) * (128 + R) * kWideLd;
        bf16_t *ps = xs + 128 * kWideLd;
#pragma unroll
        for (int q = 0; q < XJ; q++)
            *reinterpret_cast<uint4 *>(xs + (lrow + RSTEP * q) * kWideLd + seg * 8) = rg[j][q];
#pragma unroll
        for (int q = 0; q < PJ; q++) {
            uint4 p = rg[j][XJ + q * PS];
            if constexpr (PF32) {
                const uint4 p2 = rg[j][XJ + q * PS + 1];
                p = make_uint4(pack_bf16x2(__uint_as_float(p.x), __uint_as_float(p.y)),
                               pack_bf16x2(__uint_as_float(p.z), __uint_as_float(p.w)),
                               pack_bf16x2(__uint_as_float(p2.x), __uint_as_float(p2.y)),
                               pack_bf16x2(__uint_as_float(p2.z), __uint_as_float(p2.w)));
                if (sg == 0 && pv[q])  // every (row group, K slab) stores its part of the packed phi once
                    *reinterpret_cast<uint4 *>(static_cast<bf16_t *>(src.phi_out) + (size_t)(group * R + lrow + RSTEP * q) * nC + cur * 64 + seg * 8) = p;
            }
            *reinterpret_cast<uint4 *>(ps + (lrow + RSTEP * q) * kWideLd + seg * 8) = p;
        }
        if (want_ssq) {
#pragma unroll
            for (int q = 0; q < XJ; q++) {
                const uint32_t w4[4] = {rg[j][q].x, rg[j][q].y, rg[j][q].z, rg[j][q].w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float lo = bf16lo_to_f32(w4[i]), hi = bf16hi_to_f32(w4[i]);
                    ssq[q] += lo * lo + hi * hi;
                }
            }
        }
        __syncthreads();
        if constexpr (decltype(prefetch)::value) issue(j, next);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            bf16x8_t af[MT], bfr[NT];
#pragma unroll
            for (int m = 0; m < MT; m++)
                af[m] = *reinterpret_cast<const bf16x8_t *>(
                    xs + (wm * 32 * MT + m * 32 + row) * kWideLd + s * 16 + kh * 8);
#pragma unroll
            for (int t = 0; t < NT; t++)
                bfr[t] = *reinterpret_cast<const bf16x8_t *>(
                    ps + (wn * NT * 32 + t * 32 + row) * kWideLd + s * 16 + kh * 8);
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    acc[m][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[m], bfr[t], acc[m][t], 0, 0, 0);
        }
    };

    if constexpr (PF32)
        if (item == 0) gather_small(src, tid, NTHR, D);
    // prologue: fill the FIFO (indices beyond the slab are clamped: redundant, never consumed)
#pragma unroll
    for (int j = 0; j < P; j++) issue(j, min(cbeg + j, cend - 1));
    int c = cbeg;
    for (; c + P <= cend; c += P) {
#pragma unroll
        for (int j = 0; j < P; j++) step(j, c + j, min(c + j + P, cend - 1), std::true_type{});
    }
    const int rem = cend - c;  // < P chunks left, all already in flight
#pragma unroll
    for (int j = 0; j < P - 1; j++)
        if (j < rem) step(j, c + j, 0, std::false_type{});

    // accumulator layout of a 32x32 tile: lane -> column (lane & 31),
    // register i -> row 8 * (i / 4) + 4 * (lane / 32) + (i % 4)
    float *out = Ppart + (size_t)ks * B * DP;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int d = group * R + wn * NT * 32 + t * 32 + row;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int bs = sg * 128 + wm * 32 * MT + m * 32 + 8 * (i >> 2) + 4 * kh + (i & 3);
                if (bs < B && d < D) out[(size_t)bs * DP + d] = acc[m][t][i];
            }
        }
    if (want_ssq) {
#pragma unroll
        for (int j = 0; j < XJ; j++) {
            float v = ssq[j];  // the 8 lanes of one row are consecutive
            v += __shfl_xor(v, 1, kWave);
            v += __shfl_xor(v, 2, kWave);
            v += __shfl_xor(v, 4, kWave);
            if (seg == 0 && xv[j]) ssqpart[(size_t)ks * B + sg * 128 + lrow + RSTEP * j] = v;
        }
    }
}

template <int NT, int P, int NWM = 2, int NWN = 2, bool PF32 = false>
static hipError_t launch_wide(const void *x, const void *phi, float *Ppart, float *ssqpart, int KS,
                              int B, int D, int DP, int nC, hipStream_t stream, const PhiSrc &src = PhiSrc{}) {
    const int sgroups = (B + 127) / 128;
    constexpr int R = NT * 32 * NWN;
    const int groups = (DP + R - 1) / R;
    const int nch_all = (nC + 63) / 64;
    const int cpk = (nch_all + KS - 1) / KS;
    const int grid = 8 * ((groups * sgroups * KS + 7) / 8);
    const size_t smem = sizeof(bf16_t) * 2 * (128 + R) * kWideLd;
    if (hipError_t e = allow_dynamic_lds<&proj_fwd_wide_kernel<NT, P, NWM, NWN, PF32>>(smem); e != hipSuccess) return e;
    proj_fwd_wide_kernel<NT, P, NWM, NWN, PF32><<<grid, 64 * NWM * NWN, smem, stream>>>(
        static_cast<const bf16_t *>(x), static_cast<const bf16_t *>(phi), Ppart, ssqpart, B, D, DP,
        nC, groups, sgroups, KS, cpk, src);
    return hipGetLastError();
}

// --------------------------------------------------------------------------------------------
// shape-dependent split and launch
// --------------------------------------------------------------------------------------------
static int mfma_nt(int n) {
    const int tiles = padded_D(n) / 32;
    return tiles <= 4 ? tiles : 2;
}

// wide projections (more than four 32-row tiles) with whole 64-element K chunks take the
// LDS-staged kernel
static bool use_wide(int n, int C) { return padded_D(n) / 32 > 4 && (n * C) % 64 == 0; }

// fp32 tier, n <= 8: the narrow kernel in fp32 arithmetic
static bool use_exact(int x_dtype, int phi_dtype, int n, int C) {
    return n <= 8 && x_dtype == kF32 && phi_dtype == kF32 && n * C >= 256;
}

int proj_fwd_ksplit(int x_dtype, int phi_dtype, int B, int n, int C) {
    // The generic path always uses one split.  MFMA path: enough workgroups to fill 256 CUs
    // several times over (the K loop is latency-bound per wave), at least 64 K elements per wave.
    const bool exact = use_exact(x_dtype, phi_dtype, n, C);
    if (!exact && gemm_f32_supported(x_dtype, phi_dtype, n, C)) return gemm_f32_proj_ksplit(B, n, C, kMaxKSplit);
    if (!exact && !use_mfma(x_dtype, phi_dtype, n, C)) return 1;
    const int nC = n * C, DP = padded_D(n);
    if (!exact && use_wide(n, C)) {
        // Workgroups = (64-row groups) x (128-sample tiles) x splits.  The chip has 256 CUs and a workgroup
        // (8 waves) loads one: the count that fills every CU once, or twice where that still keeps the
        // splits within the 24 that the coefficient kernel sums in one round of loads, beats the counts in
        // between, which leave some CUs with twice the work of others
        // (forward us, B n C: 128 32 1280  15 splits 41.8 | 24: 43.0 | 30: 44.2 | 16: 48.7;
        //  256 32 1280  15: 62.1 | 12: 66.2 | 7: 67.5;  512 12 512  16: 28.1 | 3: 35.8).
        const int wgs = ((DP + 63) / 64) * ((B + 127) / 128);
        int ks = 512 / wgs <= 24 ? 512 / wgs : 256 / wgs;
        if (ks > 24) ks = 24;
        const int cap_chunks = nC / 64 / 8;  // a slab is at least 8 chunks
        if (ks > cap_chunks) ks = cap_chunks;
        // the partial sums (written here, read by the coefficient kernel) stay below the bytes streamed,
        // unless that would leave half the CUs without a workgroup
        const int cap_bytes = (int)((2.0 * B * nC + 2.0 * DP * nC) / (8.0 * B * DP));
        if (ks > cap_bytes) {
            const int half_chip = (128 + wgs - 1) / wgs;
            ks = cap_bytes > (ks < half_chip ? ks : half_chip) ? cap_bytes : (ks < half_chip ? ks : half_chip);
        }
        if (ks < 1) ks = 1;
        if (const int forced = tuning_get(kTuneSpareB); forced > 0) ks = forced;  // experiment hook
        return ks;
    }
    const int tiles_s = (B + 31) / 32;
    const int groups = DP / 32 / mfma_nt(n);
    int ks = (1024 + tiles_s * groups - 1) / (tiles_s * groups);
    const int chunk = exact ? 32 : 64;
    const double esize = exact ? 4.0 : 2.0;
    const int cap_slab = nC / (4 * chunk);
    // partial sums (KS * B * DP fp32) at most ~1/3 of the bytes this kernel streams (x and phi)
    const int cap_bytes = (int)(0.35 * (esize * B * nC + esize * DP * nC) / (4.0 * B * DP));
    if (ks > cap_slab) ks = cap_slab;
    if (ks > cap_bytes) ks = cap_bytes;
    // the fused forward kernel (n <= 8) sums that many splits with loads that it issues ahead of the sample's
    // tile; more splits would queue behind the tile.  (The cap is that of bf16 rows: with 4-byte x a thread has two
    // chunks from C = 1025 on and sums 16 at once, the rest in a second round.  Capped at 16 instead: float32 storage of
    // bf16 arithmetic n=4 C=1280 B=512 14.0 -> 13.2 us, but float32 B=200 12.2 -> 13.5, 320 13.4 -> 14.4.)
    if (const int cap = fwd_splits_summed_at_once(n, C); n <= 8 && ks > cap) ks = cap;
    if (ks > 64) ks = 64;
    if (ks < 1) ks = 1;
    // splits with work when ks are asked for (see below)
    auto effective = [&](int k) { const int s_ = round_up((nC + k * 4 - 1) / (k * 4), chunk); return (nC + 4 * s_ - 1) / (4 * s_); };
    if (mfma_nt(n) == 1) {
        // one row tile of phi: a multiple of 8 gives every XCD whole slabs of phi (forward us, default count -> 8:
        // B=8192 C=2560 4: 112.7 -> 107.5, B=3001 C=2560 5: 43.3 -> 41.9, fp32 B=2560 C=1280 13: 41.4 -> 38.8)
        const int k8 = ks < 8 ? 8 : ks / 8 * 8;
        if (ks >= 4 && k8 <= cap_slab && effective(k8) == k8) ks = k8;
    } else if (const int wgs = tiles_s * groups; wgs * effective(ks) > 256) {
        // more row tiles (two workgroups per CU): once per CU instead of once and a bit, but not below 8 (forward us,
        // n=8 C=1280: bf16 B=1024 16 -> 8 splits 33.7 -> 30.1, B=2048 49.2 -> 44.8, fp32 B=512 20 -> 16 36.9 -> 30.6)
        const int k = 256 / wgs > 8 ? 256 / wgs : 8;
        if (k < ks) ks = k;
    }
    if (const int forced = tuning_get(kTuneSpareB); forced > 0) ks = forced;  // experiment hook
    // a wave's share is whole 64-element chunks (launch_mfma): with that share fixed, only as many
    // splits as have work (B=1280 n=4 C=2560: 16 splits of 4 x 192 elements would leave the last two
    // and a half empty; 14 do the same work and the forward sums two partial rows fewer per sample)
    const int sub = round_up((nC + ks * 4 - 1) / (ks * 4), chunk);
    ks = (nC + 4 * sub - 1) / (4 * sub);
    return ks;
}

template <typename TX, typename TP>
static hipError_t launch_generic(const void *x, const void *phi, float *Ppart, float *ssqpart, int B,
                                 int D, int DP, int nC, hipStream_t stream) {
    dim3 grid(B, (D + kGenDB - 1) / kGenDB);
    proj_fwd_generic_kernel<TX, TP><<<grid, 256, 0, stream>>>(
        static_cast<const TX *>(x), static_cast<const TP *>(phi), Ppart, ssqpart, B, D, DP, nC);
    return hipGetLastError();
}

// Waves per workgroup of the narrow kernel.  Few samples and a long row (the split count is capped by what the
// forward kernel sums in one round): a wave's chunks are one dependent round trip to memory each, so eight waves
// share the slab where that shortens the walk and at most one workgroup falls to a CU anyway (147 KB of LDS at n = 8).
// Kernel us, four -> eight: n=6 B=2 C=2752 11.3 -> 10.3, n=8 B=64 C=3072 17.0 -> 15.3, n=4 B=64 C=4096 7.2 -> 6.3.
static int narrow_waves(int workgroups, int KS, int nC, int chunk) {
    return workgroups <= 256 && (nC + KS * 4 - 1) / (KS * 4) > chunk ? 8 : 4;
}

template <int NT, bool XF32 = false, bool PF32 = false, bool EXACT = false, bool RAG = false, int NW = 4>
static hipError_t launch_mfma(const void *x, const void *phi, float *Ppart, float *ssqpart, int KS,
                              int B, int D, int DP, int nC, hipStream_t stream, const PhiSrc &src = PhiSrc{}) {
    if constexpr (NT <= 3 && !RAG) {
        if (nC % (EXACT ? 4 : 8) != 0) {
            if constexpr (XF32) return hipErrorInvalidValue;  // fp32 storage: whole pieces only (capi.hip)
            else return launch_mfma<NT, XF32, PF32, EXACT, true>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
        }
    }
    const int tiles_s = (B + 31) / 32;
    const int groups = (DP / 32 + NT - 1) / NT;
    constexpr int kChunk = EXACT ? 32 : 64;
    if constexpr (NT <= 3 && !RAG && NW == 4) {
        // (n <= 8: counted without the groups.  Row tiles in workgroups of their own (narrow_nt) add up in the same order as all
        // in one; four waves, whose chains are twice as long, are off by 14 to 28 % more in float32 and 2 to 8 % in bf16, for 0 to 10 % of time)
        if (narrow_waves(tiles_s * KS * (DP <= 96 ? 1 : groups), KS, nC, kChunk) == 8)
            return launch_mfma<NT, XF32, PF32, EXACT, RAG, 8>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
    }
    const int sub = round_up((nC + KS * NW - 1) / (KS * NW), kChunk);  // whole chunks: 128-byte lines
    dim3 grid(8 * ((tiles_s * KS + 7) / 8), groups);
    const size_t smem_chunks = sizeof(bf16_t) * NW * (1 + NT) * 32 * kNarrowPitch;
    const size_t smem_sum = sizeof(float) * NW * (NT * 16 + 1) * 64;
    const size_t smem = smem_chunks > smem_sum ? smem_chunks : smem_sum;
    if (hipError_t e = allow_dynamic_lds<&proj_fwd_mfma_kernel<NT, XF32, PF32, EXACT, RAG, NW>>(smem); e != hipSuccess) return e;
    proj_fwd_mfma_kernel<NT, XF32, PF32, EXACT, RAG, NW><<<grid, 64 * NW, smem, stream>>>(x, phi, Ppart,
                                                                 ssqpart, B, D, DP, nC, tiles_s, KS, sub, src);
    return hipGetLastError();
}

// Where the projection reads the caller's fp32 parameters itself.  In a narrow projection every tile of 32
// samples reads all of phi, so fp32 doubles what the tiles pull through L1 and a large batch pays more than the
// packing launch costs; the more row tiles of phi (n), the sooner.  In a wide one a workgroup covers 128 samples
// and every element of phi is read once per 128.  Forward in graphs of ten, packing launch -> in the projection (us):
//   n=4 C=1280: B=8 12.3 -> 10.7, 320 13.4 -> 11.9, 4096 37.1 -> 36.1;  C=2560: B=3001 43.8 -> 43.4, 8192 113.6 -> 116.4
//   n=6 C=1280: B=1024 27.2 -> 26.7, 2048 41.2 -> 42.5
//   n=8 C=1280: B=256 17.9 -> 18.3, 512 23.0 -> 23.5, 1024 34.0 -> 36.5  (and one launch less on the host)
//   n=32 C=1280: B=64 89.0 -> 66.5, 128 91.5 -> 75.0, 256 112.5 -> 109.5, 384 137.9 -> 140.2;  n=16: B=128 39.2 -> 30.6
// The wide case is decided on whole steps, forward + backward in graphs of ten: each row of 128 samples reads the fp32
// phi again, and in a step dphi (as many bytes) has gone through the memory-side cache (256 MB) since the last one.
//   n=32 C=1280 (178 MB of phi): B=32 170 -> 150, 64 176 -> 154, 128 188 -> 175, 192 261 -> 253, 256 272 -> 275, 320 350 -> 367
//   n=24 C=1280 (77 MB): B=128 120 -> 106, 320 209 -> 195;  n=16 (24 MB): B=128 87 -> 80, 320 139 -> 128
bool proj_fwd_gathers(const ParamGather &g, int x_dtype, int B, int n, int C) {
    auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (g.phi_dtype != kF32 || !al16(g.phi[0]) || !al16(g.phi[1]) || !al16(g.phi[2])) return false;
    if (g.out_dtype == kF32) return use_exact(x_dtype, kF32, n, C) && B <= 4096 && tuning_get(kTuneGather) != 1;
    if (!use_mfma(x_dtype, kBF16, n, C)) return false;
    // the narrow kernel finds the rows of pre and post among its first 16 (n <= 8); beyond, rows that are not
    // whole 64-element chunks keep the packing launch
    if (!use_wide(n, C) && n > 8) return false;
    if (const int hook = tuning_get(kTuneGather)) return hook == 2;
    // (128 MB: phi and dphi together fit that cache)
    if (use_wide(n, C)) return B <= ((size_t)padded_D(n) * n * C * 4 > (128u << 20) ? 192 : 320);
    const int nt = mfma_nt(n);
    return B <= (nt == 1 ? 4096 : (nt == 2 ? 1024 : 512));
}

// Row tiles of phi per workgroup of the narrow kernel, n = 5 .. 8: one, in as many groups, where all of them (two or three) would
// leave the chip few workgroups that each walk three times the bytes, and while reading x once per group costs less than that.
// Forward us, all tiles -> one: n=8 B=1 C=4096 14.8 -> 12.3, 16 2560 15.2 -> 12.8, 100 1280 12.9 -> 11.4, 100 2560 15.9 -> 14.5, 150 4096
// 17.1 -> 15.9, 600 512 13.7 -> 12.9; n=6 B=32 C=1024 11.4 -> 10.7; n=5 B=10 C=777 13.7 -> 12.8; float32 n=8 B=16 C=2560 23.6 -> 16.2,
// 100 1280 20.1 -> 17.3, 100 2560 25.1 -> 21.0, 150 4096 30.5 -> 26.1.  Beyond: n=6 B=2000 C=1024 (25 MB) 20.6 -> 21.3, n=8 B=700 C=2560
// (29 MB) 26.3 -> 27.7, 2000 2560 54.9 -> 70.2.
static int narrow_nt(int x_dtype, int B, int n, int C, int KS) {
    const int tiles = mfma_nt(n), wgs = (B + 31) / 32 * KS;
    // (eight waves: 74 KB of LDS, two workgroups per CU; n=8, all tiles -> one: float32 B=600 C=512 20.6 -> 21.5, B=512 C=1024
    // 22.2 -> 24.3, bf16 B=800 C=512 14.0 -> 15.3)
    const int most = narrow_waves(wgs, KS, n * C, x_dtype == kF32 ? 32 : 64) == 8 ? 512 : 1024;
    const bool few = wgs * tiles <= most && (size_t)B * n * C * (x_dtype == kBF16 ? 2 : 4) <= (22u << 20);
    return n <= 8 && few ? 1 : tiles;
}

hipError_t launch_proj_fwd(const void *x, int x_dtype, const void *phi, int phi_dtype, float *Ppart,
                           float *ssqpart, int KS, int B, int n, int C, hipStream_t stream,
                           const ParamGather *gather) {
    const int nC = n * C, D = n * n + 2 * n, DP = padded_D(n), nt = narrow_nt(x_dtype, B, n, C, KS);
    if (gather) {
        const PhiSrc src = phi_src_of(*gather, n);
        if (x_dtype == kF32) {
            switch (nt) {
                case 1: return launch_mfma<1, false, true, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
                case 2: return launch_mfma<2, false, true, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
                case 3: return launch_mfma<3, false, true, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
                default: return hipErrorInvalidValue;
            }
        }
        if (use_wide(n, C)) return launch_wide<1, 2, 4, 2, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
        if (n > 8) return hipErrorInvalidValue;  // see proj_fwd_gathers
        const bool xf32 = x_dtype == kF32AsBF16;
        switch (nt) {
            case 1: return xf32 ? launch_mfma<1, true, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src)
                                : launch_mfma<1, false, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
            case 2: return xf32 ? launch_mfma<2, true, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src)
                                : launch_mfma<2, false, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
            case 3: return xf32 ? launch_mfma<3, true, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src)
                                : launch_mfma<3, false, true>(x, nullptr, Ppart, ssqpart, KS, B, D, DP, nC, stream, src);
            default: return hipErrorInvalidValue;
        }
    }
    if (use_mfma(x_dtype, phi_dtype, n, C)) {
        if (x_dtype == kF32AsBF16) {  // fp32 storage, rounded on load: the narrow kernel only (n <= 8)
            switch (use_wide(n, C) ? 0 : nt) {
                case 1: return launch_mfma<1, true>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
                case 2: return launch_mfma<2, true>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
                case 3: return launch_mfma<3, true>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
                default: return hipErrorInvalidValue;
            }
        }
        if (use_wide(n, C)) return launch_wide<1, 2, 4>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
        switch (nt) {
            case 1: return launch_mfma<1>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
            case 2: return launch_mfma<2>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
            case 3: return launch_mfma<3>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
            default: return launch_mfma<4>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
        }
    }
    if (use_exact(x_dtype, phi_dtype, n, C)) {
        switch (nt) {
            case 1: return launch_mfma<1, false, false, true>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
            case 2: return launch_mfma<2, false, false, true>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
            case 3: return launch_mfma<3, false, false, true>(x, phi, Ppart, ssqpart, KS, B, D, DP, nC, stream);
            default: return hipErrorInvalidValue;
        }
    }
    if (gemm_f32_supported(x_dtype, phi_dtype, n, C))
        return launch_gemm_f32_proj(static_cast<const float *>(x), static_cast<const float *>(phi), Ppart,
                                    ssqpart, KS, B, n, C, stream);
    if (KS != 1) return hipErrorInvalidValue;  // the generic path produces exactly one split
    if (x_dtype == kF32 && phi_dtype == kF32) return launch_generic<float, float>(x, phi, Ppart, ssqpart, B, D, DP, nC, stream);
    if (x_dtype == kF32 && phi_dtype == kBF16) return launch_generic<float, bf16_t>(x, phi, Ppart, ssqpart, B, D, DP, nC, stream);
    if (x_dtype == kBF16 && phi_dtype == kF32) return launch_generic<bf16_t, float>(x, phi, Ppart, ssqpart, B, D, DP, nC, stream);
    return launch_generic<bf16_t, bf16_t>(x, phi, Ppart, ssqpart, B, D, DP, nC, stream);
}

}  // namespace mhc
