// Backward, second (and last) launch behind the sample-resident kernel (bwd_resident.hip), bf16 tier,
// D <= 96 (n <= 8): a workgroup owns a slab of 32 columns of x_flat / phi for ALL samples, so that
//
//   dphi[d, k] = sum_b dP[b, d] x_flat[b, k]                      (reference ops.py:332-334)
//
// is finished here without batch-split partial sums, and completes dx,
//
//   dx[b, k] = dxp[b, k] + sum_d dP[b, d] phi[d, k] - cx[b] x_flat[b, k]      (reference ops.py:336-351)
//
// where dxp = M^T dy + Hpre (x) da was left by the first launch, in the dx buffer or in fp32 beside it.  A few extra
// workgroups (one more grid row) add up dw, dbias and dalpha (batch_sums.h), so the backward needs no
// third launch.
//
// Samples are walked in blocks of 128, 256 or 384 (4, 8 or 12 waves of 32 samples).  Per block every thread requests its 16-byte
// chunks of x and dxp up front (row-contiguous, next block in flight while this one is worked on); x is
// parked in LDS as [sample][column] and read back transposed as the B operand of
// v_mfma_f32_32x32x16_bf16 (the contraction of dphi runs over samples, the strided axis).  Wave w owns a
// quarter of the block's samples: it accumulates their share of every dphi tile (dP^T from global memory in fragment
// order, rounded value + remainder), forms dP phi for them (phi fragments from the slab in LDS),
// hands the result through a wave-private LDS tile to a row-major epilogue - 16-byte loads of dxp,
// 16-byte stores of dx - and at the very end the four waves' dphi shares are summed through LDS.
#include "launchers.h"

#include <type_traits>
#include "mhc_common.h"
#include "phase_profiler.h"

namespace mhc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

struct ProjAddxArgs {
    const void *x;       // [B][nC], bf16 or (F32) fp32 rounded to bf16 on its way into LDS
    const bf16_t *phi;   // [D][nC]
    const bf16_t *dPb;   // dP, fragment-major (frag_dpb); columns >= D are zero
    const bf16_t *dPT;   // dP^T hi and lo bf16 planes, fragment-major (frag_dpt); rows >= D, columns >= B zero
    const float *cx;     // [B]
    float *dphi;         // [D][nC], one such plane per batch split
    const void *dxp;     // [B][nC]: dx itself, or fp32 (kAxFine, kAxRagged)
    void *dx;            // [B][nC], stored like x
    int B, BP, D, DP, nC;
    int per_split;       // samples of a batch split (whole blocks); blockIdx.y < splits
    int tail_row;        // first blockIdx.y of the workgroups that compute `tail` (-1: none)
    int tail_rows;       // samples per workgroup of the tail (all of them, or a part with partial sums as the result)
    int tail_parts;
    BatchSumArgs tail;
};

// Columns per workgroup of the batch sums: 16 leave sixteen row groups in four waves (a walk of 1000 samples is 4
// rounds of loads; with 64 columns and four groups it was 16, longer than the slabs': B=789 n=8 C=1984 30.1 -> 27.0 us)
constexpr int kAxSumCols = 16;
constexpr int kAxSumRows = 128;    // samples per part of the sums beside a split batch
constexpr int kAxKW = 32;          // slab width (columns)
constexpr int kAxLD = kAxKW + 8;   // LDS pitch of the bf16 tiles (elements): rows stay 16-byte aligned
constexpr int kAxLDO = kAxKW + 4;  // LDS pitch of the fp32 tile of dP phi
constexpr int kAxLDR = 36;         // LDS pitch of the dphi tiles in the final cross-wave sum (rows 16-byte aligned)

// NTD: 32-row tiles of dphi (D <= 32 NTD).  SPW: samples a wave owns per block (32 or 64; a block is
// 4 SPW samples).  PFOP: the dP operands of the next block are requested a block ahead like x and dxp.
// Measured at B=320, C=1280, n=4 (backward, graphs of ten): SPW 32 without / with PFOP 16.1 / 16.1 us,
// SPW 64 without PFOP 19.1 us, with PFOP 23.0 us (registers spill).
// ST: how the activations are stored and dxp is handed over
//   kAxBf16    bf16, dxp in place (dx is rounded twice)
//   kAxF32     fp32, dxp in place (x is rounded to bf16 for the products and for the -cx x term, as in the bf16
//              storage case; dxp is read and dx written as fp32)
//   kAxFine    bf16, dxp fp32 in a buffer of its own (dx is rounded once)
//   kAxRagged  the same for rows of any length (C % 8 != 0): the last chunk of a row is loaded from nC - 8 on and
//              shifted down; dP in one more bf16 plane each (dphi: three, 24 bits; dP phi: two), so that the
//              gradients are as good as from the fp32 arithmetic of the general kernels (dphi off by 2e-7, with
//              two planes 3e-6; B=333 n=3 C=1230 backward 19.7 us with two planes and dxp in bf16, 21.9 with
//              three and dxp in fp32, 46.1 in the general kernels; B=130 n=8 C=643 21.1, 33.4, 160.7)
// NW: waves per workgroup (a block is NW * SPW samples).
// SPLIT: blockIdx.y is a batch split (a template argument: with a run-time first sample the compiler keeps fewer
// loads in flight, B=1000 n=6 C=1024 17.2 -> 21.2 us without any split).
enum { kAxBf16 = 0, kAxF32 = 1, kAxFine = 2, kAxRagged = 3 };

template <int NTD, int SPW, bool PFOP, int ST, int NW = 4, bool SPLIT = false>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void proj_bwd_addx_kernel(ProjAddxArgs a) {
    constexpr int NT_ = 64 * NW;  // threads
    constexpr bool F32 = ST == kAxF32, RAG = ST == kAxRagged, P32 = ST != kAxBf16;  // P32: dxp is fp32
    using TS = typename std::conditional<F32, float, bf16_t>::type;
    using TP = typename std::conditional<P32, float, bf16_t>::type;
    constexpr int AW = F32 ? 8 : 4, PW = P32 ? 8 : 4;  // words of an 8-element chunk as stored: of x, of dxp
    constexpr int SBR = NW * SPW;  // samples per block
    constexpr int KS = SPW / 16;   // k-steps (16 samples) of a wave per block = its 16-byte chunks of x and of dxp
    constexpr int TT = SPW / 32;   // 32-sample tiles of a wave per block
    extern __shared__ __align__(16) unsigned char ax_smem[];
    bf16_t *phi_s = reinterpret_cast<bf16_t *>(ax_smem);                 // [32 NTD][LD]
    bf16_t *x_s = phi_s + (size_t)32 * NTD * kAxLD;                       // [SBR][LD]
    float *o_s = reinterpret_cast<float *>(x_s + (size_t)SBR * kAxLD);    // [SBR][LDO]
    float *red_s = reinterpret_cast<float *>(ax_smem);                    // final sum: [NW][NTD][32][LDR], over everything
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (a.tail_row >= 0 && (int)blockIdx.y >= a.tail_row) {
        // the extra rows of the grid: the first workgroups do the batch sums, the others have nothing to do
        const int id = ((int)blockIdx.y - a.tail_row) * (int)gridDim.x + (int)blockIdx.x, part = id / a.tail.nblk;
        if (part >= a.tail_parts) return;
        BatchSumArgs s = a.tail;
        const int r0 = part * a.tail_rows, rows = min(a.tail_rows, a.B - r0);
        s.rows_u = s.rows_dt = rows;
        s.u = static_cast<const float *>(s.u) + (size_t)r0 * s.C;
        s.dt = static_cast<const float *>(s.dt) + (size_t)r0 * (s.D + 3);
        double *red = reinterpret_cast<double *>(ax_smem);
        if constexpr (SPLIT) {  // rows of float64, added up by the launch that follows
            if (s.dw) s.dw = static_cast<double *>(s.dw) + (size_t)part * s.C;
            s.dbias = reinterpret_cast<float *>(reinterpret_cast<double *>(s.dbias) + (size_t)part * (s.D + 3));
            batch_sum_block<NT_ / kAxSumCols, kAxSumCols, false, true>(s, id % s.nblk, tid, red);
        } else {
            batch_sum_block<NT_ / kAxSumCols, kAxSumCols>(s, id % s.nblk, tid, red);
        }
        return;
    }
    // Workgroup ids go round robin over the 8 XCDs (each with its own L2, 128-byte lines).  A slab
    // row of 32 columns is half a line: neighbouring slabs are given to the same XCD (ids x and
    // x + 8 of a group of 16), otherwise two L2s fetch every line of x, dxp and phi.
    const int slab = (blockIdx.x >> 4) * 16 + (blockIdx.x & 7) * 2 + ((blockIdx.x >> 3) & 1);
    const int k0 = slab * kAxKW;
    if (k0 >= a.nC) return;  // ids of the padded grid; the whole workgroup, before any barrier
    const int row = lane & 31, kg = lane >> 5;
    const int D = a.D, nC = a.nC, b_begin = SPLIT ? (int)blockIdx.y * a.per_split : 0, B = SPLIT ? min(a.B, b_begin + a.per_split) : a.B;  // the split's samples
    const int pwg = slab;
    (void)pwg;
    MHC_PHASE_ZERO(kPhaseColSlab, pwg);
    MHC_PHASE_BEGIN(pclk);

    // ---- per-block loads: x for the LDS tile (thread -> chunks tid + 256 u) and, for the epilogue,
    // the chunks of dxp this thread completes: sample SPW wave + lane / 4 + 16 t, chunk lane % 4 ------
    const int ech = lane & 3, erow = SPW * wave + (lane >> 2);
    const int kc = k0 + ech * 8;
    const bool kok = kc < nC;
    // a thread owns the same column chunk in all of its loads (they are multiples of four chunks apart), so the
    // shift of a ragged row is one value per thread
    const int kl = k0 + (tid & 3) * 8;  // the chunk of x and phi
    const int kls = RAG && kl < nC && kl + 8 > nC ? kl + 8 - nC : 0, kcs = RAG && kok && kc + 8 > nC ? kc + 8 - nC : 0;
    // dxp of the next block is requested a block ahead like x, except where that costs the registers that
    // keep two workgroups on a CU (fp32 dxp with a wide projection): there it is requested at the top
    // of its own block and arrives under the matrix-core phase
    constexpr int PS = (P32 && NTD >= 2) ? 1 : 2;
    uint32_t xr[2][KS][AW], pr[PS][KS][PW];
    float cxr[PS][KS];
    const TS *xg = static_cast<const TS *>(a.x);
    TS *dxg = static_cast<TS *>(a.dx);
    const TP *dxpg = static_cast<const TP *>(a.dxp);
    auto load_chunk = [&](const auto *p, auto &q, bool ok) {
        const uint4 v = ldg16<RAG>(p);
        q[0] = ok ? v.x : 0u; q[1] = ok ? v.y : 0u; q[2] = ok ? v.z : 0u; q[3] = ok ? v.w : 0u;
        if constexpr (sizeof(*p) == 4) {
            const uint4 v2 = ldg16<RAG>(p + 4);
            q[4] = ok ? v2.x : 0u; q[5] = ok ? v2.y : 0u; q[6] = ok ? v2.z : 0u; q[7] = ok ? v2.w : 0u;
        }
    };
    auto load_block = [&](int sb, auto slot) {
        constexpr int S = decltype(slot)::value;
#pragma unroll
        for (int u = 0; u < KS; u++) {
            const int ch = tid + u * NT_;
            const int b = sb + (ch >> 2);
            const bool ok = b < B && kl < nC;
            load_chunk(xg + (ok ? (size_t)b * nC + kl - kls : 0), xr[S][u], ok);
        }
        if constexpr (PS == 2) {
#pragma unroll
            for (int t = 0; t < KS; t++) {
                const int b = sb + erow + 16 * t;
                const bool ok = b < B && kok;
                load_chunk(dxpg + (ok ? (size_t)b * nC + kc - kcs : 0), pr[S][t], ok);
                cxr[S][t] = a.cx[b < B ? b : 0];
            }
        }
    };
    auto load_prev = [&](int sb) {  // PS == 1: the block's own dxp chunks
#pragma unroll
        for (int t = 0; t < KS; t++) {
            const int b = sb + erow + 16 * t;
            const bool ok = b < B && kok;
            load_chunk(dxpg + (ok ? (size_t)b * nC + kc - kcs : 0), pr[0][t], ok);
            cxr[0][t] = a.cx[b < B ? b : 0];
        }
    };
    // Operands that come straight from global memory in fragment order: dP^T (rounded value and
    // remainder) of this wave's samples for every dphi tile, and dP of its sample tiles.  Steps and
    // tiles beyond the padded batch read zeros.
    // (the planes that only ragged rows have - the third of dP^T, the second of dP - are fetched where they are used: held
    // from here they spill)
    constexpr int HELD = RAG && NTD == 3 ? 1 : 2;  // planes of dP^T requested here
    const size_t plane = (size_t)a.DP * a.BP;
    auto load_at = [&](int sb, int p, int m, int ks) {
        const int nsteps = a.BP >> 4, step = (sb >> 4) + KS * wave + ks;
        const bool ok = step < nsteps;
        return load16_masked(reinterpret_cast<const uint4 *>(a.dPT + p * plane + (ok ? frag_base(m, nsteps, step) : 0) + lane * 8), ok);
    };
    auto load_av = [&](int sb, int p, int t, int ks) {
        const int tile = (sb >> 5) + TT * wave + t;
        const bool ok = tile < (a.BP >> 5);
        return load16_masked(reinterpret_cast<const uint4 *>(a.dPb + p * plane + (ok ? frag_base(tile, a.DP >> 4, ks) : 0) + lane * 8), ok);
    };
    struct Ops {
        uint4 ah[NTD][KS], al[NTD][KS], av[TT][2 * NTD];
    };
    Ops ops[PFOP ? 2 : 1];
    auto load_ops = [&](int sb, Ops &o) {
        const int step0 = (sb >> 4) + KS * wave, nsteps = a.BP >> 4;
#pragma unroll
        for (int m = 0; m < NTD; m++)
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const bool ok = step0 + ks < nsteps;
                const bf16_t *ap = a.dPT + (ok ? frag_base(m, nsteps, step0 + ks) : 0) + lane * 8;
                o.ah[m][ks] = load16_masked(reinterpret_cast<const uint4 *>(ap), ok);
                if constexpr (HELD == 2)
                    o.al[m][ks] = load16_masked(reinterpret_cast<const uint4 *>(ap + (size_t)a.DP * a.BP), ok);
            }
#pragma unroll
        for (int t = 0; t < TT; t++) {
            const int tile = (sb >> 5) + TT * wave + t;
            const bool ok = tile < (a.BP >> 5);
#pragma unroll
            for (int ks = 0; ks < 2 * NTD; ks++)
                o.av[t][ks] = load16_masked(
                    reinterpret_cast<const uint4 *>(a.dPb + (ok ? frag_base(tile, a.DP >> 4, ks) : 0) + lane * 8), ok);
        }
    };
    using Slot0 = std::integral_constant<int, 0>;
    using Slot1 = std::integral_constant<int, 1>;

    // ---- every load of the first block (and the next one) is requested before anything is waited for ---
    constexpr int PCH = 32 * NTD * 4;  // 16-byte chunks of the phi slab (rows >= D, columns >= nC read as zero)
    uint4 phir[(PCH + NT_ - 1) / NT_];
#pragma unroll
    for (int u = 0; u < (PCH + NT_ - 1) / NT_; u++) {
        const int ch = tid + u * NT_;
        const int d = ch >> 2;
        const bool ok = ch < PCH && d < D && kl < nC;
        const uint4 v = ldg16<RAG>(a.phi + (ok ? (size_t)d * nC + kl - kls : 0));
        phir[u] = make_uint4(ok ? v.x : 0u, ok ? v.y : 0u, ok ? v.z : 0u, ok ? v.w : 0u);
    }
    load_block(b_begin, Slot0{});
    load_ops(b_begin, ops[0]);
    if (b_begin + SBR < B) {
        load_block(b_begin + SBR, Slot1{});
        if constexpr (PFOP) load_ops(b_begin + SBR, ops[1]);
    }
#pragma unroll
    for (int u = 0; u < (PCH + NT_ - 1) / NT_; u++) {
        const int ch = tid + u * NT_;
        if constexpr (RAG) phir[u] = drop8(phir[u], kls);
        if (ch < PCH) *reinterpret_cast<uint4 *>(phi_s + (size_t)(ch >> 2) * kAxLD + (ch & 3) * 8) = phir[u];
    }

    f32x16_t acc[NTD];
#pragma unroll
    for (int m = 0; m < NTD; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[m][i] = 0.f;
    MHC_PHASE_ADD(kPhaseColSlab, pwg, 0, pclk);

    auto process_block = [&](int sb, auto slot) {
        constexpr int S = decltype(slot)::value;
        Ops &op = ops[PFOP ? S : 0];
        constexpr int P = PS == 2 ? S : 0;
        if constexpr (PS == 1) load_prev(sb);
        if (sb != b_begin) {
            if constexpr (!PFOP) load_ops(sb, op);
            __syncthreads();  // every wave is done with the previous block's tile
        }
        // ---- x block -> LDS (the first barrier also covers the phi slab) -------------------------------
#pragma unroll
        for (int u = 0; u < KS; u++) {
            const int ch = tid + u * NT_;
            uint4 xb;
            if constexpr (RAG) drop_elems<(int)sizeof(TS)>(xr[S][u], kls);
            if constexpr (F32)
                xb = make_uint4(pack_bf16x2(__uint_as_float(xr[S][u][0]), __uint_as_float(xr[S][u][1])),
                                pack_bf16x2(__uint_as_float(xr[S][u][2]), __uint_as_float(xr[S][u][3])),
                                pack_bf16x2(__uint_as_float(xr[S][u][4]), __uint_as_float(xr[S][u][5])),
                                pack_bf16x2(__uint_as_float(xr[S][u][6]), __uint_as_float(xr[S][u][7])));
            else xb = make_uint4(xr[S][u][0], xr[S][u][1], xr[S][u][2], xr[S][u][3]);
            *reinterpret_cast<uint4 *>(x_s + (size_t)(ch >> 2) * kAxLD + (ch & 3) * 8) = xb;
        }
        __syncthreads();
        MHC_PHASE_ADD(kPhaseColSlab, pwg, 1, pclk);
        // ---- dphi: this wave's samples, every row tile ------------------------------------------------
        {
            bf16x8_t xf[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
                xf[ks] = __builtin_bit_cast(bf16x8_t, lds_frag_tr(x_s, kAxLD, (KS * wave + ks) * 16, 0, lane));
#pragma unroll
            for (int m = 0; m < NTD; m++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, op.ah[m][ks]), xf[ks], acc[m], 0, 0, 0);
                    if constexpr (HELD == 2)
                        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, op.al[m][ks]), xf[ks], acc[m], 0, 0, 0);
                    if constexpr (RAG) {
#pragma unroll
                        for (int p = HELD; p < 3; p++)
                            acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, load_at(sb, p, m, ks)), xf[ks], acc[m], 0, 0, 0);
                    }
                }
        }
        // ---- dP phi of this wave's sample tiles -> its own rows of o_s (phi fragments from the slab) -----
#pragma unroll
        for (int t = 0; t < TT; t++) {
            f32x16_t o;
#pragma unroll
            for (int i = 0; i < 16; i++) o[i] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 2 * NTD; ks++) {
                const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, lds_frag_tr(phi_s, kAxLD, ks * 16, 0, lane));
                o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, op.av[t][ks]), pf, o, 0, 0, 0);
                if constexpr (RAG)
                    o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, load_av(sb, 1, t, ks)), pf, o, 0, 0, 0);
            }
            // accumulator layout: column = lane & 31, register i -> row 8*(i/4) + 4*(lane/32) + i%4
#pragma unroll
            for (int i = 0; i < 16; i++)
                o_s[(size_t)(SPW * wave + 32 * t + 8 * (i >> 2) + 4 * kg + (i & 3)) * kAxLDO + row] = o[i];
        }
        MHC_PHASE_ADD(kPhaseColSlab, pwg, 2, pclk);
        // ---- epilogue, row-major: the wave reads back only rows it wrote itself (its LDS accesses
        // complete in order), x from the block's tile ------------------------------------------------------
#pragma unroll
        for (int t = 0; t < KS; t++) {
            const int r = erow + 16 * t, b = sb + r;
            const float4 o0 = *reinterpret_cast<const float4 *>(o_s + (size_t)r * kAxLDO + ech * 8);
            const float4 o1 = *reinterpret_cast<const float4 *>(o_s + (size_t)r * kAxLDO + ech * 8 + 4);
            const uint4 xv = *reinterpret_cast<const uint4 *>(x_s + (size_t)r * kAxLD + ech * 8);
            const float cxv = cxr[P][t];
            if constexpr (RAG) drop_elems<(int)sizeof(TP)>(pr[P][t], kcs);
            const float ov[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
            const uint32_t xw[4] = {xv.x, xv.y, xv.z, xv.w};
            float res[8];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const float plo = P32 ? __uint_as_float(pr[P][t][P32 ? 2 * p : p]) : bf16lo_to_f32(pr[P][t][p]);
                const float phi_ = P32 ? __uint_as_float(pr[P][t][P32 ? 2 * p + 1 : p]) : bf16hi_to_f32(pr[P][t][p]);
                res[2 * p] = plo + ov[2 * p] - cxv * bf16lo_to_f32(xw[p]);
                res[2 * p + 1] = phi_ + ov[2 * p + 1] - cxv * bf16hi_to_f32(xw[p]);
            }
            if (b < B && kok) {
                if constexpr (RAG) store_vec_any<TS, 8, true>(dxg + (size_t)b * nC + kc, res, nC - kc);
                else store_vec<TS, 8, true>(dxg + (size_t)b * nC + kc, res);
            }
        }
        if (sb + 2 * SBR < B) {
            load_block(sb + 2 * SBR, slot);
            if constexpr (PFOP) load_ops(sb + 2 * SBR, op);
        }
        MHC_PHASE_ADD(kPhaseColSlab, pwg, 3, pclk);
    };
    for (int sb = b_begin; sb < B; sb += 2 * SBR) {
        process_block(sb, Slot0{});
        if (sb + SBR < B) process_block(sb + SBR, Slot1{});
    }

    float *dphi = a.dphi + (SPLIT ? (size_t)blockIdx.y * D * nC : 0);
    // ---- dphi: sum the four waves' shares through LDS, store row-major --------------------------------
    __syncthreads();  // all tiles consumed; the memory becomes red_s
#pragma unroll
    for (int m = 0; m < NTD; m++)
#pragma unroll
        for (int i = 0; i < 16; i++)
            red_s[((size_t)(wave * NTD + m) * 32 + 8 * (i >> 2) + 4 * kg + (i & 3)) * kAxLDR + row] = acc[m][i];
    __syncthreads();
    for (int e = tid; e < NTD * 32 * 8; e += NT_) {  // four columns per thread: 16-byte LDS reads and stores
        const int d = e >> 3, c = (e & 7) * 4;
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float4 v = *reinterpret_cast<const float4 *>(red_s + ((size_t)w * NTD * 32 + d) * kAxLDR + c);
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
        if (d < D && k0 + c < nC) {
            if constexpr (RAG) {
                const float out[4] = {s.x, s.y, s.z, s.w};
                store_vec_any<float, 4>(dphi + (size_t)d * nC + k0 + c, out, nC - (k0 + c));
            } else {  // k0 % 32 == 0: a quad of columns is inside or outside
                *reinterpret_cast<float4 *>(dphi + (size_t)d * nC + k0 + c) = s;
            }
        }
    }
    MHC_PHASE_ADD(kPhaseColSlab, pwg, 4, pclk);
}

bool proj_bwd_addx_supported(int n) { return padded_D(n) / 32 <= 3; }

template <int NTD, int SPW, bool PFOP, int ST, int NW = 4, bool SPLIT = false>
static hipError_t launch_addx(const ProjAddxArgs &a, hipStream_t stream) {
    if constexpr (NW == 4 && !SPLIT) {
        if (a.per_split < a.B) return launch_addx<NTD, SPW, PFOP, ST, NW, true>(a, stream);
    }
    constexpr int SBR = NW * SPW;
    const size_t tiles = sizeof(bf16_t) * (size_t)kAxLD * (32 * NTD + SBR) + sizeof(float) * SBR * kAxLDO;
    const size_t red = sizeof(float) * NW * NTD * 32 * kAxLDR;  // the final cross-wave sum reuses the tiles' memory
    const size_t smem = tiles > red ? tiles : red;
    hipError_t e = allow_dynamic_lds<&proj_bwd_addx_kernel<NTD, SPW, PFOP, ST, NW, SPLIT>>(smem);
    if (e != hipSuccess) return e;
    const int slabs = (a.nC + kAxKW - 1) / kAxKW;
    dim3 grid(round_up(slabs, 16), (a.B + a.per_split - 1) / a.per_split + (a.tail_row >= 0 ? (a.tail.nblk * a.tail_parts + round_up(slabs, 16) - 1) / round_up(slabs, 16) : 0));
    proj_bwd_addx_kernel<NTD, SPW, PFOP, ST, NW, SPLIT><<<grid, 64 * NW, smem, stream>>>(a);
    return hipGetLastError();
}

// Short rows make few slabs, and one workgroup of each then walks a large batch by itself.  Where the walk is long
// and the slabs leave room for it (two workgroups per CU), the batch is split and the finalize launch adds up the
// partial dphi (kernels us, one workgroup per slab -> split with
// its finalize launch: n=8 B=6000 C=256 94.9 -> 30.2, B=2048 C=512 36.0 -> 22.9; float32 storage n=4 B=6835 C=320
// 91.2 -> 34.7, B=2560 C=1280 41.0 -> 38.6).
int proj_bwd_addx_splits(int B, int n, int C) {
    const int slabs = (n * C + kAxKW - 1) / kAxKW, D = n * n + 2 * n;
    const int walk = padded_D(n) == 32 && slabs <= 256 ? (B + 383) / 384 : (B + 127) / 128;  // blocks without a split
    int S = 512 / slabs, blocks = (B + 127) / 128;
    if (S > blocks / 2) S = blocks / 2;
    // the partial copies (written and read once) stay below half of the activation bytes of this launch
    const int cap = (int)(0.375 * B / D);
    if (S > cap) S = cap;
    // (one launch more: B=2000 n=8 C=1024, walk 16, S = 2 40.2 -> 39.3; B=1000 n=6 C=1024, walk 8 17.9 -> 21.6)
    if (S < 2 || walk < (S == 2 ? 20 : (padded_D(n) == 32 ? 5 : 10))) return 1;
    const int per = (blocks + S - 1) / S;  // blocks of the longest split
    return (blocks + per - 1) / per;
}

// Parts of the batch sums beside a split batch: a workgroup per 64 columns that walks thousands of samples would be
// the longest of the launch (B=6835 n=4 C=320: 66 us, the split slabs 30).
int proj_bwd_addx_sum_parts(int B, int S) { return S > 1 ? (B + kAxSumRows - 1) / kAxSumRows : 1; }

hipError_t launch_proj_bwd_addx(const void *x, int x_dtype, const void *phi, const void *dPb, const void *dPT, int BP,
                                const float *cx, float *dphi, int S, const float *dxp, void *dx, int B, int n, int C,
                                const BatchSumArgs *tail, bool *tail_taken, hipStream_t stream) {
    const int nC = n * C, D = n * n + 2 * n, DP = padded_D(n), NTD = DP / 32;
    ProjAddxArgs a{x, static_cast<const bf16_t *>(phi), static_cast<const bf16_t *>(dPb),
                   static_cast<const bf16_t *>(dPT), cx, dphi, dxp ? dxp : dx, dx, B, BP, D, DP, nC, S > 1 ? ((B + 127) / 128 + S - 1) / S * 128 : B, -1, B, 1, {}};
    if (tail_taken) *tail_taken = false;
    if (tail) {
        a.tail = *tail;
        a.tail.nblk = ((tail->dw ? C : 0) + D + 3 + kAxSumCols - 1) / kAxSumCols;
        a.tail_row = S;
        a.tail_parts = proj_bwd_addx_sum_parts(B, S);
        if (a.tail_parts > 1) a.tail_rows = kAxSumRows;
        if (tail_taken) *tail_taken = true;
    }
    const int st = x_dtype == kF32AsBF16 ? kAxF32 : (!dxp ? kAxBf16 : (C % 8 == 0 ? kAxFine : kAxRagged));
    if (C % 8 != 0 && st != kAxRagged) return hipErrorInvalidValue;
    // D <= 32: the workgroup is sized so that it walks its samples in as few blocks as possible (4, 8 or
    // 12 waves of 32 samples; every block costs two barriers and a round of dependent LDS traffic).
    // Backward at B=320, C=1280, n=4, graphs of ten: 4 waves (three blocks) 16.5 us, 8 waves 16.0, 12 waves
    // (one block) 14.9; B=128: 9.5 / 9.9 with 4 / 8 waves; B=512: 19.7 / 19.0 / 19.5.  Wider projections
    // keep four waves: their registers allow two workgroups per CU only that way.
    // More than 256 slabs: workgroups of four waves, of which three fit a CU, keep the grid in one round
    // (B=1280, C=2560, n=4: 24.4 us with 4 waves, 31.7 with 12).
    int nw = 4;
    if (S == 1 && NTD == 1 && (nC + kAxKW - 1) / kAxKW <= 256) {
        int best = (B + 127) / 128;
        if ((B + 255) / 256 < best) { nw = 8; best = (B + 255) / 256; }
        if ((B + 383) / 384 < best) nw = 12;
    }
#define MHC_ADDX(NTD, NW)                                                                                            \
    return st == kAxBf16 ? launch_addx<NTD, 32, false, kAxBf16, NW>(a, stream)                                       \
                         : (st == kAxFine ? launch_addx<NTD, 32, false, kAxFine, NW>(a, stream)                      \
                                          : (st == kAxRagged ? launch_addx<NTD, 32, false, kAxRagged, NW>(a, stream) \
                                                             : launch_addx<NTD, 32, false, kAxF32, NW>(a, stream)))
    switch (NTD) {
        case 1:
            // (fp32 dxp needs more registers per wave: eight waves at most)
            if (nw == 12 && st == kAxBf16) return launch_addx<1, 32, false, kAxBf16, 12>(a, stream);
            if (nw >= 8) MHC_ADDX(1, 8);
            MHC_ADDX(1, 4);
        case 2: MHC_ADDX(2, 4);
        case 3: MHC_ADDX(3, 4);
        default: return hipErrorInvalidValue;
    }
#undef MHC_ADDX
}

}  // namespace mhc
