// Slab backward for n = 5 .. 8 in the bf16 tier, behind the channel sums (gram_small_kernel): dx, df and the batch-split
// partial sums of dphi, dw and dt in one pass over dy and x, as bwd_slab.hip does it for n <= 4:
//
//   dx[b,j,c]  = sum_i M_b[i,j] dy[b,i,c] + Hpre_b[j] da[b,c] - cx_b x[b,j,c] + sum_d dP[b,d] phi[d, jC+c]
//   dphi[d,k] += sum_b dP[b,d] x_flat[b,k]            dw[c] += sum_b df[b,c] a[b,c] / q_b
//   (reference stream_ops.cuh:761-850, :646-663, ops.py:319-351, rmsnorm.cuh:282-294)
//
// A workgroup owns 64 channels of every stream, walks the samples of its batch split 16 at a time and has a CU to
// itself.  Everything goes from global memory straight into LDS, two tiles ahead; dP phi is formed transposed, so that
// it stays with the lane that mixes the sample; dx replaces dy in LDS and leaves a tile later in whole 128-byte rows.
// What differs from n <= 4 is what the registers hold: the projection has up to 96 rows here (80 at n = 8), so phi takes
// 12 registers per stream and dphi 48 per 32 columns.  Four waves mix (phi in their registers, the rows of M fetched from
// LDS one at a time), four others hold dphi and request the tiles; eight waves of 256 registers fill the CU.
//
// What bounds it: bytes (x, dy in, dx out) and the partial sums of dphi, up to 256 * 64 columns of every stream and D rows in
// fp32 (up to 42 MB at n = 8), written here and added up by the finalize launch.  n=8 B=2000 C=2560: 62 us for 246 MB and
// 39 MB of partial sums (4.6 TB/s); the whole backward 182 us (resident path) -> 102, n=5 B=2000 C=1280 89 -> 50, n=6 B=3000
// C=768 80 -> 54.  One walk of the batch per 64 channels took the resident path's second launch 120 us there.
#include "launchers.h"

#include <algorithm>

#include "lds_stage.h"
#include "phase_profiler.h"
#include "tuning.h"

namespace mhc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

struct BwdSlab8Args {
    const bf16_t *dy, *x;    // [B, N, C]
    const void *w;           // [C]
    const bf16_t *phi;       // [D, N C]
    const float *Hpre, *Hpost, *M, *q, *s1, *cx;  // per sample
    const bf16_t *dPb, *dPT; // dP and dP^T hi / lo, fragment-major (frag_dpb, frag_dpt)
    const float *dt;         // [B, D+3]
    void *dx;                // [B, N, C], in the type of x's storage
    bf16_t *df;              // [B, C] or nullptr
    float *dphi_part;        // [S][D][N C]
    double *dw_part;         // [S][C]
    double *dt_part;         // [S slabs][D+3]
    int w_bf16, B, BP, C, tiles;  // tiles of 16 samples
};

// F32: float32 storage, as in bwd_slab.hip: the channel sums have left x and dy in bf16 where dx will be, and the bytes of CW channels
// of dx hold CW of x, then CW of dy.  x and dy are one tile, two ahead, and dx leaves through two places of its own; at n = 7 and 8
// the LDS holds that for 32 channels (two mixers); n = 8 keeps 19 registers in scratch memory, 80 bytes a lane.  Whole backward, resident
// path -> this: n=5 B=2000 C=2560 198 -> 116 us, n=6 B=3000 C=1024 146 -> 83, n=7 B=3000 C=1024 160 -> 109, n=8 B=4369 C=1024 269 -> 211.
template <int N, bool F32> struct Slab8Stage {
    static constexpr int CW = F32 ? f32_piece_channels(N) : 64, TB = 16, kMixers = CW / 16, kHolders = 4, kThreads = 64 * (kMixers + kHolders);  // waves
    static constexpr int kRowBytes = CW * (F32 ? 4 : 2), kChunks = kRowBytes / 16, kRows = 1024 / kRowBytes;  // of a tile's row; rows per KiB
    static constexpr int kRing8 = kChunks * 8;                         // what slab_swizzle() goes by
    static constexpr int D = N * N + 2 * N, NTD = (D + 31) / 32, DP = 32 * NTD;
    static constexpr int kXRing = 3, kGRing = F32 ? 2 : 4;             // two tiles ahead
    static constexpr int kTile = N * TB * kRowBytes;                   // bytes of x or dy, or of both; of dx
    // behind x: dP^T hi and lo of every 32 rows, dP of every 32 columns (1 KiB each), then blocks of 64 floats: M (a block
    // per sample, rows of 8), Hpre and Hpost (8 samples a block, 8 floats each), cx | q | s1
    static constexpr int kP = kTile, kPBlocks = 3 * NTD, kCoef = kP + kPBlocks * 1024, kCoefBlocks = TB + 2 + 2 + 3;
    static constexpr int kXBytes = kCoef + kCoefBlocks * 256;
    static constexpr int kG = kXRing * kXBytes, kW = kG + kGRing * kTile, kLds = kW + CW * 4;
    // KiB of x (and of dy), or of both, per holder: eight rows of every second stream, or (256-byte rows) four rows of every stream
    static constexpr int kStreams = kRows == 8 ? (N + 1) / 2 : N, kLoads = kStreams * (F32 ? 1 : 2);
    static constexpr int kShare = (kPBlocks + kCoefBlocks + kHolders - 1) / kHolders;
    static constexpr int kCols = N * CW / 32, kAcc = (kCols + kHolders - 1) / kHolders;  // 32-column tiles of dphi, per holder
    static constexpr int kPhiAt = kG + (kGRing - 2) * kTile;           // prologue: 32 rows of phi, in two places of the dy / dx ring
    static_assert(32 * N * CW * 2 <= 2 * kTile && kLds <= 160 * 1024, "32 rows of phi fit two places of the ring");
};

template <int N, bool INJECT, bool F32>
__global__ __launch_bounds__((Slab8Stage<N, F32>::kThreads), 2) void bwd_slab8_kernel(BwdSlab8Args a) {
    static_assert(!(INJECT && F32), "an injected f takes the other kernels");
    using ST = Slab8Stage<N, F32>;
    constexpr int CW = ST::CW, TB = ST::TB, D = ST::D, NTD = ST::NTD;
    constexpr int kChunks = ST::kChunks, kRows = ST::kRows, kRowBytes = ST::kRowBytes;
    typedef __attribute__((address_space(3))) lds_tr_v4i16 *lds_tr_ptr;
    extern __shared__ float smem_f[];
    char *const smem = reinterpret_cast<char *>(smem_f);
    const uint32_t smem_at = lds_address(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int C = a.C, nC = N * C;
    const int slab = blockIdx.x, slabs = gridDim.x, c0 = slab * CW;
    const unsigned nsplit = gridDim.y;
    // tiles y, y + S, ..: all splits go through the batch together and begin where the channel sums, which go through it from its end,
    // have just read x and dy: the memory-side cache (256 MB) still holds that part.  Backward us, splits of consecutive tiles | this: n=8 C=2560
    // B=4096 206.2 | 196.3 (the order of either kernel alone: 204.3, 210.9);  C=1280 3000 84.8 | 84.1;  C=512 8192 98.2 | 95.1;  n=5 C=1024
    // 8192 94.6 | 90.9;  n=6 C=2560 1024 49.6 | 49.0
    const int b_begin = blockIdx.y * TB, b_step = nsplit * TB, b_end = a.B;
    const int T = (a.tiles - 1 - (int)blockIdx.y) / (int)nsplit + 1;
    const int pwg = blockIdx.y * gridDim.x + blockIdx.x;
    (void)pwg;
    MHC_PHASE_ZERO(kPhaseBwdSlab, pwg);
    MHC_PHASE_BEGIN(pclk);
    const bool holder = wave >= ST::kMixers;
    const int hw = wave - ST::kMixers;  // holder index

    const auto lane_row = [&](int row0) { return row0 + lane / kChunks; };
    const auto lane_chunk = [&](int row) { return (lane % kChunks) ^ slab_swizzle<ST::kRing8>(row); };
    const auto lane_col = [&](int row) { return c0 + lane_chunk(row) * (F32 ? 4 : 8); };  // of x or dy; F32: of dx

    // ---- loads of a tile (holders) -------------------------------------------------------------------
    // holder h brings eight rows (h % 2) of the streams h / 2, h / 2 + 2 .. (the last one twice where they do not come out
    // even: every holder has the same number of instructions in flight) and its share of the blocks behind x
    const int ld_row0 = kRows == 8 ? (hw & 1) * 8 : hw * 4, ld_row = lane_row(ld_row0);
    const int ld_at = F32 ? c0 * 4 + lane_chunk(ld_row) * 16 : min(lane_col(ld_row), C - 8) * 2;  // bytes behind the row's first
    auto load_tile = [&](const void *src, int t, uint32_t dst) {
        constexpr int ES = F32 ? 4 : 2;
        const int sb = b_begin + t * b_step;
        const char *base = static_cast<const char *>(src) + (size_t)sb * nC * ES;
        // slots beyond the batch alias its last sample, columns beyond C the last ones: they only meet zero columns of
        // dP^T or land in rows and columns that are not stored (F32: C is a multiple of 64)
        const uint32_t off = (uint32_t)min(ld_row, b_end - sb - 1) * nC * ES + ld_at;
#pragma unroll
        for (int i = 0; i < ST::kStreams; i++) {
            const int j = kRows == 8 ? min((hw >> 1) + 2 * i, N - 1) : i;
            load_to_lds<16>(base + (size_t)j * C * ES, off, dst + (j * TB + ld_row0) * kRowBytes);
        }
    };
    struct Block {
        const char *src;          // for the first sample of the batch
        uint32_t step, at, dst;   // bytes per sample; this lane's bytes behind the tile's first; place behind the tile's x
        bool wide;                // a KiB of dP operands; otherwise 64 floats of the coefficients
    };
    auto block_of = [&](int k) {
        k = min(k, ST::kPBlocks + ST::kCoefBlocks - 1);
        const size_t plane = (size_t)ST::DP * a.BP;
        if (k < 2 * NTD)  // rows 32 (k / 2) ..: value (k even) or remainder
            return Block{reinterpret_cast<const char *>(a.dPT + (k & 1) * plane + frag_base(k >> 1, a.BP >> 4, 0)), 64u, lane * 16u,
                         ST::kP + k * 1024u, true};
        if (k < ST::kPBlocks) {  // columns 32 kk ..: [d / 8][16 samples][8] out of the fragments of 32 samples
            const int kk = k - 2 * NTD;
            return Block{reinterpret_cast<const char *>(a.dPb + frag_base(0, ST::DP >> 4, 2 * kk)), ST::DP * 2u,
                         (lane >> 5) * 1024u + ((lane >> 4) & 1) * 512u + (lane & 15) * 16u, ST::kP + k * 1024u, true};
        }
        const int s = k - ST::kPBlocks;
        const uint32_t dst = ST::kCoef + s * 256u;
        if (s < TB) {
            // sample s: element (i, j) of M at (8 i + j + 4 s) mod 64, so that sixteen samples' rows lie in different banks
            const int e = (lane - 4 * s) & 63, i = min(e >> 3, N - 1), j = min(e & 7, N - 1);
            return Block{reinterpret_cast<const char *>(a.M), N * N * 4u, (uint32_t)(s * N * N + i * N + j) * 4u, dst, false};
        }
        const int v = s - TB;
        if (v < 4) {
            const int row = (v & 1) * 8 + (lane >> 3);
            return Block{reinterpret_cast<const char *>(v < 2 ? a.Hpre : a.Hpost), N * 4u, (uint32_t)(row * N + min(lane & 7, N - 1)) * 4u, dst, false};
        }
        return Block{reinterpret_cast<const char *>(INJECT || v == 4 ? a.cx : (v == 5 ? a.q : a.s1)), 4u, (lane & 15) * 4u, dst, false};
    };
    auto load_all = [&](int t, const Block (&mine)[ST::kShare]) {
        const uint32_t st = smem_at + t % ST::kXRing * ST::kXBytes;
        const int sb = b_begin + t * b_step;
        const uint32_t left = min(b_end - sb, TB);
        load_tile(F32 ? a.dx : static_cast<const void *>(a.x), t, st);
#pragma unroll
        for (int i = 0; i < ST::kShare; i++) {
            const Block &m = mine[i];
            if (m.wide) {  // (the second half of a 32-sample fragment of dP lies 256 bytes behind the first)
                const bool half = m.dst >= ST::kP + 2 * NTD * 1024u && (sb & 16);
                load_to_lds<16>(m.src + (size_t)(half ? sb - 16 : sb) * m.step + (half ? 256 : 0), m.at, st + m.dst);
            } else {
                // slots beyond the batch: the last float of the batch, whatever it is
                load_to_lds<4>(m.src + (size_t)sb * m.step, min(m.at, left * m.step - 4), st + m.dst);
            }
        }
        if constexpr (!F32) load_tile(a.dy, t, smem_at + ST::kG + t % ST::kGRing * ST::kTile);
    };

    // ---- prologue: the first tiles requested; phi -> LDS, 32 rows at a time, row-major [32 d][N][CW] -> the mixers' fragments
    if (holder) {
        Block mine[ST::kShare];
#pragma unroll
        for (int i = 0; i < ST::kShare; i++) mine[i] = block_of(hw + i * ST::kHolders);
        load_all(0, mine);
        if (T > 1) load_all(1, mine);
    }
    char *const phi_s = smem + ST::kPhiAt;
    // mixer lane (l16, kq): the four channels from c0 + cl of sample l16
    const int l16 = lane & 15, kq = lane >> 4, cl = 16 * (wave % ST::kMixers) + 4 * kq;
    bf16x8_t phif[N][NTD];  // mixers: A operand, rows = this wave's 16 channels of a stream, contraction over 32 d
    // The mixers alone bring phi and w, all of it asked for at once, and none of these barriers waits for global memory: holders
    // that brought a part of it waited for their first tiles before they could hand it on.  Backward in graphs of ten: n=5 B=3000
    // C=1024 55.4 -> 54.3 us, n=7 B=700 C=2552 56.1 -> 55.1, n=8 B=2048 C=2560 99.5 -> 99.2.
    constexpr int kPhiThreads = 64 * ST::kMixers, kPc = CW / 8, kPhiIters = N * 32 * kPc / kPhiThreads;
    static_assert(kPhiIters * kPhiThreads == N * 32 * kPc, "whole chunks of phi for every mixer");
    uint4 phir[NTD][kPhiIters];
    if (!holder) {
#pragma unroll
        for (int kk = 0; kk < NTD; kk++)
#pragma unroll
            for (int i = 0; i < kPhiIters; i++) {
                const int e = tid + i * kPhiThreads;
                const int d = 32 * kk + e / (N * kPc), j = e / kPc % N, c = c0 + e % kPc * 8;
                const bool ok = d < D && c < C;
                phir[kk][i] = load16_masked(reinterpret_cast<const uint4 *>(a.phi + (ok ? (size_t)d * nC + (size_t)j * C + c : 0)), ok);
            }
        if (tid < CW)
            reinterpret_cast<float *>(smem + ST::kW)[tid] =
                (c0 + tid < C && !INJECT) ? (a.w_bf16 ? bf16_to_f32(static_cast<const bf16_t *>(a.w)[c0 + tid])
                                                      : static_cast<const float *>(a.w)[c0 + tid]) : 0.f;
    }
#pragma unroll
    for (int kk = 0; kk < NTD; kk++) {
        if (kk > 0) stage_barrier();  // the rows before have been read
        if (!holder) {
#pragma unroll
            for (int i = 0; i < kPhiIters; i++) *reinterpret_cast<uint4 *>(phi_s + (tid + i * kPhiThreads) * 16) = phir[kk][i];
        }
        stage_barrier();
        if (!holder) {
            const int q = lane & 3, jj = (lane >> 2) & 3;
#pragma unroll
            for (int j = 0; j < N; j++) {
                const char *p = phi_s + ((kq * 8 + jj) * N + j) * CW * 2 + (16 * wave + 4 * q) * 2;
                const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)p));
                const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(p + 4 * N * CW * 2)));
                phif[j][kk] = __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
            }
        }
    }
    stage_barrier();  // the places that held phi may be filled

    double *const red_w = reinterpret_cast<double *>(smem);  // at the end: [16][CW + 1]
    double *const red_dt = red_w + 16 * (CW + 1);            // and [mixers][128]
    if (holder) {
        // ---- requests the tiles, accumulates dphi: 32-column tiles hw, hw + 4 .. (stream, channel half) ----------
        Block mine[ST::kShare];  // (formed again: kept across the prologue they spill)
#pragma unroll
        for (int i = 0; i < ST::kShare; i++) {
            int k = hw + i * ST::kHolders;
            asm volatile("" : "+s"(k));
            mine[i] = block_of(k);
        }
        f32x16_t acc[ST::kAcc][NTD];
#pragma unroll
        for (int k = 0; k < ST::kAcc; k++)
#pragma unroll
            for (int m = 0; m < NTD; m++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[k][m][i] = 0.f;
        // transposed reads of x: this lane's row (lo; hi: + 4) and its 8 bytes of the 32-channel group
        constexpr int kHalves = CW / 32;  // 32-column tiles of a stream
        const int q = lane & 3, row = (lane >> 5) * 8 + ((lane >> 2) & 3), ch = 4 * (hw % kHalves) + ((lane >> 4) & 1) * 2 + (q >> 1);
        const int at_lo = row * kRowBytes + (ch ^ slab_swizzle<ST::kRing8>(row)) * 16 + (q & 1) * 8;
        const int at_hi = (row + 4) * kRowBytes + (ch ^ slab_swizzle<ST::kRing8>(row + 4)) * 16 + (q & 1) * 8;
        for (int p = 0; p < T; p++) {
            // tile p has landed: all but the next tile's instructions; for everybody behind the barrier, where everybody is
            // done with x of tile p - 1 and with dx of tile p - 2 as well, whose places tile p + 2 takes
            if (p + 1 < T) wait_vmem<ST::kLoads + ST::kShare>();
            else wait_vmem<0>();
            stage_barrier();
            if (p + 2 < T) load_all(p + 2, mine);
            const char *st = smem + p % ST::kXRing * ST::kXBytes;
            bf16x8_t xf[ST::kAcc];
#pragma unroll
            for (int k = 0; k < ST::kAcc; k++) {
                const int tile = min(hw + 4 * k, ST::kCols - 1);  // (64 channels: both have the half hw & 1, kCols is even)
                const char *xs = st + tile / kHalves * TB * kRowBytes;
                const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(xs + at_lo)));
                const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(xs + at_hi)));
                xf[k] = __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
            }
#pragma unroll
            for (int m = 0; m < NTD; m++) {
                const bf16x8_t ah = *reinterpret_cast<const bf16x8_t *>(st + ST::kP + 2 * m * 1024 + lane * 16);
                const bf16x8_t al = *reinterpret_cast<const bf16x8_t *>(st + ST::kP + (2 * m + 1) * 1024 + lane * 16);
#pragma unroll
                for (int k = 0; k < ST::kAcc; k++) {
                    acc[k][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, xf[k], acc[k][m], 0, 0, 0);
                    acc[k][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, xf[k], acc[k][m], 0, 0, 0);
                }
            }
        }
        stage_barrier();  // the mixers' last dx
        float *dphi_out = a.dphi_part + (size_t)blockIdx.y * D * nC;
#pragma unroll
        for (int k = 0; k < ST::kAcc; k++) {
            const int tile = hw + 4 * k, c = c0 + tile % kHalves * 32 + (lane & 31);
            if (tile < ST::kCols && c < C) {
#pragma unroll
                for (int m = 0; m < NTD; m++)
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int d = 32 * m + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                        if (d < D) dphi_out[(size_t)d * nC + (size_t)(tile / kHalves) * C + c] = acc[k][m][i];
                    }
            }
        }
        __syncthreads();
        __syncthreads();
    } else {
        // ---- forms dx, stores the tile before ---------------------------------------------------------------------
        const float4 w4 = *reinterpret_cast<const float4 *>(smem + ST::kW + cl * 4);
        const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
        const float inv_c = 1.0f / (float)C;
        double usum[4] = {0.0, 0.0, 0.0, 0.0};  // float32 terms, a sample each: the walk may be hundreds of tiles long
        double dtsum[2] = {0.0, 0.0};  // columns lane, lane + 64 of dt
        // this lane's 8 bytes of its sample's row of x, of dy (F32: behind x), and what it writes of dx
        const auto row_place = [&](int chunk) { return l16 * kRowBytes + ((chunk ^ slab_swizzle<ST::kRing8>(l16)) * 16); };
        const int row_at = row_place(cl >> 3) + (kq & 1) * 8, row_dy = F32 ? row_place(kChunks / 2 + (cl >> 3)) + (kq & 1) * 8 : row_at;
        constexpr int kPieces = N * TB / kRows, kOut = (kPieces + ST::kMixers - 1) / ST::kMixers;
        auto store_dx = [&](int t) {
            const int sb = b_begin + t * b_step;
            const char *g = smem + ST::kG + t % ST::kGRing * ST::kTile;
#pragma unroll
            for (int i = 0; i < kOut; i++) {
                const int at = wave + i * ST::kMixers, piece = min(at, kPieces - 1), j = piece / (TB / kRows);
                const int row = lane_row(piece % (TB / kRows) * kRows), c = lane_col(row);
                const uint4 v = *reinterpret_cast<const uint4 *>(g + piece * 1024 + lane * 16);
                if (at < kPieces && sb + row < b_end && c < C) {  // C % 8 == 0: eight channels are inside or outside
                    if constexpr (F32) st16<true>(static_cast<float *>(a.dx) + (size_t)sb * nC + (uint32_t)(row * nC + j * C + c), v.x, v.y, v.z, v.w);
                    else st16<true>(static_cast<bf16_t *>(a.dx) + (size_t)sb * nC + (uint32_t)(row * nC + j * C + c), v.x, v.y, v.z, v.w);
                }
            }
        };
        for (int t = 0; t < T; t++) {
            const char *st = smem + t % ST::kXRing * ST::kXBytes;
            char *const gs = smem + ST::kG + t % ST::kGRing * ST::kTile;
            const int sb = b_begin + t * b_step;
            const float *co = reinterpret_cast<const float *>(st + ST::kCoef);
            MHC_PHASE_ADD(kPhaseBwdSlab, pwg, t > 0 ? 2 : 0, pclk);
            stage_barrier();
            MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 1, pclk);
            if (t > 0) store_dx(t - 1);
            // dt is summed by the slabs in turn: this tile's rows by slab t % slabs, as many rows per mixer
            constexpr int kDtRows = TB / ST::kMixers;
            const bool my_dt = t % slabs == slab;
            float dtv[kDtRows][2];
            if (my_dt) {
#pragma unroll
                for (int r = 0; r < kDtRows; r++) {
                    const int b = min(sb + kDtRows * wave + r, b_end - 1);
                    const float *p = a.dt + (size_t)b * (D + 3);
                    dtv[r][0] = p[min(lane, D + 2)];
                    dtv[r][1] = p[min(lane + 64, D + 2)];
                }
            }
            // projection term: columns = samples, rows = this lane's channels.  What the mixing needs first is requested before
            // it, and below every stream of dy with its row of M one stream ahead: left to itself the scheduler puts the reads
            // where their waits are not hidden as soon as registers get short (n=8 B=2000 C=2560, whole backward: 105.6 -> 101.5 us)
            f32x4_t o[N];
            float hpre[8], hpost[8];
            const float *const Mb = co + l16 * 64;
            struct Row { uint2 g; float4 m0, m1; };
            auto row_of = [&](int i) {
                return Row{*reinterpret_cast<const uint2 *>((F32 ? st : gs) + i * TB * kRowBytes + row_dy),
                           *reinterpret_cast<const float4 *>(Mb + ((8 * i + 4 * l16) & 63)),
                           *reinterpret_cast<const float4 *>(Mb + ((8 * i + 4 + 4 * l16) & 63))};
            };
            Row row;
            {
                bf16x8_t pf[NTD];
#pragma unroll
                for (int kk = 0; kk < NTD; kk++) pf[kk] = *reinterpret_cast<const bf16x8_t *>(st + ST::kP + (2 * NTD + kk) * 1024 + lane * 16);
                lds_floats<8>(co + (TB + (l16 >> 3)) * 64 + (l16 & 7) * 8, hpre);
                lds_floats<8>(co + (TB + 2 + (l16 >> 3)) * 64 + (l16 & 7) * 8, hpost);
                row = row_of(0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < N; j++) o[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(phif[j][0], pf[0], f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int kk = 1; kk < NTD; kk++)
#pragma unroll
                    for (int j = 0; j < N; j++) o[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(phif[j][kk], pf[kk], o[j], 0, 0, 0);
            }
            const float *sc = co + (TB + 4) * 64 + l16;
            const float cxv = sc[0];
            float qinv = 0.f, k2 = 0.f;
            const bool real = sb + l16 < b_end;  // a slot beyond the batch adds nothing to usum, whatever its sample holds
            if constexpr (!INJECT) {
                qinv = 1.0f / sc[64];
                k2 = sc[128] * qinv * qinv * qinv * inv_c;
            }
            // streams of dy one after the other: df, and the rows of M^T dy added into the accumulators
            float s_df[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < N; i++) {
                const Row next = row_of(min(i + 1, N - 1));
                __builtin_amdgcn_sched_barrier(0);
                const uint2 g = row.g;
                const float gv[4] = {bf16lo_to_f32(g.x), bf16hi_to_f32(g.x), bf16lo_to_f32(g.y), bf16hi_to_f32(g.y)};
                const float mr[8] = {row.m0.x, row.m0.y, row.m0.z, row.m0.w, row.m1.x, row.m1.y, row.m1.z, row.m1.w};
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    s_df[c] += hpost[i] * gv[c];
#pragma unroll
                    for (int j = 0; j < N; j++) o[j][c] += mr[j] * gv[c];
                }
                row = next;
            }
            uint2 xr[N];
            float s_a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < N; j++) {
                xr[j] = *reinterpret_cast<const uint2 *>(st + j * TB * kRowBytes + row_at);
                s_a[0] += hpre[j] * bf16lo_to_f32(xr[j].x); s_a[1] += hpre[j] * bf16hi_to_f32(xr[j].x);
                s_a[2] += hpre[j] * bf16lo_to_f32(xr[j].y); s_a[3] += hpre[j] * bf16hi_to_f32(xr[j].y);
            }
            float da[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float dq = s_df[c] * qinv;
                da[c] = INJECT ? 0.f : dq * wv[c] - s_a[c] * k2;
                if constexpr (!INJECT) usum[c] += (double)(real ? dq * s_a[c] : 0.f);
            }
#pragma unroll
            for (int j = 0; j < N; j++) {
                const float xv[4] = {bf16lo_to_f32(xr[j].x), bf16hi_to_f32(xr[j].x), bf16lo_to_f32(xr[j].y), bf16hi_to_f32(xr[j].y)};
                float r[4];
#pragma unroll
                for (int c = 0; c < 4; c++) r[c] = o[j][c] + hpre[j] * da[c] - cxv * xv[c];
                if constexpr (F32) *reinterpret_cast<float4 *>(gs + j * TB * kRowBytes + row_place(cl >> 2)) = make_float4(r[0], r[1], r[2], r[3]);
                else *reinterpret_cast<uint2 *>(gs + j * TB * kRowBytes + row_at) = make_uint2(pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]));
            }
            if (my_dt) {
#pragma unroll
                for (int r = 0; r < kDtRows; r++)
                    if (sb + kDtRows * wave + r < b_end) { dtsum[0] += dtv[r][0]; dtsum[1] += dtv[r][1]; }
            }
            if (INJECT && a.df && sb + l16 < b_end && c0 + cl < C)
                store_vec<bf16_t, 4>(a.df + (size_t)sb * C + (uint32_t)(l16 * C + c0 + cl), s_df);
        }
        MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 2, pclk);
        stage_barrier();
        store_dx(T - 1);
        // vmcnt(0), for the compiler: it sees the loads of dt above as pending on every path out of here, and would wait for
        // them - and with them for all that the holders have requested - in the holders' loop
        __builtin_amdgcn_s_waitcnt(0x0f70);
        MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 3, pclk);
        __syncthreads();  // everyone is done with the rings
        if constexpr (!INJECT) {
#pragma unroll
            for (int v = 0; v < 4; v++) red_w[l16 * (CW + 1) + cl + v] = usum[v];
        }
        red_dt[wave * 128 + lane] = dtsum[0];
        red_dt[wave * 128 + 64 + lane] = dtsum[1];
        __syncthreads();
    }

    // ---- small outputs of the split -------------------------------------------------------------------
    if (!INJECT && tid < CW && c0 + tid < C) {
        double s = 0.0;
#pragma unroll
        for (int r = 0; r < 16; r++) s += red_w[r * (CW + 1) + tid];
        a.dw_part[(size_t)blockIdx.y * C + c0 + tid] = s;
    }
    if (tid < D + 3) {
        double s = 0.0;
#pragma unroll
        for (int r = 0; r < ST::kMixers; r++) s += red_dt[r * 128 + tid];
        a.dt_part[((size_t)blockIdx.y * slabs + slab) * (D + 3) + tid] = s;
    }
    MHC_PHASE_ADD(kPhaseBwdSlab, pwg, 4, pclk);
}

bool bwd_slab8_supported(int x_dtype, int y_dtype, int phi_dtype, int n, int C) {
    return x_dtype == kBF16 && y_dtype == kBF16 && phi_dtype == kBF16 && n >= 5 && n <= 8 && C % 8 == 0;
}

static int slab8_width(int n, bool f32) { return f32 ? f32_piece_channels(n) : 64; }
int bwd_slab8_slabs(int n, int C, bool f32) { return (C + slab8_width(n, f32) - 1) / slab8_width(n, f32); }

// At most one workgroup per CU and at least three tiles each, and within that the splits that cost least: a tile is some 0.2 n us
// of a walk, and from two splits on their partial dphi are written, read and added up, D n C elements each, while a single one
// leaves the result.  Backward us, one split | two | as many as the CUs (and tiles) allow:
//   n=8 C=256  B=100 36.6 | 32.3 | 32.3 (2), 300 58.0 | 42.7 | 32.7 (6), 2000 two tiles each 50.3, three 47.3, four 47.1, seven 51.4
//   n=8 C=2560 B=100 41.8 | 50.8 | 50.8 (2), 200 52.3 | 52.5 | 47.9 (4);  C=4104 100 46.2 | 57.7, 200 55.5 | 62.3 | 61.2 (3), 300 67.4 |
//              69.0 | 66.6 (3);  C=8192 100 50.2 | 74.9, 300 77.0 | 92.5
//   n=5 C=2560 B=100 33.6 | 32.3, 200 36.8 | 34.1 | 32.1 (4);  C=6144 100 35.2 | 40.9, 200 42.9 | 43.7, 300 51.7 | 48.4
int bwd_slab8_batch_splits(int B, int n, int C, bool f32) {
    const int slabs = bwd_slab8_slabs(n, C, f32), tiles = (B - 1) / 16 + 1;
    const auto per_split = [&](int s) { return (tiles + s - 1) / s; };
    int S = 1;
    if (const int hook = tuning_get(kTuneSlabSplits); hook > 0) {  // experiment hook
        S = std::min(hook, tiles);
    } else {
        const double part = 6.4e-6 * (n * n + 2 * n) * n * C;
        double least = 0.2 * n * tiles;
        for (int s = 2; s <= std::min(256 / slabs, tiles / 3); s++) {
            const double us = 0.2 * n * per_split(s) + part * (0.7 + 0.15 * s);
            if (us < least) { least = us; S = s; }
        }
    }
    // the longest split decides: the fewest splits that keep its tile count
    return (tiles + per_split(S) - 1) / per_split(S);
}

hipError_t launch_bwd_slab8(const void *dy, const void *x, const void *w, int w_dtype, const void *f_inject, const void *phi,
                            const float *Hpre, const float *Hpost, const float *M, const float *q, const BwdCoefOut &co,
                            void *dx, void *df, float *dphi_part, double *dw_part, double *dt_part, int S, int B, int n, int C,
                            hipStream_t stream, bool f32) {
    const int tiles = (B - 1) / 16 + 1;
    if (S < 1 || S > tiles || (f32 && (f_inject || C % 64 != 0))) return hipErrorInvalidValue;
    const BwdSlab8Args a{static_cast<const bf16_t *>(dy), static_cast<const bf16_t *>(x), w, static_cast<const bf16_t *>(phi),
                         Hpre, Hpost, M, q, co.s1, co.cx, co.dPb, co.dPT, co.dt, dx,
                         static_cast<bf16_t *>(df), dphi_part, dw_part, dt_part, w_dtype == kBF16, B, co.BP, C, tiles};
    const dim3 grid(bwd_slab8_slabs(n, C, f32), S);
#define MHC_SLAB8(N, INJ, F32)                                                                                \
    do {                                                                                                      \
        constexpr size_t lds = Slab8Stage<N, F32>::kLds;                                                      \
        if (hipError_t e = allow_dynamic_lds<&bwd_slab8_kernel<N, INJ, F32>>(lds); e != hipSuccess) return e; \
        bwd_slab8_kernel<N, INJ, F32><<<grid, Slab8Stage<N, F32>::kThreads, lds, stream>>>(a);                \
    } while (0)
#define MHC_SLAB8_N(N)                                                                                        \
    do {                                                                                                      \
        if (f32) MHC_SLAB8(N, false, true);                                                                   \
        else if (f_inject) MHC_SLAB8(N, true, false);                                                         \
        else MHC_SLAB8(N, false, false);                                                                      \
    } while (0)
    switch (n) {
        case 5: MHC_SLAB8_N(5); break;
        case 6: MHC_SLAB8_N(6); break;
        case 7: MHC_SLAB8_N(7); break;
        default: MHC_SLAB8_N(8); break;
    }
#undef MHC_SLAB8_N
#undef MHC_SLAB8
    return hipGetLastError();
}

}  // namespace mhc
