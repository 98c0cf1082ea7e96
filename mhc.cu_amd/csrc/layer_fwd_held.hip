// Dynamic-H layer forward of large batches, n = 2 .. 4: projection, coefficients and mix (reference bindings.cu:421-477) in
// one pass over x.
//
// The two-launch forward (proj_fwd.hip, mix_fwd.hip) reads x twice, and once x no longer fits the L2 both passes are bound
// by memory.  Here a workgroup takes a tile of sixteen samples, the columns of one matrix-core tile, and holds its x in
// registers (up to 160 of 256 per lane, 320 KB per CU) from the load to the store:
//   projection    a wave owns a range of channels of all streams; its pieces go through its own LDS from rows into operand
//                 layout, phi comes from the L2 in operand layout (held_pack_kernel), 491 KB per tile at n = 4, C = 2560
//   coefficients  the waves' sums meet in LDS, 16 lanes per sample run activations and Sinkhorn on four of the waves
//   mix           from the registers the tile was loaded into, whole 128-byte lines per store; the workgroup then goes on to
//                 its next tile, whose first pieces are requested as registers fall free
// sixteen samples and no fewer, because every tile reads all of phi; whole lines, because a store of half a line costs
// as much as a whole one (operand layout instead of rows, n=4 B=8192 C=2560: 88 us, 70 with this one).
// The registers are full: 19 of the 84 forms keep 1 to 18 of them in scratch memory (bf16 n=4 at five chunks per wave, the form of
// C=2560: 5; float32 storage, whose loads wait unrounded beside the held rows: up to 18).
// It is bound by memory in its load and store phases (the tile's arithmetic overlaps with them only between the workgroups of a
// CU, which is why rows of at most 1280 channels, two or more workgroups per CU, gain most).  Forward us, two launches ->
// this one, the packing of phi included: bf16 n=4 B=8192 C=2560 87.8 -> 68.8 (4.9 TB/s on x and y), 8192 1280 52.2 -> 38.2,
// 3001 2560 39.5 -> 33.0, 4096 1920 40.7 -> 31.5, n=3 3000 2048 27.8 -> 21.3, n=2 3000 4096 36.7 -> 27.6; float32 n=4 2560 1280
// 37.5 -> 31.4, 4096 640 34.7 -> 24.3, n=2 2200 2048 32.1 -> 22.1; float32 storage of bf16 arithmetic n=4 8192 832 66 -> 48,
// 3500 2560 74 -> 62.
#include "launchers.h"
#include "mhc_common.h"
#include "sinkhorn_device.h"
#include "tuning.h"

#include <algorithm>

namespace mhc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;

constexpr int kHeldS = 16;  // samples per tile: the columns of one 16 x 16 product

// How the contraction is cut into products.
//   chunk     128 bytes of every stream of a sample; half of it is what one product takes per sample
//   unit      what is requested together: one stream of a chunk, FU fragments of phi (1 KB each, in operand layout)
//   fragment  16 rows of phi; rows left over from a multiple of 16 (n = 4: 8 of 24, n = 2: all 8) are paired, the
//             same rows for both halves in one fragment, and each half is used with its own x
template <typename TX, int N> struct HeldShape {  // TX: what is multiplied (bf16, or float in the exact tier)
    static constexpr int VE = 16 / (int)sizeof(TX), CH = 8 * VE;  // channels of a lane's piece, of a chunk
    static constexpr int D = N * N + 2 * N;
    static constexpr int FU = N - 1;
    static constexpr int kTiles = N == 4 ? 2 : 1;  // tiles of partial sums that a wave leaves
    // row of phi and half of the chunk for row r of fragment f; rows >= D hold zeros
    __host__ __device__ static constexpr int row(int f, int r) { return N == 2 ? (r & 7) : (N == 4 && f == 2 ? 16 + (r & 7) : r); }
    __host__ __device__ static constexpr int half(int f, int r) { return N == 2 || (N == 4 && f == 2) ? r >> 3 : f; }
};

// ---- phi in operand layout ----------------------------------------------------------------------
struct HeldPackArgs {
    const void *src[3];   // pre | post | res (or three parts of one array)
    const float *b[3], *alpha_in[3];
    void *phi_out, *frag;  // phi_out: row-major copy, or nullptr
    float *bias, *alpha;   // or nullptr
    int C, units;
};

// Fragment f of unit u, lane l = (row l & 15, piece l >> 4 of the half).  The caller's own parameters are also left behind in
// their packed form (as pack_params.hip does) for the backward.  2.5 us, a launch; bound by its latency.
template <typename TS, typename TX, int N>
__global__ __launch_bounds__(256) void held_pack_kernel(HeldPackArgs a) {
    using H = HeldShape<TX, N>;
    constexpr int VE = H::VE;
    const int C = a.C, nC = N * C;
    const int id = blockIdx.x * 256 + threadIdx.x;
    if (a.bias && blockIdx.x == 0) {
        const int t = threadIdx.x;
        if (t < 3) a.alpha[t] = a.alpha_in[t][0];
        if (t < H::D) a.bias[t] = t < N ? a.b[0][t] : (t < 2 * N ? a.b[1][t - N] : a.b[2][t - 2 * N]);
    }
    const int lane = id & 63, f = (id >> 6) % H::FU, u = (id >> 6) / H::FU;
    if (u >= a.units) return;
    const int r = lane & 15, d = H::row(f, r), j = u % N;
    const int c = (u / N) * H::CH + (H::half(f, r) * 4 + (lane >> 4)) * VE;
    float v[VE];
#pragma unroll
    for (int i = 0; i < VE; i++) v[i] = 0.f;
    if (d < H::D && c < C) {  // C is a multiple of VE
        const int g = alpha_group(d, N), d0 = g == 0 ? 0 : (g == 1 ? N : 2 * N);
        load_vec<TS, VE>(static_cast<const TS *>(a.src[g]) + (size_t)(d - d0) * nC + (size_t)j * C + c, v);
        if (a.phi_out) store_vec<TX, VE>(static_cast<TX *>(a.phi_out) + (size_t)d * nC + (size_t)j * C + c, v);
    }
    store_vec<TX, VE>(static_cast<TX *>(a.frag) + (size_t)id * VE, v);
}

struct HeldArgs {
    const void *x, *w, *frag;
    void *y;
    const float *alpha, *bias;
    float *Hpre, *Hpost, *M, *P, *r, *q, *sk_state;
    int w_bf16, B, C, T, S, tiles, frag_bytes;  // S: samples per tile, at most kHeldS
    float eps;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t held_rsrc(const void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00020000);
}

// Sum of the waves' values, pair by pair.
template <int K, typename F> __device__ __forceinline__ float held_wave_sum(F at) {
    float v[K];
#pragma unroll
    for (int i = 0; i < K; i++) v[i] = at(i);
#pragma unroll
    for (int d = K / 2; d > 0; d /= 2)
#pragma unroll
        for (int i = 0; i < d; i++) v[i] += v[i + d];
    return v[0];
}

// waves per SIMD, by the units that a wave holds (8 registers each)
constexpr int held_waves(int units) { return units <= 5 ? 4 : (units <= 10 ? 3 : 2); }

template <typename TS, typename TX, int N, int CB, int NW, int WX, int WP, int ST>
__global__ __launch_bounds__(NW * 64, held_waves(N * CB)) void layer_fwd_held_kernel(HeldArgs a) {
    using H = HeldShape<TX, N>;
    using SK = SkSmall<4>;
    constexpr int VE = H::VE, D = H::D, U = CB * N, ES = (int)sizeof(TS);
    constexpr bool kExact = std::is_same<TX, float>::value;
    constexpr bool kRound = sizeof(TS) > sizeof(TX);            // fp32 storage, rounded to bf16 behind the load
    constexpr bool kFine = std::is_same<TS, float>::value;      // fp32 results: library functions, IEEE divisions, mix in fp32
    constexpr int kFold = kExact ? 1 : 2, kSums = kRound || N < 4 ? 2 : 1;
    constexpr int LP = kRound ? 2 : 1;                          // loads per piece: 16 bytes of either half of the chunk's channels
    constexpr int kCoef = 28;                  // floats of a sample's coefficients (pitch)
    constexpr int kPitch = 144;                // bytes of a staged row
    constexpr int kStage = kHeldS * kPitch;    // a staged unit; two per wave
    __shared__ float ssx_s[NW][16], ssa_s[NW][16];
    __shared__ __align__(16) float coef_s[kHeldS * kCoef];                          // M (4 x 4) | Hpre | Hpost
    __shared__ __align__(16) unsigned char stage_s[NW][2 * kStage];                 // later the wave's partial sums
    extern __shared__ __align__(16) float w_s[];                                    // [channels of all waves' chunks]
    const int C = a.C, nC = N * C, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    auto red = [&](int w2, int t, int r, int l) -> float & { return *reinterpret_cast<float *>(&stage_s[w2][((t * 4 + r) * 64 + l) * 4]); };
    const int chunk0 = ((wave + (blockIdx.x >> 3)) % NW) * CB;  // first of the wave's chunks
    for (int c = tid; c < NW * CB * H::CH; c += NW * 64)
        w_s[c] = c < C ? (a.w_bf16 ? bf16_to_f32(static_cast<const bf16_t *>(a.w)[c]) : static_cast<const float *>(a.w)[c]) : 0.f;
    // coefficient lanes: 16 per sample, four samples per wave on the first four waves
    const int g = lane & 15, sc = (wave & 3) * 4 + (lane >> 4), r0 = SK::row(g), c0 = SK::col0(g);
    const bool mv = r0 < N && c0 < N, vv = g < 2 * N;
    const float al0 = a.alpha[vv ? (g < N ? 0 : 1) : 2], al2 = a.alpha[2];
    const float bvec = a.bias[vv ? g : 0], bres = a.bias[mv ? 2 * N + r0 * N + c0 : 0];

    // x: lane (row r8 of either half of the tile, 16 bytes at seg of the chunk's 128)
    const int r8 = lane >> 3, seg = lane & 7;
    const int c_lane = chunk0 * H::CH + seg * (VE / LP), off0 = (r8 * nC + c_lane) * ES, stream = C * ES, rows8 = 8 * nC * ES;
    uint32_t xr[CB][N][2][4];
    auto rsrc_of = [&](const void *p, int tile) {
        const int left = tile < a.tiles ? min(a.B - tile * a.S, a.S) : 0;
        const int t = tile < a.tiles ? tile : 0;
        return held_rsrc(static_cast<const char *>(p) + (size_t)t * a.S * nC * ES, left * nC * ES);
    };
    // offset of part l of the lane's piece of chunk cb, stream 0, first half of the tile; beyond the row's end: outside
    // every buffer (formed where it is used: the compiler would otherwise keep one per chunk in registers)
    auto piece = [&](int cb, int l) {
        int c = c_lane, o = off0;
        asm volatile("" : "+v"(c), "+v"(o));
        return (c + cb * H::CH + l * (H::CH / 2) < C ? o : (int)0x80000000) + (cb * LP + l) * 128;
    };
    u32x4_t raw[kRound ? WX : 1][2][LP];
    auto load_x = [&](const __amdgpu_buffer_rsrc_t &rs, int u, int h) {
        const int cb = u / N, j = u % N;
#pragma unroll
        for (int l = 0; l < LP; l++) {
            const u32x4_t t = __builtin_amdgcn_raw_buffer_load_b128(rs, piece(cb, l) + j * stream + h * rows8, 0, 0);
            if constexpr (kRound) {
                raw[u % WX][h][l] = t;
            } else {
                xr[cb][j][h][0] = t[0]; xr[cb][j][h][1] = t[1]; xr[cb][j][h][2] = t[2]; xr[cb][j][h][3] = t[3];
            }
        }
    };
    u32x4_t ph[WP][H::FU];
    const __amdgpu_buffer_rsrc_t prs = held_rsrc(a.frag, a.frag_bytes);
    const int poff = chunk0 * N * H::FU * 1024 + lane * 16;
    auto load_phi = [&](int u) {
#pragma unroll
        for (int f = 0; f < H::FU; f++) ph[u % WP][f] = __builtin_amdgcn_raw_buffer_load_b128(prs, poff + (u * H::FU + f) * 1024, 0, 0);
    };
    // a unit on its way from rows to operand layout, through the wave's own LDS (no barrier)
    unsigned char *const st_w = &stage_s[wave][r8 * kPitch + seg * (16 / LP)];
    const unsigned char *const st_r = &stage_s[wave][(lane & 15) * kPitch + (lane >> 4) * 16];
    auto stage = [&](int u) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            auto &x = xr[u / N][u % N][h];
            unsigned char *to = st_w + (u & 1) * kStage + h * 8 * kPitch;
            if constexpr (kRound) {
#pragma unroll
                for (int l = 0; l < LP; l++) {
                    const u32x4_t t = raw[u % WX][h][l];
                    x[2 * l] = pack_bf16x2(__uint_as_float(t[0]), __uint_as_float(t[1]));
                    x[2 * l + 1] = pack_bf16x2(__uint_as_float(t[2]), __uint_as_float(t[3]));
                    *reinterpret_cast<uint2 *>(to + l * 64) = make_uint2(x[2 * l], x[2 * l + 1]);
                }
            } else {
                *reinterpret_cast<uint4 *>(to) = make_uint4(x[0], x[1], x[2], x[3]);
            }
        }
    };
    u32x4_t xf[2];
    auto operands = [&](int u) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < 2; h++) xf[h] = *reinterpret_cast<const u32x4_t *>(st_r + (u & 1) * kStage + h * 64);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto product = [&](const u32x4_t &p, const u32x4_t &x, f32x4_t acc) {
        if constexpr (kExact) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(p[e]), __uint_as_float(x[e]), acc, 0, 0, 0);
            return acc;
        } else {
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, p), __builtin_bit_cast(bf16x8_t, x), acc, 0, 0, 0);
        }
    };
    // the words of a piece as values of their own: nothing computed from them before is kept in registers until here
    auto opaque = [&](int cb, int h) {
#pragma unroll
        for (int j = 0; j < N; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) asm volatile("" : "+v"(xr[cb][j][h][i]));
    };
    // the streams of channel v of a piece as an operand of the 4 x 4 x 4 products
    auto channel = [&](int cb, int h, int v) {
        const int p = v >> 1;
        const uint32_t w0 = xr[cb][0][h][p], w1 = xr[cb][1][h][p], w2 = N > 2 ? xr[cb][N > 2 ? 2 : 0][h][p] : 0u,
                       w3 = N > 3 ? xr[cb][N > 3 ? 3 : 0][h][p] : 0u;
        return (v & 1) ? streams_of_channel<true>(w0, w1, w2, w3) : streams_of_channel<false>(w0, w1, w2, w3);
    };
    auto value = [&](int cb, int j, int h, int v) {
        if constexpr (kExact) return __uint_as_float(xr[cb][j][h][v]);
        else return (v & 1) ? bf16hi_to_f32(xr[cb][j][h][v >> 1]) : bf16lo_to_f32(xr[cb][j][h][v >> 1]);
    };
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};

    int tile = blockIdx.x;
    {
        const __amdgpu_buffer_rsrc_t rs = rsrc_of(a.x, tile);
#pragma unroll
        for (int u = 0; u < WX; u++) {
            load_x(rs, u, 0);
            load_x(rs, u, 1);
        }
    }
    for (; tile < a.tiles; tile += gridDim.x) {
        const __amdgpu_buffer_rsrc_t rs = rsrc_of(a.x, tile);
        // ---- projection and sum of squares -------------------------------------------------------
#pragma unroll
        for (int u = 0; u < WP; u++) load_phi(u);
        // The products of kFold units are summed on the matrix cores and then added to the wave's sums, to each of kSums in turn: a
        // chain over all units loses bits (error of P against float64, one chain | this | the two-launch forward: bf16 n=4 B=3001 C=2560
        // 2.0e-7 | 1.1e-7 | 1.4e-7, float32 2560 1280 4.2e-7 | 1.5e-7 | 2.4e-7)
        f32x4_t sum[kSums][H::kTiles], acc[N == 4 ? 3 : (N == 2 ? 2 : 1)];
#pragma unroll
        for (auto &k : sum)
#pragma unroll
            for (auto &t : k) t = zero;
        float ssx[2] = {0.f, 0.f};
        stage(0);
        operands(0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u + 1 < U) stage(u + 1);
            const auto &p = ph[u % WP];
            if (u % kFold == 0) {
#pragma unroll
                for (auto &t : acc) t = zero;
            }
            if constexpr (N == 4) {
                acc[0] = product(p[0], xf[0], acc[0]);
                acc[1] = product(p[2], xf[0], acc[1]);
                acc[0] = product(p[1], xf[1], acc[0]);
                acc[2] = product(p[2], xf[1], acc[2]);
            } else if constexpr (N == 3) {
                acc[0] = product(p[0], xf[0], acc[0]);
                acc[0] = product(p[1], xf[1], acc[0]);
            } else {
                acc[0] = product(p[0], xf[0], acc[0]);
                acc[1] = product(p[0], xf[1], acc[1]);
            }
            if (u % kFold == kFold - 1 || u == U - 1) {
                auto &to = sum[u / kFold % kSums];
                if constexpr (N != 2) to[0] += acc[0];
                if constexpr (N != 3) {  // paired rows: one half of the lanes holds either product
                    const f32x4_t &lo = acc[N == 4 ? 1 : 0], &hi = acc[N == 4 ? 2 : 1];
#pragma unroll
                    for (int r = 0; r < 4; r++) to[H::kTiles - 1][r] += lane < 32 ? lo[r] : hi[r];
                }
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float t = 0.f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (kExact) {
                        const float v = __uint_as_float(xr[u / N][u % N][h][i]);
                        t = __builtin_fmaf(v, v, t);
                    } else {
                        const bf16x2_t pr = __builtin_bit_cast(bf16x2_t, xr[u / N][u % N][h][i]);
                        t = __builtin_amdgcn_fdot2_f32_bf16(pr, pr, t, false);
                    }
                }
                ssx[h] += t;
            }
            if (u + WX < U) {
                load_x(rs, u + WX, 0);
                load_x(rs, u + WX, 1);
            }
            if (u + WP < U) load_phi(u + WP);
            if (u + 1 < U) operands(u + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 0; t < H::kTiles; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) red(wave, t, r, lane) = kSums == 2 ? sum[0][t][r] + sum[kSums - 1][t][r] : sum[0][t][r];
        auto row_sum = [&](float v) {  // over the eight lanes that hold a row
            v += dpp_mov<kDppQuadXor1>(v);
            v += dpp_mov<kDppQuadXor2>(v);
            return v + dpp_mov<kDppRowHalfMirror>(v);
        };
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float v = row_sum(ssx[h]);
            if (seg == 0) ssx_s[wave][h * 8 + r8] = v;
        }
        __syncthreads();

        // ---- coefficients on the first four waves ------------------------------------------------
        const int b = tile * a.S + sc;
        const bool sv = sc < a.S && b < a.B;
        const size_t bb = (size_t)(sv ? b : a.B - 1);
        float m[1] = {0.f};
        if (wave < 4) {
            // row d of the product for sample sc, summed over the waves
            auto psum = [&](int d) {
                constexpr int last = H::kTiles - 1;
                const bool paired = N == 2 || (N == 4 && d >= 16);
                const int t = paired ? last : 0, rr = paired ? (d & 7) : d;
                const int o0 = (rr >> 2) * 16 + sc, o1 = ((8 + rr) >> 2) * 16 + sc;
                return held_wave_sum<NW>([&](int w2) {
                    float v = red(w2, t, rr & 3, o0);
                    if constexpr (N != 3) {
                        const float o = red(w2, t, rr & 3, o1 & 63);
                        v += paired ? o : 0.f;
                    }
                    return v;
                });
            };
            const float pvec = psum(vv ? g : 0), pe = psum(mv ? 2 * N + r0 * N + c0 : 0);
            const float ssq = held_wave_sum<NW>([&](int w2) { return ssx_s[w2][sc]; });
            const float ms = kFine ? ssq / (float)nC + a.eps : ssq * (1.0f / (float)nC) + a.eps;
            const float r = kFine ? sqrtf(ms) : __builtin_amdgcn_sqrtf(ms);
            const float rinv = kFine ? 1.0f / r : fast_rcp(r);
            if (sv && g == 0) a.r[bb] = r;
            if (vv) {
                const bool pre = g < N;
                const float p = pvec * rinv, z = al0 * p + bvec;
                const float sg = kFine ? sigmoidf_acc(z) : sigmoid_fast(z);
                const float h = pre ? sg : 2.0f * sg;
                coef_s[sc * kCoef + 16 + (pre ? g : 4 + g - N)] = h;
                if (sv) {
                    (pre ? a.Hpre : a.Hpost)[bb * N + (pre ? g : g - N)] = h;
                    a.P[bb * D + g] = p;
                }
            } else if (g < 8) {  // the padded entries, met by zero streams only
                const int k = g - 2 * N;
                coef_s[sc * kCoef + 16 + (k < 4 - N ? N + k : 4 + N + (k - (4 - N)))] = 0.f;
            }
            if (mv) {
                const float p = pe * rinv;
                if (sv) a.P[bb * D + 2 * N + r0 * N + c0] = p;
                m[0] = kFine ? expf(al2 * p + bres) : exp_fast(al2 * p + bres);
            }
        }
        __syncthreads();
        if (wave < 4) {
            if (a.sk_state) {  // (whole groups of 16 lanes: samples beyond the batch keep no state)
                if (sv) SK::template forward_save<kFine>(m, g, N, a.T, a.eps, a.sk_state + bb * SK::state_floats(a.T));
            } else {
                SK::template forward<kFine, false>(m, g, N, a.T, a.eps, nullptr, lane);
            }
            coef_s[sc * kCoef + r0 * 4 + c0] = m[0];
            if (sv && mv) a.M[bb * N * N + r0 * N + c0] = m[0];
        }
        // ---- RMS of the aggregate ----------------------------------------------------------------
        const bool jq0 = (lane & 3) == 0;
        auto hpre_of = [&](int h, float (&hp)[4]) {
            const float4 t = *reinterpret_cast<const float4 *>(coef_s + (h * 8 + r8) * kCoef + 16);
            hp[0] = t.x; hp[1] = t.y; hp[2] = t.z; hp[3] = t.w;
        };
        auto agg_row = [&](const float (&hp)[4]) {
            CoefRow ca;
            ca.set(jq0 ? hp[0] : 0.f, jq0 ? hp[1] : 0.f, jq0 ? hp[2] : 0.f, jq0 ? hp[3] : 0.f);
            return ca;
        };
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float hp[4], ss = 0.f;
            hpre_of(h, hp);
            const CoefRow ca = agg_row(hp);
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                opaque(cb, h);
                float part[2] = {0.f, 0.f};
#pragma unroll
                for (int v = 0; v < VE; v++) {
                    float t;
                    if constexpr (kFine) {
                        t = hp[0] * value(cb, 0, h, v);
#pragma unroll
                        for (int j = 1; j < N; j++) t = __builtin_fmaf(hp[j], value(cb, j, h, v), t);
                    } else {
                        const bf16x4_t bx = channel(cb, h, v);
                        t = mfma4(ca.lo, bx, mfma4(ca.hi, bx, zero))[0];
                    }
                    part[v & 1] = __builtin_fmaf(t, t, part[v & 1]);
                }
                ss += part[0] + part[1];
                __builtin_amdgcn_sched_barrier(0);
            }
            const float v = row_sum(ss);
            if (seg == 0) ssa_s[wave][h * 8 + r8] = v;
        }
        __syncthreads();
        // ---- mix; the next tile's first units are requested as registers fall free ---------------------
        const __amdgpu_buffer_rsrc_t yrs = rsrc_of(a.y, tile), nrs = rsrc_of(a.x, tile + gridDim.x);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int row = h * 8 + r8;
            const float ss = held_wave_sum<NW>([&](int w2) { return ssa_s[w2][row]; });
            const float q = sqrtf(ss / (float)C + a.eps), qinv = 1.0f / q;
            if (wave == 0 && seg == 0 && row < a.S && tile * a.S + row < a.B) a.q[tile * a.S + row] = q;
            float hp[4], hq[4];
            hpre_of(h, hp);
            {
                const float4 t = *reinterpret_cast<const float4 *>(coef_s + row * kCoef + 20);
                hq[0] = t.x; hq[1] = t.y; hq[2] = t.z; hq[3] = t.w;
            }
            const CoefRow ca = agg_row(hp);
            CoefRow cm;
            float M[kFine ? N : 1][4];
            if constexpr (kFine) {
#pragma unroll
                for (int i = 0; i < N; i++) {
                    const float4 t = *reinterpret_cast<const float4 *>(coef_s + row * kCoef + i * 4);
                    M[i][0] = t.x; M[i][1] = t.y; M[i][2] = t.z; M[i][3] = t.w;
                }
            } else {
                const float4 t = *reinterpret_cast<const float4 *>(coef_s + row * kCoef + (lane & 3) * 4);
                cm.set(t.x, t.y, t.z, t.w);
            }
#pragma unroll
            for (int cb = 0; cb < CB; cb++) {
                opaque(cb, h);
                float wv[VE];
#pragma unroll
                for (int v = 0; v < VE / 4; v++) {
                    const float4 t = *reinterpret_cast<const float4 *>(w_s + c_lane + cb * H::CH + v * (LP == 2 ? H::CH / 2 : 4));
                    wv[4 * v] = t.x; wv[4 * v + 1] = t.y; wv[4 * v + 2] = t.z; wv[4 * v + 3] = t.w;
                }
                uint32_t yw[N][4 * LP];
                if constexpr (kFine) {
#pragma unroll
                    for (int v = 0; v < VE; v++) {
                        float xv[N];
#pragma unroll
                        for (int j = 0; j < N; j++) xv[j] = value(cb, j, h, v);
                        float t = hp[0] * xv[0];
#pragma unroll
                        for (int j = 1; j < N; j++) t = __builtin_fmaf(hp[j], xv[j], t);
                        const float f = t * qinv * wv[v];
#pragma unroll
                        for (int i = 0; i < N; i++) {
                            float o = M[i][0] * xv[0];  // (the largest term last: one rounding at its size)
#pragma unroll
                            for (int j = 1; j < N; j++) o = __builtin_fmaf(M[i][j], xv[j], o);
                            yw[i][v] = __float_as_uint(__builtin_fmaf(hq[i], f, o));
                        }
                    }
                } else {
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        f32x4_t d[2];
                        float f[2];
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            const bf16x4_t bx = channel(cb, h, 2 * p + e);
                            d[e] = mfma4(cm.lo, bx, mfma4(cm.hi, bx, zero));
                            f[e] = mfma4(ca.lo, bx, mfma4(ca.hi, bx, zero))[0] * qinv * wv[2 * p + e];
                        }
#pragma unroll
                        for (int i = 0; i < N; i++) yw[i][p] = pack_bf16x2(d[0][i] + hq[i] * f[0], d[1][i] + hq[i] * f[1]);
                    }
                }
#pragma unroll
                for (int l = 0; l < LP; l++) {
                    const int o = piece(cb, l) + h * rows8;
#pragma unroll
                    for (int i = 0; i < N; i++)
                        __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{yw[i][4 * l], yw[i][4 * l + 1], yw[i][4 * l + 2], yw[i][4 * l + 3]},
                                                               yrs, o + i * stream, 0, ST);
                }
#pragma unroll
                for (int u = cb * N; u < (cb + 1) * N; u++)
                    if (u < WX) load_x(nrs, u, h);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// Units of phi requested ahead (more, or x further ahead than four units, cost registers and gain nothing: n=4 B=8192 C=2560 69.5,
// three and six 70.6, three and eight 71.1) and the cache policy of the stores (nt: 69, without 92, y then evicts x and phi).
constexpr int kHeldWP = 2, kHeldST = 2;

template <typename TS, typename TX, int N, int CB, int NW> static hipError_t launch_held(HeldArgs a, hipStream_t stream) {
    constexpr int U = CB * N, W = sizeof(TS) > sizeof(TX) ? 2 : 4, WX = W < U ? W : U;
    constexpr auto kernel = &layer_fwd_held_kernel<TS, TX, N, CB, NW, WX, kHeldWP, kHeldST>;
    const size_t smem = (size_t)NW * CB * HeldShape<TX, N>::CH * 4;
    const int most = 256 * (held_waves(N * CB) * 4 / NW);
    const int tiles = (a.B + kHeldS - 1) / kHeldS, rounds = (tiles + most - 1) / most;
    // a last round that would leave most CUs idle: all rounds equally full instead (n=4 B=4400 C=2560 57 -> 51 us; no gain where
    // it is half full, B=6500 61 | 61, C=1280 30.8 | 32.5, nor in a single round, where it only multiplies the reads of phi)
    if (rounds > 1 && tiles - (rounds - 1) * most <= most / 2) a.S = (a.B + rounds * most - 1) / (rounds * most);
    a.tiles = (a.B + a.S - 1) / a.S;
    if (hipError_t e = allow_dynamic_lds<kernel>(smem + 64 * 1024); e != hipSuccess) return e;
    kernel<<<a.tiles < most ? a.tiles : most, NW * 64, smem, stream>>>(a);
    return hipGetLastError();
}

// units (stream of a chunk) that a wave's registers hold
constexpr int held_most_cb(int n) { return n == 4 ? 5 : (n == 3 ? 6 : 10); }
template <typename TS, typename TX, int N> static hipError_t launch_held_by_size(const HeldArgs &a, hipStream_t stream) {
    const int nch = (a.C + HeldShape<TX, N>::CH - 1) / HeldShape<TX, N>::CH;
// (eight waves for the rows that four do not hold: no form that nothing reaches)
#define MHC_HELD(CB, NW) \
    if constexpr (CB <= held_most_cb(N) && (NW == 4 || CB * NW > 4 * held_most_cb(N))) { if (nch <= CB * NW) return launch_held<TS, TX, N, CB, NW>(a, stream); }
    MHC_HELD(1, 4) MHC_HELD(2, 4) MHC_HELD(3, 4) MHC_HELD(4, 4) MHC_HELD(5, 4) MHC_HELD(6, 4) MHC_HELD(8, 4) MHC_HELD(10, 4)
    MHC_HELD(3, 8) MHC_HELD(4, 8) MHC_HELD(5, 8) MHC_HELD(6, 8) MHC_HELD(8, 8) MHC_HELD(10, 8)
#undef MHC_HELD
    return hipErrorInvalidValue;
}

static int held_chunk(int x_dtype) { return x_dtype == kF32 ? 32 : 64; }
static int held_units(int x_dtype, int n, int C) { return (C + held_chunk(x_dtype) - 1) / held_chunk(x_dtype) * n; }
size_t layer_fwd_held_bytes(int x_dtype, int n, int C) { return (size_t)held_units(x_dtype, n, C) * (n - 1) * 1024; }

// Rows of whole 128-byte lines; the lines in B stand where two launches and this one cost the same.  Forward us, the forward of
// before | this one, on either side:
//   bf16     n=4 C=704 B=2047 11.0 | 13.3, 2160 14.7 | 13.3;  1280 2047 14.8 | 18.7, 2160 21.8 | 18.5;  1536 2000 18.7 | 18.9;  1920 1500
//            18 | 22, 1613 23 | 22;  2560 1333 25 | 26, 1613 27 | 26;  n=3 1664 2047 14 | 17, 2160 22 | 17;  3072 1333 23 | 23;  n=2 5120
//            1333 38 | 26  (the two-launch forward has a step where x outgrows the L2)
//            beside the one-launch forward: n=4 512 4000 12 | 13, 4400 21 | 16;  n=3 1280 3500 17 | 17, 4000 31 | 19;  n=2 2560 2450
//            18 | 22, 2700 34 | 22;  shorter rows n=4 256 8192 12 | 13, 12000 19 | 16, 20000 28 | 28;  from the caller's fp32
//            parameters, which that one has packed by a launch there: n=4 64 8192 11.8 | 12.0, 128 4500 11.6 | 11.6, 256 4500 13.1 | 11.8, n=3
//            128 4500 11.0 | 10.6, n=2 256 8192 11.7 | 10.8, 640 4500 20.2 | 13.6
//   float32  n=2 640 1000 12.3 | 12.5, 1060 12.9 | 12.5;  768 1060 13.3 | 13.4, 1350 14.3 | 13.7;  896 1150 13.8 | 15.0, 1350 15.0 | 15.1, 1500
//            15.5 | 15.3;  1152 1100 16.2 | 16.6, 1250 16.6 | 16.6;  1664 1200 17.5 | 18.3, 1250 18.5 | 18.4;  2048 1030 18.6 | 19.4, 1150 19.5
//            | 18.4;  2560 1000 20.2 | 21.3, 1030 26.0 | 21.3;  n=3 384 1000 12.2 | 12.1, 1060 13.2 | 12.1;  576 1150 13.5 | 14.5, 1200 14.9 |
//            14.6;  640 1000 13.4 | 14.5, 1100 15.1 | 14.5;  768 1300 15.4 | 15.9, 1400 16.7 | 16.0;  832 1060 15.7 | 15.8, 1200 15.6 | 15.5;
//            1152 1150 17.0 | 17.4, 1200 18.5 | 17.5;  1536 1000 19.5 | 19.3, 1060 20.7 | 19.4;  n=4 384 1500 14.7 | 15.0, 1900 15.4 | 15.0;
//            448 1950 17.0 | 17.4, 2100 18.0 | 17.4;  1024 1500 21.9 | 23.5, 1850 29.3 | 24.6;  1152 1950 26.9 | 28.3, 2100 32.9 | 28.4;  1280
//            1500 25.6 | 26.5, 1850 29.7 | 28.4
//   float32 storage  n=2 640 1330 12.5 | 12.3, 1600 13.0 | 12.5;  896 1500 14.1 | 14.4, 1700 14.5 | 14.3;  1280 1500 15.9 | 16.7, 1600 20.0 |
//            16.5;  n=3 512 1500 13.4 | 12.8, 1650 13.7 | 12.9;  640 1900 15.1 | 15.4, 2100 17.3 | 15.5;  704 1600 15.0 | 15.7, 1750 16.6 |
//            15.6;  1024 1700 18.3 | 19.5, 1800 22.1 | 19.3;  1152 1500 18.6 | 19.3, 1600 23.0 | 19.1;  1344 1650 25.8 | 26.5, 1850 26.6 | 26.1;
//            2048 1150 23.4 | 21.5, 1300 29.5 | 21.5;  n=4 320 2200 14.6 | 15.0, 2400 15.2 | 15.3;  512 2300 17.4 | 17.7, 2400 17.7 | 17.0;
//            1024 2100 28.4 | 24.3, 2200 29.0 | 24.4;  1280 2100 30.6 | 30.9, 2400 32.2 | 32.3;  1536 1150 23.2 | 22.5, 1330 25.2 | 23.0;  2304
//            1150 32.3 | 34.0, 1400 36.5 | 35.2
// In float32 and float32 storage the lines go by the registers of a row's form: where another number of chunks per wave begins (768 ->
// 832 channels at n = 2) a tile costs as much as one of the longest rows of that form.
constexpr BatchLine kHeldF32N2[] = {{448, 1000}, {640, 1030}, {768, 1150}, {1024, 1350}, {1280, 1200}, {1536, 1000}, {1856, 1250}, {2048, 1080}, {kAnyRow, 1030}};
constexpr BatchLine kHeldF32N3[] = {{256, 1000}, {384, 1030}, {576, 1200}, {640, 1050}, {768, 1400}, {1024, 1100}, {1344, 1175}, {kAnyRow, 1050}};
constexpr BatchLine kHeldF32N4[] = {{384, 1850}, {512, 2050}, {1024, 1850}, {1152, 2050}, {kAnyRow, 1850}};
constexpr BatchLine kHeldStoredN2[] = {{3071, 1600}, {kAnyRow, 1300}};
constexpr BatchLine kHeldStoredN3[] = {{512, 1600}, {640, 2050}, {768, 1720}, {1024, 1800}, {1280, 1600}, {1344, 1800}, {2047, 1600}, {kAnyRow, 1300}};
constexpr BatchLine kHeldStoredN4[] = {{256, 2200}, {320, 2400}, {512, 2350}, {1024, 2200}, {1280, 2300}, {1535, 2200}, {kAnyRow, 1300}};
bool layer_fwd_held_supported(int x_dtype, int y_dtype, int phi_dtype, int B, int n, int C, bool from_params) {
    if (n < 2 || n > 4 || C % held_chunk(x_dtype) != 0 || C / held_chunk(x_dtype) > 8 * held_most_cb(n)) return false;
    const bool types = (x_dtype == kBF16 && y_dtype == kBF16 && phi_dtype == kBF16) || (x_dtype == kF32 && y_dtype == kF32 && phi_dtype == kF32) ||
                       (x_dtype == kF32AsBF16 && y_dtype == kF32 && phi_dtype == kBF16);
    if (!types) return false;
    const int hook = tuning_get(kTuneOnepassOff);
    if (hook) return hook == 3;
    const int nC = n * C;
    if (x_dtype == kF32) return B >= (n == 4 ? batch_line(kHeldF32N4, C) : n == 3 ? batch_line(kHeldF32N3, C) : batch_line(kHeldF32N2, C));
    if (x_dtype == kF32AsBF16) return B >= (n == 4 ? batch_line(kHeldStoredN4, C) : n == 3 ? batch_line(kHeldStoredN3, C) : batch_line(kHeldStoredN2, C));
    // (where the one-launch forward of layer_fwd_onepass.hip stands beside it: from its second round of workgroups on)
    if (layer_fwd_onepass_supported(x_dtype, phi_dtype, B, n, C))
        return (nC >= 1536 || (from_params && C >= 128)) && B > 256 * layer_fwd_onepass_most_samples(n, C);
    return B >= (nC <= 6144 ? 2100 : (n < 4 && nC >= 9216 ? 1333 : 1600));
}

hipError_t launch_layer_fwd_held(const void *x, int x_dtype, const void *w, int w_dtype, void *y, const ParamGather *gather, const void *phi,
                                 const float *alpha, const float *bias, void *frag, float *Hpre, float *Hpost, float *M, float *P,
                                 float *r, float *q, float *sk_state, int B, int n, int C, int T, float eps, hipStream_t stream) {
    const bool exact = x_dtype == kF32;
    const size_t nC = (size_t)n * C, es = exact ? 4 : 2;
    HeldPackArgs pa{};
    const char *base = static_cast<const char *>(phi);
    for (int i = 0; i < 3; i++) {
        pa.src[i] = gather ? gather->phi[i] : base + (size_t)(i == 0 ? 0 : (i == 1 ? n : 2 * n)) * nC * es;
        if (gather) { pa.b[i] = gather->b[i]; pa.alpha_in[i] = gather->alpha[i]; }
    }
    if (gather) { pa.phi_out = gather->phi_out; pa.bias = gather->bias_out; pa.alpha = gather->alpha_out; }
    pa.frag = frag; pa.C = C; pa.units = held_units(x_dtype, n, C);
    const unsigned grid = (unsigned)((pa.units * (n - 1) * 64 + 255) / 256);
    const bool sf32 = gather ? gather->phi_dtype == kF32 : exact;
    const HeldArgs a{x, w, frag, y, alpha, bias, Hpre, Hpost, M, P, r, q, sk_state, w_dtype == kBF16, B, C, T, kHeldS, 0,
                     (int)layer_fwd_held_bytes(x_dtype, n, C), eps};
#define MHC_HELD_N(TX, N)                                                       \
    do {                                                                        \
        if (sf32) held_pack_kernel<float, TX, N><<<grid, 256, 0, stream>>>(pa); \
        else held_pack_kernel<bf16_t, TX, N><<<grid, 256, 0, stream>>>(pa);     \
    } while (0)
#define MHC_HELD_TYPES(N)                                                                       \
    do {                                                                                        \
        if (exact) {                                                                            \
            MHC_HELD_N(float, N);                                                               \
            return launch_held_by_size<float, float, N>(a, stream);                             \
        }                                                                                       \
        MHC_HELD_N(bf16_t, N);                                                                  \
        if (x_dtype == kF32AsBF16) return launch_held_by_size<float, bf16_t, N>(a, stream);     \
        return launch_held_by_size<bf16_t, bf16_t, N>(a, stream);                               \
    } while (0)
    if (n == 4) MHC_HELD_TYPES(4);
    if (n == 3) MHC_HELD_TYPES(3);
    MHC_HELD_TYPES(2);
#undef MHC_HELD_TYPES
#undef MHC_HELD_N
}

}  // namespace mhc
