// C ABI of libmhc_hip.so (declared in include/mhc_hip.h): argument validation, workspace
// carving and the launch sequence of each entry point.  No allocation, no synchronisation,
// no global state; every call only enqueues kernels on the caller's stream.  The one exception
// is mhc_layer_fwd_dynamic_static_scratch at the end of this file, whose scratch memory is a
// device array owned by the library.
#include "../../include/mhc_hip.h"

#include "launchers.h"
#include "phase_profiler.h"
#include "tuning.h"

#include <algorithm>
#include <mutex>
#include <stdint.h>

using namespace mhc;

#ifdef MHC_TUNING
namespace mhc {
int g_tuning[kTuneCount];
}
#endif

namespace {

struct Carver {
    char *base;
    size_t off = 0;
    explicit Carver(void *p) : base(static_cast<char *>(p)) {}
    float *floats(size_t count) {
        float *p = base ? reinterpret_cast<float *>(base + off) : nullptr;
        off += (count * sizeof(float) + 255) / 256 * 256;
        return p;
    }
};

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool valid_dtype(int d) { return d == MHC_F32 || d == MHC_BF16; }
inline bool valid_io(int x_dtype, int y_dtype) {
    // activations in / out: (f32, f32), (bf16, bf16), (bf16 in, f32 out), (f32 consumed as bf16 in, f32 out)
    return (x_dtype == MHC_F32 && y_dtype == MHC_F32) || (x_dtype == MHC_BF16 && valid_dtype(y_dtype)) ||
           (x_dtype == MHC_F32_AS_BF16 && y_dtype == MHC_F32);
}

int check_shape(int B, int n, int C, int iters) {
    if (n < 1 || n > MHC_MAX_N) return MHC_ERR_BAD_N;
    if (B < 1 || C < 1 || iters < 0 || iters > max_layer_sinkhorn_iters(n)) return MHC_ERR_BAD_SHAPE;
    if ((long long)B * n * C > (1ll << 40)) return MHC_ERR_BAD_SHAPE;
    if (C > MHC_MAX_C) return MHC_ERR_BAD_SHAPE;       // the generic kernels keep a [C] float row in LDS
    return MHC_OK;
}

int ws_check(void *ws, size_t have, size_t need) {
    if (need == 0) return MHC_OK;
    if (!ws || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0 || have < need) return MHC_ERR_WORKSPACE;
    return MHC_OK;
}

#define MHC_LAUNCH(expr)                              \
    do {                                              \
        if ((expr) != hipSuccess) return MHC_ERR_LAUNCH; \
    } while (0)

// ---- dynamic workspace layout ----------------------------------------------------------------
struct DynFwdWs { float *Ppart, *ssqpart, *agg; size_t part_bytes, bytes; };  // Ppart (part_bytes): partial sums, or phi for the held forward
struct DynBwdWs { float *dt, *dP, *cx, *s1, *u, *upart, *dtpart, *raw, *s1part, *dx_part, *dxp, *dphi_part; unsigned short *dPb, *dPT; int BP; size_t bytes; };

// Whether the sample-resident backward (bwd_resident.hip + the column-slab kernel) is taken where it is
// supported.  Its second launch walks all samples of a column slab in one workgroup, which stops paying once the batch is
// large enough to fill the chip with batch splits; the fewer streams, the fewer slabs.
// Measured, backward in graphs of ten, tiled (Gram + slab) path | resident path (us), in each row from below the line to above it.
// Single rows jump by a few us with B mod 32 and the tiles per split; the lines are fitted to 1500 shapes of all remainders.
//   n=1 C=128:  B=850 17.1 | 18.4, 1500 16.7 | 23.2, 2000 19.5 | 17.5, 2800 18.9 | 20.4;  C=256: 652 18.8 | 17.8, 850 17.8 | 19.0,
//               1500 17.8 | 24.9, 2000 21.2 | 19.0, 2800 20.8 | 22.6;  C=640: 559 18.9 | 17.5, 671 15.7 | 16.0
//       C=1280: 437 17.3 | 15.6, 614 20.9 | 22.4;  C=1920: 354 20.6 | 18.0, 543 17.2 | 20.2;  C=3200: 206 17.9 | 15.7, 300 19.3 | 19.8
//   n=2 C=128:  850 19.2 | 19.0, 1000 21.3 | 21.7, 1500 19.5 | 24.2, 2800 22.5 | 21.7, 3700 23.7 | 25.1;  C=256: 850 19.6 | 19.6,
//               1000 21.6 | 22.3, 1500 19.8 | 25.7, 2000 23.2 | 20.0, 2800 23.3 | 24.7;  C=384: 676 22.5 | 19.9, 960 17.2 | 19.0
//       C=1280: 495 19.9 | 17.3, 659 19.9 | 21.3;  C=1920: 354 21.9 | 18.2, 447 16.5 | 17.4;  C=3200: 212 17.9 | 16.9, 265 21.3 | 23.0
//       C=4096: 172 20.0 | 19.0, 212 18.5 | 20.1
//   n=3 C=128:  1000 23.4 | 22.2, 1500 21.7 | 24.8, 2800 24.8 | 22.9, 3700 26.1 | 26.5;  C=256: 1200 24.0 | 24.2, 1500 21.9 | 27.2,
//               2000 25.5 | 22.0, 2800 26.2 | 27.1;  C=384: 721 22.0 | 17.7, 816 22.3 | 20.3 (rounded twice), 1152 22.0 | 22.6
//       C=1280: 593 23.5 | 21.7, 764 21.7 | 23.2;  C=1920: 472 21.0 | 19.7, 577 27.6 | 27.3, 700 22.2 | 24.5;  C=2560: 310 21.3 | 22.7,
//               444 21.6 | 25.1;  C=4096: 242 23.4 | 22.3, 266 27.0 | 30.4
//   n=4 C=128:  1000 22.1 | 21.2, 1500 21.1 | 24.9, 2800 24.1 | 23.2, 3700 26.6 | 26.6, 4300 29.4 | 31.1;  C=256: 1200 23.5 | 24.0, 1500
//               21.9 | 27.4, 2000 25.5 | 23.1, 2800 26.2 | 26.8;  C=264: 687 21.9 | 17.2, 816 22.0 | 19.5 (rounded twice), 1152
//               22.9 | 22.0, 1392 25.3 | 26.1;  C=384: 816 21.7 | 20.4, 960 19.7 | 20.6 (the step at 256 channels: up to there a
//               workgroup of the resident path has two tile waves instead of four, and more workgroups fit a CU)
//       C=1280: 473 21.0 | 18.1, 624 24.2 | 23.6, 729 22.3 | 24.1;  C=1920: 424 25.0 | 22.9, 489 24.6 | 24.4, 611 28.2 | 30.7
//       C=2560: 331 25.8 | 24.7, 450 27.9 | 29.2;  C=3200: 247 23.6 | 22.4, 364 27.7 | 28.4;  C=4096: 235 26.6 | 23.9, 270 28.0 | 31.8
// (from about 2000 channels and five streams on, and 4096 and three, one workgroup of the resident path fills a CU: the step at 256)
// n = 5 .. 8, where the slab is bwd_slab8.hip:
//   n=5 C=64: 1200 23.9 | 22.1, 1600 25.2 | 26.7, 8192 49.0 | 58.4; C=256: 1200 25.9 | 26.0, 4000 36.0 | 47.6, 8192 51.4 | 80.7
//       C=384: 565 24.7 | 23.7, 655 26.8 | 26.9, 829 26.0 | 30.0; C=1280: 382 25.9 | 25.1, 518 31.4 | 36.7; C=2560: 245 30.3 |
//       25.1, 273 30.8 | 35.0; C=4096: 225 36.7 | 30.9, 291 39.6 | 46.9
//   n=6 C=64: 4000 37.2 | 37.4, 4125 42.3 | 39.6, 8192 51.8 | 59.1; C=256: 1200 28.9 | 27.1, 1600 30.4 | 32.1, 8192 55.4 | 76.9
//       C=384: 655 29.3 | 27.2, 765 27.3 | 29.0; C=768: 647 32.8 | 32.0, 790 30.8 | 35.0; C=1280: 472 29.9 | 27.8, 527 33.5 |
//       36.1; C=2560: 256 31.8 | 25.1, 307 35.4 | 36.4; C=4096: 227 41.3 | 33.3, 291 44.7 | 48.9
//   n=7 C=64: 4000 40.1 | 37.8, 8192 54.6 | 60.5; C=256: 1600 32.4 | 32.6, 4000 42.8 | 49.7, 8192 60.7 | 83.0 (with the
//       forward: C=192 2126 53.8 | 51.3, 2400 54.5 | 53.3, 3000 55.9 | 63.7; C=256 2400 56.0 | 55.0, 3000 56.6 | 62.6); C=384: 777 35.6 |
//       31.4, 1024 31.8 | 32.9, 1163 39.3 | 36.9; C=768: 680 36.0 | 32.7, 832 34.2 | 35.2, 1087 40.4 | 41.4; C=1280: 455 37.4 |
//       32.3, 705 42.0 | 44.9; C=2560: 361 42.7 | 41.7, 448 41.5 | 45.1
//   n=8 C=128: 4000 43.8 | 41.2, 8192 61.7 | 66.4; C=256: 2200 40.8 | 36.5, 4000 48.1 | 50.4, 8192 69.4 | 87.0; C=384: 1200 37.4
//       | 35.0, 1600 39.9 | 42.8 (with the forward: C=320 1500 58.1 | 55.9, 1600 58.2 | 62.6); C=512: 1200 42.2 | 40.0, 1600 43.7 | 49.5; C=1280: 569 43.5 | 42.0, 815 49.3 | 55.7; C=2560:
//       387 52.5 | 49.6, 532 56.4 | 64.1; C=4096: 344 60.8 | 58.2, 539 73.1 | 85.6
// Experiment hook: 1 = never, 2 = always.
bool bwd_resident_preferred(int B, int n, int C) {
    if (const int hook = tuning_get(kTuneResident)) return hook == 2;
    if (n > 4) {
        // (large batches of short rows: the channel sums are gram_wave_kernel there)
        const int upto128[4] = {1500, 5000, 6000, 7000}, upto256[4] = {1200, 1500, 2450, 3700};
        if (C <= 256) return B <= (C <= 128 ? upto128 : upto256)[n - 5];
        const int per_row[4] = {500'000, 680'000, 880'000, 940'000}, least[4] = {256, 256, 256, 448}, most[4] = {640, 704, 832, C <= 384 ? 1500 : 1400};
        return B <= std::min(most[n - 5], std::max(least[n - 5], per_row[n - 5] / C));
    }
    if (C <= 256) {
        // up to 1536 samples one workgroup of the second launch walks all of them, beyond the batch is split
        const int walk[4] = {768, 896, 1216, 1216}, upto128[4] = {2432, 3200, 3968, 3840}, upto256[4] = {2432, 2432, 2432, 2432};
        return B <= (B <= 1536 ? walk : (C <= 128 ? upto128 : upto256))[n - 1];
    }
    // (never beyond kResTwiceMaxB samples where dxp is handed over in bf16: dx would be rounded twice, on the tiled path once)
    const int per_row[4] = {640'000, 740'000, 900'000, 860'000}, least[4] = {0, 0, 256, 256};
    return B <= std::min(kResTwiceMaxB, std::max(least[n - 1], per_row[n - 1] / C));
}

// Whether the tiled path of n = 5 .. 8 ends in the slab kernel or in the general ones.  Small batches of rows that the resident
// path would hold get here with more than 32 Sinkhorn iterations only (backward us, general kernels | slab):
//   n=5 C=1280 B=100 26.2 | 27.0, 170 28.8 | 26.6;  n=6 C=1280 100 26.5 | 30.1, 170 29.3 | 29.9, 300 34.4 | 32.8;  n=7 C=512 170 27.4 | 29.0,
//   300 30.9 | 30.5, C=2560 100 36.4 | 37.2, 170 42.4 | 40.9;  n=8 C=512 300 31.8 | 36.1, 500 36.0 | 37.2, 700 36.7 | 36.1, C=1280
//   170 32.9 | 41.6, 300 39.8 | 41.9, 500 47.9 | 41.5, C=2560 170 44.3 | 48.3, 300 56.3 |
//   49.7, C=4096 100 43.1 | 44.5;  C=4608 64 40.0 | 35.7, 100 48.3 | 45.9
bool bwd_slab8_preferred(int B, int n, int C) {
    if (const int hook = tuning_get(kTuneSlab8)) return hook == 2;
    const int least[4] = {112, 176, 208, C <= 1280 ? 400 : 208};
    return C > kResWholeMaxC || B > least[n - 5];
}

// Shapes for which the dynamic entry points take fp32 activations that are consumed as bf16
// (MHC_F32_AS_BF16): the kernels that load fp32 storage directly are the narrow projection, the fused
// n <= 8 forward, the two launches of the sample-resident backward and, for large batches of whole lines, the tiled backward
// (bwd_f32_tiled).  Every batch size is taken: the alternative is a cast pass over x and dy.
bool f32_as_bf16_accepted(int B, int n, int C, int iters) {
    return n <= 8 && C % 8 == 0 && layer_fwd_fused_supported(n, C, kF32) &&
           bwd_resident_supported(kF32AsBF16, kF32, kBF16, n, C, iters) && proj_bwd_addx_supported(n);
}

// Whether the backward of float32 storage takes the tiled path (channel sums that leave x and dy in bf16, slab) instead of the resident
// one.  The resident path's time is a staircase: a workgroup per sample, two to eight of them on a CU by the registers and waves
// that the row takes, and it is at its best where its last round of workgroups is full (256 x 2, x 3, x 4 samples).  The lines stand behind
// the full rounds that it wins, between row lengths at which another form of it begins (items of 512 channels, with n > 4 also of 896
// and 1280).  n = 8 has slabs of 32 channels (shorter runs of a row, more partial sums) and a slab kernel with 19 registers in scratch
// memory.  Forward + backward us in graphs of ten, tiled | resident, on either side of the lines:
//   n=1 C=512: 600 27.4 | 27.6, 680 27.7 | 28.4;  C=1536: 512 30.6 | 29.9, 540 31.5 | 35.4;  C=1600: 256 26.5 | 23.3, 300 28.5 | 30.0;  C=2624:
//       340 34.2 | 33.3, 1024 51.1 | 48.1, 1060 54.2 | 59.8;  C=3584: 460 40.4 | 39.0, 540 43.3 | 46.4
//   n=2 C=512: 600 29.4 | 28.8, 768 29.3 | 30.4;  C=1024: 540 32.6 | 33.0, 600 32.6 | 33.8;  C=2048: 512 37.4 | 36.7, 540 39.8 | 43.8;  C=2624:
//       512 41.1 | 37.9, 800 51.1 | 53.0;  C=3584: 512 46.2 | 45.9, 540 50.5 | 53.2;  C=4096: 256 38.2 | 35.8, 300 42.9 | 45.4
//   n=3 C=1024: 800 40.7 | 41.1, 1024 41.5 | 43.6;  C=1280: 512 38.0 | 34.8, 540 39.4 | 40.4;  C=1536: 680 43.6 | 43.2, 800 47.0 | 50.2;
//       C=2048: 512 43.2 | 41.3, 540 46.6 | 48.1;  C=2560: 300 42.5 | 42.6, 460 45.2 | 46.0;  C=2624: 512 46.6 | 44.8, 600 53.0 | 54.1;  C=3584:
//       384 49.6 | 48.8, 420 50.7 | 52.2
//   n=4 C=1024: 1024 46.6 | 45.4, 1060 49.8 | 52.0;  C=1536: 512 44.1 | 38.4, 768 50.9 | 50.0, 800 53.8 | 55.4;  C=1600: 512 44.2 | 41.1, 600
//       47.3 | 48.5;  C=2048: 512 46.7 | 45.9, 600 52.0 | 55.7;  C=2560: 384 50.3 | 49.0, 460 52.6 | 54.4;  C=2624: 512 55.7 | 53.0, 768 69.6 |
//       72.6;  C=3584: 460 62.9 | 61.2, 540 73.7 | 74.5
//   n=5 C=384: 600 41.7 | 41.1, 680 42.5 | 44.2;  C=512: 1150 53.4 | 59.4, 1250 55.9 | 54.4, 1300 56.0 | 57.9;  C=896: 768 51.4 | 49.9, 900 57.6
//       | 59.2;  C=1664: 460 56.8 | 55.0, 540 68.7 | 74.1;  C=2560: 384 71.8 | 71.5, 460 72.3 | 75.4
//   n=6 C=384: 680 45.0 | 45.1, 768 43.5 | 45.7, 1300 56.8 | 55.6;  C=512: 768 47.4 | 48.5, 1280 58.8 | 57.0, 1300 59.0 | 61.4;  C=768: 768 53.3
//       | 51.1, 900 59.4 | 60.6;  C=896: 600 54.2 | 48.9, 1024 64.5 | 65.1;  C=1792: 460 64.4 | 62.2, 540 75.7 | 79.2;  C=2624: 512 82.8 | 81.5,
//       540 100 | 104
//   n=7 C=640: 820 58.6 | 57.4, 950 62.4 | 62.4;  C=768: 1024 68.0 | 66.1, 1280 75.4 | 78.1;  C=896: 768 64.0 | 58.6, 1280 86.4 | 84.9, 1536
//       94.7 | 95.3;  C=1024: 512 53.7 | 49.9, 540 59.1 | 59.6;  C=1792: 600 90.7 | 86.2, 800 108 | 110;  C=3072: 1024 205 | 202, 1060 229 | 235
//   n=8 C=1024: 1024 88.7 | 88.1, 1060 103 | 104;  C=1792: 1400 199 | 185, 1800 249 | 251;  C=2048: 1400 215 | 209, 1537 234 | 241;  C=2560:
//       1150 245 | 234, 1400 290 | 296;  C=3072: 1060 290 | 269, 2000 495 | 483;  C=3328: 1060 308 | 302, 1280 340 | 349;  C=4096: 1060 340 |
//       357
//   at most 256 channels, where the resident path splits larger batches: n=1 C=64 1600 30.0 | 28.6, 2000 29.2 | 28.3, 2100 29.4 | 32.5, n=3
//       C=128 1024 31.2 | 30.4, 1060 31.8 | 33.4, n=4 C=64 1060 32.8 | 33.7, 2000 36.9 | 33.1, 4000 44.1 | 41.9, 4200 45.5 | 46.1
//   beyond a full round of larger batches: n=4 C=512 1536 45.9 | 49.5, 1600 47.2 | 45.6, 1800 47.5 | 49.7
constexpr BatchLine kF32Tiled1[] = {{512, 700}, {1024, 620}, {1536, 513}, {2560, 280}, {2688, 1025}, {3072, 280}, {3584, 513}, {kAnyRow, 280}};
constexpr BatchLine kF32Tiled2[] = {{256, 850}, {576, 740}, {1024, 600}, {2560, 513}, {2688, 769}, {3584, 513}, {kAnyRow, 280}};
constexpr BatchLine kF32Tiled3[] = {{256, 1025}, {1024, 950}, {1280, 513}, {1536, 769}, {2048, 513}, {2560, 320}, {2688, 513}, {3072, 320}, {3584, 400}, {kAnyRow, 320}};
constexpr BatchLine kF32Tiled4[] = {{1024, 1025}, {1536, 769}, {2048, 513}, {2560, 420}, {2688, 680}, {3584, 490}, {kAnyRow, 420}};
constexpr BatchLine kF32Tiled5[] = {{256, kNever}, {384, 680}, {768, 700}, {896, 800}, {1664, 513}, {2688, 450}, {kAnyRow, 400}};
constexpr BatchLine kF32Tiled6[] = {{256, kNever}, {384, 768}, {768, 850}, {896, 1000}, {1792, 513}, {2560, 460}, {2688, 513}, {kAnyRow, 400}};
constexpr BatchLine kF32Tiled7[] = {{256, kNever}, {384, 850}, {640, 920}, {704, 1040}, {768, 1200}, {896, 1500}, {1024, 540}, {1216, 769}, {1408, 600},
                                    {1536, 680}, {1792, 769}, {2048, 600}, {2496, 769}, {2688, 640}, {3584, 1025}, {kAnyRow, 960}};
constexpr BatchLine kF32Tiled8[] = {{1023, kNever}, {1600, 1025}, {1792, 1750}, {2112, 1500}, {2688, 1350}, {3072, kNever}, {3519, 1200}, {kAnyRow, 1025}};
// further full rounds beyond a line
bool bwd_f32_resident_round(int B, int n, int C) {
    const auto in = [&](int c_min, int c_max, int b_min, int b_max) { return C >= c_min && C <= c_max && B >= b_min && B <= b_max; };
    if (n <= 4) return in(0, 256, 1537, n == 4 ? 4096 : 2048) || (n >= 3 && in(257, 512, 1537, 1700));
    return (n <= 6 && in(385, 512, 1201, 1280)) || (n == 6 && in(257, 384, 1281, 1450));
}
bool bwd_f32_tiled(int B, int n, int C) {
    if (n > 8 || C % 64 != 0) return false;
    if (const int hook = tuning_get(kTuneResident)) return hook == 1;
    const auto line = [&] {
        switch (n) {
            case 1: return batch_line(kF32Tiled1, C);
            case 2: return batch_line(kF32Tiled2, C);
            case 3: return batch_line(kF32Tiled3, C);
            case 4: return batch_line(kF32Tiled4, C);
            case 5: return batch_line(kF32Tiled5, C);
            case 6: return batch_line(kF32Tiled6, C);
            case 7: return batch_line(kF32Tiled7, C);
            default: return batch_line(kF32Tiled8, C);
        }
    };
    return B >= line() && !bwd_f32_resident_round(B, n, C);
}

int max_ksplit(int B, int n, int C) {
    const int a = proj_fwd_ksplit(kBF16, kBF16, B, n, C), b = proj_fwd_ksplit(kF32, kF32, B, n, C);
    return a > b ? a : b;
}

DynFwdWs carve_dyn_fwd(void *ws, int B, int n, int C) {
    Carver c(ws);
    const int ks = max_ksplit(B, n, C);
    DynFwdWs w;
    w.part_bytes = (size_t)ks * B * padded_D(n) * sizeof(float);
#ifdef MHC_TUNING  // batches below the line of the held forward, whose partial sums are smaller than phi
    if (n >= 2 && n <= 4) w.part_bytes = std::max({w.part_bytes, layer_fwd_held_bytes(kBF16, n, C), layer_fwd_held_bytes(kF32, n, C)});
#endif
    w.Ppart = c.floats(w.part_bytes / sizeof(float));
    w.ssqpart = c.floats((size_t)ks * B);
    w.agg = c.floats(n > 8 ? (size_t)B * C : 0);  // stream aggregate of the matrix-core mix
    w.bytes = c.off;
    return w;
}

// How the dynamic forward goes.  direct: the caller's own parameters are whole 16-byte pieces, which a kernel can read (the others are
// packed by a launch of their own).
enum ForwardKind { kTwoLaunches, kOneLaunch, kOneLaunchReadsParams, kHeldForward };
struct ForwardRoute { ForwardKind kind; bool direct; };
ForwardRoute forward_route(int x_dtype, int y_dtype, int phi_dtype, int B, int n, int C, bool inject, const ParamGather *gather, size_t part_bytes) {
    const bool direct = gather && aligned16(gather->phi[0]) && aligned16(gather->phi[1]) && aligned16(gather->phi[2]) &&
                        tuning_get(kTuneGather) != 1;
    if (!inject && layer_fwd_held_supported(x_dtype, y_dtype, phi_dtype, B, n, C, direct && gather->phi_dtype == kF32) &&
        layer_fwd_held_bytes(x_dtype, n, C) <= part_bytes)
        return {kHeldForward, direct};
    const bool can_gather = gather && layer_fwd_onepass_gathers(*gather);
    if (!layer_fwd_onepass_supported(x_dtype, phi_dtype, B, n, C, can_gather)) return {kTwoLaunches, direct};
    return {can_gather && layer_fwd_onepass_reads_params(B, n, C) ? kOneLaunchReadsParams : kOneLaunch, direct};
}

// Wide projections (n > 18) without batch split of dphi: four launches, see mhc_layer_bwd_dynamic.
// Up to 16 M activation elements: the fp32 hand-over costs 4 more bytes per element than completing dx
// in place, which the shorter chain repays only while the coefficient launch leaves CUs idle
// (backward us, four launches | five: B=128 n=32 C=1280 92 | 100, 384 n=32 C=1280 214 | 215,
//  512 n=32 C=1280 283 | 269, 256 n=32 C=2560 338 | 312).
bool wide_dx_beside(int B, int n, int C) {
    return proj_bwd_is_wide(n) && C % 8 == 0 && proj_bwd_batch_splits(B, n, C) == 1 &&
           (long long)B * n * C <= (16ll << 20);
}

DynBwdWs carve_dyn_bwd(void *ws, int B, int n, int C) {
    Carver c(ws);
    const int D = n * n + 2 * n, nC = n * C;
    DynBwdWs w;
    w.dt = c.floats((size_t)B * (D + 3));
    w.dP = c.floats((size_t)B * padded_D(n));
    w.cx = c.floats(B);
    w.s1 = c.floats(B);
    // partial sums of dw and dt: float32 rows of at most B, float64 rows of the slab kernels or of the resident
    // backward's second launch with a split batch
    const int bs3 = n <= 4 ? std::max({bwd_slab_batch_splits(B, n, C, kBF16), bwd_slab_batch_splits(B, n, C, kF32), bwd_slab_batch_splits(B, n, C, kF32AsBF16)}) : 1;
    const int bs5 = n <= 4 ? bwd_slab_f32_splits(B, C) : 1, bs6 = proj_bwd_addx_supported(n) ? proj_bwd_addx_splits(B, n, C) : 1;
    // (also where the resident path is preferred: it does not take more than 32 Sinkhorn iterations)
    const bool slab8 = n >= 5 && n <= 8 && C % 8 == 0;
    const bool slab8_f32 = slab8 && C % 64 == 0;  // float32 storage
    const int bs7a = slab8 ? bwd_slab8_batch_splits(B, n, C, false) : 1, bs7b = slab8_f32 ? bwd_slab8_batch_splits(B, n, C, true) : 1;
    const int bs7 = std::max(bs7a, bs7b);
    const size_t slab64 = n <= 4 ? std::max(bs3, bs5) : (slab8 ? std::max((size_t)bs7a * bwd_slab8_slabs(n, C, false), slab8_f32 ? (size_t)bs7b * bwd_slab8_slabs(n, C, true) : 0) : 0), parts64 = bs6 > 1 ? proj_bwd_addx_sum_parts(B, bs6) : 0;
    w.u = c.floats(std::max((size_t)B, 2 * (n <= 4 ? slab64 : (size_t)(slab8 ? bs7 : 0))) * C);
    w.upart = c.floats(2 * parts64 * C);
    w.dtpart = c.floats(std::max((size_t)B, 2 * std::max(slab64, parts64)) * (D + 3));
    w.raw = c.floats(bwd_reduce_raw_floats(B, n, C));
    w.s1part = c.floats(n > 8 ? (size_t)B * bwd_reduce_parts(B, n, C) : 0);
    // wide projections: the part of dx that is formed beside the coefficient backward, fp32
    w.dx_part = c.floats(wide_dx_beside(B, n, C) ? (size_t)B * nC : 0);
    // n <= 8, sample-resident backward: dxp where it is handed over in fp32
#ifdef MHC_TUNING
    const bool resident = n <= 8 && C <= kResMaxC;  // on either side of the line: the experiment hook may be set later
#else
    const bool resident = n <= 8 && C <= kResMaxC && (bwd_resident_preferred(B, n, C) || C % 8 != 0);
#endif
    w.dxp = c.floats(resident && bwd_resident_dxp_f32(B, n, C) ? (size_t)B * nC : 0);
    int bs = dphi_batch_splits(B, n, C);
    const int bs2 = proj_bwd_batch_splits(B, n, C);
    if (bs2 > bs) bs = bs2;
    if (bs3 > bs) bs = bs3;
    if (bs7 > bs) bs = bs7;
    const int bs4 = dphi_f32_splits(B, n, C);
    if (bs4 > bs) bs = bs4;
    if (bs5 > bs) bs = bs5;
    if (bs6 > bs) bs = bs6;
    w.dphi_part = c.floats(bs > 1 ? (size_t)bs * D * nC : 0);
    w.BP = (B + 31) / 32 * 32;
    // planes of bf16: one of dP and two of dP^T, one more each for ragged rows (BP is even)
    const size_t half_plane = (size_t)w.BP / 2 * padded_D(n);
    w.dPb = reinterpret_cast<unsigned short *>(c.floats((C % 8 != 0 ? 2 : 1) * half_plane));
    w.dPT = reinterpret_cast<unsigned short *>(c.floats((C % 8 != 0 ? 3 : 2) * half_plane));
    w.bytes = c.off;
    return w;
}

// ---- static workspace layout -----------------------------------------------------------------
struct StaFwdWs { float *Hpre, *Hpost, *M, *q, *agg; size_t bytes; };
struct StaBwdWs { float *red, *s1, *u, *red_sum, *raw, *sk, *s1part; size_t bytes; };

StaFwdWs carve_sta_fwd(void *ws, int B, int n, int C) {
    Carver c(ws);
    StaFwdWs w;
    w.Hpre = c.floats(n); w.Hpost = c.floats(n); w.M = c.floats((size_t)n * n); w.q = c.floats(B);
    w.agg = c.floats(n > 8 ? (size_t)B * C : 0);
    w.bytes = c.off;
    return w;
}

StaBwdWs carve_sta_bwd(void *ws, int B, int n, int C) {
    Carver c(ws);
    const int D = n * n + 2 * n;
    StaBwdWs w;
    // a row per sample in float32, or (n <= 8) one of at least two samples in float64: (B + 1) / 2 rows at most
    w.red = c.floats(((size_t)B + 1) * (D + 3));
    w.s1 = c.floats(B);
    w.u = c.floats(((size_t)B + 1) * C);
    w.red_sum = c.floats(D + 3);
    w.raw = c.floats(n > 8 ? bwd_reduce_raw_floats(B, n, C) : 0);
    w.sk = c.floats(n > 8 ? (size_t)(2 * max_layer_sinkhorn_iters(n) + 2) * 32 : 0);
    w.s1part = c.floats(n > 16 ? (size_t)B * bwd_reduce_parts(B, n, C) : 0);  // Sinkhorn denominators of the shared logits
    w.bytes = c.off;
    return w;
}

}  // namespace

#ifdef MHC_PHASE_PROFILE
namespace mhc {
__device__ unsigned long long g_phase[kPhaseKernels][kPhaseMaxWg][kPhaseMaxMarks];
}
#endif

namespace {

int fwd_dynamic(const void *x, int x_dtype, const void *w, int w_dtype, const ParamGather *gather, const void *phi,
                int phi_dtype, const float *bias, const float *alpha, const void *f_inject, void *y, int y_dtype,
                float *H_pre, float *H_post, float *M, float *P, float *r, float *q, float *sk_state, int B, int n,
                int C, int iters, float eps, void *workspace, size_t workspace_bytes, void *stream);
int bwd_dynamic(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w, int w_dtype, const void *phi,
                int phi_dtype, const float *bias, const float *alpha, const void *f_inject, const float *H_pre,
                const float *H_post, const float *M, const float *P, const float *r, const float *q,
                const float *sk_state, void *dx, void *df, DwOut dw, float *dphi, float *dbias, float *dalpha, int B,
                int n, int C, int iters, float eps, void *workspace, size_t workspace_bytes, void *stream);
int bwd_static(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w, int w_dtype,
               const float *H_pre_logits, const float *H_post_logits, const float *H_res_logits, const void *f_inject,
               const float *H_pre, const float *H_post, const float *M, const float *q, void *dx, void *df, DwOut dw,
               float *dH_pre, float *dH_post, float *dH_res, int B, int n, int C, int iters, float eps,
               void *workspace, size_t workspace_bytes, void *stream);

}  // namespace

extern "C" {

#ifdef MHC_PHASE_PROFILE
// Profile build only (declared in csrc/phase_profiler.h's host interface, not in the product header):
// copies the stamp table of one instrumented kernel to host memory; returns the HIP status.
__attribute__((visibility("default"))) int mhc_phase_read(int kernel, unsigned long long *host, int workgroups) {
    if (kernel < 0 || kernel >= mhc::kPhaseKernels || workgroups > mhc::kPhaseMaxWg) return -1;
    return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(mhc::g_phase),
                                    sizeof(unsigned long long) * mhc::kPhaseMaxMarks * workgroups,
                                    sizeof(unsigned long long) * mhc::kPhaseMaxMarks * mhc::kPhaseMaxWg * kernel);
}
#endif

int mhc_abi_version(void) { return MHC_ABI_VERSION; }

#ifdef MHC_TUNING
// Experiment hooks (csrc/tuning.h): only in the -DMHC_TUNING build, never in the product library.
__attribute__((visibility("default"))) int mhc_tuning_set(int key, int value) {
    if (key < 0 || key >= kTuneCount) return -1;
    g_tuning[key] = value;
    return 0;
}
__attribute__((visibility("default"))) int mhc_tuning_get(int key) {
    return (key < 0 || key >= kTuneCount) ? -1 : g_tuning[key];
}
__attribute__((visibility("default"))) int mhc_tuning_route(int route, int x_dtype, int B, int n, int C) {
    switch (route) {
        case kRouteBackward: return x_dtype == kF32AsBF16 ? bwd_f32_tiled(B, n, C) : !bwd_resident_preferred(B, n, C);
        case kRouteForward: {
            const ParamGather g{{nullptr, nullptr, nullptr}, kF32};
            const bool exact = x_dtype == kF32;
            return forward_route(x_dtype, x_dtype == kBF16 ? kBF16 : kF32, exact ? kF32 : kBF16, B, n, C, false, &g, carve_dyn_fwd(nullptr, B, n, C).part_bytes).kind;
        }
        case kRouteSums: return x_dtype == kF32 ? bwd_reduce_form_f32(B, n, C) : -1;
        default: return -1;
    }
}
#endif

int mhc_max_sinkhorn_iters(int n) { return (n < 1 || n > MHC_MAX_N) ? 0 : max_layer_sinkhorn_iters(n); }

int mhc_layer_dynamic_accepts_f32_as_bf16(int B, int n, int C, int iters) {
    return check_shape(B, n, C, iters) == MHC_OK && f32_as_bf16_accepted(B, n, C, iters) ? 1 : 0;
}

const char *mhc_status_string(int status) {
    switch (status) {
        case MHC_OK: return "ok";
        case MHC_ERR_NULL_POINTER: return "a required pointer is NULL";
        case MHC_ERR_BAD_N: return "expansion rate n must be in 1..32";
        case MHC_ERR_BAD_SHAPE:
            return "B, C or iters out of range (C <= 32768; B * n * C <= 2^40; iters <= mhc_max_sinkhorn_iters(n))";
        case MHC_ERR_BAD_DTYPE: return "unsupported dtype combination";
        case MHC_ERR_MISALIGNED: return "tensor base pointer is not 16-byte aligned";
        case MHC_ERR_WORKSPACE: return "workspace NULL, not 256-byte aligned or too small";
        case MHC_ERR_LAUNCH: return "HIP kernel launch failed";
        case MHC_ERR_SCRATCH_LIMIT:
            return "shape needs more scratch than the library's static array holds (mhc_static_scratch_capacity)";
        default: return "unknown status";
    }
}

// ===============================================================================================
// dynamic H
// ===============================================================================================
size_t mhc_layer_dynamic_workspace_bytes(int B, int n, int C) {
    if (check_shape(B, n, C, 0) != MHC_OK) return 0;
    const size_t f = carve_dyn_fwd(nullptr, B, n, C).bytes;
    const size_t b = carve_dyn_bwd(nullptr, B, n, C).bytes;
    return f > b ? f : b;
}

size_t mhc_layer_sinkhorn_state_floats(int B, int n, int iters) {
    if (n < 1 || n > MHC_MAX_N || B < 1 || iters < 0) return 0;
    return (size_t)B * (iters + 1) * 2 * sinkhorn_state_np(n);
}

int mhc_layer_fwd_dynamic(const void *x, int x_dtype, const void *w, int w_dtype, const void *phi,
                          int phi_dtype, const float *bias, const float *alpha,
                          const void *f_inject, void *y, int y_dtype, float *H_pre, float *H_post,
                          float *M, float *P, float *r, float *q, float *sk_state, int B, int n, int C,
                          int iters, float eps, void *workspace, size_t workspace_bytes, void *stream) {
    return fwd_dynamic(x, x_dtype, w, w_dtype, nullptr, phi, phi_dtype, bias, alpha, f_inject, y, y_dtype, H_pre, H_post, M, P,
                       r, q, sk_state, B, n, C, iters, eps, workspace, workspace_bytes, stream);
}

int mhc_layer_fwd_dynamic_params(const void *x, int x_dtype, const void *w, int w_dtype,
                                 const struct mhc_dynamic_params *p, void *phi, int phi_dtype, float *bias, float *alpha,
                                 const void *f_inject, void *y, int y_dtype, float *H_pre, float *H_post, float *M,
                                 float *P, float *r, float *q, float *sk_state, int B, int n, int C, int iters,
                                 float eps, void *workspace, size_t workspace_bytes, void *stream) {
    if (!p || !p->phi_pre || !p->phi_post || !p->phi_res || !p->b_pre || !p->b_post || !p->b_res || !p->alpha_pre ||
        !p->alpha_post || !p->alpha_res)
        return MHC_ERR_NULL_POINTER;
    if (!valid_dtype(p->phi_dtype)) return MHC_ERR_BAD_DTYPE;
    const ParamGather g{{p->phi_pre, p->phi_post, p->phi_res}, p->phi_dtype, {p->b_pre, p->b_post, p->b_res},
                        {p->alpha_pre, p->alpha_post, p->alpha_res}, phi, phi_dtype, bias, alpha};
    return fwd_dynamic(x, x_dtype, w, w_dtype, &g, phi, phi_dtype, bias, alpha, f_inject, y, y_dtype, H_pre, H_post, M, P,
                       r, q, sk_state, B, n, C, iters, eps, workspace, workspace_bytes, stream);
}

int mhc_layer_bwd_dynamic(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w,
                          int w_dtype, const void *phi, int phi_dtype, const float *bias,
                          const float *alpha, const void *f_inject, const float *H_pre,
                          const float *H_post, const float *M, const float *P, const float *r,
                          const float *q, const float *sk_state, void *dx, void *df, float *dw, float *dphi,
                          float *dbias, float *dalpha, int B, int n, int C, int iters, float eps,
                          void *workspace, size_t workspace_bytes, void *stream) {
    return bwd_dynamic(dy, y_dtype, x, x_dtype, w, w_dtype, phi, phi_dtype, bias, alpha, f_inject, H_pre, H_post, M, P, r, q,
                       sk_state, dx, df, DwOut{dw, false}, dphi, dbias, dalpha, B, n, C, iters, eps, workspace,
                       workspace_bytes, stream);
}

int mhc_layer_bwd_dynamic_dw(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w,
                          int w_dtype, const void *phi, int phi_dtype, const float *bias,
                          const float *alpha, const void *f_inject, const float *H_pre,
                          const float *H_post, const float *M, const float *P, const float *r,
                          const float *q, const float *sk_state, void *dx, void *df, void *dw, int dw_dtype,
                          float *dphi,
                          float *dbias, float *dalpha, int B, int n, int C, int iters, float eps,
                          void *workspace, size_t workspace_bytes, void *stream) {
    if (!valid_dtype(dw_dtype)) return MHC_ERR_BAD_DTYPE;
    return bwd_dynamic(dy, y_dtype, x, x_dtype, w, w_dtype, phi, phi_dtype, bias, alpha, f_inject, H_pre, H_post, M, P, r, q,
                       sk_state, dx, df, DwOut{dw, dw_dtype == MHC_BF16}, dphi, dbias, dalpha, B, n, C, iters, eps,
                       workspace, workspace_bytes, stream);
}

int mhc_pack_dynamic_params(const void *phi_pre, const void *phi_post, const void *phi_res, int src_dtype,
                            const float *b_pre, const float *b_post, const float *b_res,
                            const float *alpha_pre, const float *alpha_post, const float *alpha_res,
                            void *phi, int phi_dtype, float *bias, float *alpha, int n, int C, void *stream) {
    if (n < 1 || n > MHC_MAX_N) return MHC_ERR_BAD_N;
    if (C < 1 || C > MHC_MAX_C) return MHC_ERR_BAD_SHAPE;
    if (!phi_pre || !phi_post || !phi_res || !b_pre || !b_post || !b_res || !alpha_pre || !alpha_post ||
        !alpha_res || !phi || !bias || !alpha)
        return MHC_ERR_NULL_POINTER;
    if (!valid_dtype(src_dtype) || !valid_dtype(phi_dtype)) return MHC_ERR_BAD_DTYPE;
    MHC_LAUNCH(launch_pack_params(ParamGather{{phi_pre, phi_post, phi_res}, src_dtype, {b_pre, b_post, b_res},
                                              {alpha_pre, alpha_post, alpha_res}, phi, phi_dtype, bias, alpha},
                                  n, C, static_cast<hipStream_t>(stream)));
    return MHC_OK;
}

// ===============================================================================================
// static H
// ===============================================================================================
size_t mhc_layer_static_workspace_bytes(int B, int n, int C) {
    if (check_shape(B, n, C, 0) != MHC_OK) return 0;
    const size_t f = carve_sta_fwd(nullptr, B, n, C).bytes;
    const size_t b = carve_sta_bwd(nullptr, B, n, C).bytes;
    return f > b ? f : b;
}

int mhc_layer_fwd(const void *x, int x_dtype, const void *w, int w_dtype,
                  const float *H_pre_logits, const float *H_post_logits,
                  const float *H_res_logits, const void *f_inject, void *y, int y_dtype,
                  float *H_pre, float *H_post, float *M, float *q, int B, int n, int C, int iters,
                  float eps, void *workspace, size_t workspace_bytes, void *stream) {
    if (int s = check_shape(B, n, C, iters)) return s;
    if (!x || !H_pre_logits || !H_post_logits || !H_res_logits || !y) return MHC_ERR_NULL_POINTER;
    if (!f_inject && !w) return MHC_ERR_NULL_POINTER;
    if (!valid_io(x_dtype, y_dtype) || (w && !valid_dtype(w_dtype))) return MHC_ERR_BAD_DTYPE;
    if (!aligned16(x) || !aligned16(y) || (f_inject && !aligned16(f_inject))) return MHC_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (layer_fwd_fused_supported(n, C, x_dtype)) {
        // one launch; every workgroup derives the shared coefficients itself, none need storing
        MHC_LAUNCH(launch_layer_fwd_fused(x, x_dtype, w, w_dtype, f_inject, y, y_dtype, nullptr, nullptr,
                                          0, 0, nullptr, H_pre_logits, H_post_logits, H_res_logits,
                                          H_pre, H_post, M, nullptr, nullptr, q, nullptr, B, n, C, iters, eps,
                                          st));
        return MHC_OK;
    }
    const StaFwdWs ws = carve_sta_fwd(workspace, B, n, C);
    const bool need_ws = !H_pre || !H_post || !M || !q || n > 8;
    if (need_ws)
        if (int s = ws_check(workspace, workspace_bytes, ws.bytes)) return s;
    float *hp = H_pre ? H_pre : ws.Hpre, *ho = H_post ? H_post : ws.Hpost;
    float *m = M ? M : ws.M, *qq = q ? q : ws.q;
    // n > 8, up to two samples per CU: the coefficient launch runs once per sample, each workgroup with
    // the shared Sinkhorn chain and its sample's aggregate and RMS under it, instead of one workgroup
    // followed by an aggregate launch (forward, cold, B=128 n=32 C=1280: 26 -> 20 us)
    const bool agg = !f_inject && n > 8 && B <= 512 && coef_fwd_aggregates(n, C, x_dtype);
    MHC_LAUNCH(launch_coef_fwd(nullptr, nullptr, 0, 0, nullptr, H_pre_logits, H_post_logits,
                               H_res_logits, hp, ho, m, nullptr, nullptr, agg ? B : 1, n, n * C, iters, eps,
                               x_dtype == kF32, agg ? x : nullptr, agg ? ws.agg : nullptr, agg ? qq : nullptr,
                               nullptr, st));
    MHC_LAUNCH(launch_mix_fwd(x, x_dtype, w, w_dtype, f_inject, y, y_dtype, hp, ho, m, 0, qq,
                              n > 8 ? ws.agg : nullptr, B, n, C, eps, agg, st));
    return MHC_OK;
}

int mhc_layer_bwd(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w,
                  int w_dtype, const float *H_pre_logits, const float *H_post_logits,
                  const float *H_res_logits, const void *f_inject, const float *H_pre,
                  const float *H_post, const float *M, const float *q, void *dx, void *df,
                  float *dw, float *dH_pre, float *dH_post, float *dH_res, int B, int n, int C,
                  int iters, float eps, void *workspace, size_t workspace_bytes, void *stream) {
    return bwd_static(dy, y_dtype, x, x_dtype, w, w_dtype, H_pre_logits, H_post_logits, H_res_logits, f_inject, H_pre, H_post,
                      M, q, dx, df, DwOut{dw, false}, dH_pre, dH_post, dH_res, B, n, C, iters, eps, workspace,
                      workspace_bytes, stream);
}

int mhc_layer_bwd_dw(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w,
                  int w_dtype, const float *H_pre_logits, const float *H_post_logits,
                  const float *H_res_logits, const void *f_inject, const float *H_pre,
                  const float *H_post, const float *M, const float *q, void *dx, void *df,
                  void *dw, int dw_dtype, float *dH_pre, float *dH_post, float *dH_res, int B, int n, int C,
                  int iters, float eps, void *workspace, size_t workspace_bytes, void *stream) {
    if (!valid_dtype(dw_dtype)) return MHC_ERR_BAD_DTYPE;
    return bwd_static(dy, y_dtype, x, x_dtype, w, w_dtype, H_pre_logits, H_post_logits, H_res_logits, f_inject, H_pre, H_post,
                      M, q, dx, df, DwOut{dw, dw_dtype == MHC_BF16}, dH_pre, dH_post, dH_res, B, n, C, iters, eps, workspace,
                      workspace_bytes, stream);
}

// ===============================================================================================
// stand-alone operators
// ===============================================================================================
int mhc_sinkhorn_knopp_fwd(const float *inp, float *out, int batch, int rows, int cols, int iters,
                           float eps, void *stream) {
    if (!inp || !out) return MHC_ERR_NULL_POINTER;
    if (batch < 1 || rows < 1 || cols < 1 || rows > 128 || cols > 128 || iters < 0 || iters > 1024)
        return MHC_ERR_BAD_SHAPE;
    MHC_LAUNCH(launch_sinkhorn_plain_fwd(inp, out, batch, rows, cols, iters, eps,
                                         static_cast<hipStream_t>(stream)));
    return MHC_OK;
}

size_t mhc_sinkhorn_knopp_bwd_workspace_bytes(int batch, int rows, int cols, int iters) {
    if (batch < 1 || rows < 1 || cols < 1 || rows > 128 || cols > 128 || iters < 0 || iters > 1024)
        return 0;
    return ((size_t)batch * (iters > 0 ? iters : 1) * 2 * 128 * sizeof(float) + 255) / 256 * 256;
}

int mhc_sinkhorn_knopp_bwd(const float *grad_out, const float *inp, float *d_inp, int batch,
                           int rows, int cols, int iters, float eps, void *workspace,
                           size_t workspace_bytes, void *stream) {
    if (!grad_out || !inp || !d_inp) return MHC_ERR_NULL_POINTER;
    const size_t need = mhc_sinkhorn_knopp_bwd_workspace_bytes(batch, rows, cols, iters);
    if (need == 0) return MHC_ERR_BAD_SHAPE;
    if (int s = ws_check(workspace, workspace_bytes, need)) return s;
    MHC_LAUNCH(launch_sinkhorn_plain_bwd(grad_out, inp, d_inp, batch, rows, cols, iters, eps,
                                         static_cast<float *>(workspace),
                                         static_cast<hipStream_t>(stream)));
    return MHC_OK;
}

int mhc_rmsnorm_fwd(const void *inp, int dtype, const void *w, int w_dtype, void *out, float *rms,
                    int rows, int C, float eps, void *stream) {
    if (!inp || !w || !out) return MHC_ERR_NULL_POINTER;
    if (rows < 1 || C < 1) return MHC_ERR_BAD_SHAPE;
    if (!valid_dtype(dtype) || !valid_dtype(w_dtype)) return MHC_ERR_BAD_DTYPE;
    MHC_LAUNCH(launch_rmsnorm_fwd(inp, dtype, w, w_dtype, out, rms, rows, C, eps,
                                  static_cast<hipStream_t>(stream)));
    return MHC_OK;
}

size_t mhc_rmsnorm_bwd_workspace_bytes(int rows, int C) {
    if (rows < 1 || C < 1) return 0;
    Carver c(nullptr);
    c.floats((size_t)(rows + 3) * C);  // dw terms: a row per input row, or per row slot of the persistent kernel
    c.floats(colsum_workspace_floats(rows + 3, C));
    return c.off;
}

int mhc_rmsnorm_bwd(const void *grad_out, const void *inp, int dtype, const void *w, int w_dtype,
                    const float *rms, void *d_inp, float *d_w, int rows, int C, void *workspace,
                    size_t workspace_bytes, void *stream) {
    if (!grad_out || !inp || !w || !rms || !d_inp || !d_w) return MHC_ERR_NULL_POINTER;
    if (rows < 1 || C < 1) return MHC_ERR_BAD_SHAPE;
    if (!valid_dtype(dtype) || !valid_dtype(w_dtype)) return MHC_ERR_BAD_DTYPE;
    if (int s = ws_check(workspace, workspace_bytes, mhc_rmsnorm_bwd_workspace_bytes(rows, C))) return s;
    Carver c(workspace);
    float *u = c.floats((size_t)(rows + 3) * C);
    float *part = c.floats(colsum_workspace_floats(rows + 3, C));
    hipStream_t st = static_cast<hipStream_t>(stream);
    int u_rows = rows;  // rows of u whose column sums are dw (fewer when the kernel sums its own rows)
    MHC_LAUNCH(launch_rmsnorm_bwd(grad_out, inp, dtype, w, w_dtype, rms, d_inp, u, rows, C, &u_rows, st));
    MHC_LAUNCH(launch_colsum(u, u_rows, C, C, d_w, part, st));
    return MHC_OK;
}

}  // extern "C"

// ===============================================================================================
// Dynamic forward for callers that cannot allocate (HIP graph capture, serving loops, harnesses
// that forbid hipMalloc): the scratch of the split-K projection lives in a device array of this
// library instead of a caller workspace.  Every GPU holds its own copy of the array at its own
// address; the address is looked up once per device and only that pointer is handed to kernels
// (the array's name is a host-side stand-in, not a device address).
// ===============================================================================================
static __device__ __align__(256) unsigned char scratch[MHC_STATIC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices];  // device address of `scratch` per device, nullptr until looked up

int static_scratch_pointer(void **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return MHC_ERR_LAUNCH;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return MHC_ERR_LAUNCH;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return MHC_OK;
}

}  // namespace

extern "C" {

size_t mhc_static_scratch_capacity(void) { return MHC_STATIC_SCRATCH_BYTES; }

size_t mhc_layer_fwd_dynamic_scratch_bytes(int B, int n, int C) {
    if (check_shape(B, n, C, 0) != MHC_OK) return 0;
    return carve_dyn_fwd(nullptr, B, n, C).bytes;
}

int mhc_static_scratch_init(void) {
    void *p = nullptr;
    return static_scratch_pointer(&p);
}

int mhc_layer_fwd_dynamic_static_scratch(const void *x, int x_dtype, const void *w, int w_dtype,
                                         const void *phi, int phi_dtype, const float *bias,
                                         const float *alpha, const void *f_inject, void *y, int y_dtype,
                                         float *H_pre, float *H_post, float *M, float *P, float *r,
                                         float *q, float *sk_state, int B, int n, int C, int iters, float eps,
                                         void *stream) {
    if (int s = check_shape(B, n, C, iters)) return s;
    // every byte the kernels touch lies below `need`; nothing has to start at zero (the projection
    // writes each partial sum that the coefficient step reads), so the contents left by the last call
    // are simply overwritten
    const size_t need = carve_dyn_fwd(nullptr, B, n, C).bytes;
    if (need > MHC_STATIC_SCRATCH_BYTES) return MHC_ERR_SCRATCH_LIMIT;
    void *ptr = nullptr;
    if (int s = static_scratch_pointer(&ptr)) return s;
    return mhc_layer_fwd_dynamic(x, x_dtype, w, w_dtype, phi, phi_dtype, bias, alpha, f_inject, y, y_dtype,
                                 H_pre, H_post, M, P, r, q, sk_state, B, n, C, iters, eps, ptr,
                                 MHC_STATIC_SCRATCH_BYTES, stream);
}

}  // extern "C"

// ===============================================================================================
// the launch sequences behind the entry points above
// ===============================================================================================
namespace {

int fwd_dynamic(const void *x, int x_dtype, const void *w, int w_dtype, const ParamGather *gather, const void *phi,
                int phi_dtype, const float *bias, const float *alpha, const void *f_inject, void *y, int y_dtype,
                float *H_pre, float *H_post, float *M, float *P, float *r, float *q, float *sk_state, int B, int n,
                int C, int iters, float eps, void *workspace, size_t workspace_bytes, void *stream) {
    if (int s = check_shape(B, n, C, iters)) return s;
    if (!x || !phi || !bias || !alpha || !y || !H_pre || !H_post || !M || !P || !r || !q)
        return MHC_ERR_NULL_POINTER;
    if (!f_inject && !w) return MHC_ERR_NULL_POINTER;
    if (!valid_io(x_dtype, y_dtype) || !valid_dtype(phi_dtype) || (w && !valid_dtype(w_dtype)))
        return MHC_ERR_BAD_DTYPE;
    if (x_dtype == MHC_F32_AS_BF16 && (phi_dtype != MHC_BF16 || !f32_as_bf16_accepted(B, n, C, iters)))
        return MHC_ERR_BAD_DTYPE;
    if (!aligned16(x) || !aligned16(y) || !aligned16(phi) || (f_inject && !aligned16(f_inject)))
        return MHC_ERR_MISALIGNED;
    const DynFwdWs ws = carve_dyn_fwd(workspace, B, n, C);
    if (int s = ws_check(workspace, workspace_bytes, ws.bytes)) return s;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const ForwardRoute route = forward_route(x_dtype, y_dtype, phi_dtype, B, n, C, f_inject != nullptr, gather, ws.part_bytes);
    if (route.kind == kHeldForward) {
        if (gather && !route.direct) MHC_LAUNCH(launch_pack_params(*gather, n, C, st));
        MHC_LAUNCH(launch_layer_fwd_held(x, x_dtype, w, w_dtype, y, route.direct ? gather : nullptr, phi, alpha, bias, ws.Ppart, H_pre,
                                         H_post, M, P, r, q, sk_state, B, n, C, iters, eps, st));
        return MHC_OK;
    }
    // the caller's own parameters: read by the kernel that multiplies with them where it can, otherwise packed by a launch
    // of their own
    const bool in_one = route.kind == kOneLaunchReadsParams;
    const bool in_proj = gather && route.kind == kTwoLaunches && proj_fwd_gathers(*gather, x_dtype, B, n, C);
    if (gather && !in_one && !in_proj) MHC_LAUNCH(launch_pack_params(*gather, n, C, st));
    if (route.kind != kTwoLaunches) {
        // projection, coefficients and mix in one launch; x crosses HBM once
        MHC_LAUNCH(launch_layer_fwd_onepass(x, w, w_dtype, f_inject, y, y_dtype, phi, alpha, bias, H_pre, H_post,
                                            M, P, r, q, sk_state, B, n, C, iters, eps, st, in_one ? gather : nullptr));
        return MHC_OK;
    }
    const int KS = proj_fwd_ksplit(x_dtype, phi_dtype, B, n, C);
    MHC_LAUNCH(launch_proj_fwd(x, x_dtype, phi, phi_dtype, ws.Ppart, ws.ssqpart, KS, B, n, C, st,
                               in_proj ? gather : nullptr));
    if (layer_fwd_fused_supported(n, C, x_dtype)) {
        MHC_LAUNCH(launch_layer_fwd_fused(x, x_dtype, w, w_dtype, f_inject, y, y_dtype, ws.Ppart,
                                          ws.ssqpart, KS, padded_D(n), alpha, bias, bias + n,
                                          bias + 2 * n, H_pre, H_post, M, P, r, q, sk_state, B, n, C, iters,
                                          eps, st));
        return MHC_OK;
    }
    // n > 8 in the bf16 tier: the coefficient launch also forms the stream aggregate and its RMS
    const bool agg = !f_inject && ws.agg && coef_fwd_aggregates(n, C, x_dtype);
    MHC_LAUNCH(launch_coef_fwd(ws.Ppart, ws.ssqpart, KS, padded_D(n), alpha, bias, bias + n,
                               bias + 2 * n, H_pre, H_post, M, P, r, B, n, n * C, iters, eps,
                               x_dtype == kF32, agg ? x : nullptr, ws.agg, q, sk_state, st));
    MHC_LAUNCH(launch_mix_fwd(x, x_dtype, w, w_dtype, f_inject, y, y_dtype, H_pre, H_post, M, n, q,
                              ws.agg, B, n, C, eps, agg, st));
    return MHC_OK;
}

int bwd_dynamic(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w, int w_dtype, const void *phi,
                int phi_dtype, const float *bias, const float *alpha, const void *f_inject, const float *H_pre,
                const float *H_post, const float *M, const float *P, const float *r, const float *q,
                const float *sk_state, void *dx, void *df, DwOut dw, float *dphi, float *dbias, float *dalpha, int B,
                int n, int C, int iters, float eps, void *workspace, size_t workspace_bytes, void *stream) {
    if (int s = check_shape(B, n, C, iters)) return s;
    if (!dy || !x || !phi || !bias || !alpha || !H_pre || !H_post || !M || !P || !r || !q || !dx ||
        !dphi || !dbias || !dalpha)
        return MHC_ERR_NULL_POINTER;
    if (!f_inject && (!w || !dw)) return MHC_ERR_NULL_POINTER;
    if (!valid_io(x_dtype, y_dtype) || !valid_dtype(phi_dtype) || (w && !valid_dtype(w_dtype)))
        return MHC_ERR_BAD_DTYPE;
    if (x_dtype == MHC_F32_AS_BF16 && (phi_dtype != MHC_BF16 || !f32_as_bf16_accepted(B, n, C, iters)))
        return MHC_ERR_BAD_DTYPE;
    if (!aligned16(dy) || !aligned16(x) || !aligned16(dx) || !aligned16(phi) || !aligned16(dphi) ||
        (f_inject && !aligned16(f_inject)) || (df && !aligned16(df)))
        return MHC_ERR_MISALIGNED;
    const DynBwdWs ws = carve_dyn_bwd(workspace, B, n, C);
    if (int s = ws_check(workspace, workspace_bytes, ws.bytes)) return s;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int D = n * n + 2 * n, DP = padded_D(n);
    const bool mfma = proj_bwd_mfma_supported(x_dtype == kF32AsBF16 ? kBF16 : x_dtype, phi_dtype, C);
    BwdCoefOut out{ws.dt, ws.dP, ws.cx, ws.s1, nullptr, mfma ? ws.dPb : nullptr, ws.dPT, ws.BP};
    if (x_dtype == kF32AsBF16 && !f_inject && bwd_f32_tiled(B, n, C)) {
        // float32 storage, large batches: the channel sums round x and dy once and leave both where dx will be; the slab kernel
        // reads them there, half the bytes, and puts dx in their place
        MHC_LAUNCH(launch_mix_bwd_reduce_f32_as_bf16(static_cast<const float *>(dy), static_cast<const float *>(x), w, w_dtype, H_pre, H_post, M,
                                                     q, P, r, alpha, bias + 2 * n, sk_state, out, dx, B, n, C, iters, eps, st));
        if (n > 4) {
            const int S = bwd_slab8_batch_splits(B, n, C, true);
            MHC_LAUNCH(launch_bwd_slab8(nullptr, nullptr, w, w_dtype, nullptr, phi, H_pre, H_post, M, q, out, dx, nullptr,
                                        S > 1 ? ws.dphi_part : dphi, reinterpret_cast<double *>(ws.u), reinterpret_cast<double *>(ws.dtpart),
                                        S, B, n, C, st, true));
            MHC_LAUNCH(launch_finalize(ws.u, S, C, dw, ws.dtpart, S * bwd_slab8_slabs(n, C, true), D, dbias, dalpha, ws.dphi_part, S,
                                       (size_t)D * n * C, dphi, st, true));
            return MHC_OK;
        }
        const int S = bwd_slab_batch_splits(B, n, C, kF32AsBF16);
        MHC_LAUNCH(launch_bwd_slab(dx, kF32AsBF16, nullptr, w, w_dtype, nullptr, phi, H_pre, H_post, M, q, ws.s1, ws.cx, ws.dPb, ws.dPT, ws.BP,
                                   ws.dt, dx, nullptr, S > 1 ? ws.dphi_part : dphi, reinterpret_cast<double *>(ws.u),
                                   reinterpret_cast<double *>(ws.dtpart), S, B, n, C, st));
        MHC_LAUNCH(launch_finalize(ws.u, S, C, dw, ws.dtpart, S, D, dbias, dalpha, ws.dphi_part, S, (size_t)D * n * C, dphi, st, true));
        return MHC_OK;
    }
    // (rows that are no multiple of 8 elements: these two launches are the only matrix-core ones that take them)
    if (bwd_resident_supported(x_dtype, y_dtype, phi_dtype, n, C, iters) && proj_bwd_addx_supported(n) &&
        (bwd_resident_preferred(B, n, C) || x_dtype == kF32AsBF16 || C % 8 != 0)) {
        // two launches: (1) one workgroup per sample keeps the sample's rows of dy and x in registers for
        // the channel sums, the coefficient backward and the mixing part of dx; (2) a column-slab
        // kernel over all samples adds dP phi - cx x, finishes dphi without batch-split partial sums
        // and sums dw, dbias and dalpha in a few extra workgroups
        BwdCoefOut out2 = out;
        out2.dPb = ws.dPb;
        out2.dP = nullptr;  // the second launch takes dP as matrix-core operands only
        float *dxp = x_dtype == kBF16 && bwd_resident_dxp_f32(B, n, C) ? ws.dxp : nullptr;
        MHC_LAUNCH(launch_bwd_resident(dy, x, x_dtype, w, w_dtype, f_inject, H_pre, H_post, M, q, P, r, alpha, bias + 2 * n,
                                       sk_state, out2, dxp ? dxp : dx, df, ws.u, B, n, C, iters, eps, st));
        const DwOut dwo = f_inject ? DwOut{} : dw;
        const int S = proj_bwd_addx_splits(B, n, C), parts = proj_bwd_addx_sum_parts(B, S);
        bool tail_taken = false;
        if (S > 1) {
            // partial sums of dphi, dw, dbias and dalpha, added up by one more launch
            const BatchSumArgs sums = make_batch_sums(ws.u, B, C, dwo ? DwOut{ws.upart, false} : dwo, ws.dt, B, D, ws.dtpart,
                                                      nullptr);
            MHC_LAUNCH(launch_proj_bwd_addx(x, x_dtype, phi, ws.dPb, ws.dPT, ws.BP, ws.cx, ws.dphi_part, S, dxp, dx, B, n, C, &sums,
                                            &tail_taken, st));
            if (!tail_taken) return MHC_ERR_LAUNCH;  // not reached: any number of workgroups can carry the parts
            MHC_LAUNCH(launch_finalize(ws.upart, parts, C, dwo, ws.dtpart, parts, D, dbias, dalpha, ws.dphi_part, S,
                                       (size_t)D * n * C, dphi, st, true));
            return MHC_OK;
        }
        const BatchSumArgs sums = make_batch_sums(ws.u, B, C, dwo, ws.dt, B, D, dbias, dalpha);
        MHC_LAUNCH(launch_proj_bwd_addx(x, x_dtype, phi, ws.dPb, ws.dPT, ws.BP, ws.cx, dphi, 1, dxp, dx, B, n, C,
                                        tuning_get(kTuneSeparateFinalize) == 1 ? nullptr : &sums, &tail_taken, st));
        if (!tail_taken)
            MHC_LAUNCH(launch_finalize(ws.u, B, C, dwo, ws.dt, B, D, dbias, dalpha, nullptr, 1, 0, nullptr, st));
        return MHC_OK;
    }
    if (x_dtype == kF32AsBF16) return MHC_ERR_BAD_DTYPE;  // not reached: accepted shapes take the path above
    if (mfma && x_dtype == kBF16 && y_dtype == kBF16 && wide_dx_beside(B, n, C) && tuning_get(kTuneWideDxBeside) != 1) {
        // wide projection (n > 18), four launches.  The coefficient backward is one workgroup per sample,
        // all dependent chains; the part of dx that needs none of its results (M^T dy + Hpre (x) da,
        // with s1 from the channel sums) runs beside it in the same launch and is handed over in fp32;
        // the dP phi kernel then completes dx (+ dP phi - cx x, one rounding); dphi comes last and carries
        // the batch sums.
        // B=128 n=32 C=1280, backward in graphs of ten, same box: five launches 99.8 us, these four 93.0 us
        MHC_LAUNCH(launch_mix_bwd_reduce_with_dx(dy, x, w, w_dtype, f_inject, H_pre, H_post, M, n, q, P, r, alpha,
                                                 bias + 2 * n, sk_state, out, ws.raw, ws.s1part, ws.dx_part, df, ws.u, B, n, C,
                                                 iters, eps, st));
        MHC_LAUNCH(launch_dxflat_wide(phi, ws.dPb, ws.BP, dx, x, ws.cx, ws.dx_part, B, n, C, st));
        const BatchSumArgs sums = make_batch_sums(ws.u, B, C, f_inject ? DwOut{} : dw, ws.dt, B, D, dbias, dalpha);
        bool tail_taken = false;
        MHC_LAUNCH(launch_dphi_large(x, ws.dPT, ws.BP, dphi, 1, B, n, C,
                                     tuning_get(kTuneSeparateFinalize) != 1 ? &sums : nullptr, &tail_taken, st));
        if (!tail_taken)
            MHC_LAUNCH(launch_finalize(ws.u, B, C, f_inject ? DwOut{} : dw, ws.dt, B, D, dbias, dalpha, nullptr, 1,
                                       (size_t)D * n * C, dphi, st));
        return MHC_OK;
    }
    MHC_LAUNCH(launch_mix_bwd_reduce(dy, y_dtype, x, x_dtype, w, w_dtype, f_inject, H_pre, H_post, M,
                                     n, q, P, r, alpha, bias + 2 * n, sk_state, out, ws.raw, B, n, C, iters, eps,
                                     st));
    if (mfma && bwd_slab_supported(x_dtype, y_dtype, phi_dtype, n, C)) {
        // n <= 4: one slab kernel finishes dx and produces every batch-split partial sum
        const int S = bwd_slab_batch_splits(B, n, C, y_dtype);
        MHC_LAUNCH(launch_bwd_slab(dy, y_dtype, x, w, w_dtype, f_inject, phi, H_pre, H_post, M, q, ws.s1,
                                   ws.cx, ws.dPb, ws.dPT, ws.BP, ws.dt, dx, df,
                                   S > 1 ? ws.dphi_part : dphi, reinterpret_cast<double *>(ws.u),
                                   reinterpret_cast<double *>(ws.dtpart), S, B, n, C, st));
        MHC_LAUNCH(launch_finalize(ws.u, S, C, f_inject ? DwOut{} : dw, ws.dtpart, S, D, dbias, dalpha,
                                   ws.dphi_part, S, (size_t)D * n * C, dphi, st, true));
        return MHC_OK;
    }
    if (mfma && bwd_slab8_supported(x_dtype, y_dtype, phi_dtype, n, C) && bwd_slab8_preferred(B, n, C)) {
        const int S = bwd_slab8_batch_splits(B, n, C, false);
        MHC_LAUNCH(launch_bwd_slab8(dy, x, w, w_dtype, f_inject, phi, H_pre, H_post, M, q, out, dx, df,
                                    S > 1 ? ws.dphi_part : dphi, reinterpret_cast<double *>(ws.u),
                                    reinterpret_cast<double *>(ws.dtpart), S, B, n, C, st));
        MHC_LAUNCH(launch_finalize(ws.u, S, C, f_inject ? DwOut{} : dw, ws.dtpart, S * bwd_slab8_slabs(n, C, false), D, dbias, dalpha,
                                   ws.dphi_part, S, (size_t)D * n * C, dphi, st, true));
        return MHC_OK;
    }
    if (bwd_slab_f32_supported(x_dtype, phi_dtype, n, C)) {
        const int S = bwd_slab_f32_splits(B, C);
        MHC_LAUNCH(launch_bwd_slab_f32(static_cast<const float *>(dy), static_cast<const float *>(x), w, w_dtype, f_inject,
                                       static_cast<const float *>(phi), H_pre, H_post, M, q, out, static_cast<float *>(dx),
                                       static_cast<float *>(df), S > 1 ? ws.dphi_part : dphi, reinterpret_cast<double *>(ws.u),
                                       reinterpret_cast<double *>(ws.dtpart), B, n, C, st));
        MHC_LAUNCH(launch_finalize(ws.u, S, C, f_inject ? DwOut{} : dw, ws.dtpart, S, D, dbias, dalpha, ws.dphi_part, S,
                                   (size_t)D * n * C, dphi, st, true));
        return MHC_OK;
    }
    const int spg = bwd_dx_samples_per_group(B, n);
    const int groups = (B + spg - 1) / spg;
    int S = 1;
    if (mfma) {
        // matrix cores: dphi and the projection term of dx (written into dx, then completed in place)
        S = proj_bwd_batch_splits(B, n, C);
        // From D > 128 on the two products run as launches of their own (they share no operand but dP
        // and no output): dP phi first, then the dx kernel that consumes it, dphi = dP^T x last.  The
        // last launch carries the batch sums (dw, dbias, dalpha) in an extra row of workgroups, which
        // run in the shadow of the dphi stores instead of as a launch of their own.  Measured on whole
        // steps, graphs of ten (one launch for both products + finalize launch -> apart + carried sums):
        //   B=256 n=8   47.7 -> 48.8 us (not taken)    B=256 n=10   79.8 -> 80.0 (not taken)
        //   B=512 n=12 126.6 -> 125.9    B=256 n=13 101.6 -> 96.6    B=256 n=16 111.9 -> 104.4
        //   B=256 n=18 127.5 -> 119.0    B=128 n=32 148.6 -> 145.8 (always two product kernels; sums carried)
        const bool wide = proj_bwd_is_wide(n);
        const int hook = tuning_get(kTuneProjApart);
        const bool apart = wide || (hook ? hook == 2 : proj_bwd_products_apart(n));
        if (apart) {
            if (wide) MHC_LAUNCH(launch_dxflat_wide(phi, ws.dPb, ws.BP, dx, nullptr, nullptr, nullptr, B, n, C, st));
            else MHC_LAUNCH(launch_proj_bwd_mfma(x, phi, ws.dPb, ws.dPT, ws.BP, dphi, ws.dphi_part, dx, B, n, C, st, kProjPartDx));
        } else {
            MHC_LAUNCH(launch_proj_bwd_mfma(x, phi, ws.dPb, ws.dPT, ws.BP, dphi, ws.dphi_part, dx, B, n, C, st));
        }
        MHC_LAUNCH(launch_mix_bwd_dx(dy, y_dtype, x, x_dtype, w, w_dtype, f_inject, H_pre, H_post, M,
                                     n, q, ws.s1, ws.cx, ws.dP, DP, nullptr, 0, dx, dx, df, ws.u, ws.dt,
                                     ws.dtpart, spg, B, n, C, st));
        if (apart) {
            const BatchSumArgs sums = make_batch_sums(ws.u, groups, C, f_inject ? DwOut{} : dw, ws.dtpart, groups,
                                                      D, dbias, dalpha);
            const BatchSumArgs *tail = S == 1 && tuning_get(kTuneSeparateFinalize) != 1 ? &sums : nullptr;
            bool tail_taken = false;
            if (wide) MHC_LAUNCH(launch_dphi_large(x, ws.dPT, ws.BP, S > 1 ? ws.dphi_part : dphi, S, B, n, C, tail, &tail_taken, st));
            else MHC_LAUNCH(launch_proj_bwd_mfma(x, phi, ws.dPb, ws.dPT, ws.BP, dphi, ws.dphi_part, dx, B, n, C, st,
                                                 kProjPartDphi, tail, &tail_taken));
            if (tail_taken) return MHC_OK;
        }
    } else if (dx_dphi_f32_supported(x_dtype, phi_dtype, n, C)) {
        // exact float32 tier, wide projection: both products on the fp32 matrix cores; the projection
        // term of dx is written into dx and completed in place
        MHC_LAUNCH(launch_gemm_f32_dxflat(ws.dP, static_cast<const float *>(phi), static_cast<float *>(dx), B, n, C, st));
        MHC_LAUNCH(launch_mix_bwd_dx(dy, y_dtype, x, x_dtype, w, w_dtype, f_inject, H_pre, H_post, M,
                                     n, q, ws.s1, ws.cx, ws.dP, DP, nullptr, 0, dx, dx, df, ws.u, ws.dt,
                                     ws.dtpart, spg, B, n, C, st));
        if (n <= 8) {
            S = dphi_f32_splits(B, n, C);
            MHC_LAUNCH(launch_dphi_f32(ws.dP, static_cast<const float *>(x), S > 1 ? ws.dphi_part : dphi, S, B, n, C, st));
        } else {
            MHC_LAUNCH(launch_gemm_f32_dphi(ws.dP, static_cast<const float *>(x), dphi, B, n, C, st));
        }
    } else {
        MHC_LAUNCH(launch_mix_bwd_dx(dy, y_dtype, x, x_dtype, w, w_dtype, f_inject, H_pre, H_post, M,
                                     n, q, ws.s1, ws.cx, ws.dP, DP, phi, phi_dtype, nullptr, dx, df,
                                     ws.u, ws.dt, ws.dtpart, spg, B, n, C, st));
        MHC_LAUNCH(launch_dphi(x, x_dtype, ws.dP, DP, dphi, B, n, C, ws.dphi_part, st));
    }
    MHC_LAUNCH(launch_finalize(ws.u, groups, C, f_inject ? DwOut{} : dw, ws.dtpart, groups, D, dbias,
                               dalpha, ws.dphi_part, S, (size_t)D * n * C, dphi, st));
    return MHC_OK;
}

int bwd_static(const void *dy, int y_dtype, const void *x, int x_dtype, const void *w, int w_dtype,
               const float *H_pre_logits, const float *H_post_logits, const float *H_res_logits, const void *f_inject,
               const float *H_pre, const float *H_post, const float *M, const float *q, void *dx, void *df, DwOut dw,
               float *dH_pre, float *dH_post, float *dH_res, int B, int n, int C, int iters, float eps,
               void *workspace, size_t workspace_bytes, void *stream) {
    if (int s = check_shape(B, n, C, iters)) return s;
    if (!dy || !x || !H_pre_logits || !H_post_logits || !H_res_logits || !H_pre || !H_post || !M ||
        !q || !dx || !dH_pre || !dH_post || !dH_res)
        return MHC_ERR_NULL_POINTER;
    if (!f_inject && (!w || !dw)) return MHC_ERR_NULL_POINTER;
    if (!valid_io(x_dtype, y_dtype) || (w && !valid_dtype(w_dtype))) return MHC_ERR_BAD_DTYPE;
    if (!aligned16(dy) || !aligned16(x) || !aligned16(dx) || (f_inject && !aligned16(f_inject)) ||
        (df && !aligned16(df)))
        return MHC_ERR_MISALIGNED;
    const StaBwdWs ws = carve_sta_bwd(workspace, B, n, C);
    if (int s = ws_check(workspace, workspace_bytes, ws.bytes)) return s;
    hipStream_t st = static_cast<hipStream_t>(stream);
    BwdCoefOut out{nullptr, nullptr, nullptr, ws.s1, ws.red, nullptr, nullptr, 0};
    if (bwd_resident_supported(x_dtype, y_dtype, kBF16, n, C, 0) && tuning_get(kTuneResident) != 1) {
        // bf16 activations, n <= 8: with shared coefficients nothing of dx depends on a batch-wide
        // result, so ONE pass over dy and x (a workgroup keeps a sample's rows in registers) forms
        // the channel sums, the raw coefficient gradients and the complete dx; large batches several samples per workgroup
        const bool walk = bwd_static_preferred(B, n, C);
        const int rows = walk ? bwd_static_rows(B, n, C) : B;
        if (walk) MHC_LAUNCH(launch_bwd_static(dy, x, w, w_dtype, f_inject, H_pre, H_post, M, q, dx, df, ws.u, ws.red, B, n, C, st));
        else MHC_LAUNCH(launch_bwd_resident_static(dy, x, w, w_dtype, f_inject, H_pre, H_post, M, q, out, dx, df, ws.u,
                                                   B, n, C, st));
        MHC_LAUNCH(launch_finalize_static(ws.u, rows, C, f_inject ? DwOut{} : dw, ws.red, rows, ws.red_sum, H_pre, H_post,
                                          H_res_logits, dH_pre, dH_post, dH_res, n, iters, eps, st, nullptr, walk));
        return MHC_OK;
    }
    if (n > 16 && x_dtype == kBF16 && y_dtype == kBF16 && C % 8 == 0) {
        // three launches: channel sums (+ the Sinkhorn forward recompute), the per-sample coefficient sums
        // with the complete dx beside them, batch sums + coefficient backward
        // (cold, B=128 n=32 C=1280: 44.7 us -> see profiles/native_bench_all_configs.txt)
        MHC_LAUNCH(launch_mix_bwd_reduce_with_dx_static(dy, x, w, w_dtype, f_inject, H_pre, H_post, M, q, out, ws.raw,
                                                        ws.s1part, dx, df, ws.u, B, n, C, iters, eps, st, H_res_logits,
                                                        ws.sk));
        MHC_LAUNCH(launch_finalize_static(ws.u, B, C, f_inject ? DwOut{} : dw, ws.red, B, ws.red_sum, H_pre, H_post,
                                          H_res_logits, dH_pre, dH_post, dH_res, n, iters, eps, st, ws.sk));
        return MHC_OK;
    }
    MHC_LAUNCH(launch_mix_bwd_reduce(dy, y_dtype, x, x_dtype, w, w_dtype, f_inject, H_pre, H_post, M,
                                     0, q, nullptr, nullptr, nullptr, nullptr, nullptr, out, n > 8 ? ws.raw : nullptr,
                                     B, n, C, iters, eps, st, H_res_logits, n > 8 ? ws.sk : nullptr));
    // samples per workgroup of the dx kernel: with a large batch a workgroup adds up the dw terms of a
    // few samples itself, so that the batch-sum launch reads fewer rows
    const int hook = tuning_get(kTuneStaticSpg);
    // (measured cold, bf16: B=1280 C=2560 n=4 60.5 -> 58.6 us with four; B=1024 n=8 and small batches lose)
    const int spg = n > 8 ? 1 : (hook > 0 ? hook : (n <= 4 && B >= 1024 ? 4 : 1));
    const int groups = (B + spg - 1) / spg;
    MHC_LAUNCH(launch_mix_bwd_dx(dy, y_dtype, x, x_dtype, w, w_dtype, f_inject, H_pre, H_post, M, 0,
                                 q, ws.s1, nullptr, nullptr, 0, nullptr, 0, nullptr, dx, df, ws.u, nullptr,
                                 nullptr, spg, B, n, C, st));
    // the batch sums (dw = sum_b u, sum_b red) and the coefficient backward on them: one launch for
    // n <= 8, two beyond
    MHC_LAUNCH(launch_finalize_static(ws.u, groups, C, f_inject ? DwOut{} : dw, ws.red, B, ws.red_sum, H_pre, H_post,
                                      H_res_logits, dH_pre, dH_post, dH_res, n, iters, eps, st, n > 8 ? ws.sk : nullptr));
    return MHC_OK;
}

}  // namespace
