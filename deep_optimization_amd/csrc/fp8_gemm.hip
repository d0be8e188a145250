// FP8 e4m3 scaled GEMM launcher: which kernel and tile a shape gets.
//
// Large outputs take 256 x 256 tiles (fp8_gemm.h: GROUP_M = 4 tile rows per L2 group, even MFMA / memory
// interleave; the persistent kernels with one workgroup per CU, 16x16x128 MFMAs from K = 8192, 32x32x64
// below; the non-persistent kernel for an odd number of K slabs). They leave CUs idle when the output has
// few of them, and a tile's K slabs run one after the other: M = 64, N = K = 4096 took 38 us on 16
// workgroups. Smaller outputs take smaller tiles (fp8_gemm_mid.h, fp8_gemm_small.h) by the estimate in
// `plan` below.
#include <atomic>

#include "fp8_gemm.h"
#include "fp8_gemm_mid.h"
#include "fp8_gemm_small.h"

namespace dopt {

using Fp8GemmDefault = Fp8GemmCfg<256, 256, 4, 0>;

namespace {
// compute units of the current device, queried once per device
int device_cu_count() {
    constexpr int MAX_DEV = 64;
    static std::atomic<int> cached[MAX_DEV];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEV) return 256;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n <= 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}
}  // namespace

namespace {

using Fp8Gemm128 = Fp8GemmCfg<128, 128, 4, 0>;

// Estimated time (us) of a tile shape on this part: start + per K slab the larger of a lone workgroup's
// step and the CU's throughput at its share of the tiles, + an epilogue per round of tiles. The constants
// are fitted to a sweep in which every kernel was timed on 32 shapes from 1 x 4096 x 4096 to 4096^3; on
// those the estimate picks the fastest kernel or one within 10% of it but for rows that are not a
// multiple of 128 bytes (within 25%). Times in us, before (256 x 256 tiles only) -> now: 16 x 768 x 768
// 12.1 -> 3.0, 64 x 4096 x 4096 38 -> 7.2, 256 x 256 x 8192 64 -> 8.3, 985 x 3072 x 768 15.0 -> 7.1,
// 1024^3 13.3 -> 4.2, 1024 x 4096 x 4096 38 -> 19.1, 2048^3 21.8 -> 12.0; from about 3000^3 on the
// 256 x 256 tiles are the fastest and stay.
struct TileCost {
    int bm, bn;
    float start, step, rate, epilogue;
};
enum { T_SMALL, T_32x64, T_64x64, T_128x64, T_128x128, T_128x128_NT, T_256, T_COUNT };
constexpr TileCost TILE_COST[T_COUNT] = {
    {16, 16, 2.4f, 0.09f, 0.105f, 0.1f},   // 8 waves split K (M <= 16 only)
    {32, 64, 2.2f, 0.14f, 0.14f, 0.4f},
    {64, 64, 2.4f, 0.17f, 0.18f, 0.8f},
    {128, 64, 2.9f, 0.20f, 0.29f, 1.2f},
    {128, 128, 2.9f, 0.33f, 0.50f, 1.8f},
    {128, 128, 2.9f, 0.60f, 0.50f, 1.5f},  // two workgroups per CU, double-buffered (hides part of its epilogues)
    {256, 256, 5.0f, 0.95f, 1.45f, 2.5f},
};

// the tile with the least estimate (kn: of those that read B as it lies in [K, N] rows) and that estimate
int plan(int64_t M, int64_t N, int64_t K, int n_cu, bool kn, float* us_out) {
    const float nk = (float)((K + 127) / 128);
    int best = kn ? T_128x128 : T_256;
    float least = 0.0f;
    for (int t = kn ? T_128x128 : T_COUNT - 1; t >= (kn ? T_32x64 : 0); --t) {
        const TileCost& c = TILE_COST[t];
        if (t == T_SMALL && M > 16) continue;
        const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
        if (tiles >= ((int64_t)1 << 31)) continue;
        const float rounds = (float)((tiles + n_cu - 1) / n_cu);
        const float rate = (kn ? 1.2f : 1.0f) * c.rate * rounds;  // the transposing reads: four per fragment for two
        const float step = rate > c.step ? rate : c.step;
        const float us = c.start + nk * step + c.epilogue * rounds;
        if (t == best || us < least) {
            least = us;
            best = t;
        }
    }
    *us_out = least;
    return best;
}

}  // namespace

int launch_fp8_gemm_nt(const uint8_t* A, const uint8_t* B, int64_t M, int64_t N, int64_t K, int64_t lda,
                       int64_t ldb, float out_scale, uint16_t* C, int64_t ldc, hipStream_t s) {
    const int n_cu = device_cu_count();
    const Fp8GemmArgs p{A, B, C, M, N, K, lda, ldb, ldc, out_scale, 0, 0,
                        (uint32_t)(ldc % 8 == 0 && ((uintptr_t)C & 15) == 0), K};
    float us;
    switch (plan(M, N, K, n_cu, false, &us)) {
        case T_SMALL: return fp8_gemm_small_launch<1, 1, 8>(p, s);
        case T_32x64: return fp8_gemm_mid_launch<32, 64>(p, s);
        case T_64x64: return fp8_gemm_mid_launch<64, 64>(p, s);
        case T_128x64: return fp8_gemm_mid_launch<128, 64>(p, s);
        case T_128x128: return fp8_gemm_mid_launch<128, 128>(p, s);
        case T_128x128_NT: return fp8_gemm_launch<Fp8Gemm128>(A, B, M, N, K, lda, ldb, out_scale, C, ldc, s);
    }
    return fp8_gemm_persistent_launch<Fp8GemmDefault>(A, B, M, N, K, lda, ldb, out_scale, C, ldc, n_cu, s);
}

// B in [K, N] rows
int launch_fp8_gemm_kn(const uint8_t* A, const uint8_t* B, int64_t M, int64_t N, int64_t K, int64_t b_rows, int64_t lda,
                       int64_t ldb, float out_scale, uint16_t* C, int64_t ldc, hipStream_t s) {
    const Fp8GemmArgs p{A, B, C, M, N, K, lda, ldb, ldc, out_scale, 0, 0,
                        (uint32_t)(ldc % 8 == 0 && ((uintptr_t)C & 15) == 0), b_rows};
    float us;
    switch (plan(M, N, K, device_cu_count(), true, &us)) {
        case T_32x64: return fp8_gemm_mid_launch<32, 64, true>(p, s);
        case T_64x64: return fp8_gemm_mid_launch<64, 64, true>(p, s);
        case T_128x64: return fp8_gemm_mid_launch<128, 64, true>(p, s);
    }
    return fp8_gemm_mid_launch<128, 128, true>(p, s);
}

// the index in TILE_COST of the tile a product gets
int fp8_gemm_tile(int64_t M, int64_t N, int64_t K, bool kn) {
    float us;
    return plan(M, N, K, device_cu_count(), kn, &us);
}

// Whether reading B as it lies is estimated to be faster than packing it (a launch of about 3 us and its
// bytes) for launch_fp8_gemm_nt. Both ways timed on 16 shapes from 1 x 4096 x 4096 to 8192^3; us, packed ->
// as it lies: 985 x 768 x 1536 8.5 -> 5.5, 64 x 4096 x 4096 17.1 -> 6.7, 1024^3 7.8 -> 4.8, 2048^3
// 18.0 -> 11.4, 8192 x 1024 x 1024 17.6 -> 15.3; the other way at 3000^3 (50.7 against 55.8) and 4096^3
// (57.4 against 72.2), where the 256 x 256 tiles win.
// A B that would have to be copied into aligned rows first (`copied`) is passed over once either way, by the copy
// about 0.3 us faster than by the transpose: the row-major kernel has to be that close to the other one. Over 230
// random odd N from 17 to 8191 (captured calls, copy or transpose included) the faster way is lost by 1.0% in the
// geometric mean and by more than 5% on 18; with the comparison above it was 4.8% and 60 (16 x 1001 x 8192 24.2
// against 14.4 us packed, 64 x 4097 x 4096 19.2 against 17.4, 2500 x 2501 x 1000 24.9 against 21.7).
bool fp8_gemm_kn_preferred(int64_t M, int64_t N, int64_t K, bool copied) {
    const int n_cu = device_cu_count();
    float kn, nt;
    plan(M, N, K, n_cu, true, &kn);
    plan(M, N, K, n_cu, false, &nt);
    return kn < nt + (copied ? 0.3f : 3.0f + (float)N * (float)K * (1.0f / 3.2e6f));
}

}  // namespace dopt
