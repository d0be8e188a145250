// FP8 (OCP e4m3) scaled GEMM of at most 16 rows (larger ones: fp8_gemm_mid.h, fp8_gemm.h): a workgroup computes a
// (16 MT) x (16 NT) tile and its NW waves split K between them; the launcher uses 16 x 16 tiles and 8 waves.
// Same operands, result and edge handling: C[m][n] = bf16(out_scale * sum_k A[m][k] * B[n][k]), fp32
// sums, one rounding; any M, N; K a multiple of 16.
//
// What bounds these shapes is latency and bytes, not the matrix pipe: with one 256 x 256 workgroup per
// tile, M = 16, N = 256, K = 8192 ran its 64 K slabs one after the other on a single CU (51 us). Here
// every wave walks the K chunks w, w + NW, ... of 128 bytes with its operands straight from memory to
// registers (fragment i is 16 rows x 128 bytes, whole cache lines; nothing is shared that LDS would
// save), the next chunk's loads in flight during the current one's MFMAs, and no barrier until the end.
// The NW fp32 partial tiles then meet in LDS, where each thread sums its 8 output columns over the waves
// in order (the result does not depend on timing) and stores them as one 16-byte chunk.
//
// Lanes whose row lies past M (or N) or whose 16 bytes lie past K load with an offset beyond the buffer
// resource's range, which reads zeros.
#pragma once

#include "fp8_gemm.h"

namespace dopt {

template <int MT, int NT, int NW>
__global__ __launch_bounds__(64 * NW) void fp8_gemm_small_kernel(Fp8GemmArgs p) {
    constexpr int TM = 16 * MT, TN = 16 * NT, PITCH = TN + 4;  // floats per LDS row
    __shared__ __attribute__((aligned(16))) float part[NW][TM * PITCH];
    const int64_t M = p.M, N = p.N, lda = p.lda, ldb = p.ldb, ldc = p.ldc;
    const uint32_t Kb = (uint32_t)p.K;  // K <= lda < 2^23
    // XCD x (workgroup ids x, x + 8, ...) takes a contiguous range of tiles, M tiles first, so the
    // workgroups that read the same rows of B share an L2
    const uint32_t n_tiles = p.tiles_m * p.tiles_n;
    const uint32_t xcd = blockIdx.x % GEMM_XCDS, local = blockIdx.x / GEMM_XCDS;
    const uint32_t per = n_tiles / GEMM_XCDS, rem = n_tiles % GEMM_XCDS;
    const uint32_t t = xcd * per + min(xcd, rem) + local;
    const int64_t m0 = (int64_t)(t % p.tiles_m) * TM, n0 = (int64_t)(t / p.tiles_m) * TN;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)(p.A + m0 * lda), (short)0, (int)GEMM_RANGE, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc((void*)(p.B + n0 * ldb), (short)0, (int)GEMM_RANGE, 0x00020000);
    // lane l of a fragment: row l % 16, bytes 16 (l / 16) .. + 15 and 64 + 16 (l / 16) .. + 15 of the chunk, so
    // one load covers 64 contiguous bytes of each row (the MFMA pairs A's and B's bytes by lane and
    // position, so any assignment of K to them works when both operands share it)
    const int row = lane & 15, kb = 16 * (lane >> 4);
    uint32_t offa[MT], offb[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
        offa[i] = m0 + 16 * i + row < M ? (uint32_t)((16 * i + row) * lda + kb) : GEMM_OOB;
#pragma unroll
    for (int j = 0; j < NT; ++j)
        offb[j] = n0 + 16 * j + row < N ? (uint32_t)((16 * j + row) * ldb + kb) : GEMM_OOB;

    struct Frags {
        v8i_t a[MT], b[NT];
    };
    // (the K offset is at most 2^23 and the row offsets at most 16 * 2^23 for the 16 x 16 tile: a lane past its rows
    // stays beyond the range)
    auto load = [&](__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t k0, uint32_t past0, uint32_t past1)
                    __attribute__((always_inline)) {
        const v4u_t x0 = __builtin_amdgcn_raw_buffer_load_b128(r, off | past0, (int)k0, 0);
        const v4u_t x1 = __builtin_amdgcn_raw_buffer_load_b128(r, (off + 64) | past1, (int)k0, 0);
        return __builtin_bit_cast(v8i_t, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    auto load_chunk = [&](Frags& f, uint32_t k0) __attribute__((always_inline)) {
        const uint32_t past0 = k0 + kb < Kb ? 0u : GEMM_OOB, past1 = k0 + kb + 64 < Kb ? 0u : GEMM_OOB;
#pragma unroll
        for (int j = 0; j < NT; ++j) f.b[j] = load(rb, offb[j], k0, past0, past1);
#pragma unroll
        for (int i = 0; i < MT; ++i) f.a[i] = load(ra, offa[i], k0, past0, past1);
    };
    v4f_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto mma = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = mfma_fp8_16x16x128(f.b[j], f.a[i], acc[i][j]);
    };

    constexpr uint32_t STEP = 128u * NW;
    uint32_t k0 = 128u * wave;
    if (k0 < Kb) {
        Frags f0, f1;
        load_chunk(f0, k0);
        for (;;) {
            // (a chunk past K loads zeros and is not multiplied)
            load_chunk(f1, k0 + STEP);
            mma(f0);
            k0 += STEP;
            if (k0 >= Kb) break;
            load_chunk(f0, k0 + STEP);
            mma(f1);
            k0 += STEP;
            if (k0 >= Kb) break;
        }
    }

    // lane l holds row 16 i + l % 16, columns 16 j + 4 (l / 16) .. + 3 of block (i, j)
    float* mine = part[wave];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) *(v4f_t*)(mine + (16 * i + row) * PITCH + 16 * j + 4 * (lane >> 4)) = acc[i][j];
    __syncthreads();
    constexpr int CPR = TN / 8;  // 8-column chunks per row
    for (int q = threadIdx.x; q < TM * CPR; q += 64 * NW) {
        const int r = q / CPR, c = 8 * (q % CPR);
        const int64_t m = m0 + r, n = n0 + c;
        if (m >= M || n >= N) continue;
        v4f_t s0 = *(const v4f_t*)(part[0] + r * PITCH + c), s1 = *(const v4f_t*)(part[0] + r * PITCH + c + 4);
#pragma unroll
        for (int w = 1; w < NW; ++w) {
            s0 += *(const v4f_t*)(part[w] + r * PITCH + c);
            s1 += *(const v4f_t*)(part[w] + r * PITCH + c + 4);
        }
        const v4u_t v = {pack_bf16x2(s0[0] * p.out_scale, s0[1] * p.out_scale),
                         pack_bf16x2(s0[2] * p.out_scale, s0[3] * p.out_scale),
                         pack_bf16x2(s1[0] * p.out_scale, s1[1] * p.out_scale),
                         pack_bf16x2(s1[2] * p.out_scale, s1[3] * p.out_scale)};
        uint16_t* dst = p.C + m * ldc + n;
        if (n + 8 <= N) {
            store_c8(dst, v);
        } else {
            const uint16_t e8[8] = {(uint16_t)v.x, (uint16_t)(v.x >> 16), (uint16_t)v.y, (uint16_t)(v.y >> 16),
                                    (uint16_t)v.z, (uint16_t)(v.z >> 16), (uint16_t)v.w, (uint16_t)(v.w >> 16)};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (n + e < N) dst[e] = e8[e];
        }
    }
}

template <int MT, int NT, int NW>
inline int fp8_gemm_small_launch(Fp8GemmArgs p, hipStream_t s) {
    p.tiles_m = (uint32_t)((p.M + 16 * MT - 1) / (16 * MT));
    p.tiles_n = (uint32_t)((p.N + 16 * NT - 1) / (16 * NT));
    hipLaunchKernelGGL((fp8_gemm_small_kernel<MT, NT, NW>), dim3(p.tiles_m * p.tiles_n), dim3(64 * NW), 0, s, p);
    return 0;
}

}  // namespace dopt
