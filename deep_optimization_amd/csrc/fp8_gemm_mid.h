// FP8 (OCP e4m3) scaled GEMM for the sizes between fp8_gemm_small.h and the 256 x 256 tiles of
// fp8_gemm.h: BM x BN workgroup tiles (2 x 2 waves) through a ring of 4 LDS stages.
// Same operands, result and edge handling as the other kernels.
//
// What bounds these shapes: with one workgroup on a CU and the next slab's loads issued only one slab
// ahead, a 128-byte K slab of a 128 x 128 tile took 0.6 us, three times its MFMAs: the load latency. Here
// three slabs are in flight behind the one being multiplied. Per slab and wave:
//   wait: own loads of slab k+1 landed, own operand reads returned | barrier | issue slab k+4 into
//   slab k's stage | operand reads of slab k+1 beside the MFMAs of slab k
// Every stage's A and B tiles are LDS objects of their own, so the compiler can tell an operand read from
// the loads in flight. Slabs past K issue loads beyond the buffer resource's range (zeros into stages
// nobody multiplies), so the wait count is the same in every step.
//
// LDS rows are the slab's 128 bytes; 16-byte chunk c of row r lies at c ^ f(r), f as in
// fp8_gemm16_persistent_kernel (the same 16-row fragments).
//
// KN: B lies as [K, N] rows (a weight used as x @ w) at a stride of a multiple of 16 bytes, each row readable up to
// N rounded up to one (the bytes past N only reach columns that are not stored). Its slab is
// then 128 rows of BN bytes, loaded as they lie, and the operand reads transpose: ds_read_b64_tr_b8 hands 16
// lanes an 8 x 16 block of bytes by columns, four of them make a fragment's 32 K bytes per lane (the K order of
// the other form, so the sums are the same bit for bit). 16-byte chunk c of row k lies at c ^ g(k), so the 16
// rows that 32 lanes read at once (8 i .. + 7 and 32 + 8 i .. + 7) fall into different banks. The form spares
// the transposed copy of B, a launch of its own: 985 x 3072 x 768 (M, N, K) took 4.7 us for it beside 8.1 for the GEMM,
// which takes 8.2 reading B as it lies.
#pragma once

#include "fp8_gemm.h"

namespace dopt {

typedef int v2i_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i_t lds_v2i_t;

template <int BM, int BN, bool KN>
__global__ __launch_bounds__(256, 1) void fp8_gemm_mid_kernel(Fp8GemmArgs p) {
    constexpr int BK = 128, WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
    constexpr int LA = BM / 32, LB = BN / 32, LD = LA + LB;  // 1 KB loads per wave and slab
    static_assert(BM % 32 == 0 && BN % 32 == 0 && 2 * LD < 64, "tile shape, vmcnt range");
    const int64_t M = p.M, N = p.N, lda = p.lda, ldb = p.ldb, ldc = p.ldc;
    const uint32_t Kb = (uint32_t)p.K;  // K <= lda < 2^23
    __shared__ __attribute__((aligned(1024))) uint8_t sA0[BM * BK];
    __shared__ __attribute__((aligned(1024))) uint8_t sA1[BM * BK];
    __shared__ __attribute__((aligned(1024))) uint8_t sA2[BM * BK];
    __shared__ __attribute__((aligned(1024))) uint8_t sA3[BM * BK];
    __shared__ __attribute__((aligned(1024))) uint8_t sB0[BN * BK];
    __shared__ __attribute__((aligned(1024))) uint8_t sB1[BN * BK];
    __shared__ __attribute__((aligned(1024))) uint8_t sB2[BN * BK];
    __shared__ __attribute__((aligned(1024))) uint8_t sB3[BN * BK];

    // tile order: XCD x owns a contiguous tile range, walked 4 tile rows at a time (fp8_gemm_nt_kernel)
    constexpr uint32_t GROUP_M = 4;
    const uint32_t n_tiles = p.tiles_m * p.tiles_n;
    const uint32_t xcd = blockIdx.x % GEMM_XCDS, local = blockIdx.x / GEMM_XCDS;
    const uint32_t per = n_tiles / GEMM_XCDS, rem = n_tiles % GEMM_XCDS;
    const uint32_t t = xcd * per + min(xcd, rem) + local;
    const uint32_t group = GROUP_M * p.tiles_n, first_m = (t / group) * GROUP_M;
    const uint32_t gsize = min(p.tiles_m - first_m, GROUP_M);
    const int64_t m0 = (int64_t)(first_m + (t % group) % gsize) * BM, n0 = (int64_t)((t % group) / gsize) * BN;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // global -> LDS: load j of wave w fills rows 8 (4 j + w) + lane / 8, position lane % 8 <- chunk
    // (lane % 8) ^ f(row), f(r) = r3 | r1 << 1 | r2 << 2 (rn: bit n of r)
    const int lrow = 8 * wave + (lane >> 3);
    const int lchunk = (lane & 7) ^ ((wave & 1) | (((lane >> 4) & 1) << 1) | (((lane >> 5) & 1) << 2));
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)(p.A + m0 * lda), (short)0, (int)GEMM_RANGE, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc((void*)(p.B + (KN ? 0 : n0 * ldb)), (short)0, (int)GEMM_RANGE, 0x00020000);
    uint32_t offa[LA], offb[LB];
#pragma unroll
    for (int j = 0; j < LA; ++j)
        offa[j] = m0 + 32 * j + lrow < M ? (uint32_t)((32 * j + lrow) * lda + lchunk * 16) : GEMM_OOB;
    if constexpr (KN) {
        // load j of wave w fills rows k = RPL (4 j + w) + lane / CPR of CPR chunks, position lane % CPR <- chunk
        // (lane % CPR) ^ g(k): g = k2 | k5 << 1 at 4 chunks a row, k1 | k2 << 1 | k5 << 2 at 8
        constexpr int CPR = BN / 16, RPL = 64 / CPR;
        static_assert(CPR == 4 || CPR == 8, "swizzles of 64- and 128-byte rows");
#pragma unroll
        for (int j = 0; j < LB; ++j) {
            const int k = RPL * (4 * j + wave) + lane / CPR;
            const int g = CPR == 4 ? ((k >> 2) & 1) | (((k >> 5) & 1) << 1)
                                   : ((k >> 1) & 1) | (((k >> 2) & 1) << 1) | (((k >> 5) & 1) << 2);
            const int col = ((lane & (CPR - 1)) ^ g) * 16;
            offb[j] = n0 + col < N ? (uint32_t)(k * ldb + col) : GEMM_OOB;
        }
    } else {
#pragma unroll
        for (int j = 0; j < LB; ++j)
            offb[j] = n0 + 32 * j + lrow < N ? (uint32_t)((32 * j + lrow) * ldb + lchunk * 16) : GEMM_OOB;
    }
    // (the LDS offsets carry a zero the compiler cannot see through: a read it could prove disjoint from
    // the one load it records per LDS object would wait for every load in flight)
    int opaque0;
    asm volatile("s_mov_b32 %0, 0" : "=s"(opaque0));
    auto issue = [&](uint8_t* sa, uint8_t* sb, uint32_t k) __attribute__((always_inline)) {
        uint8_t *da = sa + opaque0, *db = sb + opaque0;
        const uint32_t k0 = k * BK;
        const uint32_t past = k0 + (uint32_t)lchunk * 16 < Kb ? 0u : GEMM_OOB;  // or'ed in: no branch, no select per load
#pragma unroll
        for (int j = 0; j < LA; ++j) {
            const uint32_t off = offa[j] | past;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t*)(da + wave * 1024 + j * 4096), 16, off, (int)k0,
                                                     0, 0);
        }
        if constexpr (KN) {
            // the slab's rows end with B's last: the buffer range covers what is left of it, so rows past it
            // read zeros (a slab's offsets stay below 2^30, so a range cut to GEMM_RANGE covers whole slabs)
            const int64_t left = (p.b_rows - 1 - (int64_t)k0) * ldb + (N + 15) / 16 * 16 - n0;
            const int range = left <= 0 ? 0 : left < (int64_t)GEMM_RANGE ? (int)left : (int)GEMM_RANGE;
            const __amdgpu_buffer_rsrc_t rk =
                __builtin_amdgcn_make_buffer_rsrc((void*)(p.B + (int64_t)k0 * ldb + n0), (short)0, range, 0x00020000);
#pragma unroll
            for (int j = 0; j < LB; ++j) {
                const uint32_t off = offb[j];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_void_t*)(db + wave * 1024 + j * 4096), 16, off, 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < LB; ++j) {
                const uint32_t off = offb[j] | past;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void_t*)(db + wave * 1024 + j * 4096), 16, off,
                                                         (int)k0, 0, 0);
            }
        }
    };

    // fragment i: rows base + 16 i + lane % 16, K bytes 32 (lane / 16) .. + 31 (chunks oc, oc + 1)
    const int orow = lane & 15, oc = 2 * (lane >> 4);
    const int sw = ((lane >> 3) & 1) | (((lane >> 1) & 1) << 1) | (((lane >> 2) & 1) << 2);  // f(lane % 16)
    const int p0 = (oc ^ sw) * 16, p1 = ((oc + 1) ^ sw) * 16;
    struct Frags {
        v8i_t a[FM], b[FN];
    };
    auto read_frag = [&](const uint8_t* s, int base_row) __attribute__((always_inline)) -> v8i_t {
        const int o = (base_row + orow) * BK;
        const v4u_t x0 = *(const v4u_t*)(s + (o + p0));
        const v4u_t x1 = *(const v4u_t*)(s + (o + p1));
        return __builtin_bit_cast(v8i_t, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // KN: fragment j is columns WN wn + 16 j + lane % 16; lane l names row 8 i + (l % 16) / 2 (+ 32 (l / 16)),
    // half l % 2 of its 16 bytes, for the transposing read i
    const int crow = 32 * (lane >> 4) + ((lane & 15) >> 1), chalf = 8 * (lane & 1);
    const int cg = BN == 64 ? ((lane >> 3) & 1) | (((lane >> 4) & 1) << 1)
                            : ((lane >> 2) & 1) | (((lane >> 3) & 1) << 1) | (((lane >> 4) & 1) << 2);
    auto read_cols = [&](const uint8_t* s, int j) __attribute__((always_inline)) -> v8i_t {
        const uint8_t* q = s + (crow * BN + (((wn * FN + j) ^ cg) << 4) + chalf);
        const v2i_t x0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t*)q);
        const v2i_t x1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t*)(q + 8 * BN));
        const v2i_t x2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t*)(q + 16 * BN));
        const v2i_t x3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_t*)(q + 24 * BN));
        return v8i_t{x0[0], x0[1], x1[0], x1[1], x2[0], x2[1], x3[0], x3[1]};
    };
    auto read_frags = [&](Frags& f, const uint8_t* sa, const uint8_t* sb) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < FN; ++j) f.b[j] = KN ? read_cols(sb, j) : read_frag(sb, WN * wn + 16 * j);
#pragma unroll
        for (int i = 0; i < FM; ++i) f.a[i] = read_frag(sa, WM * wm + 16 * i);
    };
    v4f_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};

    // step k: slab k's operands are in `cur`; (sa, sb) is its stage, (na, nb) slab k+1's
    constexpr int W = 2 * LD;
    constexpr int WAIT = (W & 15) | ((W >> 4) << 14) | (7 << 4);  // vmcnt(2 LD), lgkmcnt(0)
    auto step = [&](const Frags& cur, Frags& nxt, uint8_t* sa, uint8_t* sb, const uint8_t* na, const uint8_t* nb,
                    uint32_t k) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(WAIT);
        asm volatile("s_barrier" ::: "memory");
        issue(sa, sb, k + 4);
        read_frags(nxt, na, nb);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = mfma_fp8_16x16x128(cur.b[j], cur.a[i], acc[i][j]);
        constexpr int NM = FM * FN, NR = 2 * FM + (KN ? 4 : 2) * FN;
        constexpr int PER = (NR + NM - 1) / NM;
#pragma unroll
        for (int q = 0; q < NM; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);  // LDS reads
            if (q < LD) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // one global load
        }
    };

    const uint32_t nk = (Kb + BK - 1) / BK;
    if (nk > 0) {
        issue(sA0, sB0, 0);
        issue(sA1, sB1, 1);
        issue(sA2, sB2, 2);
        issue(sA3, sB3, 3);
        constexpr int W0 = 3 * LD;
        __builtin_amdgcn_s_waitcnt((W0 & 15) | ((W0 >> 4) << 14) | (7 << 4));
        asm volatile("s_barrier" ::: "memory");
        Frags f0, f1;
        read_frags(f0, sA0, sB0);
        uint32_t k = 0;
        for (; k + 4 <= nk; k += 4) {
            step(f0, f1, sA0, sB0, sA1, sB1, k);
            step(f1, f0, sA1, sB1, sA2, sB2, k + 1);
            step(f0, f1, sA2, sB2, sA3, sB3, k + 2);
            step(f1, f0, sA3, sB3, sA0, sB0, k + 3);
        }
        if (k < nk) step(f0, f1, sA0, sB0, sA1, sB1, k);
        if (k + 1 < nk) step(f1, f0, sA1, sB1, sA2, sB2, k + 1);
        if (k + 2 < nk) step(f0, f1, sA2, sB2, sA3, sB3, k + 2);
    }
    // the trailing loads land and every wave's operand reads return before LDS is reused
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    // epilogue: scale, round once, stage the wave's WM x WN bf16 tile in an LDS array of its own, write
    // 16-byte row chunks (element stores for a ragged last chunk)
    constexpr int PITCH = WN + 8;  // bf16 per staged row
    static_assert(WM * PITCH * 2 <= BM * BK, "a wave's tile fits one LDS array");
    uint16_t* tile = (uint16_t*)(wave == 0 ? sA0 : wave == 1 ? sA1 : wave == 2 ? sA2 : sA3);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
            *(v2u_t*)(tile + (16 * i + orow) * PITCH + 16 * j + 4 * (lane >> 4)) =
                v2u_t{pack_bf16x2(acc[i][j][0] * p.out_scale, acc[i][j][1] * p.out_scale),
                      pack_bf16x2(acc[i][j][2] * p.out_scale, acc[i][j][3] * p.out_scale)};
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    constexpr int CPR = WN / 8;
    const int64_t row0 = m0 + WM * wm, col0 = n0 + WN * wn;
#pragma unroll 1
    for (int q = lane; q < WM * CPR; q += 64) {
        const int r = q / CPR, c = 8 * (q % CPR);
        const int64_t m = row0 + r, n = col0 + c;
        if (m >= M || n >= N) continue;
        uint16_t* dst = p.C + m * ldc + n;
        const uint16_t* src = tile + r * PITCH + c;
        if (n + 8 <= N) {
            store_c8(dst, *(const v4u_t*)src);
        } else {
#pragma unroll 1
            for (int e = 0; e < 8 && n + e < N; ++e) dst[e] = src[e];
        }
    }
}

template <int BM, int BN, bool KN = false>
inline int fp8_gemm_mid_launch(Fp8GemmArgs p, hipStream_t s) {
    p.tiles_m = (uint32_t)((p.M + BM - 1) / BM);
    p.tiles_n = (uint32_t)((p.N + BN - 1) / BN);
    hipLaunchKernelGGL((fp8_gemm_mid_kernel<BM, BN, KN>), dim3(p.tiles_m * p.tiles_n), dim3(256), 0, s, p);
    return 0;
}

}  // namespace dopt
