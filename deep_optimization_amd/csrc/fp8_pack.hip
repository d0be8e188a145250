// Layout conversion for the FP8 GEMM: any strided byte matrix -> K-contiguous rows.
//
// dst[r * ld_dst + c] = src[r * stride_r + c * stride_c] for r < rows, c < cols (element strides
// in bytes, any non-negative values), and zeros for cols <= c < cols_out (the columns that fill K up to
// a multiple of 16; a separate fill of the buffer was a launch of 4.6 us). The GEMM (fp8_gemm.h) reads both operands K-contiguous; the
// reference's Triton_Linear (Activation_Compression/triton_kernel/linear.py:43-95) takes A [M, K]
// and B [K, N] with arbitrary strides, so B in its natural row-major [K, N] layout (stride_r =
// 1 along N, stride_c = ldb along K) is transposed here into [N, K].
//
// Three kernels:
//   - transpose (stride_r == 1): 128 x 128 byte tiles. A lane reads 16 contiguous source bytes (rows
//     r..r+15) of four columns c..c+3, transposes the sixteen 4-byte rows in registers (v_perm_b32) and
//     writes them to LDS as dwords; after the barrier it writes 16 contiguous destination bytes of one row
//     per step. Rows of the LDS tile are 33 dwords apart, so the dword writes of 8 lanes 16 rows apart fall
//     in different banks. Bound by HBM: [8192, 8192] takes 20.8 us, 6.4 TB/s, and 31.1 us on [8191, 8191],
//     whose unaligned lines are read twice (64 x 64 tiles moved byte by byte: 31.1 and 101 us).
//   - copy (stride_c == 1): whole rows whose pitch or base does not suit the GEMM; 16 bytes per lane
//     ([8192, 8192] 20.2 us; 93.6 us through the gather).
//   - gather (anything else): one byte per lane, consecutive lanes along c.
// Source addresses need no alignment: 16-byte loads from any byte are one instruction on gfx950. The last
// chunk of a run that is no multiple of 16 bytes is the 16 bytes that end it, shifted (tail16): a loop over its
// bytes put its loads one after the other.
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dopt {

constexpr int TP = 128;          // tile edge (bytes)
constexpr int TPITCH = TP / 4 + 1;  // dwords per LDS row

// 16 bytes from any address
__device__ __forceinline__ uint4 load16_any(const uint8_t* p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

__device__ __forceinline__ uint32_t pick(bool c, uint32_t a, uint32_t b) { return c ? a : b; }

// bytes i..i+15 (i < n) of a run of n bytes, zeros past its end
__device__ __forceinline__ uint4 tail16(const uint8_t* run, int64_t i, int64_t n) {
    if (n < 16) {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 15; ++e)
            if (i + e < n) w[e >> 2] |= (uint32_t)run[i + e] << (8 * (e & 3));
        return make_uint4(w[0], w[1], w[2], w[3]);
    }
    const int64_t o = i + 16 <= n ? i : n - 16;
    const uint32_t sh = (uint32_t)(i - o);
    uint4 v = load16_any(run + o);
    if (sh) {
        const bool s8 = sh & 8u, s4 = sh & 4u;
        const uint32_t a0 = pick(s8, v.z, v.x), a1 = pick(s8, v.w, v.y), a2 = pick(s8, 0u, v.z), a3 = pick(s8, 0u, v.w);
        const uint32_t b0 = pick(s4, a1, a0), b1 = pick(s4, a2, a1), b2 = pick(s4, a3, a2), b3 = pick(s4, 0u, a3);
        v = make_uint4(__builtin_amdgcn_alignbyte(b1, b0, sh & 3u), __builtin_amdgcn_alignbyte(b2, b1, sh & 3u),
                       __builtin_amdgcn_alignbyte(b3, b2, sh & 3u), b3 >> (8 * (sh & 3u)));
    }
    return v;
}

__global__ __launch_bounds__(256) void fp8_transpose_kernel(const uint8_t* __restrict__ src, int64_t rows,
                                                            int64_t cols, int64_t stride_c, uint8_t* __restrict__ dst,
                                                            int64_t ld_dst, int64_t cols_out, uint32_t row_tiles) {
    __shared__ uint32_t t[TP * TPITCH];
    const int64_t r0 = (int64_t)(blockIdx.x % row_tiles) * TP, c0 = (int64_t)(blockIdx.x / row_tiles) * TP;
    const int tid = threadIdx.x;
    {
        const int rl = (tid & 7) * 16, cl = (tid >> 3) * 4;  // this lane's 16 x 4 block
        const int64_t r = r0 + rl;
        uint32_t w[4][4];  // [column][dword of its 16 rows]
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t c = c0 + cl + j;
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (c < cols && r < rows) v = tail16(src + c * stride_c, r, rows);
            w[j][0] = v.x;
            w[j][1] = v.y;
            w[j][2] = v.z;
            w[j][3] = v.w;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // a 4 x 4 byte block: rows 4q..4q+3 of the four columns
            const uint32_t lo01 = __builtin_amdgcn_perm(w[1][q], w[0][q], 0x05010400u);  // a0 b0 a1 b1
            const uint32_t hi01 = __builtin_amdgcn_perm(w[1][q], w[0][q], 0x07030602u);  // a2 b2 a3 b3
            const uint32_t lo23 = __builtin_amdgcn_perm(w[3][q], w[2][q], 0x05010400u);
            const uint32_t hi23 = __builtin_amdgcn_perm(w[3][q], w[2][q], 0x07030602u);
            uint32_t* at = t + (rl + 4 * q) * TPITCH + (cl >> 2);
            at[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
            at[TPITCH] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
            at[2 * TPITCH] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
            at[3 * TPITCH] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
        }
    }
    __syncthreads();
    const int cl = (tid & 7) * 16;
    const int64_t c = c0 + cl;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int rl = (tid >> 3) + 32 * h;
        const int64_t r = r0 + rl;
        if (r >= rows || c >= cols_out) continue;
        const uint32_t* s = t + rl * TPITCH + (cl >> 2);
        const uint32_t v[4] = {s[0], s[1], s[2], s[3]};
        uint8_t* d = dst + r * ld_dst + c;
        if (c + 16 <= cols_out && (((uintptr_t)d) & 15) == 0) {
            *(uint4*)d = make_uint4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (c + i < cols_out) d[i] = (uint8_t)(v[i >> 2] >> (8 * (i & 3)));
        }
    }
}

// rows of `cols` contiguous bytes: lane -> 16 bytes of one row
__global__ __launch_bounds__(256) void fp8_copy_rows_kernel(const uint8_t* __restrict__ src, int64_t cols,
                                                            int64_t stride_r, uint8_t* __restrict__ dst, int64_t ld_dst,
                                                            int64_t cols_out, uint64_t chunks, uint32_t per_row) {
    const uint64_t q = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= chunks) return;
    const int64_t r = (int64_t)(q / per_row), c = (int64_t)(q % per_row) * 16;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (c < cols) v = tail16(src + r * stride_r, c, cols);
    uint8_t* d = dst + r * ld_dst + c;
    if (c + 16 <= cols_out && (((uintptr_t)d) & 15) == 0) {
        *(uint4*)d = v;
    } else {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (c + i < cols_out) d[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
    }
}

__global__ __launch_bounds__(256) void fp8_gather_kernel(const uint8_t* __restrict__ src, int64_t rows, int64_t cols,
                                                         int64_t stride_r, int64_t stride_c, uint8_t* __restrict__ dst,
                                                         int64_t ld_dst, int64_t cols_out, uint32_t col_blocks) {
    const int64_t r = blockIdx.x / col_blocks;
    const int64_t c = (int64_t)(blockIdx.x % col_blocks) * 256 + threadIdx.x;
    if (r < rows && c < cols_out) dst[r * ld_dst + c] = c < cols ? src[r * stride_r + c * stride_c] : (uint8_t)0;
}

int launch_fp8_pack(const uint8_t* src, int64_t rows, int64_t cols, int64_t stride_r, int64_t stride_c, uint8_t* dst,
                    int64_t ld_dst, int64_t cols_out, hipStream_t s) {
    if (rows == 0 || cols_out == 0) return 0;
    if (stride_r == 1) {
        const uint64_t rt = (uint64_t)((rows + TP - 1) / TP), ct = (uint64_t)((cols_out + TP - 1) / TP);
        if (rt * ct >= (1ull << 31)) return -1;
        hipLaunchKernelGGL(fp8_transpose_kernel, dim3((uint32_t)(rt * ct)), dim3(256), 0, s, src, rows, cols, stride_c,
                           dst, ld_dst, cols_out, (uint32_t)rt);
    } else if (stride_c == 1) {
        const uint64_t pr = (uint64_t)((cols_out + 15) / 16), chunks = (uint64_t)rows * pr;
        if (pr >= (1ull << 32) || (chunks + 255) / 256 >= (1ull << 31)) return -1;
        hipLaunchKernelGGL(fp8_copy_rows_kernel, dim3((uint32_t)((chunks + 255) / 256)), dim3(256), 0, s, src, cols,
                           stride_r, dst, ld_dst, cols_out, chunks, (uint32_t)pr);
    } else {
        const uint64_t cb = (uint64_t)((cols_out + 255) / 256);
        if ((uint64_t)rows * cb >= (1ull << 31)) return -1;
        hipLaunchKernelGGL(fp8_gather_kernel, dim3((uint32_t)(rows * cb)), dim3(256), 0, s, src, rows, cols, stride_r,
                           stride_c, dst, ld_dst, cols_out, (uint32_t)cb);
    }
    return 0;
}

}  // namespace dopt
