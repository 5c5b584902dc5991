// Column sums of a bf16 matrix for gfx950: the bias gradients of the MLP
// layers (autograd's grad.sum(0) of z + b, lib_sparse/layers.py:86-94, :169-177).
//
// Bound by the one read of the matrix.  Two passes: every workgroup sums a
// block of 256 columns by up to a few hundred rows in fp32 (so that a narrow
// matrix still fills the chip) and writes one row of partial sums; a second,
// small pass adds the partial rows in order and rounds once to bf16.  The
// split is a function of the shape alone, so the sums are deterministic.
// 4096 x 16384: 28 us against 150 us for the library's column reduction, which
// gives each workgroup whole columns.
#include <algorithm>

#include "bs_device.h"
#include "bs_host.h"

namespace bs {

constexpr int kSumThreads = 256;
constexpr int kSumCols = 256;       // columns per workgroup: 32 chunks of 8, 512 contiguous bytes per row
constexpr int kSumRowLanes = kSumThreads / (kSumCols / 8);   // rows in flight per pass
constexpr int kSumUnroll = 4;       // independent 16-byte loads per thread

__device__ __forceinline__ void add_chunk(float (&s)[8], const uint4 v)
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        s[2 * i] += __uint_as_float(w[i] << 16);
        s[2 * i + 1] += __uint_as_float(w[i] & 0xffff0000u);
    }
}

// part[blockIdx.y * C + c] = sum of x[r, c] over the rows of blockIdx.y.
// C % 8 == 0 and x 16-byte aligned (host check).
template <bool NT>
__global__ __launch_bounds__(kSumThreads) void col_sum_part_kernel(const uint16_t* x, int64_t R, int64_t C,
                                                                   int64_t rows_per, float* part)
{
    __shared__ float s_acc[kSumRowLanes][kSumCols];
    const int tid = threadIdx.x, ch = tid & 31, rl = tid >> 5;
    const int64_t c = (int64_t)blockIdx.x * kSumCols + ch * 8;
    const int64_t r0 = (int64_t)blockIdx.y * rows_per, r1 = min(R, r0 + rows_per);
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (c < C) {
        int64_t r = r0 + rl;
        for (; r + (kSumUnroll - 1) * kSumRowLanes < r1; r += kSumUnroll * kSumRowLanes) {
            uint4 v[kSumUnroll];
#pragma unroll
            for (int u = 0; u < kSumUnroll; u++) v[u] = ld16<NT>(x + (r + u * kSumRowLanes) * C + c);
#pragma unroll
            for (int u = 0; u < kSumUnroll; u++) add_chunk(s, v[u]);
        }
        for (; r < r1; r += kSumRowLanes) add_chunk(s, ld16<NT>(x + r * C + c));
    }
#pragma unroll
    for (int e = 0; e < 8; e++) s_acc[rl][ch * 8 + e] = s[e];
    __syncthreads();
    const int64_t col = (int64_t)blockIdx.x * kSumCols + tid;
    if (col < C) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < kSumRowLanes; q++) t += s_acc[q][tid];
        part[(int64_t)blockIdx.y * C + col] = t;
    }
}

// Workgroups below col_blocks: out[c] = bf16(sum over rows p < S of part[p, c]),
// 64 columns each, the four waves taking every fourth partial row.  The
// others: the largest of `maxima` (bf16 magnitude bits) into the amax slot.
constexpr int kMaxBlocks = 16;
__global__ __launch_bounds__(kSumThreads) void sums_finish_kernel(const float* part, int64_t S, int64_t C,
                                                                  uint16_t* out, uint32_t col_blocks,
                                                                  const uint32_t* maxima, int64_t nmax,
                                                                  uint64_t* slot, uint32_t epoch)
{
    __shared__ float s_acc[4][64];
    __shared__ uint32_t s_mx[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.x >= col_blocks) {
        const int64_t stride = (int64_t)(gridDim.x - col_blocks) * kSumThreads;
        uint32_t m = 0;
        for (int64_t i = (int64_t)(blockIdx.x - col_blocks) * kSumThreads + threadIdx.x; i < nmax; i += stride)
            m = max(m, maxima[i]);
        m = wave_max_u32(m);
        if (lane == 0) s_mx[wave] = m;
        __syncthreads();
        if (threadIdx.x == 0)
            atomicMax((unsigned long long*)slot, (unsigned long long)(((uint64_t)epoch << 32) |
                                                                      max(max(s_mx[0], s_mx[1]), max(s_mx[2], s_mx[3]))));
        return;
    }
    const int64_t c = (int64_t)blockIdx.x * 64 + lane;
    float t = 0.f;
    if (c < C) {
        int64_t p = wave;
        for (; p + 28 < S; p += 32) {                  // eight loads in flight
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = part[(p + 4 * u) * C + c];
#pragma unroll
            for (int u = 0; u < 8; u++) t += v[u];
        }
        for (; p < S; p += 4) t += part[p * C + c];
    }
    s_acc[wave][lane] = t;
    __syncthreads();
    if (wave == 0 && c < C)
        out[c] = (uint16_t)f32_to_bf16((s_acc[0][lane] + s_acc[1][lane]) + (s_acc[2][lane] + s_acc[3][lane]));
}

// Row splits of the first pass: about 2048 workgroups (8 per CU), each of at
// least 64 rows (8 per row lane), so that the partial rows stay a small
// fraction (at most 1/32) of the bytes read.
static int64_t col_sum_splits(int64_t R, int64_t C)
{
    const int64_t groups = (C + kSumCols - 1) / kSumCols;
    return std::max<int64_t>(1, std::min<int64_t>((2048 + groups - 1) / groups, R / 64));
}

int sums_finish_launch(const float* part, int64_t S, int64_t C, void* out, const uint32_t* maxima, int64_t nmax,
                       uint64_t* slot, uint32_t epoch, hipStream_t stream)
{
    const uint32_t cb = part ? (uint32_t)((C + 63) / 64) : 0u;
    const uint32_t mb = maxima ? (uint32_t)std::min<int64_t>((nmax + 1023) / 1024, kMaxBlocks) : 0u;
    if (cb + mb == 0) return BS_OK;
    hipLaunchKernelGGL(sums_finish_kernel, dim3(cb + mb), dim3(kSumThreads), 0, stream, part, S, C, (uint16_t*)out, cb,
                       maxima, nmax, slot, epoch);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? BS_OK : set_error(BS_ERR_HIP, "sums_finish launch: %s", hipGetErrorString(e));
}

}  // namespace bs

using namespace bs;

extern "C" int64_t bs_col_sum_workspace_bytes(int64_t R, int64_t C)
{
    if (R <= 0 || C <= 0) return 0;
    return col_sum_splits(R, C) * C * 4;
}

extern "C" int bs_col_sum(const void* x, int64_t R, int64_t C, void* out, void* workspace, int64_t workspace_bytes,
                          void* stream)
{
    clear_error();
    if (R < 0 || C < 0) return set_error(BS_ERR_INVALID, "bs_col_sum: negative shape");
    if (C == 0) return BS_OK;
    if (R == 0) return set_error(BS_ERR_INVALID, "bs_col_sum: no rows");
    if (x == nullptr || out == nullptr) return set_error(BS_ERR_INVALID, "bs_col_sum: null pointer");
    if (C % 8 != 0 || (((uintptr_t)x) & 15u))
        return set_error(BS_ERR_INVALID, "bs_col_sum: needs C %% 8 == 0 and a 16-byte aligned input");
    if (((uintptr_t)out) & 1u) return set_error(BS_ERR_INVALID, "bs_col_sum: output misaligned");
    if ((uint64_t)R * (uint64_t)C >= kMaxElemsUntested)
        return set_error(BS_ERR_INVALID, "bs_col_sum: R*C must be < 2^31");
    if (workspace == nullptr || workspace_bytes < bs_col_sum_workspace_bytes(R, C) || (((uintptr_t)workspace) & 3u))
        return set_error(BS_ERR_INVALID, "bs_col_sum: workspace too small or misaligned");
    const int64_t S = col_sum_splits(R, C), rows_per = (R + S - 1) / S;
    const dim3 grid((uint32_t)((C + kSumCols - 1) / kSumCols), (uint32_t)S);
    hipStream_t st = (hipStream_t)stream;
    auto kernel = use_nontemporal(2 * R * C) ? col_sum_part_kernel<true> : col_sum_part_kernel<false>;
    hipLaunchKernelGGL(kernel, grid, dim3(kSumThreads), 0, st, (const uint16_t*)x, R, C, rows_per, (float*)workspace);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(BS_ERR_HIP, "bs_col_sum launch: %s", hipGetErrorString(e));
    return sums_finish_launch((const float*)workspace, S, C, out, nullptr, 0, nullptr, 0, st);
}
