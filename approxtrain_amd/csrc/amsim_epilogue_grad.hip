// Gradient of the fused epilogue act(z + bias) (amdenselayer.py:211-226, am_convolutional.py:248-276 run
// BiasAdd and the activation as ops of their own): d(z) = d(out) masked by the rectifier, d(bias) = sum
// of d(z) over the rows, in one pass over the gradient.
//
// HBM-bound: 4 bytes per element for a bias alone, 12 with the rectifier.  A workgroup owns a slab of
// rows of up to 64 columns; its threads run along the columns first, 16 lanes or more, and each adds every
// (256 / columns)-th row in four chains.  Rows of fewer than 16 columns leave lanes idle (6 columns: ten of
// 16) and are read in short pieces, which a narrow output's few bytes bear.  The slabs' sums go to the workspace and
// slab_sum_kernel adds them (one slab writes the bias gradient itself): no atomics, no counter to clear, the
// same bits on every run.  Chains run in 32 bits, what combines them in 64: added in 32 bits, a narrow output's
// 32 ways were the largest error (25600 x 16, terms of mean 0.3: 7.9e-8 of the result; 1.8e-8 now, torch's sum 2.9e-8).
// On the device, torch's compare, product with the mask and sum against this file: 25600 x 16 18.3 -> 7.5 us,
// 401408 x 6 30.4 -> 13.5, 8192 x 512 37.7 -> 13.7 (3.7 TB/s), 401408 x 128 257 -> 130 (4.7 TB/s); the sum alone
// 8192 x 512 18.2 -> 7.0, 401408 x 128 52.6 -> 37.7 (5.5 TB/s).  Training step of the 32 x 256 x 512 attention block
// (four biases) 2711 -> 2661 us; LeNet-5's convolutions, bound by the host, show no difference beyond their spread.
#include "amsim_internal.h"
#include "amsim_device.h"

#include <algorithm>

namespace amsim {

namespace {

constexpr int WG = 256;
constexpr int ROWS_PER_THREAD = 16;  // shortest slab: four loads in flight, four times
constexpr int MAX_SLABS = 2048;      // then slabs grow instead: eight workgroups per compute unit and column tile

struct EpilogueGradArgs {
    const float *grad, *out;  // out: only with the rectifier
    float *grad_z, *partial;  // [rows][cols]; [slabs][cols] (one slab: d(bias) itself) or null
    int64_t rows, rows_per_slab;
    int cols;
};

// The grid's first extent times the workgroup's threads stays below 2^32 (here and in the reduction of the
// slabs, four threads per column each), element indices far below 2^63.
inline bool extents_fit(int64_t rows, int cols) { return cols < (1 << 30) && (double)rows * cols <= 17592186044416.0; }

inline int threads_along_columns(int cols) { return cols > 32 ? 64 : cols > 16 ? 32 : 16; }

inline int64_t slabs_of(int64_t rows, int cols)
{
    const int64_t shortest = (int64_t)(WG / threads_along_columns(cols)) * ROWS_PER_THREAD;
    return std::min<int64_t>((rows + shortest - 1) / shortest, MAX_SLABS);
}

template <int TX, bool RELU>
__global__ __launch_bounds__(WG) void epilogue_grad_kernel(EpilogueGradArgs a)
{
    constexpr int TY = WG / TX;
    __shared__ double part[TY][TX];
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    const int64_t col = (int64_t)blockIdx.x * TX + tx;
    const int64_t beg = (int64_t)blockIdx.y * a.rows_per_slab;
    const int64_t end = beg + a.rows_per_slab < a.rows ? beg + a.rows_per_slab : a.rows;
    float c[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (col < a.cols) {
        for (int64_t r = beg + ty; r < end; r += 4 * TY) {
            float g[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t i = (r + u * TY) * a.cols + col;
                g[u] = r + u * TY < end ? a.grad[i] : 0.0f;
                // (a product with the mask, not a select: an infinite gradient of a masked element gives NaN)
                if (RELU && r + u * TY < end) g[u] = g[u] * (a.out[i] > 0.0f ? 1.0f : 0.0f);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (RELU && r + u * TY < end) a.grad_z[(r + u * TY) * a.cols + col] = g[u];
                c[u] += g[u];
            }
        }
    }
    if (a.partial == nullptr) return;  // (the same for every thread)
    part[ty][tx] = ((double)c[0] + c[1]) + ((double)c[2] + c[3]);
    __syncthreads();
    if (ty == 0 && col < a.cols) {
        double s = part[0][tx];
#pragma unroll
        for (int w = 1; w < TY; ++w) s += part[w][tx];
        a.partial[(int64_t)blockIdx.y * a.cols + col] = (float)s;
    }
}

// OUTS columns per workgroup, WG / OUTS threads ("ways") per column, eight loads of each in flight: few columns
// with many slabs use OUTS = 8, else the loop over the slabs is one long chain of memory latencies.
template <int OUTS>
__global__ __launch_bounds__(WG) void slab_sum_kernel(const float *partial, float *grad_bias, int slabs, int cols)
{
    constexpr int WAYS = WG / OUTS;
    __shared__ double part[WAYS][OUTS];
    const int o = threadIdx.x % OUTS, way = threadIdx.x / OUTS;
    const int64_t col = (int64_t)blockIdx.x * OUTS + o;
    double c[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (col < cols) {
        const float *src = partial + col;
        for (int sl = way; sl < slabs; sl += 8 * WAYS) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = src[(int64_t)min(sl + u * WAYS, slabs - 1) * cols];
#pragma unroll
            for (int u = 0; u < 8; ++u) c[u] += sl + u * WAYS < slabs ? v[u] : 0.0f;  // (no load waits for a test)
        }
    }
    part[way][o] = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
    __syncthreads();
    if (way == 0 && col < cols) {
        double s = part[0][o];
#pragma unroll
        for (int w = 1; w < WAYS; ++w) s += part[w][o];
        grad_bias[col] = (float)s;
    }
}

template <int TX>
void launch_epilogue_grad(const EpilogueGradArgs &a, int64_t slabs, bool relu, hipStream_t stream)
{
    const dim3 grid((unsigned)((a.cols + TX - 1) / TX), (unsigned)slabs);
    if (relu) epilogue_grad_kernel<TX, true><<<grid, WG, 0, stream>>>(a);
    else epilogue_grad_kernel<TX, false><<<grid, WG, 0, stream>>>(a);
}

}  // namespace

}  // namespace amsim

using namespace amsim;

extern "C" {

size_t amsim_epilogue_grad_workspace_bytes(int64_t rows, int cols)
{
    if (rows <= 0 || cols <= 0 || !extents_fit(rows, cols)) return 0;
    const int64_t slabs = slabs_of(rows, cols);
    return slabs == 1 ? 0 : (size_t)slabs * (size_t)cols * sizeof(float);
}

int amsim_epilogue_grad_f32(const float *grad, const float *out, int64_t rows, int cols, int act, float *grad_z,
                            float *grad_bias, void *workspace, size_t workspace_bytes, void *stream)
{
    if (rows < 0 || cols < 0) return fail(AMSIM_ERR_INVALID, "negative extent");
    if (act != AMSIM_ACT_NONE && act != AMSIM_ACT_RELU) return fail(AMSIM_ERR_INVALID, "unknown activation");
    if (!extents_fit(rows, cols)) return fail(AMSIM_ERR_UNSUPPORTED, "gradient exceeds the grid limit");
    const bool relu = act == AMSIM_ACT_RELU;
    if (rows == 0 || cols == 0) return fail(AMSIM_ERR_INVALID, "empty gradient");
    if (!relu && !grad_bias) return AMSIM_OK;
    if (!grad || (relu && (!out || !grad_z))) return fail(AMSIM_ERR_INVALID, "null tensor pointer");
    const size_t need = grad_bias ? amsim_epilogue_grad_workspace_bytes(rows, cols) : 0;
    if (need && (workspace == nullptr || ((uintptr_t)workspace & 255) || workspace_bytes < need))
        return fail(AMSIM_ERR_WORKSPACE, "workspace missing, not 256-byte aligned or smaller than " +
                                             std::to_string(need) + " bytes");
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t slabs = slabs_of(rows, cols);
    // one slab's sums are the bias gradient: no workspace and no second launch, which would only copy them
    float *const partial = !grad_bias ? nullptr : slabs == 1 ? grad_bias : static_cast<float *>(workspace);
    EpilogueGradArgs a{grad, out, grad_z, partial, rows, (rows + slabs - 1) / slabs, cols};
    switch (threads_along_columns(cols)) {
    case 64: launch_epilogue_grad<64>(a, slabs, relu, s); break;
    case 32: launch_epilogue_grad<32>(a, slabs, relu, s); break;
    default: launch_epilogue_grad<16>(a, slabs, relu, s); break;
    }
    AMSIM_HIP_CHECK(hipGetLastError());
    if (!grad_bias || slabs == 1) return AMSIM_OK;
    if (cols <= 16384 && slabs >= 64)
        slab_sum_kernel<8><<<(unsigned)((cols + 7) / 8), WG, 0, s>>>(partial, grad_bias, (int)slabs, cols);
    else
        slab_sum_kernel<64><<<(unsigned)((cols + 63) / 64), WG, 0, s>>>(partial, grad_bias, (int)slabs, cols);
    AMSIM_HIP_CHECK(hipGetLastError());
    return AMSIM_OK;
}

}  // extern "C"
