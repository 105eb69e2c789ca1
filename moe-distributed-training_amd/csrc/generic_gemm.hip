// Shape- and dtype-generic grouped GEMM kernels.  They accept any strides, any K/N/rank and bf16/fp16/fp32 storage, and serve every
// case the 16-bit matrix-core kernels do not take (fp32 inputs, odd sizes, unaligned views): fp32 products without adapters, from a size on,
// on the fp32 matrix instructions, the others by fp32 FMA through LDS tiles.  fp32 accumulation, fixed summation order.
#include "common.h"
#include "kernels.h"
#include <type_traits>

namespace {

constexpr int GT = 16;   // tile edge; workgroup is GT x GT threads
// Contraction elements per step.  A step costs a trip to memory and two barriers whatever its length (the tiles are small and
// so are the launches), and the next step's operands are requested before the present one is worked through.  fp32, 512 rows over 4
// experts: 128 x 256 9.6 -> 8.2 us, 256 x 128 12.6 -> 9.9 against steps of 16 without the request ahead (same sums, same order).
// Products that steps of 64 would pad by more than a quarter take steps of 16: what a step lacks is worked through as zeros (2048 rows, K x 2048, fp32,
// steps of 16 and of 64: K=8 27 and 46 us, 40 38 and 45, 72 54 and 76, 128 79 and 76).  Products with adapters do so too: their time is that of the
// loads of the factors, which more elements per thread do not overlap (rank 16, K=64 137 and 143, 128 241 and 250).
constexpr int GK = 64, GK_SHORT = 16;
inline bool short_steps(int64_t K, bool adapters) { return adapters || (K + GK - 1) / GK * GK * 4 > 5 * K; }

// PAIR: two weights without adapters (gate, up) and Y = silu(gate) * up, the arithmetic of the separate launches (fp32: bit for bit).
// Y[out_row(m)][n] = sum_k X[in_row(m)][k] * (W[e][k][n] + scaling * sum_r A[e][k][r] * B[e][r][n])
// m runs over sorted positions; tiles of GT rows never straddle experts (find_row_tile on the offsets).
template <typename T, bool PAIR, int GK>
__global__ void __launch_bounds__(GT * GT) generic_grouped_gemm_kernel(
    const T* __restrict__ X, int64_t sxm, int64_t sxk, const T* __restrict__ W, const T* __restrict__ W_up, int64_t swe, int64_t swk, int64_t swn,
    const T* __restrict__ A, int64_t sae, int64_t sak, int64_t sar, const T* __restrict__ B, int64_t sbe, int64_t sbr,
    int64_t sbn, T* __restrict__ Y, int64_t sym, int64_t syn, const void* __restrict__ pos, int pos64,
    const void* __restrict__ offsets, int off64, int E, int64_t K, int64_t N, int rank, int fan_out, float scaling,
    int x_grouped, int y_grouped)
{
    constexpr int GPT = GT * GK / (GT * GT);   // elements of an operand tile per thread
    __shared__ float xs[GT][GK + 1];   // [row][k]
    __shared__ float ws[GK][GT + 1];   // [k][n]
    __shared__ float wu[PAIR ? GK : 1][GT + 1];
    __shared__ int64_t s_in[GT];
    RowTile rt;
    if (!find_row_tile(offsets, off64, E, GT, blockIdx.x, &rt)) return;
    const int tx = threadIdx.x % GT, ty = threadIdx.x / GT;
    const int64_t n0 = (int64_t)blockIdx.y * GT;
    const int64_t m = rt.row0 + ty;   // row of this thread's output
    const bool mval = m < rt.row1;
    int64_t out_row = 0;
    if (mval) {
        const int64_t p = (x_grouped && y_grouped) ? 0 : load_idx(pos, m, pos64);
        if (tx == 0) s_in[ty] = x_grouped ? m : p / fan_out;
        out_row = y_grouped ? m : p;
    }
    __syncthreads();
    const T* We = W + (int64_t)rt.expert * swe;
    const T* Ae = A ? A + (int64_t)rt.expert * sae : nullptr;
    const T* Be = B ? B + (int64_t)rt.expert * sbe : nullptr;
    // Which elements of an operand tile a thread loads: neighbours along the operand's own contiguous direction.  An adapter's factors are fetched
    // once per rank and the weight once: a B that is contiguous along n decides, where A is not along k (rank 16, 256 x 512, 2048 rows, k-contiguous
    // weights, fp32: 145 us along n, 584 along k, where every lane of A's loads is a row of its own).
    const int tid = threadIdx.x, nrows = (int)(rt.row1 - rt.row0);
    const bool w_along_k = swk == 1 && !(Ae && sbn == 1 && sak != 1);
    const T* Wu = PAIR ? W_up + (int64_t)rt.expert * swe : nullptr;
    auto load = [&](int64_t k0, float* xv, float* wv, float* uv) {
#pragma unroll
        for (int i = 0; i < GPT; ++i) {
            const int xr = tid / GK + i * (GT * GT / GK);
            const int64_t xk = k0 + tid % GK;
            xv[i] = (xr < nrows && xk < K) ? Elem<T>::ld(X + s_in[xr] * sxm + xk * sxk) : 0.f;
            const int64_t k = k0 + (w_along_k ? tid % GK : tid / GT + i * GT), n = n0 + (w_along_k ? tid / GK + i * (GT * GT / GK) : tid % GT);
            float w = 0.f, u = 0.f;
            if (k < K && n < N) {   // effective weight
                w = Elem<T>::ld(We + k * swk + n * swn);
                if (PAIR) u = Elem<T>::ld(Wu + k * swk + n * swn);
                else if (Ae) {
                    float l = 0.f;
                    for (int r = 0; r < rank; ++r) l = fmaf(Elem<T>::ld(Ae + k * sak + r * sar), Elem<T>::ld(Be + r * sbr + n * sbn), l);
                    w = fmaf(scaling, l, w);
                }
            }
            wv[i] = w;
            uv[i] = u;
        }
    };
    float acc = 0.f, acc_up = 0.f, xv[GPT], wv[GPT], uv[GPT];
    load(0, xv, wv, uv);
    for (int64_t k0 = 0; k0 < K; k0 += GK) {
#pragma unroll
        for (int i = 0; i < GPT; ++i) {
            xs[tid / GK + i * (GT * GT / GK)][tid % GK] = xv[i];
            const int wk = w_along_k ? tid % GK : tid / GT + i * GT, wn = w_along_k ? tid / GK + i * (GT * GT / GK) : tid % GT;
            ws[wk][wn] = wv[i];
            if (PAIR) wu[wk][wn] = uv[i];
        }
        __syncthreads();
        if (k0 + GK < K) load(k0 + GK, xv, wv, uv);
#pragma unroll
        for (int kk = 0; kk < GK; ++kk) {
            acc = fmaf(xs[ty][kk], ws[kk][tx], acc);
            if (PAIR) acc_up = fmaf(xs[ty][kk], wu[kk][tx], acc_up);
        }
        __syncthreads();
    }
    if (PAIR) acc = acc / (1.f + __expf(-acc)) * acc_up;   // as swiglu_fwd_kernel
    if (mval && n0 + tx < N) Elem<T>::st(Y + out_row * sym + (n0 + tx) * syn, acc);
}

// fp32 products without adapters on the fp32 matrix instructions: 16 rows x 64 columns per workgroup, a wave per 16 columns, steps of 64 along the contraction whose loads are
// requested a step ahead.  A thread of the kernel above reads two LDS words per multiply-add, which bounds it from a few hundred rows on; here a wave reads two per 16.
// LDS pitches: the 16 rows (or columns) x 4 k of a fragment, and the row of 64 that a wave stores, meet different banks; the weight's image is [n][k] or
// [k][n] as the weight is contiguous.  fp32 products and sums; a step's sums run over k in another order than above.
// (Contractions of at most 32 take steps of 16, whose loads are all of them used: 2048 rows over 8 experts, K x 2048, us with the kernel above, steps of 64 and of 16: 8 25.2, 24.3 and 15.2.)
constexpr int FM_ROWS = 16, FM_COLS = 64, FM_K_LONG = 64, FM_K_SHORT = 16, FM_WP = FM_COLS + 16;
template <bool PAIR, int FM_K>
__global__ void __launch_bounds__(256) grouped_gemm_f32_kernel(
    const float* __restrict__ X, int64_t sxm, int64_t sxk, const float* __restrict__ W, const float* __restrict__ W_up, int64_t swe, int64_t swk, int64_t swn,
    float* __restrict__ Y, int64_t sym, int64_t syn, const void* __restrict__ pos, int pos64, const void* __restrict__ offsets, int off64, int E, int64_t K,
    int64_t N, int fan_out, int x_grouped, int y_grouped)
{
    constexpr int FM_XP = FM_K + 4, STEP = 256 / FM_K;
    constexpr int XPT = FM_ROWS * FM_K / 256, WPT = FM_COLS * FM_K / 256;   // elements per thread and step
    __shared__ float xs[FM_ROWS * FM_XP];
    __shared__ float ws[PAIR ? 2 : 1][FM_K * FM_WP];   // (64 columns of FM_XP fit as well)
    static_assert(FM_COLS * FM_XP <= FM_K * FM_WP, "either image");
    __shared__ int64_t s_in[FM_ROWS], s_out[FM_ROWS];
    RowTile rt;
    if (!find_row_tile(offsets, off64, E, FM_ROWS, blockIdx.x, &rt)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 15, g = lane >> 4;
    const int nrows = (int)(rt.row1 - rt.row0);
    const int64_t n0 = (int64_t)blockIdx.y * FM_COLS;
    if (tid < FM_ROWS) {   // rows past the group repeat its last one and are not stored
        const int64_t m = rt.row0 + (tid < nrows ? tid : nrows - 1);
        const int64_t p = (x_grouped && y_grouped) ? 0 : load_idx(pos, m, pos64);
        s_in[tid] = x_grouped ? m : p / fan_out;
        s_out[tid] = y_grouped ? m : p;
    }
    __syncthreads();
    const float* We = W + (int64_t)rt.expert * swe;
    const float* Wu = PAIR ? W_up + (int64_t)rt.expert * swe : nullptr;
    const bool along_k = swk == 1;   // neighbouring threads along the weight's contiguous direction
    const int hi = tid / FM_K, lo = tid % FM_K, nhi = tid / FM_COLS, nlo = tid % FM_COLS;
    float xv[XPT], wv[WPT], uv[PAIR ? WPT : 1];
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int q = 0; q < XPT; ++q) xv[q] = k0 + lo < K ? X[s_in[hi + STEP * q] * sxm + (k0 + lo) * sxk] : 0.f;
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
            const int64_t k = k0 + (along_k ? lo : nhi + 4 * q), n = n0 + (along_k ? hi + STEP * q : nlo);
            const bool in = k < K && n < N;
            wv[q] = in ? We[k * swk + n * swn] : 0.f;
            if (PAIR) uv[q] = in ? Wu[k * swk + n * swn] : 0.f;
        }
    };
    f32x4_t acc2[2] = {}, up2[2] = {};   // alternate groups of four k: half as long a chain of sums, in time and in rounding
    load(0);
    const int nk = along_k ? FM_XP : 1, kk1 = along_k ? 1 : FM_WP;   // strides of n and k in the weight's image
    const bool live = n0 + wave * 16 < N;
    for (int64_t k0 = 0; k0 < K; k0 += FM_K) {
#pragma unroll
        for (int q = 0; q < XPT; ++q) xs[(hi + STEP * q) * FM_XP + lo] = xv[q];
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
            const int at = along_k ? (hi + STEP * q) * FM_XP + lo : (nhi + 4 * q) * FM_WP + nlo;
            ws[0][at] = wv[q];
            if (PAIR) ws[PAIR ? 1 : 0][at] = uv[q];
        }
        __syncthreads();
        if (k0 + FM_K < K) load(k0 + FM_K);
        if (live) {
            const float* xp = xs + i * FM_XP + g;
            const int w0 = (wave * 16 + i) * nk + g * kk1;
            const int left = K - k0 < FM_K ? (int)(K - k0) : FM_K;   // (what the image holds past K is zero)
            for (int kq = 0; kq < left; kq += 16)
#pragma unroll
                for (int c = 0; c < 16; c += 4) {
                    const float x = xp[kq + c];
                    const int h = c / 4 & 1;
                    acc2[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, ws[0][w0 + (kq + c) * kk1], acc2[h], 0, 0, 0);
                    if (PAIR) up2[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, ws[PAIR ? 1 : 0][w0 + (kq + c) * kk1], up2[h], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    // element r: row 4 g + r, column i of the wave's 16
    const int64_t n = n0 + wave * 16 + i;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float a = acc2[0][r] + acc2[1][r], u = up2[0][r] + up2[1][r];
        const float v = PAIR ? a / (1.f + __expf(-a)) * u : a;   // as swiglu_fwd_kernel
        if (4 * g + r < nrows && n < N) Y[s_out[4 * g + r] * sym + n * syn] = v;
    }
}

// O[e][k][n] = scale * sum_{m in group e} X[m][k] * Y[m][n];  zero for an empty group.  The last step is worked through in pieces of GT rows, as far
// as it holds rows, and a group of one piece by itself: the products are bound by their LDS reads (8 of 2048 x 2048, fp32: one row per
// expert 82 us, 260 as a whole step; 300 rows 1214 and 1274).
template <typename T>
__global__ void __launch_bounds__(GT * GT) generic_grouped_xty_kernel(
    const T* __restrict__ X, int64_t sxm, int64_t sxk, const T* __restrict__ Yp, int64_t sym, int64_t syn,
    T* __restrict__ O, int64_t soe, int64_t sok, int64_t son, const void* __restrict__ offsets, int off64, int64_t K,
    int64_t N, float scale)
{
    constexpr int GPT = GK / GT;   // elements of an operand tile per thread
    __shared__ float xs[GK][GT + 1];  // [m][k]
    __shared__ float ys[GK][GT + 1];  // [m][n]
    const int e = blockIdx.z;
    const int64_t start = e ? load_idx(offsets, e - 1, off64) : 0;
    const int64_t end = load_idx(offsets, e, off64);
    const int tx = threadIdx.x % GT, ty = threadIdx.x / GT;
    const int64_t k0 = (int64_t)blockIdx.x * GT, n0 = (int64_t)blockIdx.y * GT;
    if (end - start <= GT) {
        const int64_t m = start + ty;
        xs[ty][tx] = (m < end && k0 + tx < K) ? Elem<T>::ld(X + m * sxm + (k0 + tx) * sxk) : 0.f;
        ys[ty][tx] = (m < end && n0 + tx < N) ? Elem<T>::ld(Yp + m * sym + (n0 + tx) * syn) : 0.f;
        __syncthreads();
        float sum = 0.f;
#pragma unroll
        for (int q = 0; q < GT; ++q) sum = fmaf(xs[q][ty], ys[q][tx], sum);
        if (k0 + ty < K && n0 + tx < N) Elem<T>::st(O + (int64_t)e * soe + (k0 + ty) * sok + (n0 + tx) * son, sum * scale);
        return;
    }
    auto load = [&](int64_t m0, float* xv, float* yv) {
#pragma unroll
        for (int i = 0; i < GPT; ++i) {
            const int64_t m = m0 + ty + i * GT;
            xv[i] = (m < end && k0 + tx < K) ? Elem<T>::ld(X + m * sxm + (k0 + tx) * sxk) : 0.f;
            yv[i] = (m < end && n0 + tx < N) ? Elem<T>::ld(Yp + m * sym + (n0 + tx) * syn) : 0.f;
        }
    };
    float acc = 0.f, xv[GPT], yv[GPT];  // output (k0+ty, n0+tx)
    load(start, xv, yv);
    for (int64_t m0 = start; m0 < end; m0 += GK) {
#pragma unroll
        for (int i = 0; i < GPT; ++i) {
            xs[ty + i * GT][tx] = xv[i];
            ys[ty + i * GT][tx] = yv[i];
        }
        __syncthreads();
        auto multiply = [&](int first, auto length) {
#pragma unroll
            for (int q = 0; q < decltype(length)::value; ++q) acc = fmaf(xs[first + q][ty], ys[first + q][tx], acc);
        };
        if (m0 + GK < end) load(m0 + GK, xv, yv);
        if (m0 + GK <= end) multiply(0, std::integral_constant<int, GK>{});
        else for (int mm = 0; m0 + mm < end; mm += GT) multiply(mm, std::integral_constant<int, GT>{});
        __syncthreads();
    }
    if (k0 + ty < K && n0 + tx < N) Elem<T>::st(O + (int64_t)e * soe + (k0 + ty) * sok + (n0 + tx) * son, acc * scale);
}

// Which of the two: by the workgroups of the one above, a tile of 16 x 16 each.  Up to two of them per compute unit run side by side and are through after one
// chain of K steps; a thread of the kernel here fetches four times the weights before it can begin and has as long a chain.  From there on the one
// above takes turns.  Measured with 256 compute units, by workgroups of the one above; us above and here, of one product (and of gate and up in one launch):
//   256: 512 rows of 4 experts, K x N = 256 x 128, 11.6 and 11.9 (11.1 and 12.0); 8 rows of 8, 512 x 512, 13.4 and 17.6 (14.5 and 20.1)
//   512: 512 rows of 4, 128 x 256, 9.9 and 9.0 (8.8 and 7.9);  768 and 2048, 512 rows of 2, 512 x 384 and 512 x 1024: 1.42 and 1.6 times as fast here
// One round more where tiles or columns are half empty (groups of less than 16 rows; 65 to 85 columns of 128): 512, 8 rows of 8, 256 x 1024 10.3 and 11.1;
// 640, 2048 rows of 4, 64 x 80 0.98 times as fast (0.94);  768, 8 rows of 8, 64 x 1536 1.04 (1.05).
// Two rounds more below 64 k, where the chain is a step or two: 768, 64 rows of 8, 40 x 1536 0.95 (0.89); 1024, 512 rows of 2, 40 x 512 1.03 (1.01).
// Groups without rows count (the host does not see them): of 1698 drawn launches beyond these lines 20 are slower by more than 3 %, most of them of few rows over 64 or more experts and with
// steps filled to less than 0.8 (80 rows over 64, 77 x 293 6.8 and 7.9); two rounds more for those would leave 9 and cost 111 others a tenth.
bool f32_on_matrix_cores(int64_t R, int E, int64_t K, int64_t N)
{
    if (N <= FM_COLS / 2) return false;   // half of the columns at least (2048 rows, 250 x 16: 10.4 and 11.4)
    const int64_t rows16 = R / FM_ROWS, groups = R < E ? R : E, workgroups = (rows16 > groups ? rows16 : groups) * ((N + GT - 1) / GT);
    const bool full = R >= (int64_t)FM_ROWS * E && 3 * N >= 2 * ((N + FM_COLS - 1) / FM_COLS * FM_COLS);
    return workgroups >= ((K < 64 ? 4 : 2) + (full ? 0 : 1)) * (int64_t)moe_device_cus();
}

}  // namespace

int moe_launch_generic_gemm(const void* X, int64_t sxm, int64_t sxk, const void* W, int64_t swe, int64_t swk,
                            int64_t swn, const void* A, int64_t sae, int64_t sak, int64_t sar, const void* B,
                            int64_t sbe, int64_t sbr, int64_t sbn, void* Y, int64_t sym, int64_t syn, const void* pos,
                            int pos64, const void* offsets, int off64, int E, int64_t R, int64_t K, int64_t N, int rank,
                            int fan_out, float scaling, int x_grouped, int y_grouped, int dtype, hipStream_t stream)
{
    if (R == 0 || N == 0) return MOE_OK;
    const int64_t mtiles = R / GT + E;  // upper bound on sum_e ceil(c_e / GT)
    dim3 grid((unsigned)mtiles, (unsigned)((N + GT - 1) / GT));
    if (dtype == MOE_F32 && !A && f32_on_matrix_cores(R, E, K, N)) {
        static_assert(FM_ROWS == GT, "the same row tiles");
        auto f32 = K <= 2 * FM_K_SHORT ? grouped_gemm_f32_kernel<false, FM_K_SHORT> : grouped_gemm_f32_kernel<false, FM_K_LONG>;
        hipLaunchKernelGGL(f32, dim3((unsigned)mtiles, (unsigned)((N + FM_COLS - 1) / FM_COLS)), dim3(256), 0, stream, (const float*)X, sxm, sxk, (const float*)W,
                           (const float*)nullptr, swe, swk, swn, (float*)Y, sym, syn, pos, pos64, offsets, off64, E, K, N, fan_out, x_grouped, y_grouped);
        return moe_launch_status();
    }
    MOE_DISPATCH_DTYPE(dtype, {
        auto kern = short_steps(K, A != nullptr) ? generic_grouped_gemm_kernel<T, false, GK_SHORT> : generic_grouped_gemm_kernel<T, false, GK>;
        hipLaunchKernelGGL(kern, grid, dim3(GT * GT), 0, stream, (const T*)X, sxm, sxk, (const T*)W, (const T*)nullptr, swe, swk, swn, (const T*)A, sae, sak,
                           sar, (const T*)B, sbe, sbr, sbn, (T*)Y, sym, syn, pos, pos64, offsets, off64, E, K, N, rank, fan_out, scaling, x_grouped, y_grouped);
    });
    return moe_launch_status();
}

int moe_launch_generic_swiglu_pair(const float* X, int64_t sxm, int64_t sxk, const float* W_gate, const float* W_up, int64_t swe, int64_t swk,
                                   int64_t swn, float* H, int64_t ldh, const void* pos, int pos64, const void* offsets, int off64, int E, int64_t R,
                                   int64_t K, int64_t N, int fan_out, hipStream_t stream)
{
    if (R == 0 || N == 0) return MOE_OK;
    if (f32_on_matrix_cores(R, E, K, N)) {
        auto f32 = K <= 2 * FM_K_SHORT ? grouped_gemm_f32_kernel<true, FM_K_SHORT> : grouped_gemm_f32_kernel<true, FM_K_LONG>;
        hipLaunchKernelGGL(f32, dim3((unsigned)(R / FM_ROWS + E), (unsigned)((N + FM_COLS - 1) / FM_COLS)), dim3(256), 0, stream, X, sxm, sxk, W_gate, W_up, swe, swk,
                           swn, H, ldh, (int64_t)1, pos, pos64, offsets, off64, E, K, N, fan_out, 0, 1);
        return moe_launch_status();
    }
    dim3 grid((unsigned)(R / GT + E), (unsigned)((N + GT - 1) / GT));
    auto kern = short_steps(K, false) ? generic_grouped_gemm_kernel<float, true, GK_SHORT> : generic_grouped_gemm_kernel<float, true, GK>;
    hipLaunchKernelGGL(kern, grid, dim3(GT * GT), 0, stream, X, sxm, sxk, W_gate, W_up, swe, swk, swn, (const float*)nullptr,
                       0, 0, 0, (const float*)nullptr, 0, 0, 0, H, ldh, 1, pos, pos64, offsets, off64, E, K, N, 0, fan_out, 0.f, 0, 1);
    return moe_launch_status();
}

int moe_launch_generic_xty(const void* X, int64_t sxm, int64_t sxk, const void* Yp, int64_t sym, int64_t syn, void* O,
                           int64_t soe, int64_t sok, int64_t son, const void* offsets, int off64, int E, int64_t K,
                           int64_t N, float scale, int dtype, hipStream_t stream)
{
    if (E == 0 || K == 0 || N == 0) return MOE_OK;
    dim3 grid((unsigned)((K + GT - 1) / GT), (unsigned)((N + GT - 1) / GT), (unsigned)E);
    MOE_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((generic_grouped_xty_kernel<T>), grid, dim3(GT * GT), 0, stream,
                                                 (const T*)X, sxm, sxk, (const T*)Yp, sym, syn, (T*)O, soe, sok, son,
                                                 offsets, off64, K, N, scale));
    return moe_launch_status();
}
