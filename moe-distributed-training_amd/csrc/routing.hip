// Router (logits GEMV, softmax/top-k/renormalise) and the integer pipeline that puts token->expert
// assignments into expert-grouped order: histogram, prefix sums, stable counting sort, padded block table.
// All integer results are exact and independent of launch geometry (no floating point, no data races:
// LDS/global atomics are only used for integer counts whose final value is order independent).
#include "common.h"
#include "kernels.h"
#include <mutex>
#include <type_traits>

namespace {

constexpr int ROUTER_EXPERT_GROUP = 8;

// 8 consecutive elements as floats; one 16-byte (2-byte types) or two 16-byte (fp32) loads when the row is aligned
template <typename T>
__device__ __forceinline__ void load8(const T* p, float* v, int kn, bool vec_ok)
{
    if (vec_ok && kn == 8) {
        if (sizeof(T) == 2) {
            const uint4 raw = *(const uint4*)p;
            const T* e = (const T*)&raw;
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = Elem<T>::ld(e + u);
        } else {
            const float4 a = *(const float4*)p, b = *((const float4*)p + 1);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        }
    } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = (u < kn) ? Elem<T>::ld(p + u) : 0.f;
    }
}

// v[0..N): sums over the 64 lanes, see router_logits_kernel
template <int N, int O>
__device__ __forceinline__ void butterfly_sums(float* v, int lane)
{
    if constexpr (O > 0) {
        if constexpr (N > 1) {
            const bool up = (lane & O) != 0;
#pragma unroll
            for (int q = 0; q < N / 2; ++q) {
                const float keep = up ? v[N / 2 + q] : v[q], send = up ? v[q] : v[N / 2 + q];
                v[q] = keep + __shfl_xor(send, O, 64);
            }
            butterfly_sums<N / 2, O / 2>(v, lane);
        } else {
            v[0] += __shfl_xor(v[0], O, 64);
            butterfly_sums<1, O / 2>(v, lane);
        }
    }
}

// logits[t][e] = sum_k x[t][k] * wg[e][k], fp32 accumulate, for the shapes router_mfma_kernel does not take (more than 8
// experts, fp32, odd hidden sizes).  One wave owns TOKENS tokens and one group of 8 experts (blockIdx.y) and walks the
// hidden dimension 8 elements per lane at a time: one wave per expert group keeps every SIMD busy where one wave for all
// groups did not (2048 tokens x 64 experts x 2048 columns: 83 -> 28 us; bound by the vector ALUs, one FMA per token,
// expert and column plus the unpacking).  The order of the additions of a logit depends neither on TOKENS nor on the grid.
// TOPK: up to 8 experts, whose logits all lie in one wave: softmax and top-k follow in the same launch (scores .. renorm; 256 tokens fp32, 4 experts:
// 4.4 + 3.5 us in two launches, 6.2 in one).
constexpr int TK_LANES = 16;
template <int PER_LANE>
__device__ __forceinline__ void softmax_topk_token(const float* __restrict__ l, float* __restrict__ s, float* __restrict__ topw, int32_t* __restrict__ topi, int E, int k,
                                                   int renorm, bool store);
template <typename T, int TOKENS, bool TOPK>
__global__ void __launch_bounds__(256) router_logits_kernel(const T* __restrict__ x, int64_t ldx,
                                                            const T* __restrict__ wg, int64_t ldw,
                                                            float* __restrict__ logits, int64_t ntok, int64_t d, int E,
                                                            bool vec_ok, float* __restrict__ scores, float* __restrict__ topw,
                                                            int32_t* __restrict__ topi, int k, int renorm)
{
    __shared__ float s_l[TOPK ? 4 : 1][TOKENS][ROUTER_EXPERT_GROUP];
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t t0 = wave * TOKENS;
    if (t0 >= ntok) return;
    const int e0 = blockIdx.y * ROUTER_EXPERT_GROUP;
    float acc[TOKENS][ROUTER_EXPERT_GROUP];
#pragma unroll
    for (int i = 0; i < TOKENS; ++i)
#pragma unroll
        for (int j = 0; j < ROUTER_EXPERT_GROUP; ++j) acc[i][j] = 0.f;
#pragma unroll 1
    for (int64_t k0 = (int64_t)lane * 8; k0 < d; k0 += 64 * 8) {
        const int kn = (d - k0 < 8) ? (int)(d - k0) : 8;
        float xv[TOKENS][8];
#pragma unroll
        for (int i = 0; i < TOKENS; ++i) {
            const int64_t t = (t0 + i < ntok) ? t0 + i : ntok - 1;
            load8<T>(x + t * ldx + k0, xv[i], kn, vec_ok);
        }
#pragma unroll
        for (int j = 0; j < ROUTER_EXPERT_GROUP; ++j) {
            const int e = (e0 + j < E) ? e0 + j : E - 1;
            float wv[8];
            load8<T>(wg + (int64_t)e * ldw + k0, wv, kn, vec_ok);
#pragma unroll
            for (int i = 0; i < TOKENS; ++i)
#pragma unroll
                for (int u = 0; u < 8; ++u) acc[i][j] = fmaf(xv[i][u], wv[u], acc[i][j]);
        }
    }
    // Sums over the 64 lanes of all NV values at once: in each step of the butterfly a lane keeps one half of its values
    // and sends the other half to its partner, so NV values cost about NV exchanges instead of 6 NV (the additions, and
    // so the bits, are those of a butterfly per value).  Lane l ends up with value l * NV / 64.
    constexpr int NV = TOKENS * ROUTER_EXPERT_GROUP;
    float v[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = acc[q / ROUTER_EXPERT_GROUP][q % ROUTER_EXPERT_GROUP];
    butterfly_sums<NV, 32>(v, lane);
    const int idx = lane * NV / 64;
    const bool writer = lane % (64 / NV) == 0;
    const int i = idx / ROUTER_EXPERT_GROUP, e = e0 + idx % ROUTER_EXPERT_GROUP;
    if (writer && t0 + i < ntok && e < E) logits[(t0 + i) * E + e] = v[0];
    if constexpr (TOPK) {
        static_assert(TOKENS * TK_LANES <= 64, "the tokens of a wave share its lanes");
        float (*l)[ROUTER_EXPERT_GROUP] = s_l[threadIdx.x >> 6];
        if (writer) l[i][idx % ROUTER_EXPERT_GROUP] = v[0];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the wave's own writes, read by its other lanes
        __builtin_amdgcn_wave_barrier();
        const int tt = lane / TK_LANES;
        if (tt < TOKENS) {   // whole groups of TK_LANES lanes
            const int64_t t = t0 + tt < ntok ? t0 + tt : ntok - 1;
            softmax_topk_token<1>(l[tt], scores + t * E, topw + t * k, topi + t * k, E, k, renorm, t0 + tt < ntok);
        }
    }
}

// fp32 softmax over the E logits of one token, k rounds of arg-max (the lowest expert index wins a tie), optional division
// by the sum of the selected scores.  s / topw / topi point at the token's output rows.  TK_LANES lanes share a token,
// lane l holding experts l, l + TK_LANES, ..: the score row is read and written coalesced and never read back from memory
// (one thread per token walking its rows in memory took 347 us for 2048 tokens x 64 experts, top-8; this takes 11).
// The exponentials are added in expert order, the selected scores in selection order: every lane of the token adds all of
// them, so the bits do not depend on the number of lanes.  All TK_LANES lanes of a token must be active.
constexpr int TK_MAX_PER_LANE = 16;   // up to TK_LANES * TK_MAX_PER_LANE = 256 experts in registers
template <int PER_LANE>
__device__ __forceinline__ void softmax_topk_token(const float* __restrict__ l, float* __restrict__ s,
                                                   float* __restrict__ topw, int32_t* __restrict__ topi, int E, int k,
                                                   int renorm, bool store)
{
    const int ln = threadIdx.x & (TK_LANES - 1);
    float v[PER_LANE];
    float mx = -__builtin_inff();
#pragma unroll
    for (int q = 0; q < PER_LANE; ++q) {
        const int e = q * TK_LANES + ln;
        v[q] = e < E ? l[e] : -__builtin_inff();
        mx = fmaxf(mx, v[q]);
    }
#pragma unroll
    for (int o = TK_LANES / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, TK_LANES));
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < PER_LANE; ++q) {
        const int e0 = q * TK_LANES;
        v[q] = e0 + ln < E ? expf(v[q] - mx) : 0.f;
#pragma unroll
        for (int i = 0; i < TK_LANES; ++i)
            if (e0 + i < E) sum += __shfl(v[q], i, TK_LANES);
    }
#pragma unroll
    for (int q = 0; q < PER_LANE; ++q) {
        const int e = q * TK_LANES + ln;
        v[q] = v[q] / sum;
        if (store && e < E) s[e] = v[q];
        if (e >= E) v[q] = -2.f;                     // never selected
        else if (!(v[q] >= 0.f)) v[q] = -1.f;        // NaN scores lose to every number and are taken in expert order
    }
    float wsum = 0.f, kept_w = 0.f;
    int kept_e = 0;
    for (int j = 0; j < k; ++j) {
        float bv = v[0];
        int be = ln;
#pragma unroll
        for (int q = 1; q < PER_LANE; ++q)
            if (v[q] > bv) { bv = v[q]; be = q * TK_LANES + ln; }
#pragma unroll
        for (int o = TK_LANES / 2; o > 0; o >>= 1) {
            const float ov = __shfl_xor(bv, o, TK_LANES);
            const int oe = __shfl_xor(be, o, TK_LANES);
            if (ov > bv || (ov == bv && oe < be)) { bv = ov; be = oe; }
        }
#pragma unroll
        for (int q = 0; q < PER_LANE; ++q)
            if (be == q * TK_LANES + ln) v[q] = -2.f;
        const float w = bv < 0.f ? __builtin_nanf("") : bv;
        wsum += w;
        // lane j % TK_LANES keeps selection j until the sum is known; a token with more selections writes them in rounds below
        if (!renorm) { if (store && ln == 0) { topw[j] = w; topi[j] = be; } }
        else if (k <= TK_LANES) { if (ln == j) { kept_w = w; kept_e = be; } }
        else if (store && ln == 0) { topw[j] = w; topi[j] = be; }
    }
    if (renorm && store) {
        if (k <= TK_LANES) { if (ln < k) { topw[ln] = kept_w / wsum; topi[ln] = kept_e; } }
        else if (ln == 0) for (int j = 0; j < k; ++j) topw[j] = topw[j] / wsum;
    }
}

template <int PER_LANE>
__global__ void __launch_bounds__(256) router_topk_kernel(const float* __restrict__ logits, float* __restrict__ scores,
                                                          float* __restrict__ topw, int32_t* __restrict__ topi, int64_t ntok, int E,
                                                          int k, int renorm)
{
    const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / TK_LANES;
    const int64_t tc = t < ntok ? t : ntok - 1;   // (lanes past the end work on the last token and store nothing)
    softmax_topk_token<PER_LANE>(logits + tc * E, scores + tc * E, topw + tc * k, topi + tc * k, E, k, renorm, t < ntok);
}

// More experts than a token's lanes hold in registers: one thread per token, rows walked in memory.
__global__ void router_topk_wide_kernel(const float* __restrict__ logits, float* __restrict__ scores,
                                        float* __restrict__ topw, int32_t* __restrict__ topi, int64_t ntok, int E, int k,
                                        int renorm)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntok) return;
    const float* l = logits + t * E;
    float* s = scores + t * E;
    topw += t * k;
    topi += t * k;
    float mx = l[0];
    for (int e = 1; e < E; ++e) mx = fmaxf(mx, l[e]);
    float sum = 0.f;
    for (int e = 0; e < E; ++e) { const float v = expf(l[e] - mx); s[e] = v; sum += v; }
    for (int e = 0; e < E; ++e) s[e] = s[e] / sum;
    float wsum = 0.f;
    for (int j = 0; j < k; ++j) {
        int best = -1;
        float bv = 0.f;
        for (int e = 0; e < E; ++e) {
            bool taken = false;
            for (int jj = 0; jj < j; ++jj) taken |= (topi[jj] == e);
            if (taken) continue;
            const float v = s[e];
            if (best < 0 || v > bv) { best = e; bv = v; }
        }
        topi[j] = best;
        topw[j] = bv;
        wsum += bv;
    }
    if (renorm) for (int j = 0; j < k; ++j) topw[j] = topw[j] / wsum;
}

// Logits, softmax and top-k in one launch for up to ROUTER_EXPERT_GROUP experts of a 2-byte type, the logits on the
// matrix cores.  A workgroup of 8 waves handles 16 tokens; wave w takes the w-th eighth of the hidden dimension: it
// requests all of its operand fragments at once -- 16 bytes per lane straight from global memory in v_mfma_f32_16x16x32
// layout (lane i + 16 g holds row i, k = 8 g .. 8 g + 7 of a 32-wide step; rows are tokens for the activations and
// experts for the router weight, whose 64 KiB stay in L2) -- so the kernel pays one memory round trip, and then runs one
// MFMA per step.  With the weight fragment as first operand a lane ends up with 4 experts' partial logits of one
// token; the eight waves' partial sums meet in LDS and are added in wave order (fixed: the result does not depend on
// timing).  The summation order differs from router_logits_kernel's, so the two agree to fp32 rounding, not bit for bit.
constexpr int RM_WAVES = 8, RM_TOKENS = 16;
constexpr int RM_MAX_EXPERTS = 96;   // beyond, a workgroup's partial sums do not fit its LDS
// SORT: one workgroup holds all tokens and sorts their assignments by expert as well, as sort_one_launch_kernel would: an assignment's place is the
// number of those before it in (expert, flat index) order, counted by a thread each.  Saves a launch and its trip to memory: one token, d = 4096, router and
// sort 7.4 + 4.5 us in two launches.
// RM_BATCH: 32-wide K steps whose loads are in flight together (16 steps x 8 waves = 4096 columns); a wave with fewer steps repeats the last one's
// loads, so narrow layers take a kernel of 4 (512 tokens, d=256: 9.5 -> 5.3 us)
struct SortedOut { int32_t *sei, *ssi, *inv, *offsets; };
template <typename T, int RM_BATCH, bool SORT>
__global__ void __launch_bounds__(RM_WAVES * 64) router_mfma_kernel(const T* __restrict__ x, int64_t ldx,
                                                                    const T* __restrict__ wg, int64_t ldw,
                                                                    float* __restrict__ logits, float* __restrict__ scores,
                                                                    float* __restrict__ topw, int32_t* __restrict__ topi,
                                                                    int64_t ntok, int d, int E, int k, int renorm, const SortedOut so)
{
    __shared__ float s_part[RM_WAVES][RM_TOKENS][16];
    __shared__ int32_t s_topi[SORT ? RM_TOKENS * ROUTER_EXPERT_GROUP : 1];   // (k <= E)
    __shared__ float s_logits[RM_TOKENS][ROUTER_EXPERT_GROUP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t t0 = (int64_t)blockIdx.x * RM_TOKENS;
    const int row = lane & 15, kc = lane >> 4;
    const int64_t tok = (t0 + row < ntok) ? t0 + row : ntok - 1;      // tokens past the end re-read the last one
    const T* xp = x + tok * ldx + kc * 8;
    const T* wp = wg + (int64_t)(row < E ? row : E - 1) * ldw + kc * 8;   // rows past the last expert enter as zeros
    const int nsteps = d / 32;
    const int s_end = nsteps * (wave + 1) / RM_WAVES;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = nsteps * wave / RM_WAVES; s0 < s_end; s0 += RM_BATCH) {
        uint4 xa[RM_BATCH], wa[RM_BATCH];
#pragma unroll
        for (int i = 0; i < RM_BATCH; ++i) {
            const int st = (s0 + i < s_end) ? s0 + i : s_end - 1;
            xa[i] = *(const uint4*)(xp + (int64_t)st * 32);
            wa[i] = *(const uint4*)(wp + (int64_t)st * 32);
        }
#pragma unroll
        for (int i = 0; i < RM_BATCH; ++i) {
            if (s0 + i < s_end) {
                uint4 w4 = wa[i];
                if (row >= E) w4 = make_uint4(0, 0, 0, 0);
                if constexpr (sizeof(T) == 2 && std::is_same<T, __hip_bfloat16>::value) {
                    union { uint4 u; bf16x8_t v; } a, b;
                    a.u = w4; b.u = xa[i];
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc, 0, 0, 0);
                } else {
                    typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
                    union { uint4 u; f16x8_t v; } a, b;
                    a.u = w4; b.u = xa[i];
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v, b.v, acc, 0, 0, 0);
                }
            }
        }
    }
    // acc[r] = partial logit of token `row`, expert 4 * kc + r
    *(f32x4_t*)&s_part[wave][row][4 * kc] = acc;
    __syncthreads();
    if (tid < RM_TOKENS * ROUTER_EXPERT_GROUP) {
        const int t = tid / ROUTER_EXPERT_GROUP, e = tid % ROUTER_EXPERT_GROUP;
        float sum = s_part[0][t][e];
#pragma unroll
        for (int w = 1; w < RM_WAVES; ++w) sum += s_part[w][t][e];
        s_logits[t][e] = sum;
        if (e < E && t0 + t < ntok) logits[(t0 + t) * E + e] = sum;
    }
    __syncthreads();
    if (tid < RM_TOKENS * TK_LANES) {   // whole waves
        const int tt = tid / TK_LANES;
        const int64_t t = t0 + tt;
        softmax_topk_token<1>(s_logits[tt], scores + t * E, topw + t * k, SORT ? s_topi + t * k : topi + t * k, E, k, renorm, t < ntok);
    }
    if constexpr (SORT) {
        __syncthreads();
        const int R = (int)ntok * k;
        if (tid < R) {
            const int e = s_topi[tid];
            int at = 0;
            for (int j = 0; j < R; ++j) at += (s_topi[j] < e || (s_topi[j] == e && j < tid)) ? 1 : 0;
            topi[tid] = e;
            so.sei[at] = e;
            so.ssi[at] = tid;
            so.inv[tid] = at;
        } else if (tid >= RM_WAVES * 64 - E) {
            const int e = RM_WAVES * 64 - 1 - tid;
            int n = 0;
            for (int j = 0; j < R; ++j) n += s_topi[j] <= e ? 1 : 0;
            so.offsets[e] = n;
        }
    }
}
static_assert(RM_TOKENS * ROUTER_EXPERT_GROUP + ROUTER_EXPERT_GROUP <= RM_WAVES * 64, "a thread per assignment and one per expert");

// The same for 9 to 96 experts, in EG groups of 16: a wave's activation fragment meets EG weight fragments per step, fewer steps' loads fit in
// flight, and the eight partial sums per logit are added in wave order as above.  The two launches of the vector kernels are bound by their
// FMAs (2048 tokens x 64 experts x 2048 columns: 26.3 + 10.2 us, this 21); the order of a logit's sum differs from theirs.  A step's 32 products are
// summed by the instruction, the steps and the waves in 64 bits: the loads hide these adds (21.1 us with fp32 accumulators too), and chained in fp32
// the logits of 2048 bf16 columns were 1.03e-7 from 64 bits (relative 2-norm) where the vector kernels are 7.5e-8 and this 4.7e-8; 96 experts, 3072
// columns 1.22e-7, 8.0e-8 and 4.6e-8; fp16 1.14e-7 (vector) and 5.7e-8.
// TOPK = false: the logits of one expert group per workgroup (blockIdx.y), the same sums, for few tokens of many experts: one workgroup for all of
// them fetches every weight through one compute unit.  A batch that is not whole leaves out its loads: as repeats of the last
// step's they made 16 experts of d=512 11.4 us where the vector kernels take 8.0 and this 5.2.  (Not with four groups and more, which
// run for many tokens only: a loop of its own for whole batches takes registers for one wave per SIMD less, 16384 x 96 x 4096 119 -> 133 us.)
template <typename T, int EG, bool TOPK>
__global__ void __launch_bounds__(RM_WAVES * 64) router_mfma_wide_kernel(const T* __restrict__ x, int64_t ldx, const T* __restrict__ wg, int64_t ldw,
                                                                         float* __restrict__ logits, float* __restrict__ scores,
                                                                         float* __restrict__ topw, int32_t* __restrict__ topi, int64_t ntok, int d,
                                                                         int E, int k, int renorm)
{
    constexpr int BATCH = EG == 1 ? 16 : EG == 2 ? 8 : 4;
    constexpr int EW = EG * 16;
    __shared__ float s_part[RM_WAVES][RM_TOKENS][EW];
    __shared__ float s_logits[TOPK ? RM_TOKENS : 1][EW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t t0 = (int64_t)blockIdx.x * RM_TOKENS;
    const int e0 = TOPK ? 0 : (int)blockIdx.y * EW;
    const int row = lane & 15, kc = lane >> 4;
    const int64_t tok = (t0 + row < ntok) ? t0 + row : ntok - 1;      // tokens past the end re-read the last one
    const T* xp = x + tok * ldx + kc * 8;
    const T* wp[EG];
#pragma unroll
    for (int g = 0; g < EG; ++g) wp[g] = wg + (int64_t)(e0 + g * 16 + row < E ? e0 + g * 16 + row : E - 1) * ldw + kc * 8;   // (rows past the last expert repeat it; nobody reads their logits)
    const int nsteps = d / 32;
    const int s_end = nsteps * (wave + 1) / RM_WAVES;
    double acc[EG][4];
#pragma unroll
    for (int g = 0; g < EG; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[g][r] = 0.0;
    using Num = typename std::conditional<std::is_same<T, __hip_bfloat16>::value, NumBf16, NumF16>::type;
    // ALL: every step of the batch is the wave's.  REPEAT: loads past the wave's steps repeat the last one's.
    auto steps = [&](int s0, auto ALL, auto REPEAT) {
        auto mine = [&](int i) { return decltype(ALL)::value || s0 + i < s_end; };
        uint4 xa[BATCH], wa[BATCH][EG];
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (decltype(REPEAT)::value || mine(i)) {
                const int st = (mine(i) ? s0 + i : s_end - 1) * 32;
                xa[i] = *(const uint4*)(xp + st);
#pragma unroll
                for (int g = 0; g < EG; ++g) wa[i][g] = *(const uint4*)(wp[g] + st);
            }
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (mine(i)) {
#pragma unroll
                for (int g = 0; g < EG; ++g) {
                    const f32x4_t p = Num::mfma(__builtin_bit_cast(bf16x8_t, wa[i][g]), __builtin_bit_cast(bf16x8_t, xa[i]), (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[g][r] += (double)p[r];
                }
            }
    };
    const int s_begin = nsteps * wave / RM_WAVES;
    if (EG > 2) {
        for (int s0 = s_begin; s0 < s_end; s0 += BATCH) steps(s0, std::false_type{}, std::true_type{});
    } else {
        for (int s0 = s_begin; s0 < s_end; s0 += BATCH) {
            if (s0 + BATCH <= s_end) steps(s0, std::true_type{}, std::false_type{});
            else steps(s0, std::false_type{}, std::false_type{});
        }
    }
    // acc[g][r] = partial logit of token `row`, expert 16 g + 4 kc + r
#pragma unroll
    for (int g = 0; g < EG; ++g) *(f32x4_t*)&s_part[wave][row][g * 16 + 4 * kc] = (f32x4_t){(float)acc[g][0], (float)acc[g][1], (float)acc[g][2], (float)acc[g][3]};
    __syncthreads();
    for (int i = tid; i < RM_TOKENS * EW; i += RM_WAVES * 64) {
        const int t = i / EW, e = i % EW;
        double dsum = s_part[0][t][e];
#pragma unroll
        for (int w = 1; w < RM_WAVES; ++w) dsum += (double)s_part[w][t][e];
        const float sum = (float)dsum;
        if (TOPK) s_logits[t][e] = sum;
        if (e0 + e < E && t0 + t < ntok) logits[(t0 + t) * E + e0 + e] = sum;
    }
    if (!TOPK) return;
    __syncthreads();
    if (tid < RM_TOKENS * TK_LANES) {   // whole waves
        const int tt = tid / TK_LANES;
        const int64_t t = t0 + tt;
        softmax_topk_token<EG>(s_logits[tt], scores + t * E, topw + t * k, topi + t * k, E, k, renorm, t < ntok);
    }
}

// Backward of softmax -> top-k -> renormalise with respect to the logits, for one token (the pointers are its rows).
// dwt (k): gradient of the returned weights; wt (k) the returned weights; s (E) the softmax.
// TK_LANES lanes share a token so that its rows move coalesced; every lane computes the token's two sums over the k
// selected experts itself, in selection order (one thread per token: 59 us for 2048 tokens x 64 experts, top-8; this: 9).
__device__ __forceinline__ void router_bwd_token(const float* dwt, const float* __restrict__ wt, const int32_t* __restrict__ it,
                                                 const float* __restrict__ s, float* __restrict__ dl, int E, int k, int renorm)
{
    const int ln = threadIdx.x & (TK_LANES - 1);
    // selected scores p_j = s[idx_j]; w_j = p_j / S (S = sum p) when renorm, else w_j = p_j.  Lane j fetches selection j
    // (of each TK_LANES selections), the token's other lanes get it by shuffle: one memory round trip for all of them.
    int my_e = 0;
    float my_p = 0.f, my_dw = 0.f, my_w = 0.f;
    auto fetch = [&](int j0) {
        if (j0 + ln < k) { my_e = it[j0 + ln]; my_dw = dwt[j0 + ln]; my_w = wt[j0 + ln]; my_p = s[my_e]; }
    };
    fetch(0);
    float S = 1.f, dot = 0.f;
    if (renorm) {
        S = 0.f;
        for (int j = 0; j < k; ++j) {
            if (j > 0 && j % TK_LANES == 0) fetch(j);
            S += __shfl(my_p, j % TK_LANES, TK_LANES);
            dot += __shfl(my_dw, j % TK_LANES, TK_LANES) * __shfl(my_w, j % TK_LANES, TK_LANES);
        }
        if (k > TK_LANES) fetch(0);
    }
    float sdot = 0.f;  // sum_e dscore_e * s_e
    for (int j = 0; j < k; ++j) {
        if (j > 0 && j % TK_LANES == 0) fetch(j);
        const float d = __shfl(my_dw, j % TK_LANES, TK_LANES);
        sdot += (renorm ? (d - dot) / S : d) * __shfl(my_p, j % TK_LANES, TK_LANES);
    }
    if (k > TK_LANES) fetch(0);
    for (int e0 = 0; e0 < E; e0 += TK_LANES) {
        const int e = e0 + ln;
        float ds = 0.f;   // dscore of expert e
        for (int j = 0; j < k; ++j) {
            if (j > 0 && j % TK_LANES == 0) fetch(j);
            const float d = __shfl(my_dw, j % TK_LANES, TK_LANES);
            if (__shfl(my_e, j % TK_LANES, TK_LANES) == e) ds = renorm ? (d - dot) / S : d;
        }
        if (k > TK_LANES) fetch(0);
        if (e < E) dl[e] = s[e] * (ds - sdot);
    }
}

__global__ void __launch_bounds__(256) router_bwd_kernel(const float* __restrict__ dw, const float* __restrict__ w,
                                                         const int32_t* __restrict__ topi, const float* __restrict__ scores,
                                                         float* __restrict__ dlogits, int64_t ntok, int E, int k, int renorm)
{
    const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / TK_LANES;
    if (t >= ntok) return;   // (whole groups of TK_LANES lanes)
    router_bwd_token(dw + t * k, w + t * k, topi + t * k, scores + t * E, dlogits + t * E, E, k, renorm);
}

// What the backward pass of a layer needs from its gates, in one launch instead of three (bound by the two rows that a pair reads): a
// wave per (token, selection) pair takes the gradient of that weight, <y[t*k+j], dout[t]> (+ d_w, a gradient that reached the returned
// weights directly), and puts the weight at the pair's place in sorted order (the row scale of the grouped GEMMs); then the token's lanes
// turn its k gradients into those of its logits.  The sums are those of combine_dgates and router_bwd, bit for bit.  As three launches
// 2048 tokens, 64 experts, top-8, d=2048 took 34.6 us, this 21.4 (eight waves per SIMD; as many registers as the compiler likes: 32.8); 4096 tokens, top-2, d=4096 28.7 and 18.8;
// 512 tokens, d=256 9.4 and 4.7.
template <typename T, int GB_WAVES>
__global__ void __launch_bounds__(GB_WAVES * 64, 8) gates_bwd_kernel(const T* __restrict__ y, int64_t ldy, const T* __restrict__ dout, int64_t ldd,
                                                                  const float* __restrict__ d_w, const float* __restrict__ w,
                                                                  const int32_t* __restrict__ topi, const float* __restrict__ scores,
                                                                  const int32_t* __restrict__ inv, float* __restrict__ dlogits,
                                                                  float* __restrict__ row_scale, int64_t ntok, int64_t d, int E, int k,
                                                                  int renorm, int tokens, bool vec_ok)
{
    extern __shared__ float s_dw[];   // [tokens][k]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t t0 = (int64_t)blockIdx.x * tokens;
    const int nt = ntok - t0 < tokens ? (int)(ntok - t0) : tokens;
    for (int p = wave; p < nt * k; p += GB_WAVES) {
        const int64_t pair = t0 * k + p;
        const T* yr = y + pair * ldy;
        const T* dr = dout + (t0 + p / k) * ldd;
        float acc = 0.f;
        int64_t c0 = (int64_t)lane * 8;
        if (vec_ok)   // whole vectors, four of each row in flight
            for (; c0 + 3 * 512 + 8 <= d; c0 += 4 * 512) {
                uint4 a[4], b[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    a[q] = *(const uint4*)(yr + c0 + q * 512);
                    b[q] = *(const uint4*)(dr + c0 + q * 512);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int u = 0; u < 8; ++u) acc = fmaf(Elem<T>::ld((const T*)&a[q] + u), Elem<T>::ld((const T*)&b[q] + u), acc);
            }
        for (; c0 < d; c0 += 64 * 8) {
            const int n = d - c0 < 8 ? (int)(d - c0) : 8;
            float a[8], b[8];
            load8<T>(yr + c0, a, n, vec_ok);
            load8<T>(dr + c0, b, n, vec_ok);
#pragma unroll
            for (int u = 0; u < 8; ++u) acc = fmaf(a[u], b[u], acc);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
        if (lane == 0) {
            s_dw[p] = d_w ? acc + d_w[pair] : acc;
            row_scale[inv[pair]] = w[pair];
        }
    }
    __syncthreads();
    const int tt = threadIdx.x / TK_LANES;
    if (tt >= nt) return;
    const int64_t t = t0 + tt;
    router_bwd_token(s_dw + tt * k, w + t * k, topi + t * k, scores + t * E, dlogits + t * E, E, k, renorm);
}

// ---------------------------------------------------------------------------------------------------------
// stable counting sort by expert id
// ---------------------------------------------------------------------------------------------------------
constexpr int SORT_THREADS = 256;
constexpr int SORT_SCAN_LDS_INTS = 8192;   // chunk histograms the scan kernel keeps in LDS (32 KiB)
constexpr int SORT_CHUNK = 512;   // assignments per workgroup: small, so that a batch of a few thousand tokens still spreads over many compute units

__global__ void __launch_bounds__(SORT_THREADS) sort_hist_kernel(const void* __restrict__ expert_idx, int in64,
                                                                 int64_t R, int E, int32_t* __restrict__ block_hist)
{
    extern __shared__ int32_t sh[];
    for (int e = threadIdx.x; e < E; e += SORT_THREADS) sh[e] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * SORT_CHUNK;
    for (int i = threadIdx.x; i < SORT_CHUNK; i += SORT_THREADS) {
        const int64_t p = base + i;
        if (p < R) {
            const int64_t e = load_idx(expert_idx, p, in64);
            if (e >= 0 && e < E) atomicAdd(&sh[e], 1);  // ids outside [0,E) are left out of the sorted order
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += SORT_THREADS) block_hist[(int64_t)blockIdx.x * E + e] = sh[e];
}

__device__ __forceinline__ void store_idx(void* p, int64_t i, int64_t v, int is64)
{
    if (is64) ((int64_t*)p)[i] = v; else ((int32_t*)p)[i] = (int32_t)v;
}

// Single workgroup: per-expert totals, exclusive bases per (expert, chunk) in expert-major order, inclusive
// offsets, and the table of block starts (block_m rows per block, blocks never straddle experts).
__global__ void __launch_bounds__(SORT_THREADS) sort_scan_kernel(int32_t* __restrict__ block_hist, int nblk, int E,
                                                                 int block_m, void* __restrict__ counts,
                                                                 void* __restrict__ offsets, int meta64,
                                                                 void* __restrict__ padded_blocks, int64_t padded_cap,
                                                                 int32_t* __restrict__ num_padded)
{
    extern __shared__ int32_t sh[];  // totals[E], then (when it fits) a copy of block_hist
    int32_t* hist = sh + E;
    const bool in_lds = (int64_t)nblk * E <= SORT_SCAN_LDS_INTS;
    // the running sums walk the chunks one after the other; from a copy in LDS that costs a few cycles per step
    // instead of a round trip to memory
    if (in_lds) {
        for (int i = threadIdx.x; i < nblk * E; i += SORT_THREADS) hist[i] = block_hist[i];
        __syncthreads();
    }
    for (int e = threadIdx.x; e < E; e += SORT_THREADS) {
        int32_t run = 0;
        if (in_lds) for (int b = 0; b < nblk; ++b) { const int32_t c = hist[b * E + e]; hist[b * E + e] = run; run += c; }
        else for (int b = 0; b < nblk; ++b) { const int32_t c = block_hist[(int64_t)b * E + e]; block_hist[(int64_t)b * E + e] = run; run += c; }
        sh[e] = run;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t run = 0, nb = 0;
        for (int e = 0; e < E; ++e) {
            const int64_t c = sh[e];
            const int64_t start = run;
            run += c;
            if (counts) store_idx(counts, e, c, meta64);
            if (offsets) store_idx(offsets, e, run, meta64);
            sh[e] = (int32_t)start;
            if (padded_blocks)
                for (int64_t s = start; s < run; s += block_m) { if (nb < padded_cap) store_idx(padded_blocks, nb, s, meta64); ++nb; }
        }
        if (num_padded) *num_padded = (int32_t)nb;
    }
    __syncthreads();
    if (in_lds) for (int i = threadIdx.x; i < nblk * E; i += SORT_THREADS) block_hist[i] = hist[i] + sh[i % E];
    else for (int i = threadIdx.x; i < nblk * E; i += SORT_THREADS) block_hist[i] += sh[i % E];
}

// Stores one group of 64 entries (flat positions p of consecutive lanes, expert e, -1: none) at its expert's cursor:
// entries of one expert keep their order (stability).  A lane's rank among the earlier lanes of its expert takes no round trip to
// memory: up to 16 experts one ballot per expert, beyond that 64 scalar broadcasts and compares, whatever the number of experts.
// Sort of 262144 rows, us, ballots / broadcasts: 2 experts 21.7 / 23.8, 8 experts 26.4 / 28.5, 16 experts 33.2 / 34.4, 32 experts
// 135.2 / 134.7, 48 experts 152.1 / 150.4.
typedef __attribute__((address_space(3))) int32_t lds_int32_t;
constexpr int SCATTER_BALLOT_EXPERTS = 16;
__device__ __forceinline__ void scatter_group(int e, int64_t p, int lane, int E, int32_t* cursor_, void* __restrict__ sorted_expert,
                                              void* __restrict__ sorted_pos, int out64, int32_t* __restrict__ inv)
{
    lds_int32_t* cursor = (lds_int32_t*)cursor_;
    int rank = 0;
    if (E <= SCATTER_BALLOT_EXPERTS) {
        uint64_t mine = 0;   // lanes of this lane's expert
#pragma unroll 1
        for (int x = 0; x < E; ++x) {
            const uint64_t m = __ballot(e == x);
            mine = e == x ? m : mine;
        }
        rank = __popcll(mine & ((1ull << lane) - 1ull));
    } else {
#pragma unroll
        for (int j = 0; j < 63; ++j) rank += (__builtin_amdgcn_readlane(e, j) == e && j < lane) ? 1 : 0;
    }
    if (e >= 0) {
        const int32_t dst = *(volatile lds_int32_t*)(cursor + e) + rank;
        store_idx(sorted_expert, dst, e, out64);
        store_idx(sorted_pos, dst, p, out64);
        if (inv) inv[p] = dst;
    }
    __builtin_amdgcn_wave_barrier();
    if (e >= 0) __hip_atomic_fetch_add(cursor + e, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // (after every lane of the wave has read its cursor)
    __builtin_amdgcn_wave_barrier();
}

// Each workgroup re-reads its chunk; wave w owns a contiguous slice of it and walks it 64 entries at a time so
// that destinations within one expert ascend with the flat position (stability).
__global__ void __launch_bounds__(SORT_THREADS) sort_scatter_kernel(const void* __restrict__ expert_idx, int in64,
                                                                    int64_t R, int E,
                                                                    const int32_t* __restrict__ block_base,
                                                                    void* __restrict__ sorted_expert,
                                                                    void* __restrict__ sorted_pos, int out64,
                                                                    int32_t* __restrict__ inv)
{
    extern __shared__ int32_t sh[];  // cursor[nwave][E]
    constexpr int NW = SORT_THREADS / 64;
    constexpr int PER_WAVE = SORT_CHUNK / NW;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < NW * E; i += SORT_THREADS) sh[i] = 0;
    __syncthreads();
    const int64_t wbase = (int64_t)blockIdx.x * SORT_CHUNK + (int64_t)w * PER_WAVE;
    // pass 1: per-wave histogram
    for (int i = lane; i < PER_WAVE; i += 64) {
        const int64_t p = wbase + i;
        if (p < R) {
            const int64_t e = load_idx(expert_idx, p, in64);
            if (e >= 0 && e < E) atomicAdd(&sh[w * E + (int)e], 1);
        }
    }
    __syncthreads();
    // exclusive prefix over waves, seeded with this chunk's base
    for (int e = threadIdx.x; e < E; e += SORT_THREADS) {
        int32_t run = block_base[(int64_t)blockIdx.x * E + e];
        for (int ww = 0; ww < NW; ++ww) { const int32_t c = sh[ww * E + e]; sh[ww * E + e] = run; run += c; }
    }
    __syncthreads();
    // pass 2: ranked scatter
    for (int i0 = 0; i0 < PER_WAVE; i0 += 64) {
        const int64_t p = wbase + i0 + lane;
        int e = -1;
        if (p < R) { const int64_t ee = load_idx(expert_idx, p, in64); e = (ee >= 0 && ee < E) ? (int)ee : -1; }
        scatter_group(e, p, lane, E, sh + w * E, sorted_expert, sorted_pos, out64, inv);
    }
}

// The whole sort in one launch, for batches small enough that every workgroup can afford to read ALL assignment ids
// itself: a workgroup counts, per expert, the entries before its own chunk and the others (LDS atomics), which gives it
// its chunk's destination bases without a histogram launch and a scan launch before it; then it scatters its chunk, one
// wave per 64 entries.  Workgroup 0 also writes the per-expert counts, the inclusive offsets and the block table.  Same
// results as the three-launch path.  Latency bound, so every step is parallel: ids are requested in batches, the scan over
// the experts runs as prefix sums of one wave (a single thread walking 64 experts took longer than all the rest).
// Rows up to which that pays: every workgroup reads all ids (6.3 us up to 8192 rows, then 0.19 us per 1000 rows whatever the number of
// experts), the three launches take 11.4 us and grow with the experts.  One launch against three, us: 32768 rows, 1 expert 10.1 / 12.0,
// 8 experts 10.3 / 11.4, 64 experts 11.3 / 28.1; 65536 rows, 1 expert 17.4 / 12.3, 8 experts 17.3 / 12.9, 16 experts 17.3 / 16.8, 64 experts
// 18.1 / 34.5.  The same within 0.3 us with nine tenths of the rows on one expert.
constexpr int64_t SORT_ONE_LAUNCH_MAX_ROWS = 65536, SORT_ONE_LAUNCH_MAX_ROWS_FEW = 32768;
constexpr int SORT_ONE_LAUNCH_FEW_EXPERTS = 15;
constexpr int SORT_ONE_LAUNCH_MAX_EXPERTS = 256;
constexpr int SORT1_THREADS = SORT_CHUNK;   // one thread per entry of the chunk
// Count rows: lane l adds into row l % SORT1_COPIES.  LDS atomics on one address are worked off a lane at a time, so with a row for all
// lanes of a wave a batch that sends most rows to one expert took 3 us more per 4096 rows (16384 rows: 19 us, so 8); rows of an odd pitch
// keep the copies of one expert in different banks.
constexpr int SORT1_COPIES = 8;
__host__ __device__ constexpr int sort1_pitch(int E) { return E | 1; }
static_assert(SORT_CHUNK % 64 == 0, "a 64-entry group of the counting pass lies wholly before a chunk or not at all");
__global__ void __launch_bounds__(SORT1_THREADS) sort_one_launch_kernel(const void* __restrict__ expert_idx, int in64,
                                                                        int64_t R, int E, int block_m,
                                                                        void* __restrict__ sorted_expert,
                                                                        void* __restrict__ sorted_pos, int out64,
                                                                        void* __restrict__ counts, void* __restrict__ offsets,
                                                                        void* __restrict__ padded_blocks, int64_t padded_cap,
                                                                        int32_t* __restrict__ num_padded, int32_t* __restrict__ inv)
{
    constexpr int NW = SORT1_THREADS / 64;
    constexpr int COPIES = SORT1_COPIES;
    extern __shared__ int32_t sh[];  // before[COPIES][pitch], rest[COPIES][pitch], cursor[NW][E]
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int pitch = sort1_pitch(E);
    int32_t* before = sh;
    int32_t* rest = sh + COPIES * pitch;
    int32_t* cur = sh + 2 * COPIES * pitch;
    for (int i = threadIdx.x; i < 2 * COPIES * pitch + NW * E; i += SORT1_THREADS) sh[i] = 0;
    __syncthreads();
    const int64_t chunk_base = (int64_t)blockIdx.x * SORT_CHUNK;
    // the own chunk's entry, and its per-wave histogram
    const int64_t pown = chunk_base + threadIdx.x;
    int eown = -1;
    if (pown < R) { const int64_t ee = load_idx(expert_idx, pown, in64); eown = (ee >= 0 && ee < E) ? (int)ee : -1; }
    // counts over the whole array: wave w walks entries [64 (w + NW j), +64), sixteen groups' ids requested together
    // (integer counts: the order of the additions does not matter)
    constexpr int SB = 16;
    int32_t* my_before = before + (lane % COPIES) * pitch;
    int32_t* my_rest = rest + (lane % COPIES) * pitch;
    for (int64_t p0 = (int64_t)w * 64; p0 < R; p0 += (int64_t)NW * 64 * SB) {
        int64_t raw[SB];
        // (one branch on the index width around all the loads, so that they are in flight together; entries past the
        // end re-read the last one and are dropped below)
        if (in64) {
#pragma unroll
            for (int j = 0; j < SB; ++j) { const int64_t p = p0 + (int64_t)j * NW * 64 + lane; raw[j] = ((const int64_t*)expert_idx)[p < R ? p : R - 1]; }
        } else {
#pragma unroll
            for (int j = 0; j < SB; ++j) { const int64_t p = p0 + (int64_t)j * NW * 64 + lane; raw[j] = ((const int32_t*)expert_idx)[p < R ? p : R - 1]; }
        }
#pragma unroll
        for (int j = 0; j < SB; ++j) {
            const int64_t p = p0 + (int64_t)j * NW * 64 + lane;
            // a 64-entry group lies wholly before the chunk or not at all (chunks are multiples of 64 entries)
            if (p < R && raw[j] >= 0 && raw[j] < E) atomicAdd(&(p0 + (int64_t)j * NW * 64 < chunk_base ? my_before : my_rest)[raw[j]], 1);
        }
    }
    if (eown >= 0) atomicAdd(&cur[w * E + eown], 1);
    __syncthreads();
    // wave 0: lane l owns experts [l * per, +per); totals, then their running sums over the lanes
    const int per = (E + 63) / 64;
    if (w == 0) {
        int32_t sum = 0;
        int64_t nblk = 0;
        for (int q = 0; q < per; ++q) {
            const int e = lane * per + q;
            int32_t b = 0, t = 0;
            if (e < E) {
#pragma unroll
                for (int c = 0; c < COPIES; ++c) { b += before[c * pitch + e]; t += rest[c * pitch + e]; }
                before[e] = b;
                rest[e] = b + t;
                sum += b + t;
                nblk += (b + t + block_m - 1) / block_m;
            }
        }
        int32_t incl = sum;
        int64_t binc = nblk;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int32_t t = __shfl_up(incl, d);
            const int64_t u = __shfl_up(binc, d);
            if (lane >= d) { incl += t; binc += u; }
        }
        const bool pub = blockIdx.x == 0;
        int32_t run = incl - sum;
        int64_t nb = binc - nblk;
        for (int q = 0; q < per; ++q) {
            const int e = lane * per + q;
            if (e >= E) break;
            const int32_t c = rest[e], start = run;
            run += c;
            if (pub) {
                if (counts) store_idx(counts, e, c, out64);
                if (offsets) store_idx(offsets, e, run, out64);
                if (padded_blocks)
                    for (int64_t s_ = start; s_ < run; s_ += block_m) { if (nb < padded_cap) store_idx(padded_blocks, nb, s_, out64); ++nb; }
            }
            rest[e] = start + before[e];   // this chunk's first destination of the expert
        }
        if (pub && num_padded && lane == 63) *num_padded = (int32_t)binc;
    }
    __syncthreads();
    // exclusive prefix over waves, seeded with the chunk's base
    for (int e = threadIdx.x; e < E; e += SORT1_THREADS) {
        int32_t run = rest[e];
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) { const int32_t c = cur[ww * E + e]; cur[ww * E + e] = run; run += c; }
    }
    __syncthreads();
    scatter_group(eown, pown, lane, E, cur + w * E, sorted_expert, sorted_pos, out64, inv);
}

// offsets[e] = number of entries of the non-decreasing array sorted_expert that are <= e  (inclusive running count)
__global__ void offsets_from_sorted_kernel(const void* __restrict__ sorted_expert, int in64, int64_t R, int E,
                                           void* __restrict__ offsets, int out64)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    int64_t lo = 0, hi = R;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (load_idx(sorted_expert, mid, in64) <= e) lo = mid + 1; else hi = mid;
    }
    store_idx(offsets, e, lo, out64);
}

__global__ void padded_blocks_kernel(const void* __restrict__ offsets, int off64, int E, int block_m,
                                     void* __restrict__ padded_blocks, int out64, int64_t cap,
                                     int32_t* __restrict__ num_padded)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int64_t start = 0, nb = 0;
    for (int e = 0; e < E; ++e) {
        const int64_t end = load_idx(offsets, e, off64);
        for (int64_t s = start; s < end; s += block_m) { if (nb < cap) store_idx(padded_blocks, nb, s, out64); ++nb; }
        start = end;
    }
    *num_padded = (int32_t)nb;
}

}  // namespace

namespace {
// topk: softmax and top-k in the same launch (E <= ROUTER_EXPERT_GROUP)
int launch_router_logits(const void* x, int64_t ldx, const void* wg, int64_t ldw, int dtype, float* logits, int64_t ntok, int64_t d, int E,
                         bool topk, float* scores, float* topw, int32_t* topi, int k, int renorm, hipStream_t stream)
{
    const int groups = (E + ROUTER_EXPERT_GROUP - 1) / ROUTER_EXPERT_GROUP;
    // 4 tokens per wave share each weight fetch, as soon as that still leaves a wave for every SIMD; 2 for fewer tokens
    const int tokens = ((ntok + 3) / 4) * groups >= 4 * (int64_t)moe_device_cus() ? 4 : 2;
    const int64_t waves = (ntok + tokens - 1) / tokens;
    const dim3 grid((unsigned)((waves + 3) / 4), (unsigned)groups);
    const int64_t per16 = dtype == MOE_F32 ? 4 : 8;
    const bool vec_ok = ((uintptr_t)x % 16 == 0) && ((uintptr_t)wg % 16 == 0) && ldx % per16 == 0 && ldw % per16 == 0;
    MOE_DISPATCH_DTYPE(dtype, {
        auto kern = tokens == 4 ? (topk ? router_logits_kernel<T, 4, true> : router_logits_kernel<T, 4, false>)
                                : (topk ? router_logits_kernel<T, 2, true> : router_logits_kernel<T, 2, false>);
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, (const T*)x, ldx, (const T*)wg, ldw, logits, ntok, d, E, vec_ok, scores, topw, topi, k, renorm);
    });
    return moe_launch_status();
}
}  // namespace

int moe_launch_router_logits(const void* x, int64_t ldx, const void* wg, int64_t ldw, int dtype, float* logits,
                             int64_t ntok, int64_t d, int E, hipStream_t stream)
{
    if (ntok == 0) return MOE_OK;
    return launch_router_logits(x, ldx, wg, ldw, dtype, logits, ntok, d, E, false, nullptr, nullptr, nullptr, 0, 0, stream);
}

// logits + softmax + top-k; one launch when the router weight fits the fused kernel, otherwise the two kernels above
static bool router_mfma_ok(const void* x, int64_t ldx, const void* wg, int64_t ldw, int dtype, int64_t d, int E)
{
    return dtype != MOE_F32 && E <= RM_MAX_EXPERTS && d % 32 == 0 && d >= 32 && d < (1 << 30) &&
           ((uintptr_t)x % 16 == 0) && ((uintptr_t)wg % 16 == 0) && ldx % 8 == 0 && ldw % 8 == 0;
}

int moe_launch_router_forward(const void* x, int64_t ldx, const void* wg, int64_t ldw, int dtype, float* logits,
                              float* scores, float* topw, int32_t* topi, int64_t ntok, int64_t d, int E, int k,
                              int renorm, hipStream_t stream)
{
    if (ntok == 0) return MOE_OK;
    if (!router_mfma_ok(x, ldx, wg, ldw, dtype, d, E)) {
        if (E <= ROUTER_EXPERT_GROUP)
            return launch_router_logits(x, ldx, wg, ldw, dtype, logits, ntok, d, E, true, scores, topw, topi, k, renorm, stream);
        const int rc = moe_launch_router_logits(x, ldx, wg, ldw, dtype, logits, ntok, d, E, stream);
        return rc != MOE_OK ? rc : moe_launch_router_topk(logits, scores, topw, topi, ntok, E, k, renorm, stream);
    }
    const unsigned grid = (unsigned)((ntok + RM_TOKENS - 1) / RM_TOKENS);
    if (E > ROUTER_EXPERT_GROUP) {
        // One launch, or one workgroup per token and expert group and top-k in a launch of its own, the same bits.  With 48 experts and more the
        // latter is sooner while its workgroups fit the chip (16 tokens, 96 experts, d=4096: 17.7 us against 33.5, and 25.7 for the
        // vector kernels; d=512 11.2, 12.1 and 12.5; 1024 tokens, 64 experts, d=4096 15.8 and 25.3, 2048 tokens 24.9 and 26), with more
        // than 64, whose one launch is the slowest, also in one and a half rounds (1024 tokens, 96 experts, d=4096: 26.1 and 34).
        const int64_t parts = (int64_t)grid * ((E + 15) / 16), cus = moe_device_cus();
        const bool apart = E > 32 && parts <= (E > 64 ? cus * 3 / 2 : cus);
        auto wide = [&](auto tag) {
            using T = decltype(tag);
            if (apart) {
                hipLaunchKernelGGL((router_mfma_wide_kernel<T, 1, false>), dim3(grid, (unsigned)((E + 15) / 16)), dim3(RM_WAVES * 64), 0, stream, (const T*)x, ldx, (const T*)wg, ldw, logits,
                                   nullptr, nullptr, nullptr, ntok, (int)d, E, 0, 0);
                return;
            }
            auto kern = E <= 16 ? router_mfma_wide_kernel<T, 1, true> : E <= 32 ? router_mfma_wide_kernel<T, 2, true> : E <= 64 ? router_mfma_wide_kernel<T, 4, true> : router_mfma_wide_kernel<T, 6, true>;
            hipLaunchKernelGGL(kern, dim3(grid), dim3(RM_WAVES * 64), 0, stream, (const T*)x, ldx, (const T*)wg, ldw, logits, scores, topw, topi, ntok, (int)d, E, k, renorm);
        };
        if (dtype == MOE_BF16) wide(__hip_bfloat16{}); else wide(__half{});
        const int rc = moe_launch_status();
        return rc != MOE_OK || !apart ? rc : moe_launch_router_topk(logits, scores, topw, topi, ntok, E, k, renorm, stream);
    }
    auto few = [&](auto tag) {
        using T = decltype(tag);
        auto kern = d <= 4 * 32 * RM_WAVES ? router_mfma_kernel<T, 4, false> : router_mfma_kernel<T, 16, false>;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(RM_WAVES * 64), 0, stream, (const T*)x, ldx, (const T*)wg, ldw, logits, scores, topw, topi, ntok, (int)d, E, k, renorm, SortedOut{});
    };
    if (dtype == MOE_BF16) few(__hip_bfloat16{}); else few(__half{});
    return moe_launch_status();
}

bool moe_router_sorts(const void* x, int64_t ldx, const void* wg, int64_t ldw, int dtype, int64_t ntok, int64_t d, int E)
{
    return ntok >= 1 && ntok <= RM_TOKENS && E <= ROUTER_EXPERT_GROUP && router_mfma_ok(x, ldx, wg, ldw, dtype, d, E);
}

int moe_launch_router_sorted(const void* x, int64_t ldx, const void* wg, int64_t ldw, int dtype, float* logits, float* scores, float* topw, int32_t* topi,
                             int64_t ntok, int64_t d, int E, int k, int renorm, int32_t* sei, int32_t* ssi, int32_t* inv, int32_t* offsets, hipStream_t stream)
{
    if (!moe_router_sorts(x, ldx, wg, ldw, dtype, ntok, d, E)) return MOE_ERR_UNSUPPORTED;
    auto go = [&](auto tag) {
        using T = decltype(tag);
        auto kern = d <= 4 * 32 * RM_WAVES ? router_mfma_kernel<T, 4, true> : router_mfma_kernel<T, 16, true>;
        hipLaunchKernelGGL(kern, dim3(1), dim3(RM_WAVES * 64), 0, stream, (const T*)x, ldx, (const T*)wg, ldw, logits, scores, topw, topi, ntok, (int)d, E, k, renorm, SortedOut{sei, ssi, inv, offsets});
    };
    if (dtype == MOE_BF16) go(__hip_bfloat16{}); else go(__half{});
    return moe_launch_status();
}

int moe_launch_router_topk(const float* logits, float* scores, float* topw, int32_t* topi, int64_t ntok, int E, int k,
                           int renorm, hipStream_t stream)
{
    if (ntok == 0) return MOE_OK;
    const dim3 grid((unsigned)((ntok * TK_LANES + 255) / 256));
#define TOPK(n) hipLaunchKernelGGL(router_topk_kernel<n>, grid, dim3(256), 0, stream, logits, scores, topw, topi, ntok, E, k, renorm)
    if (E <= TK_LANES) TOPK(1);
    else if (E <= 2 * TK_LANES) TOPK(2);
    else if (E <= 4 * TK_LANES) TOPK(4);
    else if (E <= 8 * TK_LANES) TOPK(8);
    else if (E <= TK_LANES * TK_MAX_PER_LANE) TOPK(TK_MAX_PER_LANE);
    else
        hipLaunchKernelGGL(router_topk_wide_kernel, dim3((unsigned)((ntok + 255) / 256)), dim3(256), 0, stream, logits, scores,
                           topw, topi, ntok, E, k, renorm);
#undef TOPK
    return moe_launch_status();
}

int moe_launch_router_bwd(const float* dw, const float* w, const int32_t* topi, const float* scores, float* dlogits,
                          int64_t ntok, int E, int k, int renorm, hipStream_t stream)
{
    if (ntok == 0) return MOE_OK;
    hipLaunchKernelGGL(router_bwd_kernel, dim3((unsigned)((ntok * TK_LANES + 255) / 256)), dim3(256), 0, stream, dw, w, topi,
                       scores, dlogits, ntok, E, k, renorm);
    return moe_launch_status();
}

int moe_launch_gates_bwd(const void* y, int64_t ldy, const void* dout, int64_t ldd, int dtype, const float* d_w, const float* w,
                         const int32_t* topi, const float* scores, const int32_t* inv, float* dlogits, float* row_scale, int64_t ntok,
                         int64_t d, int E, int k, int renorm, hipStream_t stream)
{
    if (dtype == MOE_F32) return MOE_ERR_UNSUPPORTED;
    if (ntok == 0) return MOE_OK;
    // Eight waves for more than four selections while the workgroups (one token each) are resident at once, and for wide rows; four otherwise
    // (top-8, four and eight waves: 500 tokens, d=1536 10.9 and 9.8 us, 1000 13.0 and 12.0, 2048 17.5 and 20.2, 8192 48.5 and 56.9; 2048 tokens,
    // d=2048 19.5 and 19.9, 4096 31.5 and 30.1; 8192 tokens, d=3072 91 and 96, 4096 117 and 111; top-5 and top-6 within 4 %).
    const int waves = k > 4 && (ntok <= 4 * (int64_t)moe_device_cus() || d > 3072) ? 8 : 4;
    const int tokens = k >= waves ? 1 : (waves + k - 1) / k;   // at least one pair per wave; at most 4 tokens, TK_LANES lanes each
    const bool vec = (uintptr_t)y % 16 == 0 && (uintptr_t)dout % 16 == 0 && ldy % 8 == 0 && ldd % 8 == 0;
    const dim3 grid((unsigned)((ntok + tokens - 1) / tokens));
    const size_t lds = (size_t)tokens * k * sizeof(float);
    auto launch = [&](auto tag) {
        using T = decltype(tag);
        hipLaunchKernelGGL((waves == 8 ? gates_bwd_kernel<T, 8> : gates_bwd_kernel<T, 4>), grid, dim3(waves * 64), lds, stream, (const T*)y, ldy, (const T*)dout, ldd, d_w, w,
                           topi, scores, inv, dlogits, row_scale, ntok, d, E, k, renorm, tokens, vec);
    };
    if (dtype == MOE_BF16) launch(__hip_bfloat16{}); else launch(__half{});
    return moe_launch_status();
}

size_t moe_sort_ws_bytes(int64_t R, int E)
{
    const int64_t nblk = (R + SORT_CHUNK - 1) / SORT_CHUNK;
    return (size_t)((nblk > 0 ? nblk : 1) * E + 4) * sizeof(int32_t);
}

int moe_launch_sort(const void* expert_idx, int in64, int64_t R, int E, int block_m, void* sorted_expert,
                    void* sorted_pos, int out64, void* counts, void* offsets, void* padded_blocks, int64_t padded_cap,
                    int32_t* num_padded, int32_t* inv, void* workspace, size_t workspace_bytes, hipStream_t stream)
{
    if (E < 1 || E > 4096 || R < 0 || block_m < 1) return MOE_ERR_BAD_ARG;
    if (workspace_bytes < moe_sort_ws_bytes(R, E)) return MOE_ERR_WORKSPACE;
    const int nblk = (int)((R + SORT_CHUNK - 1) / SORT_CHUNK);
    if (nblk > 0 && E <= SORT_ONE_LAUNCH_MAX_EXPERTS && R <= (E <= SORT_ONE_LAUNCH_FEW_EXPERTS ? SORT_ONE_LAUNCH_MAX_ROWS_FEW : SORT_ONE_LAUNCH_MAX_ROWS)) {
        hipLaunchKernelGGL(sort_one_launch_kernel, dim3(nblk), dim3(SORT1_THREADS), (2 * SORT1_COPIES * sort1_pitch(E) + SORT1_THREADS / 64 * E) * sizeof(int32_t), stream,
                           expert_idx, in64, R, E, block_m, sorted_expert, sorted_pos, out64, counts, offsets, padded_blocks,
                           padded_cap, num_padded, inv);
        return moe_launch_status();
    }
    int32_t* hist = (int32_t*)workspace;
    if (nblk > 0)
        hipLaunchKernelGGL(sort_hist_kernel, dim3(nblk), dim3(SORT_THREADS), E * sizeof(int32_t), stream, expert_idx,
                           in64, R, E, hist);
    const size_t scan_lds = ((int64_t)nblk * E <= SORT_SCAN_LDS_INTS ? (size_t)E + (size_t)nblk * E : (size_t)E) * sizeof(int32_t);
    hipLaunchKernelGGL(sort_scan_kernel, dim3(1), dim3(SORT_THREADS), scan_lds, stream, hist, nblk, E,
                       block_m, counts, offsets, out64, padded_blocks, padded_cap, num_padded);
    if (nblk > 0)
        hipLaunchKernelGGL(sort_scatter_kernel, dim3(nblk), dim3(SORT_THREADS), (SORT_THREADS / 64) * E * sizeof(int32_t),
                           stream, expert_idx, in64, R, E, hist, sorted_expert, sorted_pos, out64, inv);
    return moe_launch_status();
}

// ---------------------------------------------------------------------------------------------------------
// The same sort for callers that cannot allocate or pass a workspace: the per-chunk histograms live in a static
// device array (each GPU the library runs on holds its own copy at its own address until the process ends).
// Every call on a GPU shares that GPU's array: calls that overlap on one GPU race.  Nothing in it has to start at
// zero -- the histogram launch writes every cell the later launches read.
// ---------------------------------------------------------------------------------------------------------
constexpr int64_t SORT_STATIC_INTS = 262144;   // 1 MiB: ceil(R / 512) * E + 4 cells at most
static __device__ __align__(256) int32_t scratch[SORT_STATIC_INTS];

constexpr int SORT_STATIC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static int32_t* g_scratch_ptr[SORT_STATIC_MAX_DEVICES] = {};

// Device address of `scratch` on the current device.  In host code the array's name is only a handle: the address a
// kernel may use comes from hipGetSymbolAddress, once per device with that device current.
static int sort_static_scratch(int32_t** out)
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SORT_STATIC_MAX_DEVICES) return MOE_ERR_LAUNCH;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return MOE_ERR_LAUNCH;
        g_scratch_ptr[dev] = (int32_t*)p;
    }
    *out = g_scratch_ptr[dev];
    return MOE_OK;
}

size_t moe_sort_static_capacity_bytes() { return (size_t)SORT_STATIC_INTS * sizeof(int32_t); }

int moe_launch_sort_static(const void* expert_idx, int in64, int64_t R, int E, int block_m, void* sorted_expert,
                           void* sorted_pos, int out64, void* counts, void* offsets, void* padded_blocks,
                           int64_t padded_cap, int32_t* num_padded, int32_t* inv, hipStream_t stream)
{
    if (E < 1 || E > 4096 || R < 0 || block_m < 1) return MOE_ERR_BAD_ARG;
    if (moe_sort_ws_bytes(R, E) > moe_sort_static_capacity_bytes()) return MOE_ERR_WORKSPACE;
    int32_t* ptr = nullptr;
    const int rc = sort_static_scratch(&ptr);
    if (rc != MOE_OK) return rc;
    return moe_launch_sort(expert_idx, in64, R, E, block_m, sorted_expert, sorted_pos, out64, counts, offsets,
                           padded_blocks, padded_cap, num_padded, inv, ptr, moe_sort_static_capacity_bytes(), stream);
}

int moe_launch_offsets_from_sorted(const void* sorted_expert, int in64, int64_t R, int E, void* offsets, int out64,
                                   hipStream_t stream)
{
    hipLaunchKernelGGL(offsets_from_sorted_kernel, dim3((E + 63) / 64), dim3(64), 0, stream, sorted_expert, in64, R, E,
                       offsets, out64);
    return moe_launch_status();
}

int moe_launch_padded_blocks(const void* offsets, int off64, int E, int block_m, void* padded_blocks, int out64,
                             int64_t cap, int32_t* num_padded, hipStream_t stream)
{
    hipLaunchKernelGGL(padded_blocks_kernel, dim3(1), dim3(64), 0, stream, offsets, off64, E, block_m, padded_blocks,
                       out64, cap, num_padded);
    return moe_launch_status();
}
