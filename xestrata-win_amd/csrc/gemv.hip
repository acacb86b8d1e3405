// xestrata-win_amd/csrc/gemv.hip - the router's projections (logits = W x, W n_out rows of n_in) in the summation
// orders of the reference's kernels, so that logits, and the ids routed from them, come out bit for bit:
//
//   mmvf (f32_gemv_fp32_mmvf(_multi), bf16_gemv_fp32_mmvf(_multi); src/kernels/xe/bf16_gemv.cpp:91-147, 213-225,
//     464-517): a work-group of B threads a row, B the candidate of 32, 64, ..., 256 with the fewest pair iterations
//     (the smallest on a tie).  Thread t walks pairs t, t + B, ... with two ordered FMAs a pair (weight 2p, then
//     2p + 1) into one accumulator a token; a xor butterfly (16, 8, 4, 2, 1) over each 32 threads; for B > 32 the
//     partials of the B / 32 groups (then zeros up to 32) summed by the same butterfly.  Up to 8 tokens a launch.
//   gemm_rows (f32_gemm_rows, bf16_gemv.cpp:475-502; the prompt path's router and shared gate): one FMA chain a
//     logit, k = 0, 1, ... n_in - 1, then FMAs with zeros up to the next multiple of 16.
//   warp (bf16_gemv for n_out >= 64 and bf16_gemv_split at 32 threads a row, bf16_gemv.cpp:62-77, 300-317): bf16
//     activations and weights, 32 lanes a row, lane l over l, l + 32, ..., then the 32-lane butterfly; every product
//     of two bf16 values is exact in f32, so a fused and an unfused multiply-add agree.
//   naive (bf16_gemv for n_out < 64, bf16_gemv.cpp:50-60): one chain a row over the whole row.
//   tree (bf16_gemv_split at another power of two, bf16_gemv.cpp:318-339): lane chains as warp's, then the shared
//     memory tree s[t] += s[t + off], off = tpr / 2 ... 1.
//
// MI355X layout: a 32-lane group is half a wave64 (a xor below 32 stays inside it), so the warp form takes two rows a
// wave and the mmvf form's 32-thread groups are wave halves.  The gemm_rows form gives a work-group 16 or 64 rows of one
// side over its lanes (staged through LDS) x 16 of the other (a value a lane, broadcast by the multiply-add itself).
#include "xs_device.h"
#include "xs_kernels.h"

#include <type_traits>

namespace xs {

__device__ __forceinline__ float bf2f(uint16_t b) { return u2f((uint32_t)b << 16); }

__device__ __forceinline__ float sum32(float v) {   // the 32-lane xor butterfly, inside each wave half
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 8, 64);
    v += __shfl_xor(v, 4, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 1, 64);
    return v;
}

int mmvf_block(int64_t n_in) {
    int best = 32;
    int64_t best_it = (n_in + 63) / 64;
    for (int c = 64; c <= 256; c += 32) {
        const int64_t it = (n_in + 2 * c - 1) / (2 * c);
        if (it < best_it) {
            best_it = it;
            best = c;
        }
    }
    return best;
}

template <typename W>
__device__ __forceinline__ void weight_pair(const W* row, int64_t p, float& w0, float& w1);
template <>
__device__ __forceinline__ void weight_pair<float>(const float* row, int64_t p, float& w0, float& w1) {
    const float2 v = *(const float2*)(row + 2 * p);
    w0 = v.x;
    w1 = v.y;
}
template <>
__device__ __forceinline__ void weight_pair<uint16_t>(const uint16_t* row, int64_t p, float& w0, float& w1) {
    const uint32_t v = *(const uint32_t*)(row + 2 * p);
    w0 = u2f(v << 16);
    w1 = u2f(v & 0xFFFF0000u);
}

// sum32 by lane moves inside the VALU: the same additions (after the xor 16 and 8 steps a value repeats every 8 lanes, so
// a rotation by 4 brings the xor-4 partner's)
__device__ __forceinline__ float sum32_dpp(float v) {
    v += swz_xor16_f(v);
    v += dpp_f<kDppRor8>(v);
    v += dpp_f<kDppRor4>(v);
    v += dpp_f<kDppXor2>(v);
    v += dpp_f<kDppXor1>(v);
    return v;
}

// NT: the tokens, rounded up to 1, 2, 4 or 8 (tokens past n_tok repeat the last).  A thread's weight pairs and x values of
// four strides are in flight together: with one stride's at a time (and the token count a run-time bound) a row waited for
// memory once a stride, 4 times at 2048 values and 14 at 7168: 1 token x 128 x 2048 5.0 us, now 2.8; 8 tokens x 256 x
// 7168 39.4, now 13.9.
template <typename W, int NT>
__global__ __launch_bounds__(256) void mmvf_kernel(const float* __restrict__ x, int64_t ldx, const W* __restrict__ w,
                                                   float* __restrict__ y, int64_t ldy, int64_t n_pairs, int n_tok) {
    constexpr int U = 4;
    __shared__ float partials[NT * 32];
    const int t = threadIdx.x, B = blockDim.x;
    const int64_t o = blockIdx.x;
    const W* row = w + o * 2 * n_pairs;
    const float* xt[NT];
    float acc[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
        xt[k] = x + min(k, n_tok - 1) * ldx;
        acc[k] = 0.0f;
    }
    if (B > 32)
        for (int i = t; i < NT * 32; i += B) partials[i] = 0.0f;
    auto strides = [&](int64_t p0, auto whole_c) {   // strides p0, p0 + B, ... (U of them; past the row's end: none)
        constexpr bool WHOLE = decltype(whole_c)::value;
        float w0[U], w1[U];
        float2 xv[U][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t p = WHOLE || p0 + u * B < n_pairs ? p0 + u * B : t;
            weight_pair<W>(row, p, w0[u], w1[u]);
#pragma unroll
            for (int k = 0; k < NT; ++k) xv[u][k] = *(const float2*)(xt[k] + 2 * p);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (WHOLE || p0 + u * B < n_pairs)
#pragma unroll
                for (int k = 0; k < NT; ++k) {
                    acc[k] = __builtin_fmaf(w0[u], xv[u][k].x, acc[k]);
                    acc[k] = __builtin_fmaf(w1[u], xv[u][k].y, acc[k]);
                }
    };
    int64_t p = t;
    if (t < n_pairs) {
        for (; p + (U - 1) * B < n_pairs; p += U * B) strides(p, std::true_type{});
        if (p < n_pairs) strides(p, std::false_type{});
    }
#pragma unroll
    for (int k = 0; k < NT; ++k) acc[k] = sum32_dpp(acc[k]);
    if (B > 32) {
        __syncthreads();   // (the zeros are in place)
        if ((t & 31) == 0)
#pragma unroll
            for (int k = 0; k < NT; ++k) partials[k * 32 + t / 32] = acc[k];
        __syncthreads();
        if (t < 64) {   // lanes 32..63 run the same sums on the same values; only lane 0 stores
#pragma unroll
            for (int k = 0; k < NT; ++k) acc[k] = sum32_dpp(partials[k * 32 + (t & 31)]);
        }
    }
    if (t == 0)
#pragma unroll
        for (int k = 0; k < NT; ++k)
            if (k < n_tok) y[k * ldy + o] = acc[k];
}

template <typename W>
hipError_t launch_mmvf(const float* x, int64_t ldx, const W* w, float* y, int64_t ldy, int64_t n_in, int64_t n_out,
                       int n_tok, hipStream_t s) {
    void (*k)(const float*, int64_t, const W*, float*, int64_t, int64_t, int) =
        n_tok == 1 ? mmvf_kernel<W, 1> : n_tok == 2 ? mmvf_kernel<W, 2> : n_tok <= 4 ? mmvf_kernel<W, 4> : mmvf_kernel<W, 8>;
    hipLaunchKernelGGL(k, dim3((unsigned)n_out), dim3(mmvf_block(n_in)), 0, s, x, ldx, w, y, ldy, n_in / 2, n_tok);
    return hipGetLastError();
}
template hipError_t launch_mmvf<float>(const float*, int64_t, const float*, float*, int64_t, int64_t, int64_t, int,
                                       hipStream_t);
template hipError_t launch_mmvf<uint16_t>(const float*, int64_t, const uint16_t*, float*, int64_t, int64_t, int64_t,
                                          int, hipStream_t);

// The gemm_rows chains.  One side's rows (weights or tokens) lie over the lanes, their values staged through LDS; the
// other side's ("group rows") stay one value a lane in registers and are broadcast by the multiply-add itself, so the
// inner loop has no other instruction than its multiply-adds and the lane rows' LDS reads.  Two forms:
//   few chains: 16 lane rows x 4 group rows a wave, v_fmac_f32 whose DPP operand takes lane kk of each 16
//     (row_newbcast; lane i of the 16: the group row's value at k0 + i).  A work-group reads 32 rows: with few
//     work-groups one compute unit's share of the memory system bounds it, not the chip's (64-row tiles: 2048 x 1 x 64
//     tokens 20.3 us against 14.6).
//   many chains: v_mfma_f32_4x4x1_16b_f32, one FMA (one rounding) an output: a run of them over k = 0, 1, ... is the
//     chain itself.  64 lane rows x 4 group rows a wave; lane 4 kk + i holds group row i at k0 + kk, and CBSZ 4 / ABID
//     kk broadcast block kk.  A row is then read by fewer work-groups (8 group rows a wave in two accumulators, two
//     waves a work-group: 2048 tokens 34.6 us against 26.3).
// Chains are 1024 to 7168 steps long and few (2048 tokens x 128 experts: 4 a lane of the whole chip), so their length
// is what bounds a router: 12 ns a step as measured (25 us for 2048 steps), about 29 cycles at 2.4 GHz, in which a wave
// reads 16 bytes a lane for each 4 steps from LDS, then runs 16 dependent products.  The loads ahead must not stop it: two
// steps ahead through registers, then LDS.  A tile of 64 x 64 chains a work-group, 4 x 4 a thread, read from LDS a k at a time and waiting
// for each step's loads, took 230 us at 2048 tokens x 128 experts x 2048 (now 25; 62 against 17 TFLOP/s at 4096 x 256 x
// 7168), and 165 us for one weight row x 64 tokens x 2048 (now 13).
struct __attribute__((packed, aligned(4))) F4u {   // 16 bytes at any float's address
    float v[4];
};
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16 steps of a wave's chains, few-chains form: acc = fma(group value kk of the lane's 16, b[kk], acc), kk = 0 .. 15.
// (One block: the compiler makes a move of every broadcast.  The s_nop covers a group value written by the instruction
// before, which a DPP read has to stay two wait states behind.)
#define XS_FMAC(KK, B) "v_fmac_f32_dpp %0, %1, " B " row_newbcast:" KK " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void chain16(float& acc, float g, const float (&b)[16]) {
    asm("s_nop 1\n\t" XS_FMAC("0", "%2") XS_FMAC("1", "%3") XS_FMAC("2", "%4") XS_FMAC("3", "%5") XS_FMAC("4", "%6")
            XS_FMAC("5", "%7") XS_FMAC("6", "%8") XS_FMAC("7", "%9") XS_FMAC("8", "%10") XS_FMAC("9", "%11")
                XS_FMAC("10", "%12") XS_FMAC("11", "%13") XS_FMAC("12", "%14") XS_FMAC("13", "%15") XS_FMAC("14", "%16")
                    XS_FMAC("15", "%17")
        : "+&v"(acc)
        : "v"(g), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "v"(b[4]), "v"(b[5]), "v"(b[6]), "v"(b[7]), "v"(b[8]),
          "v"(b[9]), "v"(b[10]), "v"(b[11]), "v"(b[12]), "v"(b[13]), "v"(b[14]), "v"(b[15]));
}
#undef XS_FMAC

typedef float f32x4_t __attribute__((ext_vector_type(4)));
template <int KK>
__device__ __forceinline__ void mfma16(f32x4_t& acc, float g, const float (&b)[16]) {
    if constexpr (KK < 16) {
        acc = __builtin_amdgcn_mfma_f32_4x4x1f32(g, b[KK], acc, 4, KK, 0);
        mfma16<KK + 1>(acc, g, b);
    }
}

// y[p * yl + q * yg] = lane row p . group row q.  A work-group: LR lane rows x 16 group rows, 4 waves, KS values a
// step.  In LDS 16-byte chunk c of row r lies at c ^ (r % 16): the reads of 16 lanes cover all banks once.
template <bool MANY>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const float* __restrict__ lanes, int64_t ldl,
                                                                     int64_t n_l, const float* __restrict__ groups,
                                                                     int64_t ldg, int64_t n_g, float* __restrict__ y,
                                                                     int64_t yl, int64_t yg, int64_t n_in,
                                                                     unsigned lane_tiles) {
    constexpr int LR = MANY ? 64 : 16, KS = MANY ? 128 : 256;
    constexpr int kChunks = KS / 4, kLd = LR * kChunks / 256, kRowStep = 256 / kChunks;
    __shared__ float4 sl[2][LR * kChunks];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t l0 = (int64_t)(blockIdx.x % lane_tiles) * LR;
    const int64_t g0 = (int64_t)(blockIdx.x / lane_tiles) * 16 + 4 * wave;
    const int lrow = MANY ? lane : lane & 15;        // the lane's row of the tile
    const int lc = tid % kChunks, lr = tid / kChunks;   // the chunk it loads, and its first row (then every kRowStep)
    const float* lsrc[kLd];
#pragma unroll
    for (int i = 0; i < kLd; ++i) lsrc[i] = lanes + min(l0 + lr + kRowStep * i, n_l - 1) * ldl + 4 * lc;
    const int gk = MANY ? lane >> 2 : lane & 15;     // which of 16 k the lane's group value is, of which group row
    const float* gsrc = groups + min(g0 + (MANY ? lane & 3 : lane >> 4), n_g - 1) * ldg + gk;
    f32x4_t acc4 = {0.0f, 0.0f, 0.0f, 0.0f};
    float acc1 = 0.0f;
    F4u pre[2][kLd];
    float gv[2][KS / 16];
    const int n_full = (int)(n_in / KS);
    auto load = [&](int step, int slot) {
#pragma unroll
        for (int i = 0; i < kLd; ++i) pre[slot][i] = *(const F4u*)(lsrc[i] + (int64_t)step * KS);
    };
    auto load_g = [&](int step, int slot) {
#pragma unroll
        for (int j = 0; j < KS / 16; ++j) gv[slot][j] = gsrc[(int64_t)step * KS + 16 * j];
    };
    auto store = [&](int slot) {
#pragma unroll
        for (int i = 0; i < kLd; ++i) {
            const int r = lr + kRowStep * i;
            const F4u& v = pre[slot][i];
            sl[slot][r * kChunks + (lc ^ (r & 15))] = make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
        }
    };
    auto products = [&](int slot, int j, float g) {   // k = 16 j .. + 15 of the step in buffer `slot`
        float b[16];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float4 v = sl[slot][lrow * kChunks + ((4 * j + u) ^ (lrow & 15))];
            b[4 * u] = v.x, b[4 * u + 1] = v.y, b[4 * u + 2] = v.z, b[4 * u + 3] = v.w;
        }
        if constexpr (MANY) mfma16<0>(acc4, g, b);
        else chain16(acc1, g, b);
    };
    // step s from buffer SL; the group values of step s + 1 and the lane values of step s + 2 are issued first (past the
    // last step: the last one's again, so that no branch holds the loads up)
    auto step = [&](int s, auto slot_c) {
        constexpr int SL = decltype(slot_c)::value;
        lds_barrier();   // (the loads ahead stay in flight)
        load_g(min(s + 1, n_full - 1), SL ^ 1);
        load(min(s + 2, n_full - 1), SL);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < KS / 16; ++j) products(SL, j, gv[SL][j]);
        store(SL ^ 1);   // step s + 1; the buffer's readers (step s - 1) are past this step's barrier
    };
    if (n_full > 0) {
        load(0, 0);
        load_g(0, 0);
        load(min(1, n_full - 1), 1);
        store(0);
        for (int s = 0; s < n_full; s += 2) {
            step(s, std::integral_constant<int, 0>{});
            if (s + 1 >= n_full) break;
            step(s + 1, std::integral_constant<int, 1>{});
        }
    }
    // the values past the last whole step, and the chain's zeros up to a multiple of 16
    const int64_t k0 = (int64_t)n_full * KS, left = (n_in + 15) / 16 * 16 - k0;
    if (left > 0) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kLd; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) pre[0][i].v[u] = k0 + 4 * lc + u < n_in ? lsrc[i][k0 + u] : 0.0f;
        store(0);
        __syncthreads();
        for (int j = 0; j < left / 16; ++j) {
            const int64_t k = k0 + 16 * j;
            products(0, j, k + gk < n_in ? gsrc[k] : 0.0f);
        }
    }
    if (l0 + lrow >= n_l) return;
    if constexpr (MANY) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (g0 + i < n_g) y[(l0 + lrow) * yl + (g0 + i) * yg] = acc4[i];
    } else {
        if (g0 + (lane >> 4) < n_g) y[(l0 + lrow) * yl + (g0 + (lane >> 4)) * yg] = acc1;
    }
}

// The few-chains form up to this many work-groups (16 x 16 chains each, two a compute unit): at 512 (1024 tokens x 128
// experts x 2048) 20.1 us against 24.5 in 64-row tiles, at 1024 work-groups (2048 tokens) 29.7 against 26.3.
constexpr int64_t kFewChains = 512;
// The weight rows lie over the lanes when there are at least as many of them as tokens or a whole tile of 64, so that a
// logit row's stores are contiguous; else the tokens do (a shared expert's gate is one weight row).
hipError_t launch_gemm_rows(const float* x, int64_t ldx, const float* w, float* y, int64_t ldy, int64_t n_in,
                            int64_t n_out, int64_t n_tok, hipStream_t s) {
    const bool w_lanes = n_out >= 64 || n_out >= n_tok;
    const float *pl = w_lanes ? w : x, *pg = w_lanes ? x : w;
    const int64_t ll = w_lanes ? n_in : ldx, lg = w_lanes ? ldx : n_in, n_l = w_lanes ? n_out : n_tok;
    const int64_t n_g = w_lanes ? n_tok : n_out, yl = w_lanes ? 1 : ldy, yg = w_lanes ? ldy : 1;
    const int64_t groups = (n_g + 15) / 16;
    if ((n_l + 15) / 16 * groups <= kFewChains)
        hipLaunchKernelGGL(gemm_rows_kernel<false>, dim3((unsigned)((n_l + 15) / 16 * groups)), dim3(256), 0, s, pl, ll,
                           n_l, pg, lg, n_g, y, yl, yg, n_in, (unsigned)((n_l + 15) / 16));
    else
        hipLaunchKernelGGL(gemm_rows_kernel<true>, dim3((unsigned)((n_l + 63) / 64 * groups)), dim3(256), 0, s, pl, ll,
                           n_l, pg, lg, n_g, y, yl, yg, n_in, (unsigned)((n_l + 63) / 64));
    return hipGetLastError();
}

// x bf16 (or f32 rounded to bf16 on the fly: the same bits as converting first) against bf16 rows, 32 lanes a row
template <bool XF32>
__global__ __launch_bounds__(256) void bf16_warp_kernel(const void* __restrict__ xv, const uint16_t* __restrict__ w,
                                                        float* __restrict__ y, int64_t n_in, int64_t n_out) {
    const int lane = threadIdx.x & 31;
    const int64_t o = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
    const bool live = o < n_out;
    const uint16_t* row = w + (live ? o : 0) * n_in;
    float acc = 0.0f;
    if (live)
        for (int64_t i = lane; i < n_in; i += 32) {
            const float xf = XF32 ? bf2f(f2bf(((const float*)xv)[i])) : bf2f(((const uint16_t*)xv)[i]);
            acc = __builtin_fmaf(xf, bf2f(row[i]), acc);
        }
    acc = sum32(acc);
    if (live && lane == 0) y[o] = acc;
}

__global__ __launch_bounds__(256) void bf16_naive_kernel(const uint16_t* __restrict__ x,
                                                         const uint16_t* __restrict__ w, float* __restrict__ y,
                                                         int64_t n_in, int64_t n_out) {
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= n_out) return;
    const uint16_t* row = w + o * n_in;
    float acc = 0.0f;
    for (int64_t i = 0; i < n_in; ++i) acc = __builtin_fmaf(bf2f(x[i]), bf2f(row[i]), acc);
    y[o] = acc;
}

__global__ __launch_bounds__(1024) void bf16_tree_kernel(const uint16_t* __restrict__ x,
                                                         const uint16_t* __restrict__ w, float* __restrict__ y,
                                                         int64_t n_in) {
    extern __shared__ float tree[];
    const int t = threadIdx.x, tpr = blockDim.x;
    const int64_t o = blockIdx.x;
    const uint16_t* row = w + o * n_in;
    float acc = 0.0f;
    for (int64_t i = t; i < n_in; i += tpr) acc = __builtin_fmaf(bf2f(x[i]), bf2f(row[i]), acc);
    tree[t] = acc;
    __syncthreads();
    for (int off = tpr >> 1; off > 0; off >>= 1) {
        if (t < off) tree[t] = tree[t] + tree[t + off];
        __syncthreads();
    }
    if (t == 0) y[o] = tree[0];
}

__global__ __launch_bounds__(256) void to_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ y,
                                                      int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

hipError_t launch_to_bf16(const float* x, uint16_t* y, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, y, n);
    return hipGetLastError();
}

hipError_t launch_bf16_gemv(const void* x, bool x_f32, const uint16_t* w, float* y, int64_t n_in, int64_t n_out,
                            int form, int tpr, hipStream_t s) {
    if (form == kBf16Warp) {
        const dim3 grid((unsigned)((n_out + 7) / 8));
        if (x_f32)
            hipLaunchKernelGGL(bf16_warp_kernel<true>, grid, dim3(256), 0, s, x, w, y, n_in, n_out);
        else
            hipLaunchKernelGGL(bf16_warp_kernel<false>, grid, dim3(256), 0, s, x, w, y, n_in, n_out);
    } else if (form == kBf16Naive) {
        hipLaunchKernelGGL(bf16_naive_kernel, dim3((unsigned)((n_out + 255) / 256)), dim3(256), 0, s,
                           (const uint16_t*)x, w, y, n_in, n_out);
    } else {
        hipLaunchKernelGGL(bf16_tree_kernel, dim3((unsigned)n_out), dim3(tpr), (size_t)tpr * 4, s,
                           (const uint16_t*)x, w, y, n_in);
    }
    return hipGetLastError();
}

}  // namespace xs
