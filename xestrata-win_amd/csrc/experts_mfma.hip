// xestrata-win_amd/csrc/experts_mfma.hip - the grouped expert products of large decode batches: the canonical row
// arithmetic (xs_units.h, bit for bit the oracle) with the units' integer sums on the matrix cores.
//
// v_mfma_i32_16x16x32_i8 multiplies 16 entries' int8 activations by 16 weight rows' codes over 32 values, a sub-block:
// exact integers whatever the order, as the canonical units are.  The weight rows are the B operand, so a lane holds one
// weight row (lane % 16) and four entries (4 (lane / 16) + r): the sub-block scale is one value a lane, and a unit's
// float steps (acc = fma(d d8, S, acc), ...) run as the lane-per-row kernels run them, chain c of a row in register
// acc[c] instead of in lane c, then the same butterfly over the L chains.  Q4_K's minimums are a second product of the
// activations with the sub-block's 6-bit minimum in every place (sum of m x = m (sum of x)), Q6_K's offset a product
// with -32.
//
// Memory, as the weight-stream kernels: a wave owns a ring of LDS slots that LDS DMA fills slots - 1 steps ahead of its
// products (a step: a slice of its 16 rows, at most ~5 KB), waits on its own vmcnt only and meets no barrier; rows lie an
// odd number of 16-byte chunks apart, so that 16 rows' reads cover all banks evenly.  A work-group's waves share one
// group's 16 activation rows in LDS and take 16 weight rows in turn.
//
// Why: the lane-per-row kernels apply a staged weight row to its entries two or four at a time with v_dot4, 8 integer
// instructions an entry for each 32 values and lane; above ~2 entries a group that work, not the weights, bounded them.
// Bound here by the weight stream and each work-group's start (indices, activations, the first slice: ~5 us).  Measured,
// 512 entries of 128 experts, hidden 2048, F 768, Q4_K: gate/up 65 us (3.5 TB/s) and down 54 (2.1) against 219 and 231;
// layers, before and after: 64 tokens of that shape with a gated shared expert 885 -> 167 us, hidden 4096 IQ4_XS at 8
// tokens 254 -> 195 and at 24 663 -> 431, Q4_K/Q6_K at 8 331 -> 192, hidden 7168 Q4_K at 6 tokens 762 -> 353.  One entry a
// group and few weights: the lane-per-row kernels stay ahead (lane_rows_ahead, abi.cpp).
#include "xs_device.h"
#include "xs_kernels.h"
#include "xs_units.h"

namespace xs {

typedef int i32x4_t __attribute__((ext_vector_type(4)));

constexpr int kMfmaEnt = 16;             // entries a pass
constexpr int kMfmaNi = 6;               // DMA instructions a step at most
constexpr int kMfmaLds = 160 * 1024;

struct MfmaGeom {
    int64_t mat_off;   // the matrix's offset in a blob
    int rows_total;    // its rows
    int rb;            // bytes a row
    int n_in;          // values a row
    int segb;          // bytes of a row a step
    int steps;         // steps a task (16 rows)
    int nc;            // 16-byte chunks a row of a slot (odd)
    int ni;            // DMA instructions a step
    int slots;         // slots a wave's ring
    int tasks;         // tasks a wave
    int waves;         // waves a work-group
    int ent;           // entries a pass: 16, or the most a group can have
    int astride;       // bytes between the staged activation rows
    int ring_off;      // LDS bytes before the rings (activations and their scales)
    int F, H;
};

template <int N>
struct ChainC {
    static constexpr int value = N;
};
// blocks a step
__host__ __device__ constexpr int mfma_step_blocks(int t, bool down) {
    return t == kQ8_0 ? 8 : down || t == kQ6_K ? 1 : 2;
}

// X32 (Q8_0 gate/up): the q8_1 rows have a scale of their own in each 32-value block, kept as the fp16 it comes in (hidden
// 7168: 16 entries still fit beside the rings).  Rows of quantize_q8_1_rows repeat one scale over 256 values, which is
// read once a step (16 tokens of hidden 7168: 676 us a layer against 711 with a read a block).
template <int T, bool DOWN, int L, bool X32>
__global__ __launch_bounds__(512) void rows_mfma_kernel(GroupedArgs a, MfmaGeom G, const int8_t* __restrict__ hq,
                                                        const float* __restrict__ hd) {
    constexpr int SB = mfma_step_blocks(T, DOWN), BB = block_bytes(T);
    constexpr bool S256 = !DOWN && T != kQ8_0;            // a unit is a whole 256-value block
    static_assert(S256 ? L == 4 || L == 8 : L == 8, "a block's eight units (or eight Q8_0 blocks) are a round of 8 chains");
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = 64 * G.waves;
    const int lrow = lane & 15, oct = lane >> 4;          // the lane's weight row (and entry of A), its octet of 32 values
    uint8_t* const aq = lds;
    static_assert(!X32 || (T == kQ8_0 && !DOWN));
    float* const ad = (float*)(lds + G.ent * G.astride);   // [scale][entry]: one scale a 256 (gate/up) or 32 (down; X32: fp16)
    uint8_t* const ring = lds + G.ring_off + wave * (G.slots * G.ni * 1024);
    const uint32_t ring_lds = lds_offset(ring);
    const uint32_t iq_t[4] = {kIq4Tab[0], kIq4Tab[1], kIq4Tab[2], kIq4Tab[3]};
    uint32_t four = __builtin_amdgcn_readfirstlane(0x04040404), ident;
    asm("v_mov_b32 %0, %1" : "=v"(ident) : "n"(0x03020100u));
    const uint32_t slot_bytes = (uint32_t)G.ni * 1024u, ring_end = ring_lds + (uint32_t)G.slots * slot_bytes;
    const int nb32 = G.n_in >> 5;
    const int ng = min(*a.n_groups, (int)a.cap_groups);

    // the lane's chunk of each DMA instruction: its row's bytes past the task's first row (-1: none) and its place in
    // the row's slice
    int crow[kMfmaNi], cc[kMfmaNi];
#pragma unroll
    for (int j = 0; j < kMfmaNi; ++j) {
        const int idx = 64 * j + lane, r = idx / G.nc;
        crow[j] = j < G.ni && r < 16 ? r * G.rb : -1;
        cc[j] = 16 * (idx - r * G.nc);
    }
    const int wrow0 = (int)blockIdx.x * (16 * G.waves * G.tasks) + 16 * wave;   // the wave's first row; tasks 16 waves apart
    int n_tasks = 0;
    while (n_tasks < G.tasks && wrow0 + 16 * G.waves * n_tasks < G.rows_total) ++n_tasks;
    const int total = n_tasks * G.steps;

    for (int g = blockIdx.y; g < ng; g += gridDim.y) {
        // the blob's address in scalar registers (the DMA's base); readfirstlane gives an int: widened unsigned
        const uint64_t bp = a.grp_ptr[g];
        const uint32_t bp_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bp);
        const uint32_t bp_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(bp >> 32));
        const uint8_t* const blob = (const uint8_t*)(((uint64_t)bp_hi << 32) | (uint64_t)bp_lo);
        const int e_lo = a.grp_start[g], n_all = a.grp_start[g + 1] - e_lo;
        if (((uintptr_t)blob & 15u) != 0) {
            if (tid == 0) atomicOr(a.err, 1);
            continue;
        }
        for (int p0 = G.ent * blockIdx.z; p0 < n_all; p0 += G.ent * gridDim.z) {
            const int e0 = e_lo + p0, n = min(G.ent, n_all - p0);
            // the DMA of the wave's steps in turn (steps segb = a row's bytes, so a task's next row follows on)
            uint32_t i_so = (uint32_t)G.mat_off + (uint32_t)(wrow0 * G.rb), i_slot = ring_lds;
            int i_st = 0;
            auto issue = [&]() {
#pragma unroll
                for (int j = 0; j < kMfmaNi; ++j) {
                    if (j >= G.ni) break;
                    const uint32_t so = i_so + (uint32_t)crow[j], at = (so & ~15u) + (uint32_t)cc[j];
                    const bool live = crow[j] >= 0 && at < so + (uint32_t)G.segb;
                    dma16_nt_at(blob, live ? at : 0u, __builtin_amdgcn_readfirstlane(i_slot + 1024 * j));
                }
                i_so += (uint32_t)G.segb;
                if (++i_st == G.steps) {
                    i_st = 0;
                    i_so += (uint32_t)((16 * G.waves - 1) * G.rb);
                }
                i_slot = i_slot + slot_bytes == ring_end ? ring_lds : i_slot + slot_bytes;
            };
            __syncthreads();   // the last pass's readers of the activations are done
            const int pre = min(G.slots - 1, total);
            for (int q = 0; q < pre; ++q) issue();
            int dst[4];   // the lane's entries' output rows (loaded here: a load among the products would drain the ring)
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[r] = DOWN ? a.ent_dst[e0 + min(4 * oct + r, n - 1)] : 0;
            // the entries' activations
            if (!DOWN) {
                for (int i = tid; i < n * nb32; i += nt) {
                    const int e = i / nb32, bi = i - e * nb32;
                    const uint32_t* blk =
                        (const uint32_t*)((const uint8_t*)a.x_q8_1 + ((int64_t)a.ent_tok[e0 + e] * nb32 + bi) * 36);
                    uint32_t w[9];
#pragma unroll
                    for (int k = 0; k < 9; ++k) w[k] = blk[k];
                    uint4* dst = (uint4*)(aq + e * G.astride + 32 * bi);
                    dst[0] = make_uint4(w[1], w[2], w[3], w[4]);
                    dst[1] = make_uint4(w[5], w[6], w[7], w[8]);
                    if (X32) ((uint16_t*)ad)[bi * kMfmaEnt + e] = (uint16_t)(w[0] & 0xFFFFu);
                    else if ((bi & 7) == 0) ad[(bi >> 3) * kMfmaEnt + e] = h2f((uint16_t)(w[0] & 0xFFFFu));
                }
            } else {
                const int nc16 = G.n_in >> 4;
                for (int i = tid; i < n * nc16; i += nt) {
                    const int e = i / nc16, c = i - e * nc16;
                    *(uint4*)(aq + e * G.astride + 16 * c) = *(const uint4*)(hq + (int64_t)(e0 + e) * G.n_in + 16 * c);
                }
                for (int i = tid; i < n * nb32; i += nt) {
                    const int e = i / nb32, b = i - e * nb32;
                    ad[b * kMfmaEnt + e] = hd[(int64_t)(e0 + e) * nb32 + b];
                }
            }
            __syncthreads();

            const uint8_t* const arow = aq + min(lrow, G.ent - 1) * G.astride + 8 * oct;
            const float* const adl = ad + 4 * oct;
            auto act = [&](int gs) { return *(const long*)(arow + 32 * gs); };   // 8 values of sub-block gs of the row
            auto codes8 = [](uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); };
            auto mfma = [](long x, long w, i32x4_t c) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(x, w, c, 0, 0, 0); };
            const i32x4_t zero = {0, 0, 0, 0};
            // IQ4_XS: the levels of the low nibbles of n's bytes (table16_lookup; its constants in registers, so that
            // and-or is one instruction)
            auto iq4_codes = [&](uint32_t n) {
                const uint32_t m = n & 0x07070707u;
                uint32_t pick = ((n >> 1) & four) | ident;
                asm("" : "+v"(pick));
                return __builtin_amdgcn_perm(__builtin_amdgcn_perm(iq_t[3], iq_t[2], m),
                                             __builtin_amdgcn_perm(iq_t[1], iq_t[0], m), pick);
            };

            float acc[L][4];
            int q = 0;
            uint32_t c_slot = 0;
            for (int i = 0; i < n_tasks; ++i) {
                const int r0 = wrow0 + 16 * G.waves * i;
#pragma unroll
                for (int c = 0; c < L; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[c][r] = 0.0f;
                for (int st = 0; st < G.steps; ++st, ++q) {
                    {
                        if (q + G.slots - 1 < total) {   // into the slot that the last step read
                            lds_reads_done();
                            issue();
                        }
                        vm_wait_le(min(G.slots - 1, total - 1 - q) * G.ni);
                        const uint8_t* const slot = ring + c_slot;
                        c_slot = c_slot + slot_bytes == ring_end - ring_lds ? 0u : c_slot + slot_bytes;
                        // the row's slice in the slot: its bytes keep their address modulo 16
                        const int roff = lrow * G.nc * 16 + ((int)(G.mat_off + (int64_t)(r0 + lrow) * G.rb + st * G.segb) & 15);
                        if constexpr (T == kQ8_0) {
#pragma unroll
                            for (int c = 0; c < 8; ++c) {   // unit u = 8 st + c: block c of the slice
                                const int u = 8 * st + c;
                                uint32_t w[2];
                                lds_words_a2<2>(slot, roff + 34 * c + 2 + 8 * oct, w);
                                const float d = h2f(*(const uint16_t*)(slot + roff + 34 * c));
                                const i32x4_t D = mfma(act(u), codes8(w[0], w[1]), zero);
                                float4 d8;
                                if (X32) {
                                    const uint2 h = *(const uint2*)((const uint16_t*)ad + u * kMfmaEnt + 4 * oct);
                                    d8 = make_float4(h2f((uint16_t)(h.x & 0xFFFFu)), h2f((uint16_t)(h.x >> 16)),
                                                     h2f((uint16_t)(h.y & 0xFFFFu)), h2f((uint16_t)(h.y >> 16)));
                                } else {
                                    d8 = *(const float4*)(adl + (DOWN ? u : st) * kMfmaEnt);
                                }
                                acc[c][0] = __builtin_fmaf(d * d8.x, (float)D[0], acc[c][0]);
                                acc[c][1] = __builtin_fmaf(d * d8.y, (float)D[1], acc[c][1]);
                                acc[c][2] = __builtin_fmaf(d * d8.z, (float)D[2], acc[c][2]);
                                acc[c][3] = __builtin_fmaf(d * d8.w, (float)D[3], acc[c][3]);
                            }
                        } else {
#pragma unroll
                            for (int bb = 0; bb < SB; ++bb) {
                                const int b = SB * st + bb;         // block of the row
                                const int bo = roff + BB * bb;      // its place in the slot
                                const uint8_t* const blk = slot + bo;
                                int S[4] = {0, 0, 0, 0};
                                i32x4_t S2 = zero;
                                float d, dmin = 0.0f;
                                float4 d8;
                                if (S256) d8 = *(const float4*)(adl + b * kMfmaEnt);
                                // the integer sums v (and Q4_K's minimums' vm) of a unit with scales e8 into chain c
                                auto unit = [&](auto c, const float4& e8, const int (&v)[4], const i32x4_t& vm) {
                                    const float dd[4] = {e8.x, e8.y, e8.z, e8.w};
                                    float(&ac)[4] = acc[decltype(c)::value];
#pragma unroll
                                    for (int r = 0; r < 4; ++r) {
                                        ac[r] = __builtin_fmaf(d * dd[r], (float)v[r], ac[r]);
                                        if (T == kQ4_K) ac[r] = __builtin_fmaf(-(dmin * dd[r]), (float)vm[r], ac[r]);
                                    }
                                };
                                auto unit32 = [&](int s, const int (&v)[4], const i32x4_t& vm) {   // unit 8 b + s: chain s
                                    const float4 e8 = *(const float4*)(adl + (8 * b + s) * kMfmaEnt);
                                    switch (s) {   // (s is a constant where this is expanded)
                                        case 0: unit(ChainC<0>{}, e8, v, vm); break;
                                        case 1: unit(ChainC<1>{}, e8, v, vm); break;
                                        case 2: unit(ChainC<2>{}, e8, v, vm); break;
                                        case 3: unit(ChainC<3>{}, e8, v, vm); break;
                                        case 4: unit(ChainC<4 % L>{}, e8, v, vm); break;
                                        case 5: unit(ChainC<5 % L>{}, e8, v, vm); break;
                                        case 6: unit(ChainC<6 % L>{}, e8, v, vm); break;
                                        default: unit(ChainC<7 % L>{}, e8, v, vm); break;
                                    }
                                };
                                auto scaled = [&](int s, int sc, const i32x4_t& D) {   // S += sc D, or the unit itself
                                    if (S256) {
#pragma unroll
                                        for (int r = 0; r < 4; ++r) S[r] += __mul24(sc, D[r]);
                                    } else {
                                        const int v[4] = {__mul24(sc, D[0]), __mul24(sc, D[1]), __mul24(sc, D[2]),
                                                          __mul24(sc, D[3])};
                                        unit32(s, v, S2);
                                    }
                                };
                                if constexpr (T == kQ4_K) {
                                    const uint4 h = *(const uint4*)blk;
                                    d = h2f((uint16_t)(h.x & 0xFFFFu));
                                    dmin = h2f((uint16_t)(h.x >> 16));
                                    const uint32_t scw[2] = {h.y & 0x3F3F3F3Fu,
                                                             (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u)};
                                    const uint32_t mnw[2] = {h.z & 0x3F3F3F3Fu,
                                                             ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)};
#pragma unroll
                                    for (int p = 0; p < 4; ++p) {
                                        const uint2 w = *(const uint2*)(blk + 16 + 32 * p + 8 * oct);
#pragma unroll
                                        for (int hh = 0; hh < 2; ++hh) {
                                            const int s = 2 * p + hh;
                                            const long x = act(8 * b + s);
                                            const i32x4_t D = mfma(x, codes8((w.x >> (4 * hh)) & 0x0F0F0F0Fu,
                                                                             (w.y >> (4 * hh)) & 0x0F0F0F0Fu), zero);
                                            const uint32_t mb = __builtin_amdgcn_perm(mnw[s >> 2], mnw[s >> 2],
                                                                                      0x01010101u * (uint32_t)(s & 3));
                                            S2 = mfma(x, codes8(mb, mb), S256 ? S2 : zero);
                                            scaled(s, (int)((scw[s >> 2] >> (8 * (s & 3))) & 0xFFu), D);
                                        }
                                    }
                                } else if constexpr (T == kIQ4_XS) {
                                    const uint2 h = *(const uint2*)blk;
                                    d = h2f((uint16_t)(h.x & 0xFFFFu));
#pragma unroll
                                    for (int s = 0; s < 8; ++s) {   // octets 0, 1: low nibbles of bytes 0-7, 8-15; 2, 3: high
                                        const uint2 w = *(const uint2*)(blk + 8 + 16 * s + 8 * (oct & 1));
                                        const int sh = (oct >> 1) * 4;
                                        const uint32_t lo = iq4_codes(w.x >> sh), hi = iq4_codes(w.y >> sh);
                                        const i32x4_t D = mfma(act(8 * b + s), codes8(lo, hi), zero);
                                        const int ls = (int)((h.y >> (4 * s)) & 0xFu) |
                                                       (int)(((h.x >> (16 + 2 * s)) & 3u) << 4);
                                        scaled(s, ls - 32, D);
                                    }
                                } else {   // Q6_K: two scales a sub-block (octets 0, 1 and 2, 3), each over half the product
                                    d = h2f(*(const uint16_t*)(blk + 208));
                                    uint32_t scw[4];
                                    lds_words_a2<4>(slot, bo + 192, scw);
                                    const uint32_t m0 = oct < 2 ? 0xFFFFFFFFu : 0u, m1 = ~m0;
                                    const long off0 = codes8(m0 & 0xE0E0E0E0u, m0 & 0xE0E0E0E0u);   // -32 in every place
                                    const long off1 = codes8(m1 & 0xE0E0E0E0u, m1 & 0xE0E0E0E0u);
#pragma unroll
                                    for (int s = 0; s < 8; ++s) {
                                        const int hn = s >> 2, ss = s & 3;
                                        uint32_t ql[2], qh[2], v[2];
                                        lds_words_a2<2>(slot, bo + 64 * hn + 32 * (ss & 1) + 8 * oct, ql);
                                        lds_words_a2<2>(slot, bo + 128 + 32 * hn + 8 * oct, qh);
#pragma unroll
                                        for (int k = 0; k < 2; ++k)
                                            v[k] = ((ql[k] >> (4 * (ss >> 1))) & 0x0F0F0F0Fu) |
                                                   (((qh[k] >> (2 * ss)) & 0x03030303u) << 4);
                                        const long x = act(8 * b + s);
                                        i32x4_t D0 = mfma(x, codes8(v[0] & m0, v[1] & m0), zero);
                                        i32x4_t D1 = mfma(x, codes8(v[0] & m1, v[1] & m1), zero);
                                        D0 = mfma(x, off0, D0);
                                        D1 = mfma(x, off1, D1);
                                        const int c0 = (int)(int8_t)((scw[s >> 1] >> (16 * (s & 1))) & 0xFFu);
                                        const int c1 = (int)(int8_t)((scw[s >> 1] >> (16 * (s & 1) + 8)) & 0xFFu);
                                        int v4[4];
#pragma unroll
                                        for (int r = 0; r < 4; ++r) v4[r] = __mul24(c0, D0[r]) + __mul24(c1, D1[r]);
                                        if (S256) {
#pragma unroll
                                            for (int r = 0; r < 4; ++r) S[r] += v4[r];
                                        } else {
                                            unit32(s, v4, zero);
                                        }
                                    }
                                }
                                if (S256) {   // unit b: chain b % L (uniform; the steps unrolled over a round spilled)
                                    switch (b % L) {
                                        case 0: unit(ChainC<0>{}, d8, S, S2); break;
                                        case 1: unit(ChainC<1>{}, d8, S, S2); break;
                                        case 2: unit(ChainC<2>{}, d8, S, S2); break;
                                        case 3: unit(ChainC<3>{}, d8, S, S2); break;
                                        case 4: unit(ChainC<4 % L>{}, d8, S, S2); break;
                                        case 5: unit(ChainC<5 % L>{}, d8, S, S2); break;
                                        case 6: unit(ChainC<6 % L>{}, d8, S, S2); break;
                                        default: unit(ChainC<7 % L>{}, d8, S, S2); break;
                                    }
                                }
                            }
                        }
                    }
                }
                // the butterfly over the chains (o = L / 2 .. 1; chain 0's value), then the rows out
#pragma unroll
                for (int o = L / 2; o > 0; o >>= 1)
#pragma unroll
                    for (int c = 0; c < o; ++c)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[c][r] += acc[c + o][r];
                const int row = r0 + lrow;
                if (row < G.rows_total) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int e = 4 * oct + r;
                        if (e >= n) break;
                        if (DOWN) a.out[(int64_t)dst[r] * G.H + row] = acc[0][r];
                        else if (row < G.F) a.gate[(int64_t)(e0 + e) * G.F + row] = acc[0][r];
                        else a.up[(int64_t)(e0 + e) * G.F + (row - G.F)] = acc[0][r];
                    }
                }
            }
        }
    }
}

namespace {

template <int T, bool DOWN>
bool mfma_geom(const ExpertLayout& L, int64_t cap_groups, int64_t cap_entries, int64_t max_entries, bool x32, MfmaGeom& G) {
    constexpr int SB = mfma_step_blocks(T, DOWN), BB = block_bytes(T), BV = block_values(T);
    G.n_in = (int)(DOWN ? L.n_ff : L.n_embd);
    G.rows_total = (int)(DOWN ? L.n_embd : 2 * L.n_ff);
    G.rb = (int)(DOWN ? L.d_row : L.gu_row);
    G.mat_off = DOWN ? L.down_off : 0;
    G.F = (int)L.n_ff;
    G.H = (int)L.n_embd;
    if (L.bytes > INT32_MAX || G.n_in % (SB * BV) || G.n_in % 256) return false;
    G.segb = SB * BB;
    G.steps = G.n_in / (SB * BV);
    const bool al16 = G.rb % 16 == 0 && G.mat_off % 16 == 0 && G.segb % 16 == 0;
    G.nc = (al16 ? G.segb / 16 : (G.segb + 15) / 16 + 1) | 1;
    G.ni = (16 * G.nc + 63) / 64;
    if (G.ni > kMfmaNi) return false;
    G.astride = G.n_in + 32;
    const int scales = DOWN ? G.n_in / 32 * kMfmaEnt * 4 : x32 ? G.n_in / 32 * kMfmaEnt * 2 : G.n_in / 256 * kMfmaEnt * 4;
    G.ent = max_entries > 0 && max_entries < kMfmaEnt ? (int)max_entries : kMfmaEnt;
    G.ring_off = (G.ent * G.astride + scales + 15) & ~15;
    // work-groups of 4 waves, two or more a compute unit (one starts, its indices and activations on their way, while
    // others stream): two slots a ring, three where three work-groups still fit a unit.  Hidden 2048, 512 entries of
    // 128 experts, Q4_K: 4 waves and 2 slots 167 us a layer, 8 waves and 3 slots 184; down 3 slots 148, 2 slots 155.
    // Wide activations leave room for one work-group: 8 waves, if their rings fit.
    const int slot = G.ni * 1024;
    G.waves = G.ring_off + 4 * 2 * slot <= kMfmaLds / 2 || G.ring_off + 8 * 2 * slot > kMfmaLds ? 4 : 8;
    if (G.ring_off + 4 * 2 * slot > kMfmaLds) return false;
    G.slots = G.waves == 8 ? (kMfmaLds - G.ring_off) / (8 * slot) : G.ring_off + 4 * 3 * slot <= kMfmaLds / 3 ? 3 : 2;
    if (G.slots > 4) G.slots = 4;
    // rows a work-group: as many as keep two work-groups for every compute unit, up to 512 (384 gate/up rows and 512
    // down rows of that layer 148 us, 256 and 256 167, twice as many 181); with few groups, fewer waves too
    const int64_t each = (cap_entries + cap_groups - 1) / cap_groups, passes = (each + G.ent - 1) / G.ent;
    const int64_t work = (int64_t)(G.rows_total / 16) * cap_groups * passes;   // 16-row tasks
    while (G.waves > 2 && work < 512 * G.waves) G.waves /= 2;
    const int64_t tasks = (4 * work + 512 * G.waves) / (2048 * G.waves);   // (three quarters and more: up)
    G.tasks = (int)(tasks < 1 ? 1 : tasks > 8 ? 8 : tasks);
    // Gate/up of a call of up to 4 tokens, whose groups are nearly all distinct experts: where that leaves between one and
    // one and a half rounds of two work-groups a compute unit, the second round is nearly empty; work-groups of 16 rows a
    // wave even it out.  Layers of hidden 4096, F 1536, 3 tokens x top-8 (576 work-groups of 2): IQ4_XS 103.7 -> 96.0 us,
    // Q8_0 132 -> 120, Q4_K/Q6_K 100.3 -> 95.5; 4 x top-6 Q8_0 133 -> 120.  (At 6 tokens x top-8 F 768, whose
    // distinct experts fill one round, 91 -> 95; the down products' short rows 65.3 -> 66.8.)
    const int64_t wgs = (G.rows_total / 16 + G.waves * G.tasks - 1) / (G.waves * G.tasks) * cap_groups * passes;
    if (!DOWN && max_entries > 0 && max_entries <= 4 && wgs > 512 && wgs < 768) G.tasks = 1;
    return true;
}

template <int T, bool DOWN, int LC, bool X32 = false>
hipError_t launch_one(const GroupedArgs& a, const MfmaGeom& G, const int8_t* hq, const float* hd, hipStream_t s) {
    void (*kern)(GroupedArgs, MfmaGeom, const int8_t*, const float*) = rows_mfma_kernel<T, DOWN, LC, X32>;
    const int lds = G.ring_off + G.waves * G.slots * G.ni * 1024;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
    }
    const int per = 16 * G.waves * G.tasks;
    const int64_t gy = a.grid_groups > 0 && a.grid_groups < a.cap_groups ? a.grid_groups : a.cap_groups;
    // passes side by side (a group with fewer leaves its later ones at once)
    const int64_t most = a.max_entries > 0 ? a.max_entries : a.cap_entries_hint;
    const int64_t gz = (most + G.ent - 1) / G.ent;
    const dim3 grid((unsigned)((G.rows_total + per - 1) / per), (unsigned)gy, (unsigned)(gz < 4 ? gz : 4));
    hipLaunchKernelGGL(kern, grid, dim3(64 * G.waves), (size_t)lds, s, a, G, hq, hd);
    return hipGetLastError();
}

template <int T, bool DOWN>
hipError_t launch_t(const ExpertLayout& L, const GroupedArgs& a, hipStream_t s) {
    MfmaGeom G;
    const bool x32 = a.x_scale32 && !DOWN && T == kQ8_0;
    if (!mfma_geom<T, DOWN>(L, a.cap_groups, a.cap_entries_hint, a.max_entries, x32, G)) return hipErrorNotSupported;
    const size_t f = (size_t)a.cap_entries_hint * (size_t)L.n_ff;   // the h region: int8 values, scales, sums of 16
    int8_t* hq = (int8_t*)a.hact;
    float* hd = (float*)(hq + ((f + 255) & ~(size_t)255));
    if (DOWN) {
        int* hs = (int*)((uint8_t*)hd + (((f / 32) * 4 + 255) & ~(size_t)255));
        const hipError_t e = launch_stream_h(L, a, hq, hd, hs, s);
        if (e != hipSuccess) return e;
    }
    if constexpr (!DOWN && T != kQ8_0) {
        switch (canon_lanes(G.n_in / 256)) {
            case 8: return launch_one<T, DOWN, 8>(a, G, hq, hd, s);
            case 4: return launch_one<T, DOWN, 4>(a, G, hq, hd, s);
            default: return hipErrorNotSupported;
        }
    } else {
        if constexpr (!DOWN && T == kQ8_0)
            if (x32) return launch_one<T, DOWN, 8, true>(a, G, hq, hd, s);
        return launch_one<T, DOWN, 8>(a, G, hq, hd, s);
    }
}

template <bool DOWN>
bool geom_any(int t, const ExpertLayout& L, int64_t cap_groups, int64_t cap_entries, int64_t max_entries, bool x32) {
    MfmaGeom G;
    switch (t) {
        case kQ4_K: return mfma_geom<kQ4_K, DOWN>(L, cap_groups, cap_entries, max_entries, false, G);
        case kQ6_K: return mfma_geom<kQ6_K, DOWN>(L, cap_groups, cap_entries, max_entries, false, G);
        case kQ8_0: return mfma_geom<kQ8_0, DOWN>(L, cap_groups, cap_entries, max_entries, x32 && !DOWN, G);
        case kIQ4_XS: return mfma_geom<kIQ4_XS, DOWN>(L, cap_groups, cap_entries, max_entries, false, G);
        default: return false;
    }
}

}  // namespace

bool mfma_rows_usable(const ExpertLayout& L, int64_t cap_groups, int64_t cap_entries, int64_t max_entries, bool x_scale32) {
    if (mixed_gu(L) || cap_groups <= 0 || cap_entries < cap_groups) return false;
    // the DMA reads whole 16-byte chunks: a matrix's last chunk must stay inside the blob
    if (L.bytes % 16 || L.up_off % 16 || L.down_off % 16) return false;
    if (L.gu_type != kQ8_0 && canon_lanes((int)(L.n_embd / 256)) < 4) return false;
    return geom_any<false>(L.gu_type, L, cap_groups, cap_entries, max_entries, x_scale32) &&
           geom_any<true>(L.d_type, L, cap_groups, cap_entries, max_entries, false);
}

hipError_t launch_mfma_gu(const ExpertLayout& L, const GroupedArgs& a, hipStream_t s) {
    switch (L.gu_type) {
        case kQ4_K: return launch_t<kQ4_K, false>(L, a, s);
        case kQ6_K: return launch_t<kQ6_K, false>(L, a, s);
        case kQ8_0: return launch_t<kQ8_0, false>(L, a, s);
        case kIQ4_XS: return launch_t<kIQ4_XS, false>(L, a, s);
        default: return hipErrorNotSupported;
    }
}

hipError_t launch_mfma_down(const ExpertLayout& L, const GroupedArgs& a, hipStream_t s) {
    switch (L.d_type) {
        case kQ4_K: return launch_t<kQ4_K, true>(L, a, s);
        case kQ6_K: return launch_t<kQ6_K, true>(L, a, s);
        case kQ8_0: return launch_t<kQ8_0, true>(L, a, s);
        case kIQ4_XS: return launch_t<kIQ4_XS, true>(L, a, s);
        default: return hipErrorNotSupported;
    }
}

}  // namespace xs
