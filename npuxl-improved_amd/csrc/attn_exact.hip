// attn_exact.hip - ATTENTION_F32 in the reference's order of roundings for
// head sizes of any multiple of 8 up to 128, on the fp32 matrix cores (prefill)
// and as a scores and a chain kernel (decode).
//
// The reference's attention_range (src/kernels/llm.cpp:442-546) computes,
// per query row and 64-key block:
//   s_j = dot_avx2(q, k_j) * scale (+ mask)   eight FMA chains over
//         d = 8i + c, i ascending, then hsum256 ((c0+c4)+(c1+c5)) +
//         ((c2+c6)+(c3+c7)) (llm.cpp:332-343);
//   a block whose max is not finite is skipped; new_m = max(m, block max),
//   alpha = fast_expf(m - new_m), p_j = fast_expf(s_j - new_m), the weight
//   sum in key order, l = l * alpha + sum;
//   acc = acc * alpha, then acc = fma(v_j, p_j, acc) in key order for every
//   p_j != 0 (axpy_avx2, llm.cpp:345-355); out = acc * (1 / l).
//
// gfx950's fp32 MFMA with K = 1 (v_mfma_f32_32x32x1_2b_f32) computes
// D = A * B + C with one rounding, the same result as fmaf for every input
// (normal, denormal, infinite, NaN; checked against v_fma_f32 on MI355X over
// 8.4 million outputs per operand class, chains included).  Both sequential
// chains of the reference therefore run on the matrix core, one rank-1 step
// per instruction, in the reference's order:
//   scores   S^T[key][q] over a 32-key x 32-row tile: block 0 of the
//            instruction is chain c, block 1 chain c + 4, step i of both
//            chains per instruction (A = K, B = Q); the lane that holds
//            (key, row) in block 0 holds it in block 1, so hsum256's
//            pairing is in-lane;
//   output   O^T[d][q] += V^T[d][key] * P[key][q], one key per instruction,
//            keys ascending (A = V, B = P), 64 head elements per instruction.
// Every lane owns one query row in both products (column = lane % 32): the
// softmax state, alpha and the row's weights stay in the lane.  The weights
// of a key sit in one half of the wave; one exchange with the other half
// gives every lane its row's 64 weights, in key order for the sum and as the
// B operand of each key's instruction.
//
// The one difference from the reference is the p_j == 0 skip: the
// instruction adds v * 0 instead of skipping, which equals skipping unless
// acc is -0 (it becomes +0) or v is infinite or NaN (the sum becomes NaN).
// A sign-of-zero difference either vanishes at the next nonzero product or
// leaves a zero output element; a non-finite v leaves a NaN.  So every
// output element that is neither NaN nor zero is the reference's bit for
// bit, and a wave that finds a NaN, or a zero in a row with l > 0, among its
// outputs recomputes its rows in the reference's order on the vector ALUs.
//
// Structure: one workgroup of four waves per (batch, head) and 128 query
// rows, wave w owning rows 32w .. 32w + 31 (grids that leave CUs idle share 32
// rows between the four waves, attn_exact_coop_kernel); the 64-key K and V
// tiles are copied from HBM straight into LDS (double-buffered, the next
// block's copy in flight during this block's work); the workgroups of the
// longest causal rows are dispatched first.  The fp32 matrix instructions and
// the softmax's vector instructions share one issue, which bounds the kernel
// (32 heads x 2048 rows of 128: 388 us, 88 of 157 TFLOP/s).  Head sizes other
// than 64 and 128 took the row-wise vector kernel before: 32 heads x 2048 rows
// of 96 9014 -> 349 us, of 80 8279 -> 332; 8 x 32 heads of 96 over 4096 cached
// keys 2045 -> 147.
#include "kernels.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>
#include "device_math.hpp"
#include "lds_dma.hpp"
#include "vnpu_internal.hpp"

namespace vnpu {
namespace k {
namespace {

typedef float f32x32 __attribute__((ext_vector_type(32)));

constexpr int XT = 256;          // threads per workgroup (four waves)
constexpr int XQW = 32;          // query rows per wave
constexpr int XQ = 4 * XQW;      // query rows per workgroup
constexpr int XB = 64;           // keys per block (the reference's BK)

// Geometry for a head size of up to D (a multiple of 8).  A smaller head_dim
// runs with its missing elements as zeros: a zero step leaves a score chain
// as it is (up to the sign of a zero, which no weight sees), and the missing
// output elements are not stored.
template <int D>
struct XL {
    static constexpr int NM = (D + 63) / 64;           // output instructions per key (64 head elements each)
    static constexpr int DV = 64 * NM;                 // V row pitch (floats)
    static constexpr int KCH = D / 4 + 1;              // 16-byte slots per K row (one pad slot)
    static constexpr int KP = 4 * KCH;                 // K row pitch (floats), 4 x odd: conflict-free row reads
    static constexpr int KTILE = XB * KP;              // floats per K tile
    static constexpr int VTILE = XB * DV;              // floats per V tile
    static constexpr int KI = XB * KCH / 64;           // wave copies (64 slots each) per K tile
    static constexpr int VI = XB * DV / 4 / 64;        // per V tile
    static constexpr size_t kLds = static_cast<size_t>(2 * KTILE + 2 * VTILE) * sizeof(float);
    static_assert(D % 8 == 0, "the score chains take eight elements a step");
};

// What a copy reads for a slot past head_dim.
__device__ const float4 zero16 = {0.f, 0.f, 0.f, 0.f};

__device__ __forceinline__ f32x32 mfma1(float a, float b, f32x32 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, c, 0, 0, 0);
}

// Both halves' values of a lane's column: lo[l] = v of lane l % 32, hi[l] =
// v of lane 32 + l % 32 (one v_permlane32_swap_b32).
__device__ __forceinline__ void halves(float v, float &lo, float &hi)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    lo = __uint_as_float(r[0]);
    hi = __uint_as_float(r[1]);
}

// The weights and the output chain of one 64-key block for the lane's row
// (keys 32t + 8g + 4h + j of S[t][4g + j] in half h): per group of eight keys,
// the weights of both halves, the weight sum in key order, then one
// instruction per key and 64 head elements, keys ascending.  FULL: every key
// of the block is seen by some row of the wave (no per-key test).  Returns
// the block's weight sum.  Every S - nm is <= 0 or NaN (nm is the max).
template <int D, bool FULL>
__device__ __forceinline__ float weights_output(f32x32 (&oacc)[XL<D>::NM], const float (&S)[2][16], float nm,
                                                bool live, uint32_t kc_w, int lane, const float *Vb)
{
#pragma clang fp contract(off)
    float psum = 0.0f;
    float lo[4], hi[4], nlo[4], nhi[4];
    auto weights = [&](int t, int g, float (&wl)[4], float (&wh)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float e = dev::fast_expf_nonpos(S[t][4 * g + j] - nm);
            halves(live ? e : 0.0f, wl[j], wh[j]);
        }
    };
    weights(0, 0, nlo, nhi);
#pragma unroll
    for (int q = 0; q < 8; ++q) {   // group q: keys 8q .. 8q + 7
        // One group's V operands in registers at a time (without the fence
        // the scheduler hoists every V read of the block); the next group's
        // weights are computed while this group's instructions run.
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            lo[j] = nlo[j];
            hi[j] = nhi[j];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) psum = psum + lo[j];
#pragma unroll
        for (int j = 0; j < 4; ++j) psum = psum + hi[j];
        if (q < 7) weights((q + 1) / 4, (q + 1) % 4, nlo, nhi);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int kk = 8 * q + j;
            if (FULL || kk < static_cast<int>(kc_w)) {   // uniform
#pragma unroll
                for (int mm = 0; mm < XL<D>::NM; ++mm)
                    oacc[mm] = mfma1(Vb[kk * XL<D>::DV + 64 * mm + lane], j < 4 ? lo[j] : hi[j - 4], oacc[mm]);
            }
        }
    }
    return psum;
}

// One query row in the reference's order on the vector ALUs, by one wave:
// lane j scores key k0 + j of each block, lane e owns head elements e,
// e + 64, ... of the output row.
template <int D>
__device__ __noinline__ void exact_row_wave(Attn a, uint64_t bh, uint32_t qi, int lane)
{
#pragma clang fp contract(off)
    constexpr int E = XL<D>::NM;
    const uint32_t hd = a.head_dim;
    const uint32_t sq = a.seq_q, sk = a.seq_k;
    const uint32_t off = sk > sq ? sk - sq : 0;
    const uint64_t row = bh * sq + qi;
    const float *q = a.Q + row * hd;
    const float *Kh = a.K + bh * sk * hd;
    const float *Vh = a.V + bh * sk * hd;
    const float *Mr = a.mask ? a.mask + row * sk : nullptr;
    float acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = 0.0f;
    float m = -__builtin_inff(), l = 0.0f;
    const uint32_t kend = a.causal ? min(sk, qi + off + 1) : sk;
    for (uint32_t k0 = 0; k0 < kend; k0 += XB) {
        const uint32_t kc = min(static_cast<uint32_t>(XB), kend - k0);
        float sc = -__builtin_inff();
        if (lane < static_cast<int>(kc)) {
            sc = dev::dot_ref(q, Kh + static_cast<uint64_t>(k0 + lane) * hd, hd) * a.scale;
            if (Mr) sc = sc + Mr[k0 + lane];
        }
        const float bmax = dev::wave_max(sc);
        if (!isfinite(bmax)) continue;   // uniform
        const float nm = m < bmax ? bmax : m;
        const float alpha = dev::fast_expf_unfused(m - nm);
        const float p = dev::fast_expf_unfused(sc - nm);
        float psum = 0.0f;
        for (uint32_t j = 0; j < kc; ++j)
            psum = psum + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), static_cast<int>(j)));
        l = l * alpha + psum;
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] = acc[e] * alpha;
        for (uint32_t j = 0; j < kc; ++j) {
            const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), static_cast<int>(j)));
            if (pj == 0.0f) continue;
            const float *vr = Vh + static_cast<uint64_t>(k0 + j) * hd + lane;
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (lane + 64 * e < static_cast<int>(hd)) acc[e] = fmaf(vr[64 * e], pj, acc[e]);
        }
        m = nm;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int e = 0; e < E; ++e)
        if (lane + 64 * e < static_cast<int>(hd)) a.O[row * hd + lane + 64 * e] = acc[e] * inv;
}

template <int D>
__global__ __launch_bounds__(XT) __attribute__((amdgpu_waves_per_eu(1, 1))) void attn_exact_mfma_kernel(Attn a)
{
#pragma clang fp contract(off)
    using L = XL<D>;
    constexpr int NI = D / 8;    // steps of each dot chain
    constexpr int NM = L::NM;    // output instructions per key
    extern __shared__ float4 sm4[];
    float *Kt = reinterpret_cast<float *>(sm4);   // [2][64][KP]
    float *Vt = Kt + 2 * L::KTILE;               // [2][64][DV]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c32 = lane & 31;
    const uint64_t bh = blockIdx.x;
    const uint32_t sq = a.seq_q, sk = a.seq_k;
    // a constant for the sizes that fill their tile
    const uint32_t hd = D % 64 == 0 ? D : a.head_dim;
    const uint32_t off = sk > sq ? sk - sq : 0;
    const uint32_t q0 = (gridDim.y - 1 - blockIdx.y) * XQ;
    const uint32_t nq = min(static_cast<uint32_t>(XQ), sq - q0);
    const uint32_t qw0 = q0 + wave * XQW;       // the wave's first row
    const uint32_t qi = qw0 + c32;              // the lane's row
    const bool qvalid = qi < sq;
    const float *Kh = a.K + bh * sk * hd;
    const float *Vh = a.V + bh * sk * hd;
    const float *Mh = a.mask ? a.mask + bh * sq * sk : nullptr;

    const uint32_t kend = a.causal ? min(sk, q0 + nq - 1 + off + 1) : sk;   // keys of any row here
    uint32_t kend_w = 0;                                                    // keys of any row of the wave
    if (qw0 < sq) kend_w = a.causal ? min(sk, min(qw0 + XQW - 1, sq - 1) + off + 1) : sk;
    const uint32_t nblk = (kend + XB - 1) / XB;

    // The lane's byte offsets into a whole block of K and V for each of the
    // wave's copies (slots past the row read its start: they are not used),
    // computed once: a division by the pitch per copy and block, on the vector
    // ALUs that the matrix instructions share, cost 5% at head_dim 64 (248 ->
    // 236 us) and 1% at 128.
    constexpr int KW = (L::KI + 3) / 4, VW = L::VI / 4;
    uint32_t ko[KW], vo[VW];
#pragma unroll
    for (int i = 0; i < KW; ++i) {
        const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane, r = sl / L::KCH, c = sl % L::KCH;
        ko[i] = (r * hd + (c < D / 4 ? 4 * c : 0)) * 4;
    }
#pragma unroll
    for (int i = 0; i < VW; ++i) {
        const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane, r = sl / (L::DV / 4), c = sl % (L::DV / 4);
        vo[i] = (r * hd + (4 * c < D ? 4 * c : 0)) * 4;
    }
    // A block that ends past the last key repeats it, and a head_dim below D
    // is filled up with zeros (both uniform).
    auto copy = [&](uint32_t b) {
        int8_t *kd = reinterpret_cast<int8_t *>(Kt + (b & 1) * L::KTILE) + wave * 1024;
        int8_t *vd = reinterpret_cast<int8_t *>(Vt + (b & 1) * L::VTILE) + wave * 1024;
        const float *kb = Kh + static_cast<uint64_t>(b) * XB * hd, *vb = Vh + static_cast<uint64_t>(b) * XB * hd;
        if ((b + 1) * XB <= kend && hd == D) {
#pragma unroll
            for (int i = 0; i < KW; ++i)
                if (4 * i + wave < L::KI) lds::dma16_s(reinterpret_cast<const int8_t *>(kb), ko[i], kd + i * 4096);
#pragma unroll
            for (int i = 0; i < VW; ++i) lds::dma16_s(reinterpret_cast<const int8_t *>(vb), vo[i], vd + i * 4096);
            return;
        }
        const uint32_t last = kend - 1 - b * XB;
        for (int i = 0; 4 * i + wave < L::KI; ++i) {
            const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane;
            const uint32_t key = min(sl / L::KCH, last), c = sl % L::KCH;
            lds::dma16(4 * c < hd ? kb + static_cast<uint64_t>(key) * hd + 4 * c : &zero16.x, kd + i * 4096);
        }
        for (int i = 0; 4 * i + wave < L::VI; ++i) {
            const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane;
            const uint32_t key = min(sl / (L::DV / 4), last), c = sl % (L::DV / 4);
            lds::dma16(4 * c < hd ? vb + static_cast<uint64_t>(key) * hd + 4 * c : &zero16.x, vd + i * 4096);
        }
    };
    if (nblk) copy(0);

    // B operands of the score products: lane (h, c32) holds the row's
    // elements 8i + 4h .. 8i + 4h + 3 (chains 4h .. 4h + 3 at step i).
    float4 qop[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
        qop[i] = qvalid && 8 * i < static_cast<int>(hd)
                     ? *reinterpret_cast<const float4 *>(a.Q + (bh * sq + qi) * hd + 8 * i + 4 * h)
                     : make_float4(0.f, 0.f, 0.f, 0.f);

    float m = -__builtin_inff(), l = 0.0f;
    f32x32 oacc[NM];
#pragma unroll
    for (int mm = 0; mm < NM; ++mm)
#pragma unroll
        for (int r = 0; r < 32; ++r) oacc[mm][r] = 0.0f;

    for (uint32_t b = 0; b < nblk; ++b) {
        lds::wait_vmcnt<0>();
        lds::block_barrier();                  // block b's tiles are in; block b-1's buffers are free
        if (b + 1 < nblk) copy(b + 1);
        const uint32_t k0 = b * XB;
        if (k0 >= kend_w) continue;           // no row of this wave sees these keys (uniform)
        const uint32_t kc_w = min(static_cast<uint32_t>(XB), kend_w - k0);
        const float *Kb = Kt + (b & 1) * L::KTILE;
        const float *Vb = Vt + (b & 1) * L::VTILE;

        // Scores: S[t][r] is (key k0 + 32t + 8(r/4) + 4h + r%4, row qi).  Both
        // 32-key tiles are computed (a tile no row sees is masked below), so
        // the two tiles' products and sums share one scheduling region.
        float S[2][16];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            // Two passes of two chain pairs each: (0,4) and (1,5), then (2,6)
            // and (3,7); hsum256's ((c0+c4) + (c1+c5)) + ((c2+c6) + (c3+c7)).
            const float *kr = Kb + (32 * t + c32) * L::KP + 4 * h;
            float s01[16];
            f32x32 acc0, acc1;
#pragma unroll
            for (int r = 0; r < 32; ++r) acc0[r] = acc1[r] = 0.0f;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const float2 kv = *reinterpret_cast<const float2 *>(kr + 8 * i);
                acc0 = mfma1(kv.x, qop[i].x, acc0);
                acc1 = mfma1(kv.y, qop[i].y, acc1);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) s01[r] = (acc0[r] + acc0[r + 16]) + (acc1[r] + acc1[r + 16]);
#pragma unroll
            for (int r = 0; r < 32; ++r) acc0[r] = acc1[r] = 0.0f;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const float2 kv = *reinterpret_cast<const float2 *>(kr + 8 * i + 2);
                acc0 = mfma1(kv.x, qop[i].z, acc0);
                acc1 = mfma1(kv.y, qop[i].w, acc1);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r)
                S[t][r] = (s01[r] + ((acc0[r] + acc0[r + 16]) + (acc1[r] + acc1[r + 16]))) * a.scale;
        }
        // Every row of the wave sees every key of the block: no masking.
        const bool dense = qw0 + XQW <= sq && k0 + XB <= kend && (!a.causal || k0 + XB - 1 <= qw0 + off);
        if (!dense) {   // uniform
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t key = k0 + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
                    const bool valid = qvalid && key < kend && !(a.causal && key > qi + off);
                    S[t][r] = valid ? S[t][r] : -__builtin_inff();
                }
        }
        if (Mh) {   // the additive mask on the scores the row sees (uniform)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t key = k0 + 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (qvalid && key < kend && !(a.causal && key > qi + off))
                        S[t][r] = S[t][r] + Mh[static_cast<uint64_t>(qi) * sk + key];
                }
        }

        // Softmax state of the lane's row (both halves hold the same).
        float bmax = -__builtin_inff();
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) bmax = fmaxf(bmax, S[t][r]);
        {
            float b0, b1;
            halves(bmax, b0, b1);
            bmax = fmaxf(b0, b1);
        }
        const bool live = isfinite(bmax);
        const float nm = m < bmax ? bmax : m;
        const float alpha = live ? dev::fast_expf_unfused(m - nm) : 1.0f;
        if (__ballot(alpha != 1.0f)) {   // acc * 1 is acc: skipped when no row's max moved
#pragma unroll
            for (int mm = 0; mm < NM; ++mm)
#pragma unroll
                for (int r = 0; r < 32; ++r) oacc[mm][r] = oacc[mm][r] * alpha;
        }

        // Keys in groups of eight (32t + 8g .. +7); keys no row of the wave
        // sees are skipped.
        const float psum = kc_w == XB ? weights_output<D, true>(oacc, S, nm, live, kc_w, lane, Vb)
                                      : weights_output<D, false>(oacc, S, nm, live, kc_w, lane, Vb);
        if (live) {
            l = l * alpha + psum;
            m = nm;
        }
    }

    // Output: oacc[mm][r] is element 64mm + 32(r/16) + 8((r%16)/4) + 4h + r%4 of row qi.
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    bool bad = false;
#pragma unroll
    for (int mm = 0; mm < NM; ++mm)
#pragma unroll
        for (int r = 0; r < 32; ++r) {
            const float o = oacc[mm][r] * inv;
            oacc[mm][r] = o;
            const bool stored = 64 * mm + 32 * (r >> 4) + 8 * ((r & 15) >> 2) < static_cast<int>(hd);
            bad |= stored && ((o != o) || (o == 0.0f && l > 0.0f));
        }
    bad = bad && qvalid;
    if (__ballot(bad) == 0) {
        if (qvalid) {
            float *orow = a.O + (bh * sq + qi) * hd + 4 * h;
#pragma unroll
            for (int mm = 0; mm < NM; ++mm)
#pragma unroll
                for (int g = 0; g < 8; ++g) {
                    const int e = 64 * mm + 32 * (g >> 2) + 8 * (g & 3);
                    if (e < static_cast<int>(hd))
                        *reinterpret_cast<float4 *>(orow + e) = make_float4(
                            oacc[mm][4 * g], oacc[mm][4 * g + 1], oacc[mm][4 * g + 2], oacc[mm][4 * g + 3]);
                }
        }
    } else {
        for (uint32_t j = 0; j < XQW && qw0 + j < sq; ++j) exact_row_wave<D>(a, bh, qw0 + j, lane);
    }
}

// ---------------------------------------------------------------------------
// The same arithmetic with the four waves of a workgroup sharing 32 query
// rows.
// A wave's chains are sequential, so a grid of few 128-row workgroups is as
// slow as its longest row however idle the chip is.  Here the work of one
// 64-key block is split four ways instead of the rows, on the fp32 MFMA of
// four 16 x 16 blocks (v_mfma_f32_16x16x1_4b_f32, one rounding per step like
// the two-block form; lane l holds row 4(l / 16) + i, column l % 16 of block b
// in register 4b + i):
//   scores   wave w: keys 16w .. 16w + 15 by all 32 rows; block b of
//            instruction j is chain j + 4(b / 2) of rows 16(b % 2) .. + 15, so
//            hsum256's pairing is in-lane and a lane ends with four keys of
//            the two rows l % 16 and 16 + l % 16;
//   weights  wave w: its 16 keys, into LDS as [key / 4][row][4];
//   output   wave w: head elements 32w .. 32w + 31, one instruction per key:
//            block b is elements 16(b / 2) .. + 15 by rows 16(b % 2) .. + 15;
//            every wave adds the 64 weights in key order (the sum is a chain).
// Two barriers a block: after the score maxima (which also orders the copied
// tiles) and after the weights.  The next block's score chains run between the
// output chain's instructions; each chain alone would wait for itself.
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma4(float a, float b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 0);
}

// Maximum over the four lanes of equal l % 16, in each of them.
__device__ __forceinline__ float max16(float v)
{
    float lo, hi;
    halves(v, lo, hi);
    v = fmaxf(lo, hi);
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <int D>
struct XC {
    static constexpr int DV = (D + 31) / 32 * 32;      // V row pitch (floats)
    static constexpr int VTILE = XB * DV;
    static constexpr int VI = XB * DV / 4 / 64;        // wave copies per V tile
    static constexpr int PW = XB * XQW;                // floats of a block's weights
    static constexpr size_t kLds =
        static_cast<size_t>(2 * XL<D>::KTILE + 2 * VTILE + PW + 4 * XQW) * sizeof(float);
};

template <int D>
__global__ __launch_bounds__(XT) void attn_exact_coop_kernel(Attn a)
{
#pragma clang fp contract(off)
    using L = XL<D>;
    using C = XC<D>;
    constexpr int NI = D / 8;
    constexpr int KW = (L::KI + 3) / 4, VW = (C::VI + 3) / 4;   // copies per wave
    extern __shared__ float4 sm4[];
    float *Kt = reinterpret_cast<float *>(sm4);   // [2][64][KP]
    float *Vt = Kt + 2 * L::KTILE;               // [2][64][DV]
    float *P = Vt + 2 * C::VTILE;                // weights [key / 4][32 rows][4]
    float *Mx = P + C::PW;                       // [4][32] row maxima of each wave's keys

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c32 = lane & 31, c16 = lane & 15, g16 = lane >> 4;
    const uint64_t bh = blockIdx.x;
    const uint32_t sq = a.seq_q, sk = a.seq_k;
    const uint32_t hd = D % 64 == 0 ? D : a.head_dim;
    const uint32_t off = sk > sq ? sk - sq : 0;
    const uint32_t q0 = (gridDim.y - 1 - blockIdx.y) * XQW;
    const float *Kh = a.K + bh * sk * hd;
    const float *Vh = a.V + bh * sk * hd;
    const float *Mh = a.mask ? a.mask + bh * sq * sk : nullptr;
    const uint32_t kend = a.causal ? min(sk, min(q0 + XQW - 1, sq - 1) + off + 1) : sk;
    const uint32_t nblk = (kend + XB - 1) / XB;

    // The lane's byte offsets into a whole block of K and V for each of the
    // wave's copies (slots past the row read its start: they are not used).
    uint32_t ko[KW], vo[VW];
#pragma unroll
    for (int i = 0; i < KW; ++i) {
        const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane, r = sl / L::KCH, c = sl % L::KCH;
        ko[i] = (r * hd + (c < D / 4 ? 4 * c : 0)) * 4;
    }
#pragma unroll
    for (int i = 0; i < VW; ++i) {
        const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane, r = sl / (C::DV / 4), c = sl % (C::DV / 4);
        vo[i] = (r * hd + (4 * c < D ? 4 * c : 0)) * 4;
    }
    // A block that ends past the last key repeats it, and a head_dim below D
    // is filled up with zeros (both uniform).
    auto whole = [&](uint32_t b) { return (b + 1) * XB <= kend && hd == D; };
    auto copy_k = [&](uint32_t b) {
        int8_t *kd = reinterpret_cast<int8_t *>(Kt + (b & 1) * L::KTILE) + wave * 1024;
        const float *base = Kh + static_cast<uint64_t>(b) * XB * hd;
        if (whole(b)) {
#pragma unroll
            for (int i = 0; i < KW; ++i)
                if (4 * i + wave < L::KI) lds::dma16_s(reinterpret_cast<const int8_t *>(base), ko[i], kd + i * 4096);
        } else {
            for (int i = 0; 4 * i + wave < L::KI; ++i) {
                const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane;
                const uint32_t r = sl / L::KCH, c = sl % L::KCH;
                const uint32_t key = min(r, kend - 1 - b * XB);
                lds::dma16(4 * c < hd ? base + static_cast<uint64_t>(key) * hd + 4 * c : &zero16.x, kd + i * 4096);
            }
        }
    };
    auto copy_v = [&](uint32_t b) {
        int8_t *vd = reinterpret_cast<int8_t *>(Vt + (b & 1) * C::VTILE) + wave * 1024;
        const float *base = Vh + static_cast<uint64_t>(b) * XB * hd;
        if (whole(b)) {
#pragma unroll
            for (int i = 0; i < VW; ++i)
                if (4 * i + wave < C::VI) lds::dma16_s(reinterpret_cast<const int8_t *>(base), vo[i], vd + i * 4096);
        } else {
            for (int i = 0; 4 * i + wave < C::VI; ++i) {
                const uint32_t sl = static_cast<uint32_t>(4 * i + wave) * 64 + lane;
                const uint32_t c = sl % (C::DV / 4), key = min(sl / (C::DV / 4), kend - 1 - b * XB);
                lds::dma16(4 * c < hd ? base + static_cast<uint64_t>(key) * hd + 4 * c : &zero16.x, vd + i * 4096);
            }
        }
    };
    if (nblk) {
        copy_k(0);
        copy_v(0);
        if (nblk > 1) copy_k(1);
    }

    // B operands of the score products: row q0 + c32, elements 8i + 4h .. + 3
    // (a row past the last repeats it and is not stored).
    float4 qop[NI];
    {
        const float *qr = a.Q + (bh * sq + min(q0 + c32, sq - 1)) * hd + 4 * h;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            qop[i] = 8 * i < static_cast<int>(hd) ? *reinterpret_cast<const float4 *>(qr + 8 * i)
                                                  : make_float4(0.f, 0.f, 0.f, 0.f);
    }

    const bool writes = 32 * wave < static_cast<int>(hd);   // the wave has head elements
    float m[2] = {-__builtin_inff(), -__builtin_inff()};    // rows q0 + c16, q0 + 16 + c16
    float l = 0.0f;                                         // row q0 + c32
    f32x16 oacc, sacc[4];
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[r] = 0.0f;

    // A whole block's output chain (OUT) with the next block's score chains
    // threaded through it.  Eight keys at a time, the LDS operands of the next
    // eight read before this group's instructions: reads issued where they are
    // used stall the chain for an LDS round trip each.
    auto phase = [&](auto out, auto score, const float *vr, const float *kr, int kc, float &psum) {
        constexpr bool OUT = decltype(out)::value, SCORE = decltype(score)::value;
        constexpr int NS = (NI + 7) / 8;      // score steps per group
        const float *pr = P + 4 * c32;
        float4 p4[2][2], k4[2][NS];
        float v8[2][8];
        if constexpr (SCORE) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) sacc[j][r] = 0.0f;
        }
        auto load = [&](int q) {
            if constexpr (OUT) {
#pragma unroll
                for (int u = 0; u < 2; ++u) p4[q & 1][u] = *reinterpret_cast<const float4 *>(pr + (2 * q + u) * 4 * XQW);
#pragma unroll
                for (int j = 0; j < 8; ++j) v8[q & 1][j] = vr[(8 * q + j) * C::DV];
            }
#pragma unroll
            for (int i = 0; i < (SCORE ? NS : 0); ++i)
                if (NS * q + i < NI) k4[q & 1][i] = *reinterpret_cast<const float4 *>(kr + 8 * (NS * q + i));
        };
        load(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (!SCORE && 8 * q >= kc) break;   // the weights past the last key are zeros
            __builtin_amdgcn_sched_barrier(0);
            if (q < 7) load(q + 1);
            __builtin_amdgcn_sched_barrier(0);
            const float *p = reinterpret_cast<const float *>(p4[q & 1]);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if constexpr (OUT) {
                    psum = psum + p[j];
                    oacc = mfma4(v8[q & 1][j], p[j], oacc);
                }
                // one score instruction after each, two where a group has two steps
#pragma unroll
                for (int u = 0; u < (SCORE ? 4 * NS : 0); ++u)
                    if (u * 8 / (4 * NS) == j && NS * q + u / 4 < NI) {
                        const int i = NS * q + u / 4;
                        const float *kv = reinterpret_cast<const float *>(&k4[q & 1][u / 4]);
                        const float *qv = reinterpret_cast<const float *>(&qop[i]);
                        sacc[u % 4] = mfma4(kv[u % 4], qv[u % 4], sacc[u % 4]);
                    }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto k_row = [&](uint32_t b) { return Kt + (b & 1) * L::KTILE + (16 * wave + c16) * L::KP + 4 * h; };
    if (nblk) {
        lds::wait_vmcnt<0>();
        lds::block_barrier();
        float none = 0.0f;
        phase(std::false_type{}, std::true_type{}, Vt, k_row(0), XB, none);
    }

    for (uint32_t b = 0; b < nblk; ++b) {
        const uint32_t k0 = b * XB;
        // S[u][i]: key k0 + 16 wave + 4 g16 + i, row q0 + 16u + c16.
        float S[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 4 * u + i;
                S[u][i] = (((sacc[0][r] + sacc[0][r + 8]) + (sacc[1][r] + sacc[1][r + 8])) +
                           ((sacc[2][r] + sacc[2][r + 8]) + (sacc[3][r] + sacc[3][r + 8]))) * a.scale;
            }
        // Every row sees every key of the block: no masking (uniform).
        if (Mh || !(q0 + XQW <= sq && k0 + XB <= kend && (!a.causal || k0 + XB - 1 <= q0 + off))) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t key = k0 + 16 * wave + 4 * g16 + i, qi = q0 + 16 * u + c16;
                    const bool valid = qi < sq && key < kend && !(a.causal && key > qi + off);
                    if (Mh && valid) S[u][i] = S[u][i] + Mh[static_cast<uint64_t>(qi) * sk + key];
                    S[u][i] = valid ? S[u][i] : -__builtin_inff();
                }
        }
        float bmax[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
            bmax[u] = max16(fmaxf(fmaxf(S[u][0], S[u][1]), fmaxf(S[u][2], S[u][3])));
        if (h == 0) Mx[wave * XQW + c32] = g16 ? bmax[1] : bmax[0];
        lds::wait_vmcnt<0>();
        lds::block_barrier();                  // maxima, K of b + 1 and V of b are in; the other tiles are free
        float w[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) w[u][i] = Mx[i * XQW + 16 * u + c16];
        if (b + 1 < nblk) copy_v(b + 1);
        if (b + 2 < nblk) copy_k(b + 2);
        float alpha[2];
        bool live[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            // a wave whose keys are all NaN is left out, as by fmaxf
            const float bm = fmaxf(-__builtin_inff(), fmaxf(fmaxf(w[u][0], w[u][1]), fmaxf(w[u][2], w[u][3])));
            live[u] = isfinite(bm);
            const float nm = m[u] < bm ? bm : m[u];
            alpha[u] = live[u] ? dev::fast_expf_nonpos(m[u] - nm) : 1.0f;
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = live[u] ? dev::fast_expf_nonpos(S[u][i] - nm) : 0.0f;
            reinterpret_cast<float4 *>(P)[(4 * wave + g16) * XQW + 16 * u + c16] = make_float4(e[0], e[1], e[2], e[3]);
            if (live[u]) m[u] = nm;
        }
        if (__ballot(alpha[0] != 1.0f || alpha[1] != 1.0f)) {   // acc * 1 is acc
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[r] = oacc[r] * alpha[(r >> 2) & 1];
        }
        lds::block_barrier();                  // the block's weights are in

        // Every branch here is uniform; a block with one after it is whole.
        float psum = 0.0f;
        const float *vr = Vt + (b & 1) * C::VTILE + 32 * wave + 16 * h + c16;
        const bool more = b + 1 < nblk;
        if (more && writes) phase(std::true_type{}, std::true_type{}, vr, k_row(b + 1), XB, psum);
        else if (more) phase(std::false_type{}, std::true_type{}, vr, k_row(b + 1), XB, psum);
        else if (writes) phase(std::true_type{}, std::false_type{}, vr, vr, static_cast<int>(kend - k0), psum);
        const bool odd = g16 & 1;              // l is of row c32
        l = (odd ? live[1] : live[0]) ? l * (odd ? alpha[1] : alpha[0]) + psum : l;
    }

    // oacc[4q + i]: element 32 wave + 16(q / 2) + 4 g16 + i of row 16(q % 2) + c16.
    const float l0 = __shfl(l, c16, 64), l1 = __shfl(l, 16 + c16, 64);
    const float i0 = l0 > 0.0f ? 1.0f / l0 : 0.0f, i1 = l1 > 0.0f ? 1.0f / l1 : 0.0f;
    const uint32_t e0 = 32 * wave + 4 * g16;
    bool bad = false;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const bool odd = (r >> 2) & 1;
        const float o = oacc[r] * (odd ? i1 : i0);
        oacc[r] = o;
        const bool stored = q0 + 16 * odd + c16 < sq && e0 + 16 * (r >> 3) < hd;
        bad |= stored && ((o != o) || (o == 0.0f && (odd ? l1 : l0) > 0.0f));
    }
    bool again = __ballot(bad) != 0;
    const bool in_place = a.O == a.Q;
    if (in_place) {
        // The rows are read again: no wave may store its part before all know,
        // and one wave recomputes a row.  (The maxima in Mx were read before the
        // last barrier.)  0.1 to 0.3 us, so not where O is elsewhere.
        if (lane == 0) Mx[wave] = again ? 1.0f : 0.0f;
        lds::block_barrier();
        again = Mx[0] + Mx[1] + Mx[2] + Mx[3] != 0.0f;
    }
    if (!again) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t row = q0 + 16 * (q & 1) + c16, e = e0 + 16 * (q >> 1);
            if (row < sq && e < hd)
                *reinterpret_cast<float4 *>(a.O + (bh * sq + row) * hd + e) =
                    make_float4(oacc[4 * q], oacc[4 * q + 1], oacc[4 * q + 2], oacc[4 * q + 3]);
        }
    } else {
        for (uint32_t j = in_place ? wave : 0; j < XQW && q0 + j < sq; j += in_place ? 4 : 1)
            exact_row_wave<D>(a, bh, q0 + j, lane);
    }
}

// Time of a grid of workgroups of `rows` query rows in 64-key blocks: the
// longest workgroup's, or an even share of them all per CU, where a workgroup
// costs `start` blocks besides its own.
double grid_blocks(const Attn &a, uint32_t rows, double start)
{
    const uint64_t off = a.seq_k > a.seq_q ? a.seq_k - a.seq_q : 0;
    auto blocks = [&](uint64_t last) {   // of the workgroup whose last row is `last`
        const uint64_t keys = a.causal ? std::min<uint64_t>(a.seq_k, last + off + 1) : a.seq_k;
        return static_cast<double>((keys + XB - 1) / XB);
    };
    const double longest = blocks(a.seq_q - 1) + start, shortest = blocks(std::min(rows, a.seq_q) - 1) + start;
    const double groups = static_cast<double>(a.batch) * a.heads * ((a.seq_q + rows - 1) / rows);
    return std::max(longest, groups * (longest + shortest) / 2 / cu_count());
}

// Whether 32-row workgroups finish first.  At head_dim 128 a 64-key block
// costs a 128-row workgroup 11.5 us and a 32-row one 4.1, and starting and
// storing about 5 us either (head_dim 64: 7.3, 2.6 and 4): a 32-row workgroup
// is a third as long but a quarter of the rows, so it wins where the grid does
// not fill the chip.  8 heads, 256 rows, 2000 keys: 351 -> 120 us; 32 heads x
// 512^2 95 -> 44, x 1024^2 182 -> 143, x 2048^2 392 against 540.
bool share_rows(const Attn &a) { return 4.1 * grid_blocks(a, XQW, 1.2) < 11.5 * grid_blocks(a, XQ, 0.45); }

template <int D>
void launch(hipStream_t s, const Attn &a)
{
    using L = XL<D>;
    static std::atomic<bool> lds_optin{false};
    if (!lds_optin)
        lds_optin = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_exact_mfma_kernel<D>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(L::kLds)) == hipSuccess &&
                    hipFuncSetAttribute(reinterpret_cast<const void *>(attn_exact_coop_kernel<D>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(XC<D>::kLds)) == hipSuccess;
    const uint32_t bh = a.batch * a.heads;
    if (share_rows(a))
        attn_exact_coop_kernel<D><<<dim3(bh, (a.seq_q + XQW - 1) / XQW), XT, XC<D>::kLds, s>>>(a);
    else
        attn_exact_mfma_kernel<D><<<dim3(bh, (a.seq_q + XQ - 1) / XQ), XT, L::kLds, s>>>(a);
}

// ---------------------------------------------------------------------------
// Reference-order decode.  In attention_range only the output
// chain is sequential over keys; the scores are independent per key and the
// chain is independent per head element.  So decode runs as two kernels:
//   attn_dec_scores  s[row][key] = dot_avx2(q_row, k_key) * scale, then -inf
//                    for a causally masked key or + mask, every key in
//                    parallel (one lane per key running its eight chains);
//   attn_dec_chain   one wave per (row, 64 head elements): per 64-key block
//                    the block max, m, alpha and the weights from the saved
//                    scores (every wave of a row derives the same ones), the
//                    weight sum and acc = fma(v_j, p_j, acc) in key order for
//                    p_j != 0, with the V slices and the scores of the next
//                    three blocks copied from HBM into LDS meanwhile.
// The scores live in a workspace of rows x pitch floats (pitch = seq_k
// rounded up to 64); calls whose scores exceed kDecScoreCap run over
// consecutive (batch, head) ranges.
// ---------------------------------------------------------------------------
constexpr uint32_t DTPW = 4;                // 64-key K tiles per scores wave at most
constexpr int DNB = 4;                      // blocks in flight per chain wave
constexpr int DTV = XB * 64;                // floats per V tile (64 keys x 64 head elements)
constexpr int DOPS = 17;                    // copies per block: 16 of V, one of scores
constexpr size_t kDecLds = static_cast<size_t>(DNB) * (DTV + XB) * sizeof(float) + XB * sizeof(float);
constexpr uint64_t kDecScoreCap = 32ull << 20;
constexpr uint32_t kDecMaxRows = 8;           // query rows per (batch, head) that decode takes

uint32_t dec_pitch(const Attn &a) { return (a.seq_k + XB - 1) / XB * XB; }
// Score bytes of one (batch, head).
uint64_t dec_scores_bytes(const Attn &a) { return static_cast<uint64_t>(a.seq_q) * dec_pitch(a) * sizeof(float); }

template <int D>
size_t dec_scores_lds(uint32_t sq) { return (static_cast<size_t>(XB) * XL<D>::KP + sq * D) * sizeof(float); }

// Maximum over the wave's 64 lanes, in every lane (order-free: NaN operands
// are ignored as by fmaxf, and the sign of a zero maximum never matters).
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_f(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(x), __float_as_int(x), CTRL, ROWS, 0xf, false));
}

__device__ __forceinline__ float wave_max_dpp(float v)
{
    v = fmaxf(v, dpp_f<0xB1, 0xf>(v));    // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_f<0x4E, 0xf>(v));    // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_f<0x141, 0xf>(v));   // row_half_mirror
    v = fmaxf(v, dpp_f<0x140, 0xf>(v));   // row_mirror: every lane holds its row's max
    v = fmaxf(v, dpp_f<0x142, 0xa>(v));   // row_bcast15 into rows 1 and 3
    v = fmaxf(v, dpp_f<0x143, 0xc>(v));   // row_bcast31 into rows 2 and 3: lane 63 holds the max
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Scores: one wave per (batch, head) and tpw tiles of 64 keys (four such
// workgroups per CU by LDS); the wave copies a tile's K rows into LDS (row
// pitch D + 4 floats: lane j's 16-byte reads of key j are conflict-free) and
// lane j runs key j's eight chains for every query row (the rows' elements
// as broadcast reads).
template <int D>
__global__ __launch_bounds__(64) void attn_dec_scores(Attn a, float *S, uint32_t pitch, uint32_t tpw)
{
#pragma clang fp contract(off)
    using L = XL<D>;
    constexpr int NI = D / 8;
    extern __shared__ float4 sm4[];
    const int lane = threadIdx.x;
    float *Kt = reinterpret_cast<float *>(sm4);          // [64][KP]
    float *Qs = Kt + XB * L::KP;                         // [sq][D]
    const uint64_t bh = blockIdx.y;
    const uint32_t sq = a.seq_q, sk = a.seq_k;
    const uint32_t hd = D % 64 == 0 ? D : a.head_dim;
    const uint32_t off = sk > sq ? sk - sq : 0;
    const float *Kh = a.K + bh * sk * hd;
    for (uint32_t r = 0; r < sq; ++r)
        for (uint32_t i = lane; i < D; i += 64) Qs[r * D + i] = i < hd ? a.Q[(bh * sq + r) * hd + i] : 0.0f;
    __syncthreads();
    const uint32_t t0 = blockIdx.x * tpw;
    for (uint32_t tt = 0; tt < tpw; ++tt) {
        const uint32_t k0 = (t0 + tt) * XB;
        if (k0 >= sk) break;   // uniform over the wave; no barrier follows
        for (int i = 0; i < L::KCH; ++i) {
            const uint32_t sl = static_cast<uint32_t>(i) * 64 + lane;
            const uint32_t r = sl / L::KCH, c = sl % L::KCH;
            const uint32_t key = min(k0 + r, sk - 1);
            const float *src = Kh + static_cast<uint64_t>(key) * hd + (c < D / 4 ? 4 * c : 0);
            if (D % 64 != 0 && 4 * c >= hd) src = &zero16.x;
            lds::dma16_nt(src, reinterpret_cast<int8_t *>(Kt) + i * 1024);
        }
        lds::wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        const uint32_t key = k0 + lane;
        const float *kr = Kt + lane * L::KP;
        for (uint32_t r = 0; r < sq; ++r) {
            const float *qr = Qs + r * D;
            float c8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const float4 ka = *reinterpret_cast<const float4 *>(kr + 8 * i);
                const float4 kb = *reinterpret_cast<const float4 *>(kr + 8 * i + 4);
                const float4 qa = *reinterpret_cast<const float4 *>(qr + 8 * i);
                const float4 qb = *reinterpret_cast<const float4 *>(qr + 8 * i + 4);
                c8[0] = fmaf(qa.x, ka.x, c8[0]);
                c8[1] = fmaf(qa.y, ka.y, c8[1]);
                c8[2] = fmaf(qa.z, ka.z, c8[2]);
                c8[3] = fmaf(qa.w, ka.w, c8[3]);
                c8[4] = fmaf(qb.x, kb.x, c8[4]);
                c8[5] = fmaf(qb.y, kb.y, c8[5]);
                c8[6] = fmaf(qb.z, kb.z, c8[6]);
                c8[7] = fmaf(qb.w, kb.w, c8[7]);
            }
            const float dot = ((c8[0] + c8[4]) + (c8[1] + c8[5])) + ((c8[2] + c8[6]) + (c8[3] + c8[7]));
            const uint64_t row = bh * sq + r;
            if (key < sk) {
                float sc = dot * a.scale;
                if (a.causal && key > r + off) sc = -__builtin_inff();
                else if (a.mask) sc = sc + a.mask[row * sk + key];
                S[row * pitch + key] = sc;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the tile is read before the next copy
    }
}

// Output chain: one wave per (row, 64 head elements).
template <int D>
__global__ __launch_bounds__(64) void attn_dec_chain(Attn a, const float *S, uint32_t pitch)
{
#pragma clang fp contract(off)
    extern __shared__ float4 sm4[];
    float *Vt = reinterpret_cast<float *>(sm4);   // [DNB][64 keys][64]
    float *St = Vt + DNB * DTV;                   // [DNB][64] scores
    float *Pw = St + DNB * XB;                    // [64] weights of the current block
    const int lane = threadIdx.x;
    const uint64_t row = blockIdx.x;
    const uint32_t sq = a.seq_q, sk = a.seq_k;
    const uint32_t hd = D % 64 == 0 ? D : a.head_dim;
    const uint32_t e0 = blockIdx.y * 64;          // the wave's head elements e0 .. e0 + 63
    const uint32_t off = sk > sq ? sk - sq : 0;
    const uint64_t bh = row / sq;
    const uint32_t qi = static_cast<uint32_t>(row % sq);
    const uint32_t kend = a.causal ? min(sk, qi + off + 1) : sk;
    const uint32_t nblk = (kend + XB - 1) / XB;
    const float *Vh = a.V + bh * sk * hd + e0;
    const float *Sr = S + row * pitch;

    // Block t's copies: 16 of four keys x 64 head elements each, then the
    // block's 64 scores by lanes 0-15 (the row pitch keeps them in the row).
    auto copy = [&](uint32_t t) {
        int8_t *vd = reinterpret_cast<int8_t *>(Vt + (t % DNB) * DTV);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const uint32_t key = min(t * XB + 4 * u + (lane >> 4), kend - 1);
            const float *src = Vh + static_cast<uint64_t>(key) * hd + 4 * (lane & 15);
            lds::dma16_nt(D % 64 == 0 || e0 + 4 * (lane & 15) < hd ? src : &zero16.x, vd + u * 1024);
        }
        if (lane < 16) lds::dma16(Sr + t * XB + 4 * lane, reinterpret_cast<int8_t *>(St + (t % DNB) * XB));
    };
    for (uint32_t t = 0; t < DNB - 1 && t < nblk; ++t) copy(t);

    float m = -__builtin_inff(), l = 0.0f, acc = 0.0f;
    for (uint32_t t = 0; t < nblk; ++t) {
        if (t + DNB - 1 < nblk) {
            copy(t + DNB - 1);
            lds::wait_vmcnt<DOPS * (DNB - 1)>();
        } else {
            lds::wait_vmcnt<0>();
        }
        asm volatile("" ::: "memory");
        const uint32_t k0 = t * XB, kc = min(static_cast<uint32_t>(XB), kend - k0);
        const float *vt = Vt + (t % DNB) * DTV + lane;
        const float sc = lane < static_cast<int>(kc) ? St[(t % DNB) * XB + lane] : -__builtin_inff();
        const float bmax = wave_max_dpp(sc);
        if (isfinite(bmax)) {   // uniform
            const float nm = m < bmax ? bmax : m;
            const float alpha = dev::fast_expf_unfused(m - nm);
            const float p = dev::fast_expf_unfused(sc - nm);   // 0 past kc
            Pw[lane] = p;
            const uint64_t nz = __ballot(p != 0.0f);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            float psum = 0.0f;
            acc = acc * alpha;
            if (kc == XB && nz == ~0ull) {
                // Every weight of a whole block is nonzero: the chains without
                // a test, every read of the block issued up front.
                float v[XB], pj[XB];
#pragma unroll
                for (int j = 0; j < XB; j += 4) {
                    const float4 w4 = *reinterpret_cast<const float4 *>(Pw + j);
                    pj[j] = w4.x; pj[j + 1] = w4.y; pj[j + 2] = w4.z; pj[j + 3] = w4.w;
                }
#pragma unroll
                for (int j = 0; j < XB; ++j) v[j] = vt[j * 64];
#pragma unroll
                for (int j = 0; j < XB; ++j) {
                    psum = psum + pj[j];
                    acc = fmaf(v[j], pj[j], acc);
                }
            } else {
                for (uint32_t j = 0; j < kc; j += 4) {
                    const float4 w4 = *reinterpret_cast<const float4 *>(Pw + j);
                    const float pq[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (j + u < kc) psum = psum + pq[u];
                        if ((nz >> (j + u)) & 1ull) acc = fmaf(vt[(j + u) * 64], pq[u], acc);
                    }
                }
            }
            l = l * alpha + psum;
            m = nm;
        }
        // This wave's reads of slot t % DNB are done before block t + DNB's
        // copies land in it.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    if (D % 64 == 0 || e0 + lane < hd) a.O[row * hd + e0 + lane] = acc * inv;
}

template <int D>
void launch_decode(hipStream_t s, const Attn &a, float *ws)
{
    static std::atomic<bool> lds_optin{false};
    if (!lds_optin)
        lds_optin = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_dec_chain<D>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(kDecLds)) == hipSuccess &&
                    hipFuncSetAttribute(reinterpret_cast<const void *>(attn_dec_scores<D>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(dec_scores_lds<D>(kDecMaxRows))) == hipSuccess;
    const uint32_t pitch = dec_pitch(a);
    const uint64_t per_bh = dec_scores_bytes(a);
    const uint64_t nbh = static_cast<uint64_t>(a.batch) * a.heads;
    const uint64_t step = std::max<uint64_t>(1, kDecScoreCap / per_bh);
    for (uint64_t b0 = 0; b0 < nbh; b0 += step) {
        const uint32_t n = static_cast<uint32_t>(std::min(step, nbh - b0));
        Attn c = a;   // the (batch, head) range [b0, b0 + n) as a batch of n single heads
        const uint64_t qo = b0 * a.seq_q * a.head_dim, ko = b0 * a.seq_k * a.head_dim;
        c.Q = a.Q + qo; c.K = a.K + ko; c.V = a.V + ko; c.O = a.O + qo;
        c.mask = a.mask ? a.mask + b0 * a.seq_q * a.seq_k : nullptr;
        c.batch = n;
        c.heads = 1;
        const uint32_t tiles = (a.seq_k + XB - 1) / XB;
        // As many tiles a wave as make one round of the workgroups that LDS lets the
        // CUs hold: with more, the waves of a short context take their tiles in turn
        // on an idle chip, with fewer a second round runs part empty (64 heads x 2
        // rows of 4000 keys at head_dim 128: three a wave 99.9 us, four 95).
        const size_t lds = dec_scores_lds<D>(a.seq_q);
        const uint64_t slots = 160 * 1024 / lds * cu_count();
        const uint32_t tpw = static_cast<uint32_t>(std::min<uint64_t>(DTPW, (static_cast<uint64_t>(tiles) * n + slots - 1) / slots));
        attn_dec_scores<D><<<dim3((tiles + tpw - 1) / tpw, n), 64, lds, s>>>(c, ws, pitch, tpw);
        attn_dec_chain<D><<<dim3(n * a.seq_q, XL<D>::NM), 64, kDecLds, s>>>(c, ws, pitch);
    }
}

// The smallest tile of head elements that takes head_dim (at most 128); the
// tiles of 64 and 128 take exactly that head_dim.
template <typename F>
void with_tile(uint32_t head_dim, F &&f)
{
    if (head_dim <= 32) f(std::integral_constant<int, 32>{});
    else if (head_dim <= 56) f(std::integral_constant<int, 56>{});
    else if (head_dim <= 64) f(std::integral_constant<int, 64>{});
    else if (head_dim <= 80) f(std::integral_constant<int, 80>{});
    else if (head_dim <= 96) f(std::integral_constant<int, 96>{});
    else if (head_dim <= 120) f(std::integral_constant<int, 120>{});
    else f(std::integral_constant<int, 128>{});
}

bool aligned16(const Attn &a)
{
    for (const float *p : {a.Q, a.K, a.V, static_cast<const float *>(a.O)})
        if (reinterpret_cast<uintptr_t>(p) % 16) return false;
    return true;
}

// Up to kDecMaxRows rows run as decode or in the 32-row workgroups; the two
// times, us, fitted to both kernels over 1 to 300 (batch, head) pairs, 1 to 8
// rows, 8 to 5000 keys and all head sizes (of 1017 calls the rule takes the
// side that is more than 5% slower for 7; 96 pairs x 4 rows x 4000 keys at
// head_dim 128 204 against 259, 256 pairs x 4 x 1500 182 against 112).
//
// Decode: two launches, K from memory once, and rounds of the chains that fit
// the chip (two per CU), each longer as they share the CUs.
double decode_us(const Attn &a)
{
    const bool small = a.head_dim <= 64;
    const double pairs = static_cast<double>(a.batch) * a.heads, cus = cu_count();
    const double chains = pairs * a.seq_q * ((a.head_dim + 63) / 64);
    const double load = std::min(1.0, std::max(0.0, (chains / cus - 0.5) / 1.5));
    const double block = small ? 1.0 + 0.4 * load : 0.95 + 0.6 * load;
    return (small ? 6.7 : 8.3) + 0.6 * a.seq_q + std::ceil(chains / (2 * cus)) * a.seq_k / XB * block +
           pairs * a.seq_k * a.head_dim * sizeof(float) * 0.14e-6;
}

// 32-row workgroups: one for each pair, its blocks in turn; a second one on a
// CU costs as much again where LDS holds one (head_dim above 64), else half; at
// the largest head sizes a full chip waits for memory as well.
double few_rows_us(const Attn &a)
{
    const bool small = a.head_dim <= 64;
    const double fill = static_cast<double>(a.batch) * a.heads / cu_count();
    const double block = small ? 3.05 : a.head_dim <= 96 ? 4.0 : 4.0 + 0.35 * std::min(1.0, fill);
    return 3.5 + block * ((a.seq_k + XB - 1) / XB) * (1.0 + (std::ceil(fill) - 1.0) * (small ? 0.55 : 1.0));
}

}  // namespace

bool attention_exact_supported(const Attn &a)
{
    if (a.head_dim == 64 || a.head_dim == 128) return true;
    if (a.head_dim % 8 || a.head_dim > 128) return false;
    if (!aligned16(a)) return false;
    // a handful of keys and few rows: the general kernel's one pass over them
    // (4 heads of 32 x 4 rows, 8 keys, head_dim 80 5.4 us against 6.5)
    if (a.seq_k <= 12 && static_cast<uint64_t>(a.batch) * a.heads * a.seq_q <= 1024) return false;
    return a.seq_q > 4 || dec_scores_bytes(a) <= kDecScoreCap;
}

bool attention_exact_decodes(const Attn &a)
{
    if (a.seq_q <= 4 && !aligned16(a)) return true;   // the chains read Q and write O by dwords
    // Where the workspace is shared with calls on other streams, which race for
    // it, only the rows that have always taken it do (the output is the same).
    if (!a.own_ws && !(a.seq_q <= 4 && (a.head_dim == 64 || a.head_dim == 128))) return false;
    return a.seq_q <= kDecMaxRows && (a.seq_q <= 4 || dec_scores_bytes(a) <= kDecScoreCap) &&
           decode_us(a) < few_rows_us(a);
}

double attention_exact_us(const Attn &a)
{
    if (attention_exact_decodes(a)) return decode_us(a);
    // share_rows' estimates, 4.1 and 11.5 us a block at head_dim 128; a mask's loads
    // stand in each block's way (64 heads of 48, 21 rows, 1500 keys 109 us)
    double t = (a.head_dim <= 64 ? 3.05 : 4.0) * std::min(grid_blocks(a, XQW, 1.2), 2.8 * grid_blocks(a, XQ, 0.45));
    if (a.seq_q <= kDecMaxRows) t = std::max(t, few_rows_us(a));
    return a.mask ? 1.15 * t : t;
}

const char *attention_exact_route(const Attn &a)
{
    return attention_exact_decodes(a) ? "exact_decode" : share_rows(a) ? "exact_rows32" : "exact_rows128";
}

void attention_exact_prefill(hipStream_t s, const Attn &a)
{
    with_tile(a.head_dim, [&](auto d) { launch<decltype(d)::value>(s, a); });
}

size_t attention_exact_decode_ws_bytes(const Attn &a)
{
    const uint64_t per_bh = dec_scores_bytes(a);
    const uint64_t nbh = static_cast<uint64_t>(a.batch) * a.heads;
    const uint64_t step = std::max<uint64_t>(1, kDecScoreCap / per_bh);
    return static_cast<size_t>(std::min(step, nbh) * per_bh);
}

void attention_exact_decode(hipStream_t s, const Attn &a, float *ws)
{
    with_tile(a.head_dim, [&](auto d) { launch_decode<decltype(d)::value>(s, a, ws); });
}

}  // namespace k
}  // namespace vnpu
