// skinny_f32.hip - MATMUL_F32 and MTP_HEAD_F32 with few rows: one read of B at
// the memory's rate; and, up to 2048 rows, small weights and rows that are not
// 16-byte aligned (the rules are at plan()).
//
// Replaces the reference's f32 decode kernels (src/kernels/kernels.cpp:454-520)
// and, for an output head, execute_mtp_head (src/core/scheduler.cpp:610-641).
//
// Design (HBM-bound: 4 K N bytes of weights, each used M times):
//   * v_mfma_f32_16x16x4_f32 does the products: full f32, and at 157 TFLOP/s
//     16 rows take a third of the time that their weights take to arrive, so
//     the vector ALUs and the 4 M multiplications per weight are out of the way;
//   * a workgroup of W waves owns 16 CB columns over all of K, wave w the
//     chunks w, w + W, ... of 16 U depths; the waves' sums meet in LDS, in wave
//     order, so the result does not depend on timing; narrow outputs split K
//     over workgroups as well, added in order by a second launch;
//   * lane 16g + c multiplies depths 16u + 4g .. + 3: four consecutive
//     floats of one row of A, and of B
//       stored [N][K]: four consecutive floats of row (column of the output) c,
//       one 16-byte load; a wave reads 64 U bytes in a run of each of 16 CB rows;
//       stored [K][N]: CB consecutive columns of each of the four depths; a
//       wave reads 64 CB bytes in a run of each of 16 U rows;
//   * both operands come straight from memory (A from L2), the next chunk's
//     loads issued before this chunk's products; raw buffers return zero past
//     the matrix, so there are no branches around loads.
#include "kernels.hpp"
#include "device_math.hpp"

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <type_traits>

namespace vnpu {
namespace k {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBufferWord3 = 0x00020000;  // raw buffer, 32-bit data format
constexpr int kNontemporal = 2;           // B is read once
constexpr uint32_t kOut = 0x80000000u;    // an offset past any buffer

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const float *p, uint64_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0,
                                             static_cast<int>(bytes < 0x7fffffffull ? bytes : 0x7fffffffull),
                                             kBufferWord3);
}

template <int V, int POLICY>
__device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t off, float *v)
{
    if constexpr (V == 4) {
        const float4 t = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, POLICY));
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else if constexpr (V == 2) {
        const float2 t = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, POLICY));
        v[0] = t.x; v[1] = t.y;
    } else {
        v[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, POLICY));
    }
}

__device__ __forceinline__ void store_out(const F32Gemm &p, uint32_t m, uint32_t n, float v)
{
    float *dst = p.C + static_cast<uint64_t>(m) * p.ldc + n;
    float out = p.alpha * v;
    if (p.bias) out += p.bias[n];
    if (p.beta != 0.0f) out += p.beta * *dst;
    *dst = dev::epilogue(out, p.epilogue);
}

// MG groups of 16 rows (from row 16 MG blockIdx.z on), CB blocks of 16 columns,
// NT: B stored [N][K].  Loads of four floats need no more than 4-byte
// alignment.  The last K % 4 depths, which a vector would run past (what
// follows them may be NaN), are one step of their own; a vector that runs past
// N only feeds columns that are not stored.
template <int MG, int CB, bool NT, int W, int U>
__global__ __launch_bounds__(64 * W) void skinny_f32_kernel(F32Gemm p, uint32_t k_per_split, float *ws)
{
    extern __shared__ float red[];   // [W][16 MG][16 CB]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const uint32_t n0 = blockIdx.x * (16 * CB);

    const uint32_t K4 = p.K & ~3u;
    const uint32_t m0 = blockIdx.z * (16 * MG), mrows = min(16u * MG, p.M - m0);
    const auto ra = buffer(p.A + static_cast<uint64_t>(m0) * p.lda, (static_cast<uint64_t>(mrows - 1) * p.lda + p.K) * 4);
    uint32_t arow[MG], brow[CB];
#pragma unroll
    for (int m = 0; m < MG; ++m) arow[m] = min(16u * m + c, mrows - 1) * p.lda;   // rows past M are not stored
    if constexpr (NT) {
#pragma unroll
        for (int b = 0; b < CB; ++b) brow[b] = min(16u * b + c, p.N - 1 - n0) * p.ldb;
    }
    const uint32_t ncol = n0 + CB * c < p.N ? CB * c * 4 : kOut;
    const auto rt = buffer(p.B + static_cast<uint64_t>(n0) * p.ldb,
                           (static_cast<uint64_t>(min(16u * CB, p.N - n0) - 1) * p.ldb + p.K) * 4);

    // One chunk's operands: a[u][m][s] and b[u][..] of depth kc + 16u + 4g + s.
    struct Chunk {
        float a[U][MG][4];
        float b[U][NT ? CB : 4][NT ? 4 : CB];
    };
    auto fetch = [&](Chunk &t, uint32_t kc) {
        const auto rn = buffer(p.B + static_cast<uint64_t>(kc < K4 ? kc : 0) * p.ldb + n0,
                               kc < K4 ? (static_cast<uint64_t>(K4 - kc - 1) * p.ldb + (p.N - n0)) * 4 : 0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t k = kc + 16 * u + 4 * g;
            if constexpr (NT) {
#pragma unroll
                for (int b = 0; b < CB; ++b)
                    load<4, kNontemporal>(rt, k < K4 ? (brow[b] + k) * 4 : kOut, t.b[u][b]);
            } else {
                // rows past K4 lie past the buffer's end
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    load<CB, kNontemporal>(rn, ncol + (16 * u + 4 * g + s) * p.ldb * 4, t.b[u][s]);
            }
#pragma unroll
            for (int m = 0; m < MG; ++m) load<4, 0>(ra, k < K4 ? (arow[m] + k) * 4 : kOut, t.a[u][m]);
        }
    };
    f32x4 acc[MG][CB];
#pragma unroll
    for (int m = 0; m < MG; ++m)
#pragma unroll
        for (int b = 0; b < CB; ++b) acc[m][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Chunk &t) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int b = 0; b < CB; ++b)
#pragma unroll
                    for (int m = 0; m < MG; ++m)
                        acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(t.a[u][m][s], NT ? t.b[u][b][s] : t.b[u][s][b],
                                                                         acc[m][b], 0, 0, 0);
    };
    const uint32_t kb = blockIdx.y * k_per_split, ke = min(K4, kb + k_per_split);
    constexpr uint32_t step = 16 * U * W;
    Chunk x, y;
    uint32_t kc = kb + 16 * U * wave;
    if (kc < ke) fetch(x, kc);
    for (; kc < ke; kc += 2 * step) {
        fetch(y, kc + step < ke ? kc + step : K4);
        multiply(x);
        if (kc + step >= ke) break;
        fetch(x, kc + 2 * step < ke ? kc + 2 * step : K4);
        multiply(y);
    }

    if (K4 < p.K && blockIdx.y + 1 == gridDim.y && wave == W - 1) {   // uniform
        const uint32_t k = K4 + g;
        const auto rl = buffer(p.B + static_cast<uint64_t>(K4) * p.ldb + n0,
                               NT ? 0 : (static_cast<uint64_t>(p.K - 1 - K4) * p.ldb + (p.N - n0)) * 4);
        float a[MG], b[CB];
#pragma unroll
        for (int m = 0; m < MG; ++m) load<1, 0>(ra, k < p.K ? (arow[m] + k) * 4 : kOut, &a[m]);
        if constexpr (NT) {
#pragma unroll
            for (int i = 0; i < CB; ++i) load<1, 0>(rt, k < p.K ? (brow[i] + k) * 4 : kOut, &b[i]);
        } else {
            load<CB, 0>(rl, k < p.K ? ncol + g * p.ldb * 4 : kOut, b);
        }
#pragma unroll
        for (int i = 0; i < CB; ++i)
#pragma unroll
            for (int m = 0; m < MG; ++m) acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], b[i], acc[m][i], 0, 0, 0);
    }

    // acc[m][b][i]: row 16m + 4g + i, column 16b + c ([N][K]) or CB c + b.
#pragma unroll
    for (int m = 0; m < MG; ++m)
#pragma unroll
        for (int b = 0; b < CB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                red[(wave * 16 * MG + 16 * m + 4 * g + i) * 16 * CB + (NT ? 16 * b + c : CB * c + b)] = acc[m][b][i];
    __syncthreads();
    for (uint32_t o = tid; o < 16 * MG * 16 * CB; o += 64 * W) {
        const uint32_t m = m0 + o / (16 * CB), n = n0 + o % (16 * CB);
        if (m >= p.M || n >= p.N) continue;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) v += red[w * 16 * MG * 16 * CB + o];
        if (ws) ws[(static_cast<uint64_t>(blockIdx.y) * p.M + m) * p.N + n] = v;
        else store_out(p, m, n, v);
    }
}

// How a call runs: CB column blocks a workgroup, K in `splits` ranges of k_per.
struct Plan {
    enum Kind { kNone, kMatrix, kLanes } kind = kNone;   // not here, skinny_f32_kernel, gemv_f32_nt_kernel
    int cb = 4;
    uint32_t splits = 1, k_per = 0;
};

template <int MG, int CB, bool NT, int W, int U>
void launch(hipStream_t s, const F32Gemm &p, const Plan &x, float *ws)
{
    constexpr size_t lds = static_cast<size_t>(W) * 16 * MG * 16 * CB * sizeof(float);
    static_assert(lds <= 160 * 1024, "the waves' sums fit in LDS");
    if constexpr (lds > 65536) {
        static std::atomic<bool> optin{false};   // launches may come from several host threads
        if (!optin)
            optin = hipFuncSetAttribute(reinterpret_cast<const void *>(skinny_f32_kernel<MG, CB, NT, W, U>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) == hipSuccess;
    }
    const dim3 grid((p.N + 16 * CB - 1) / (16 * CB), x.splits, (p.M + 16 * MG - 1) / (16 * MG));
    skinny_f32_kernel<MG, CB, NT, W, U><<<grid, 64 * W, lds, s>>>(p, x.k_per, x.splits > 1 ? ws : nullptr);
}

// Waves of a 64 x 64 workgroup.  A wave takes 32 depths at a time: over a short K
// most of eight have nothing to multiply, but hold LDS that another workgroup of
// the same CU could have, and their zeros are added.  Two to K = 64, four to 128,
// where the workgroups are more than the CUs (us with eight, four, two: 932 x 32 x
// 9408 46, 34, 30; 700 x 32 x 2000 11.4, 8.4, 10.4; 300 x 96 x 10000 24, 20, 18).
// Eight where they are not (512 x 100 x 1243 8.0 against 9.1 with four) and beyond
// (290 x 202 x 7636 24.9 against 28.0).
int waves_64x64(const F32Gemm &p, const Plan &x)
{
    const uint64_t wgs = static_cast<uint64_t>((p.N + 63) / 64) * ((p.M + 63) / 64) * x.splits;
    if (x.k_per > 128 || wgs <= cu_count()) return 8;
    return x.k_per <= 64 && wgs > 2ull * cu_count() ? 2 : 4;
}

// Otherwise sixteen waves a workgroup where their registers allow it (128 a lane),
// and as many depths in flight as eight waves' 256 hold.
int waves(const F32Gemm &p, const Plan &x)
{
    return x.cb == 4 && p.M > 32 ? waves_64x64(p, x) : x.cb == 1 && p.M <= 32 ? 16 : 8;
}

template <int MG, bool NT>
void launch_matrix(hipStream_t s, const F32Gemm &p, const Plan &x, float *ws)
{
    const int w = waves(p, x);
    if constexpr (MG == 4) {
        if (x.cb == 4 && w == 2) return launch<MG, 4, NT, 2, 2>(s, p, x, ws);
        if (x.cb == 4 && w == 4) return launch<MG, 4, NT, 4, 2>(s, p, x, ws);
    }
    if (x.cb == 4) launch<MG, 4, NT, 8, 2>(s, p, x, ws);
    else if (x.cb == 2) launch<MG, 2, NT, 8, 4>(s, p, x, ws);
    else launch<MG, 1, NT, MG <= 2 ? 16 : 8, 4>(s, p, x, ws);
}

// ---------------------------------------------------------------------------
// B stored [N][K], up to 8 rows: the lanes of a wave lie along K, so every load
// is 1 KiB in a run of one row of B (the matrix-core form reads 16 rows 64
// bytes at a time, which the memory serves at two thirds of that rate: 4 x 4096
// x 32000 122 us).  The vector ALUs do 4 M products per 16 bytes, a third of
// the time that they take to arrive at M = 8.  A wave holds R rows of B, so one
// LDS read of the staged activations serves R of them, and the 64 lanes' sums
// of R x M outputs are added by halving: each step a lane keeps half of them.
// ---------------------------------------------------------------------------
constexpr int NTW = 16;                    // waves per workgroup
constexpr int NTR = 4;                     // rows of B per wave
constexpr uint32_t kNtLds = 128 * 1024;    // staged activations

// Sums of a wave's 64 lanes of each of H values by halving: after the step of
// distance S, lanes with bit S set hold the upper half of the values.
template <int H, int S, int NV>
__device__ __forceinline__ void halve(float (&v)[NV], int lane)
{
    if constexpr (H > 1) {
        const bool up = lane & S;
#pragma unroll
        for (int i = 0; i < H / 2; ++i) {
            const float keep = up ? v[i + H / 2] : v[i], give = up ? v[i] : v[i + H / 2];
            v[i] = keep + __shfl_xor(give, S, 64);
        }
    } else {
        v[0] += __shfl_xor(v[0], S, 64);
    }
    if constexpr (S > 1) halve<(H > 1 ? H / 2 : 1), S / 2>(v, lane);
}

// waves_per: waves that share a group of R rows, each every waves_per-th block
// of 256 depths; chunk_k: depths staged at a time (a multiple of 256).
template <int M>
__global__ __launch_bounds__(64 * NTW) void gemv_f32_nt_kernel(F32Gemm p, uint32_t waves_per, uint32_t chunk_k)
{
    constexpr int MP = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : 8;
    constexpr int NV = NTR * MP;           // outputs of a wave (a power of two)
    constexpr int SPREAD = 64 / NV;        // lanes that end with the same output
    extern __shared__ float4 nt_lds[];
    float *at = reinterpret_cast<float *>(nt_lds);   // [M][chunk_k]
    __shared__ float part[NTW][NV];
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t per_wg = NTW / waves_per, slot = wave / waves_per, share = wave % waves_per;
    const uint32_t groups = (p.N + NTR - 1) / NTR, step = 256 * waves_per;
    const auto ra = buffer(p.A, (static_cast<uint64_t>(M - 1) * p.lda + p.K) * 4);

    // Rows past the last and depths past kend lie past the buffer's end.
    auto fetch = [&](float4 (&b)[NTR], uint32_t g0, uint32_t k, uint32_t kend) {
        const uint32_t n0 = (g0 + slot) * NTR;
        const uint32_t rows = n0 < p.N && k < kend ? min(static_cast<uint32_t>(NTR), p.N - n0) : 0;
        const auto rb = buffer(p.B + static_cast<uint64_t>(min(n0, p.N - 1)) * p.ldb,
                               rows ? (static_cast<uint64_t>(rows - 1) * p.ldb + p.K) * 4 : 0);
        const uint32_t kl = k + 4 * lane, off = kl < p.K ? kl * 4 : kOut;
#pragma unroll
        for (int r = 0; r < NTR; ++r)
            b[r] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rb, off + r * p.ldb * 4, 0,
                                                                                    kNontemporal));
    };
    uint32_t g0 = blockIdx.x * per_wg, kc = 0;
    float4 x[NTR], y[NTR];
    float acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.0f;
    fetch(x, g0, 256 * share, min(p.K, chunk_k));
    fetch(y, g0, 256 * share + step, min(p.K, chunk_k));
    bool staged = false;
    while (g0 < groups) {                  // (group, chunk) pairs, uniform over the workgroup
        const uint32_t ke = min(p.K, kc + chunk_k);
        if (!staged) {
            __syncthreads();               // the previous chunk is consumed
            const uint32_t vecs = chunk_k / 4;
#pragma unroll
            for (int m = 0; m < M; ++m)
                for (uint32_t i = tid; i < vecs; i += 64 * NTW)
                    load<4, 0>(ra, kc + 4 * i < p.K ? (m * p.lda + kc + 4 * i) * 4 : kOut, at + (m * vecs + i) * 4);
            __syncthreads();
            staged = chunk_k >= p.K;
        }
        auto multiply = [&](float4 (&b)[NTR], uint32_t kk) {
            const float *ar = at + (kk - kc) + 4 * lane;
            // a vector that K ends in (what follows it may be NaN)
            const uint32_t left = p.K - (kk + 4 * lane);   // huge past K, where the loads gave zeros
            const bool cut = (p.K & 3u) != 0 && kk + 256 > p.K;   // uniform
            if (cut) {
#pragma unroll
                for (int r = 0; r < NTR; ++r) {
                    if (left < 2) b[r].y = 0.0f;
                    if (left < 3) b[r].z = 0.0f;
                    if (left < 4) b[r].w = 0.0f;
                }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                float4 a = *reinterpret_cast<const float4 *>(ar + m * chunk_k);
                if (cut) {
                    if (left < 2) a.y = 0.0f;
                    if (left < 3) a.z = 0.0f;
                    if (left < 4) a.w = 0.0f;
                }
#pragma unroll
                for (int r = 0; r < NTR; ++r) {
                    float &t = acc[r * MP + m];
                    t = fmaf(a.x, b[r].x, t);
                    t = fmaf(a.y, b[r].y, t);
                    t = fmaf(a.z, b[r].z, t);
                    t = fmaf(a.w, b[r].w, t);
                }
            }
        };
        // The loads past this (group, chunk) are the next one's first.
        const bool last = ke >= p.K;
        const uint32_t g1 = last ? g0 + gridDim.x * per_wg : g0, kc1 = last ? 0 : ke, ke1 = min(p.K, kc1 + chunk_k);
        uint32_t k = kc + 256 * share;
        while (true) {
            if (k < ke) multiply(x, k);
            const bool more = k + 2 * step < ke;
            fetch(x, more ? g0 : g1, more ? k + 2 * step : kc1 + 256 * share, more ? ke : ke1);
            if (k + step < ke) multiply(y, k + step);
            const bool more2 = k + 3 * step < ke;
            fetch(y, more ? g0 : g1, more ? k + 3 * step : kc1 + 256 * share + step, more ? (more2 ? ke : 0) : ke1);
            if (!more) break;
            k += 2 * step;
        }
        if (last) {
            halve<NV, 32>(acc, lane);
            const uint32_t i = lane / SPREAD, m = i % MP;
            if (waves_per == 1) {
                const uint32_t n = (g0 + slot) * NTR + i / MP;
                if (lane % SPREAD == 0 && m < M && n < p.N) store_out(p, m, n, acc[0]);
            } else {
                if (lane % SPREAD == 0) part[wave][i] = acc[0];
                __syncthreads();
                for (uint32_t o = tid; o < per_wg * NV; o += 64 * NTW) {
                    const uint32_t sl = o / NV, j = o % NV, n = (g0 + sl) * NTR + j / MP;
                    if (j % MP >= M || n >= p.N) continue;
                    float v = 0.0f;
                    for (uint32_t w = 0; w < waves_per; ++w) v += part[sl * waves_per + w][j];
                    store_out(p, j % MP, n, v);
                }
                __syncthreads();           // part[] is read before the next groups' sums
            }
#pragma unroll
            for (int j = 0; j < NV; ++j) acc[j] = 0.0f;
        }
        g0 = g1;
        kc = kc1;
    }
}

template <int M>
void launch_nt(hipStream_t s, const F32Gemm &p)
{
    static std::atomic<bool> optin{false};
    if (!optin)
        optin = hipFuncSetAttribute(reinterpret_cast<const void *>(gemv_f32_nt_kernel<M>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kNtLds) == hipSuccess;
    const uint32_t groups = (p.N + NTR - 1) / NTR, cus = cu_count();
    uint32_t per = NTW;
    while (per > 1 && (groups * per + NTW - 1) / NTW > cus) per /= 2;
    const uint32_t chunk = std::min<uint32_t>((p.K + 255) / 256 * 256, kNtLds / 4 / M / 256 * 256);
    const uint32_t wgs = std::min<uint32_t>(cus, (groups * per + NTW - 1) / NTW);
    gemv_f32_nt_kernel<M><<<dim3(wgs), 64 * NTW, static_cast<size_t>(M) * chunk * 4, s>>>(p, per, chunk);
}
}  // namespace

namespace {

// Partial sums written and read again: bytes that the second launch's 3.5 us cover
// (481 x 3808 x 1042, 32 MB in eight ranges 65 us, 16 MB in four 70.5), and those per
// microsecond beyond (988 x 3378 x 7616 in two ranges, 120 MB, 572 us, in one 534;
// 382 x 1535 x 14208 217 against 197).
constexpr double kPartialsFree = 40e6, kPartials = 2.2e6;

// Microseconds of the matrix-core kernel with 16 x.cb columns a workgroup, K in
// the number of ranges that ends first.  A workgroup alone on a CU takes 2 and
// its bytes at `cu` or its products at 0.2, 0.28 or 0.44e6 flops (wider ones
// reuse more); a round of one per CU takes no less than its bytes at `mem`
// (bytes per microsecond, measured on this kernel's reads); ranges cost the
// second launch that adds them (3.5) and their partial sums.  [K][N]
// N = K = 4096 at one range 28, two 19.2, four 15.5, eight 15.6; K = 11008 N =
// 4096 70, 42, 31.9, 32.3; K = 4096 N = 20000 64, 56, 51.7.
double split(const F32Gemm &p, double cu, double mem, Plan &x)
{
    const uint32_t cols = 16 * x.cb, mg = p.M <= 16 ? 1 : p.M <= 32 ? 2 : 4, cus = cu_count();
    const uint64_t tiles = static_cast<uint64_t>((p.N + cols - 1) / cols) * ((p.M + 16 * mg - 1) / (16 * mg));
    double best = 0.0;
    const uint64_t out_bytes = 4ull * p.M * p.N;
    for (uint32_t s = 1; s == 1 || (s <= 16 && p.K / s >= 240 && s * out_bytes <= kMaxSplitWs); s *= 2) {
        const uint32_t k_per = ((p.K + s - 1) / s + 63) / 64 * 64;   // whole chunks
        const double bytes = 4.0 * k_per * cols, flops = 32.0 * mg * k_per * cols;
        const double alone = 2.0 + std::max(bytes / cu, flops / (x.cb == 1 ? 0.2e6 : x.cb == 2 ? 0.28e6 : 0.44e6));
        const uint64_t wgs = tiles * s;
        double t = static_cast<double>(wgs / cus) * std::max(alone, cus * bytes / mem);
        if (wgs % cus) t += std::max(alone, static_cast<double>(wgs % cus) * bytes / mem);
        if (s > 1) t += 3.5 + std::max(0.0, 2.0 * s * out_bytes - kPartialsFree) / kPartials;
        if (s == 1 || t < best) {
            best = t;
            x.k_per = k_per;
            x.splits = (p.K + k_per - 1) / k_per;
        }
    }
    return best;
}

// Which calls run here; the others keep the kernels of gemm_f32.hip.  Both
// sides of each line measured on MI355X, weights from HBM (us, before -> here):
//   [N][K] M <= 8: 128-column tiles of split products before, or where rows are
//     not 16-byte aligned the fp32 tile kernel.  4 x 4096 x 32000 182 -> 87, x
//     4096 35 -> 14, 4 x 2047 x 11007 97 -> 19; below 8M weights the
//     matrix-core kernel starts faster (8 x 1024 x 4096 14 -> 6.1 against 8.3
//     with lanes along K).
//   [N][K] M <= 32: 16 x 4096 x 4096 36 -> 22, x 32000 184 -> 145; 32 x 8192 x
//     8192 101 -> 86, but x 11008 x 4096 71 against 75.  Aligned M <= 64 only up to
//     8M weights: 64 x 2048 x 2048 18.5 -> 15, but x 4096 x 11008 81 against 93.
//   [K][N] M <= 4: up to N = 4096 or 8M weights (4 x 4096 x 4096 19.8 -> 15.6,
//     x 1024 x 1024 13 -> 6); wider, or with unaligned rows from 2M weights, the
//     split kernel's 1 KiB rows are as fast or faster (1 x 4096 x 11008 31
//     against 35, 1 x 4096 x 4095 16.5 against 20).
//   [K][N] M <= 8: up to N = 20480 (8 x 4096 x 16384 55 -> 42); wider, the wide
//     kernel (8 x 4096 x 32000 84 against 87).  That one starts at 25600 even
//     columns: between the two, and at odd widths, gemv_f32_kernel runs, as it did
//     (1 x 1071 x 21049 21 against 25, but 6 x 212 x 21456 15 against 6.5).
//   [K][N] M <= 64: 16 x 4096 x 4096 39 -> 16.5, 32 x 4096 x 32000 195 -> 105,
//     64 x 8192 x 8192 109 -> 82.
//   Aligned M > 64 only while the weights are so few that tiles of 128 leave the
//     chip idle: 400 x 512 x 512 15 -> 8, 128 x 1024 x 1024 15 -> 10, 128 x 1024 x
//     4096 24 -> 19; but 256 x 4096 x 1024 26 against 27, 200 x 2048 x 2048 24
//     against 27.  Over a short K and wide outputs those tiles are faster still
//     (796 x 128 x 7584 14 against 37, 932 x 32 x 9408 16 against 30), with ten times
//     the error (4.4e-6 against 1e-7): such calls stay in full f32.
//   Unaligned rows ran on the fp32 tile kernel from M = 9 on: 16 x 4096 x 4095
//     70 -> 21, 128 x 4095 x 4096 90 -> 47, 700 x 4095 x 4096 577 -> 228, 2000 x
//     1000 x 1001 154 -> 48.  Its 128-row tiles win back many rows over a short K
//     or, [N][K], wide weights (2048 x 333 x 4000 93 against 96; [N][K] 1000 x
//     2047 x 11007 684 against 777); up to 15% on either side of these lines.
Plan plan(const F32Gemm &p)
{
    Plan x;
    // 32-bit offsets: 64 rows of A and of B
    if (p.M > 2048 || p.trans_a || p.cull || p.ktile_state || p.k_split_depth || p.ldb >= (1u << 22) ||
        p.lda >= (1u << 22))
        return x;
    const uint64_t weights = static_cast<uint64_t>(p.K) * p.N;
    auto even = [](const float *q, uint32_t ld) { return ld % 4 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0; };
    const bool even_b = even(p.B, p.ldb), even_ab = even_b && even(p.A, p.lda);
    if (p.trans_b && p.M <= 8 && weights >= (8u << 20)) {
        x.kind = Plan::kLanes;
        return x;
    }
    if (even_ab) {   // the split-bf16 tiles' ground from 65 rows on, and in part before
        if (p.M > 64 && weights > (p.M <= 128 ? 9u << 19 : p.M <= 1024 ? 1u << 20 : 0)) return x;
        if (p.trans_b && (p.M > 32 ? weights > (8u << 20) : p.M > 16 && p.K > 8192)) return x;
    } else if (p.M > (p.trans_b ? 768 : 1024)) {
        if (p.K < 512 || (p.trans_b && weights > (17u << 20))) return x;
    }
    if (!p.trans_b) {
        if (p.M <= 4 && weights > (even_b ? 8u << 20 : 2u << 20) && !(even_b && p.N <= 4096)) return x;
        if (p.M <= 8 && p.N > 20480) return x;
    }
    x.kind = Plan::kMatrix;
    // 64 columns a workgroup read the longest runs and share A the most; narrower
    // ones fill the chip where the output is small, and [N][K] up to 16 rows,
    // whose runs do not grow with the columns, likewise below N = 8192 (16 x 4096
    // x 4096 22 against 24).
    static const double kRate[2][3][2] = {{{18e3, 2.8e6}, {30e3, 5.0e6}, {35e3, 6.0e6}},    // [K][N]
                                          {{25e3, 3.4e6}, {25e3, 3.5e6}, {25e3, 3.6e6}}};   // [N][K]
    const bool small = weights <= (4u << 20);
    const int most = !small && p.trans_b && p.M <= 16 && p.N < 8192 ? 0 : 2;
    double best = 0.0;
    for (int i = most; i >= (small ? 0 : most); --i) {
        Plan y = x;
        y.cb = 1 << i;
        const double t = split(p, kRate[p.trans_b][i][0], kRate[p.trans_b][i][1], y);
        if (i == most || t < best) {
            best = t;
            x = y;
        }
    }
    return x;
}

}  // namespace

bool skinny_f32_takes(const F32Gemm &p) { return plan(p).kind != Plan::kNone; }

void skinny_f32_route(const F32Gemm &p, char *out, size_t size)
{
    const Plan x = plan(p);
    const int mg = p.M <= 16 ? 1 : p.M <= 32 ? 2 : 4;
    if (x.kind == Plan::kLanes) std::snprintf(out, size, "lanes<%u>", p.M);
    else
        std::snprintf(out, size, "skinny<%d,%d,%s,%d> splits=%u", mg, x.cb, p.trans_b ? "NK" : "KN", waves(p, x), x.splits);
}

size_t skinny_f32_ws_bytes(const F32Gemm &p)
{
    const Plan x = plan(p);
    return x.splits > 1 ? static_cast<size_t>(x.splits) * p.M * p.N * sizeof(float) : 0;
}

void skinny_f32(hipStream_t s, const F32Gemm &p, float *ws)
{
    const Plan x = plan(p);
    if (x.kind == Plan::kLanes) {
        switch (p.M) {
        case 1: launch_nt<1>(s, p); break;
        case 2: launch_nt<2>(s, p); break;
        case 3: launch_nt<3>(s, p); break;
        case 4: launch_nt<4>(s, p); break;
        case 5: launch_nt<5>(s, p); break;
        case 6: launch_nt<6>(s, p); break;
        case 7: launch_nt<7>(s, p); break;
        default: launch_nt<8>(s, p); break;
        }
        return;
    }
    auto rows = [&](auto mg) {
        constexpr int MG = decltype(mg)::value;
        if (p.trans_b) launch_matrix<MG, true>(s, p, x, ws);
        else launch_matrix<MG, false>(s, p, x, ws);
    };
    if (p.M <= 16) rows(std::integral_constant<int, 1>{});
    else if (p.M <= 32) rows(std::integral_constant<int, 2>{});
    else rows(std::integral_constant<int, 4>{});
    if (x.splits > 1) splitk_reduce(s, p, ws, x.splits);
}

}  // namespace k
}  // namespace vnpu
