// direct_i8.hip - MATMUL_I8 between decode and prefill: tens to hundreds of
// rows, and rows of any length and alignment, straight from memory.
//
// Replaces the reference's AVX2 packed-panel tiles
// (src/kernels/kernels.cpp:635-869) there.  Same semantics as its store_i8_c
// (kernels.cpp:526-535): exact int32 sums, then
// C = epi(((float)acc * scale_a[m]) * scale_b[n] + bias[n]).
//
// Design.  The staged tiles of gemm_i8.hip are 256 x 128: a chunk of 256 rows by
// 4096 columns is 32 of them on 256 CUs.  Here a workgroup owns 16 MG rows by 16
// CB columns (64 x 64 at most) over all of K, and its W waves split K, wave w
// taking the pairs of 64-deep blocks w, w + W, ...:
//   * both operands of v_mfma_i32_16x16x64_i8 are loaded as they lie: a packed
//     1 KiB weight block is one load of 16 bytes a lane, and so are 16 rows x 64
//     depths of A (lane 16g + r: 16 bytes of row r at depth 16g), a pair of
//     blocks covering whole 128-byte lines.  A wave loads MG + CB KiB for MG CB
//     products, and no two waves of a workgroup load the same;
//   * nothing is staged, so nothing waits at a barrier until the waves' int32
//     sums meet in LDS; the next pair's loads are issued before this pair's
//     products;
//   * the packed weights are zero past K, so what A's lanes read there (the next
//     row) does not matter; a buffer ends the reads at A's last byte.  Rows that
//     are not 4-byte aligned are read from the dword below and shifted.
// What bounds it is the ~45 bytes/ns that one CU takes in (a 64 x 64 workgroup at
// K = 4096 reads 0.5 MiB) and, with one row tile and wide N, the weights from
// HBM.  Starting the workgroups that share rows or columns at different depths,
// so that each finds the others' lines in L2, was slower (18.6 -> 21.0 us at
// 256 x 4096 x 4096): in step they already share them.
//
// Measured, us, before (gemv_i8.hip's matrix-core kernel to 64 rows, then the
// staged tiles, or the generic kernel where K % 64 or the alignment rules these
// out) and here, K x N, each with the QUANTIZE_I8 of its rows (2 to 4 us) and the
// launches, as all times below:
//     rows     4096x4096    11008x4096   4096x11008   4096x32000   1024x1024
//       8      (8.2)        (13.9)       (12.2)       26.1  24.2   (7.4)
//      16       8.7   8.5   16.2  14.8   12.8  12.4   26.2  25.4    7.5   7.3
//      32      11.4   8.9   23.8  15.2   19.8  13.3   55.2  30.4    7.5   7.3
//      64      16.8  10.4   38.9  19.3   26.1  18.5   41.9 (42.0)   8.3   7.3
//     128      24.3  12.7   50.0  24.0   25.1 (25.9)  45.7 (70)    12.9   7.3
//     256      25.4  18.6   54.2  35.8   26.7 (43.9)  50.4 (125)   13.2   7.7
//     384      26.1 (26.3)  55.5 (56.2)  31.7 (62)    80.9 (177)   13.5   8.1
// (in brackets: the side not taken), and 1376 x 5003 (K % 64 != 0) 96 / 331 / 1024
// rows 44 / 50 / 54 -> 8.6 / 17.8 / 31, 1001 x 4100 (rows from any byte) 24 / 96 /
// 1024 rows 21 / 58 / 93 -> 7.9 / 8.5 / 27.6.
#include "kernels.hpp"
#include "device_math.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>

namespace vnpu {
namespace k {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kBufferWord3 = 0x00020000;  // raw buffer, 32-bit data format
constexpr uint32_t kOut = 0x80000000u;    // an offset past any buffer
constexpr int kNontemporal = 2;           // cache policy bits

// SHIFT: rows of A at any alignment (else 4 bytes).  STREAM: the weights are read
// nontemporally.  A CU holds three 32 x 64 workgroups of four waves (168 registers;
// two of them, as the compiler would have it, took 35.5 instead of 31.1 us for
// 1024 x 1376 x 5003), and two such of eight with shifts; 64 x 64 does not fit twice
// without spills (18.8 -> 22.9 us at 256 x 4096 x 4096).
template <int MG, int W, bool SHIFT>
constexpr int kWavesPerSimd = MG == 4 ? 1 : MG == 2 && W == 4 ? 3 : MG == 2 && !SHIFT ? 2 : 4;
template <int MG, int CB, int W, bool SHIFT, bool STREAM, bool SPREAD>
__global__ __launch_bounds__(64 * W)
__attribute__((amdgpu_waves_per_eu(kWavesPerSimd<MG, W, SHIFT>))) void direct_i8_kernel(I8Gemm p, uint32_t last)
{
    constexpr int TILE = 256 * MG * CB;   // sums of a wave
    static_assert(W * TILE <= 16384, "the waves' sums take 64 KiB of LDS at most");
    __shared__ int red[W][16 * MG][16 * CB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const uint32_t NT = p.Np >> 4, KT = p.Kp >> 6;
    // Workgroups are dealt to the eight XCDs in turn: the row tiles of a column
    // tile are neighbours on one, so its L2 fetches the weights once (with the
    // row tiles a whole pass over the columns apart 331 x 1376 x 5003 took 22.5
    // instead of 17.8 us, 48 x 4096 x 32000 61 instead of 45).  The column tiles
    // go to the XCDs in turn too; with SPREAD the tiles of the last, less than
    // eight, are dealt out evenly, `last` to each XCD.
    uint32_t nt0 = (blockIdx.y * 8 + (blockIdx.x & 7u)) * CB, m0 = (blockIdx.x >> 3) * (16 * MG);
    if constexpr (SPREAD) {
        if (blockIdx.y + 1 == gridDim.y) {
            const uint32_t row_tiles = gridDim.x >> 3, i = blockIdx.x >> 3;
            if (i >= last) return;
            const uint32_t tile = (blockIdx.x & 7u) * last + i;
            nt0 = (blockIdx.y * 8 + tile / row_tiles) * CB;
            m0 = tile % row_tiles * (16 * MG);
        }
    }
    if (nt0 >= NT) return;
    const uint32_t rows = min(16u * MG, p.M - m0);

    // A from the dword that holds its first byte to the one that holds its last
    const int8_t *a0 = p.A + static_cast<uint64_t>(m0) * p.lda;
    const uint32_t skew = SHIFT ? static_cast<uint32_t>(reinterpret_cast<uintptr_t>(a0) & 3u) : 0u;
    const uint32_t abytes = ((rows - 1) * p.lda + p.K + skew + 3u) & ~3u;
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(a0 - skew), 0, static_cast<int>(abytes),
                                                      kBufferWord3);
    uint32_t arow[MG], shift[MG];
#pragma unroll
    for (int m = 0; m < MG; ++m) {   // rows past M repeat the last and are not stored
        const uint32_t o = min(16u * m + c, rows - 1) * p.lda + skew + 16 * g;
        arow[m] = SHIFT ? o & ~3u : o;
        shift[m] = 8 * (o & 3u);
    }
    const uint32_t strips = min(static_cast<uint32_t>(CB), NT - nt0), strip_bytes = KT * 1024;
    const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p.frag) + static_cast<uint64_t>(nt0) * strip_bytes,
                                                      0, static_cast<int>(strips * strip_bytes), kBufferWord3);

    struct Pair {
        v4i a[2][MG], b[2][CB];
        uint32_t next[SHIFT ? 2 : 1][SHIFT ? MG : 1];
    };
    auto fetch = [&](Pair &t, uint32_t kt) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const bool in = kt + u < KT;
#pragma unroll
            for (int b = 0; b < CB; ++b)
                t.b[u][b] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                    rb, in ? b * strip_bytes + (kt + u) * 1024 + lane * 16 : kOut, 0, STREAM ? kNontemporal : 0));
#pragma unroll
            for (int m = 0; m < MG; ++m) {
                const uint32_t o = in ? arow[m] + (kt + u) * 64 : kOut;
                t.a[u][m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ra, o, 0, 0));
                if constexpr (SHIFT)
                    t.next[u][m] = __builtin_amdgcn_raw_buffer_load_b32(ra, in ? o + 16 : kOut, 0, 0);
            }
        }
    };
    v4i acc[MG][CB];
#pragma unroll
    for (int m = 0; m < MG; ++m)
#pragma unroll
        for (int b = 0; b < CB; ++b) acc[m][b] = (v4i){0, 0, 0, 0};
    auto multiply = [&](const Pair &t) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int m = 0; m < MG; ++m) {
                v4i a = t.a[u][m];
                if constexpr (SHIFT) {
                    const uint32_t n = t.next[u][m], s = shift[m];
                    a = (v4i){static_cast<int>(__builtin_amdgcn_alignbit(a.y, a.x, s)),
                              static_cast<int>(__builtin_amdgcn_alignbit(a.z, a.y, s)),
                              static_cast<int>(__builtin_amdgcn_alignbit(a.w, a.z, s)),
                              static_cast<int>(__builtin_amdgcn_alignbit(n, a.w, s))};
                }
#pragma unroll
                for (int b = 0; b < CB; ++b)
                    acc[m][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, t.b[u][b], acc[m][b], 0, 0, 0);
            }
        }
    };
    Pair x, y;
    uint32_t kt = 2 * wave;
    if (kt < KT) fetch(x, kt);
    for (; kt < KT; kt += 4 * W) {
        fetch(y, kt + 2 * W);
        multiply(x);
        if (kt + 2 * W >= KT) break;
        fetch(x, kt + 4 * W);
        multiply(y);
    }

    // acc[m][b][i]: row 16m + 4g + i, column 16b + c.
#pragma unroll
    for (int m = 0; m < MG; ++m)
#pragma unroll
        for (int b = 0; b < CB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[wave][16 * m + 4 * g + i][16 * b + c] = acc[m][b][i];
    __syncthreads();
    for (int o = tid; o < TILE; o += 64 * W) {
        const uint32_t m = m0 + o / (16 * CB), n = nt0 * 16 + o % (16 * CB);
        if (m >= p.M || n >= p.N) continue;
        int v = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) v += red[w][o / (16 * CB)][o % (16 * CB)];
        float out = dev::mul_rn(dev::mul_rn(static_cast<float>(v), p.scale_a ? p.scale_a[m] : 1.0f), p.scale_b[n]);
        if (p.bias) out = dev::add_rn(out, p.bias[n]);
        p.C[static_cast<uint64_t>(m) * p.ldc + n] = dev::epilogue(out, p.epilogue);
    }
}

// Workgroup shapes: 16 mg rows x 16 cb columns, `waves` waves.  The time of a call
// is start + rounds (round + per_kib K / 1024), us, with rounds = the workgroups of
// an XCD / its CUs, rounded up; fitted to the shapes' sweeps over 16..1024 rows at the sizes above
// (they miss by some 15% at most where they are chosen).  Few rows want narrow
// workgroups on every CU, more rows larger ones that load less per product; four
// waves instead of eight let a CU hold more workgroups.  odd_round: `round` for
// rows that are not 4-byte aligned, 0 where the shifts' registers cost the shape
// more than its size gains (it is not built).
struct Shape {
    uint32_t mg, cb, waves;
    double start, round, per_kib, odd_round;
};
constexpr Shape kShapes[] = {
    {1, 1, 16, 5.7, 0.4, 0.60, 0.4}, {1, 2, 8, 5.6, 0.45, 0.70, 0.45}, {1, 4, 8, 5.5, 0.75, 0.95, 0.95},
    {2, 4, 8, 4.8, 2.0, 1.40, 1.1},  {2, 4, 4, 6.6, 0.5, 1.45, 0.0},   {4, 4, 4, 4.3, 5.9, 2.20, 0.0},
};
// Weights of this size, read once, do not stay in the 256 MiB last-level cache
// beside whatever a program runs between two calls, and are read past it: 8 / 32
// rows of 4096 x 32000 27.5 -> 24.2 / 32.7 -> 28.9 us, but 16 rows of 4096 x 11008
// (43 MiB, resident) 12.3 -> 13.4 us; even at 4096 x 22016 (86 MiB).
constexpr uint64_t kStreamBytes = 96ull << 20;

// us that memory needs for `col_tiles` times rows of `tile_rows`: the weights once
// at 6.5 TB/s (6.5e6 bytes/us), the rows of A again for every column tile at 20 TB/s
// from the L2s.
double memory_us(const I8Gemm &p, uint64_t col_tiles, uint32_t tile_rows)
{
    const uint32_t row_tiles = (p.M + tile_rows - 1) / tile_rows;
    return static_cast<double>(p.Kp) * p.Np / 6.5e6 +
           static_cast<double>(col_tiles) * row_tiles * std::min(tile_rows, p.M) * p.K / 20e6;
}

bool streams(const I8Gemm &p, uint32_t tile_rows)
{
    return p.M <= tile_rows && static_cast<uint64_t>(p.Kp) * p.Np >= kStreamBytes;
}

bool odd_rows(const I8Gemm &p) { return p.lda % 4 || reinterpret_cast<uintptr_t>(p.A) % 4; }

// The most tiles that an XCD gets, `last` of them from the column tiles past the
// last whole eight.  Of 9 column tiles in turn one XCD gets two, and of 2 six XCDs
// get none: their tiles are spread where that saves a round of workgroups (331 x
// 4096 x 576 11.4 -> 7.6 us, 781 x 8320 x 1088 46.4 -> 26.0, 2048 x 4096 x 128 21.2 ->
// 8.0).  Elsewhere it would only have more XCDs read their weights (256 x 11008 x 576
// 13.8 against 14.6 us) and a workgroup wait for one more argument (0.2 us).
struct Grid {
    uint64_t tiles;
    uint32_t xcd_tiles, last;
    bool spread;
};
Grid grid_of(const I8Gemm &p, uint32_t mg, uint32_t cb)
{
    const uint64_t cols = (p.Np / 16 + cb - 1) / cb, row_tiles = (p.M + 16 * mg - 1) / (16 * mg);
    const uint64_t last = (cols % 8 * row_tiles + 7) / 8, even = cols / 8 * row_tiles + last;
    const uint64_t in_turn = (cols + 7) / 8 * row_tiles, cus = std::max(1u, cu_count() / 8);
    const bool spread = !streams(p, 16 * mg) && (in_turn + cus - 1) / cus > (even + cus - 1) / cus;
    return {cols * row_tiles, static_cast<uint32_t>(spread ? even : in_turn), static_cast<uint32_t>(last), spread};
}

// The shape that should finish first, and its time.
const Shape &choose(const I8Gemm &p, double &best)
{
    const bool odd = odd_rows(p);
    const uint32_t cus = cu_count();
    const Shape *pick = nullptr;
    for (const Shape &h : kShapes) {
        if ((odd && h.odd_round == 0.0) || (h.mg > 1 && p.M <= 8 * h.mg)) continue;
        const uint32_t rows = 16 * h.mg;
        const Grid g = grid_of(p, h.mg, h.cb);
        const uint64_t cols = (p.Np / 16 + h.cb - 1) / h.cb, wgs = g.tiles;
        const uint64_t rounds = (8ull * g.xcd_tiles + cus - 1) / cus;
        // memory and the CUs' own pace overlap, but not wholly where they are alike;
        // a last round that is part empty leaves bandwidth unused as well
        const double fill = rounds > 1 ? std::sqrt(static_cast<double>(wgs) / (rounds * cus)) : 1.0;
        const double t = h.start + std::hypot(rounds * ((odd ? h.odd_round : h.round) + h.per_kib * p.Kp / 1024),
                                              memory_us(p, cols, rows) / fill * (streams(p, rows) ? 0.85 : 1.0));
        if (!pick || t < best) {
            pick = &h;
            best = t;
        }
    }
    return *pick;
}

template <int MG, int CB, int W, bool UNALIGNED>
void launch(hipStream_t s, const I8Gemm &p)
{
    const uint32_t row_tiles = (p.M + 16 * MG - 1) / (16 * MG);
    const Grid g = grid_of(p, MG, CB);
    const dim3 grid(8 * row_tiles, (p.Np / 16 + 8 * CB - 1) / (8 * CB));
    if constexpr (UNALIGNED) {
        if (odd_rows(p)) {
            if (g.spread) direct_i8_kernel<MG, CB, W, true, false, true><<<grid, 64 * W, 0, s>>>(p, g.last);
            else direct_i8_kernel<MG, CB, W, true, false, false><<<grid, 64 * W, 0, s>>>(p, 0);
            return;
        }
    }
    if (streams(p, 16 * MG))
        direct_i8_kernel<MG, CB, W, false, true, false><<<grid, 64 * W, 0, s>>>(p, 0);
    else if (g.spread)
        direct_i8_kernel<MG, CB, W, false, false, true><<<grid, 64 * W, 0, s>>>(p, g.last);
    else
        direct_i8_kernel<MG, CB, W, false, false, false><<<grid, 64 * W, 0, s>>>(p, 0);
}

}  // namespace

bool direct_i8_takes(const I8Gemm &p)
{
    // five to eight rows: only where the column strips need several rounds of
    // gemv_i8.hip's workgroups (8 rows 4096 x 22016 22.8 -> 20.1, 4096 x 32000
    // 26.1 -> 24.2 us; within 5% either way below that)
    if (p.M <= 8 && (p.M < 5 || p.Np < 1024 * 16)) return false;
    // 32-bit offsets in a workgroup's rows and strips; the grid's second dimension
    if (63ull * p.lda + p.K + 64 >= (1ull << 31) || 4ull * p.Kp * 16 >= (1ull << 31)) return false;
    if (p.Np > 65535u * 8 * 16) return false;
    // The staged tiles are for 64 rows and more, and so are a requested kernel
    // and the one that skips zero tiles of sparse weights.
    if (p.M < 64) return true;
    if (p.variant != kI8Auto || gemm_i8_ws_bytes(p)) return false;
    if (p.K % 64 || p.lda % 16 || reinterpret_cast<uintptr_t>(p.A) % 16) return true;
    // The staged tiles, 256 x 128: 8.8 us and 4 us for 1024 depths of a round of
    // the 128-deep ones, 10.5 and 10.7 of the 64-deep ones that K % 128 = 64
    // leaves, fitted to 96..512 rows at the sizes above and to K = 320 to 8256; the
    // latter less for fewer rows to store, which shows over a short K (98 x 64 x 24512
    // 7.6 us against 9.1 here).  The call is theirs unless the estimates differ by 10%.
    const uint64_t cols = (p.N + 127) / 128, tiles = cols * ((p.M + 255) / 256);
    const uint64_t rounds = (tiles + cu_count() - 1) / cu_count();
    const bool deep = p.K % 128 == 0;
    const double staged = (deep ? 8.8 : 7.9 + 2.6 * std::min(p.M, 256u) / 256) +
                          std::hypot(rounds * (deep ? 4.0 : 10.7) * p.K / 1024, memory_us(p, cols, 256));
    double direct;
    choose(p, direct);
    return direct * 1.1 < staged;
}

void direct_i8_route(const I8Gemm &p, char *out, size_t size)
{
    double t;
    const Shape &h = choose(p, t);
    const Grid g = grid_of(p, h.mg, h.cb);
    std::snprintf(out, size, "direct<%u,%u,%u%s%s> tiles=%llu xcd_tiles=%u", h.mg, h.cb, h.waves,
                  odd_rows(p) ? ",shift" : streams(p, 16 * h.mg) ? ",stream" : "", g.spread ? ",spread" : "",
                  static_cast<unsigned long long>(g.tiles), g.xcd_tiles);
}

void direct_i8(hipStream_t s, const I8Gemm &p)
{
    double t;
    const Shape &h = choose(p, t);
    if (h.mg == 4) launch<4, 4, 4, false>(s, p);
    else if (h.mg == 2 && h.waves == 4) launch<2, 4, 4, false>(s, p);
    else if (h.mg == 2) launch<2, 4, 8, true>(s, p);
    else if (h.cb == 4) launch<1, 4, 8, true>(s, p);
    else if (h.cb == 2) launch<1, 2, 8, true>(s, p);
    else launch<1, 1, 16, true>(s, p);
}

}  // namespace k
}  // namespace vnpu
