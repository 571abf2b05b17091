// Reduced-precision Correlation on MFMA (gfx950): BF16 / FP16 / FP8-e4m3
// features, FP32 accumulation.  Same output layout and zero-padding semantics
// as the reference op (correlation.cc:147-275; legacy: correlation_cuda.cu:182-331).
//
// Matrix form.  For output row h, a segment of 16 pixels w0..w0+15 and one
// vertical displacement dy, the 16 x 24 product
//     G[i][j] = sum_c f1[c][h][w0+i] * f2[c][h+dy][w0-4+j]
// holds all horizontal displacements on its diagonals: out[dy][dx][h][w0+i] =
// G[i][i+dx+4].  G is computed as two 16 x 16 MFMA tiles (columns 0..15 and
// 8..23) with K = 32 channels per instruction (v_mfma_f32_16x16x32_{bf16,f16,
// fp8_fp8}); 9 of every 16 columns are used, which is fine because the op is
// bound by the 81 output planes it writes, not by the products.
//
// Block: 8 waves; wave q computes one 16-pixel segment (q & 1) of output row
// h0 + q/2 for DG vertical displacements and all horizontal ones, 8*DG FP32
// accumulators per lane.  Channels stream through LDS in chunks of 32: the f1
// tile (4 rows x 32 px) and the f2 rows that the displacements reach (40 px,
// zeros outside the image), read from the NCHW operands 4 pixels at a time and
// turned channels-last with byte permutes, with a padded pixel stride, so that
// each lane's 8-channel MFMA operand is one 16-byte (8-byte for FP8) LDS read
// and 8 lanes cover all banks.  (Widths that are not a multiple of 4 used to be
// copied channels-last first, into memory allocated for the call: 213x119x64 in
// BF16 45.6 us with the two copies, 13.9 without.)
// After the channel loop, each wave moves the diagonals of its tiles through a
// small LDS stage and writes every (dy, dx) output row as 32 consecutive floats.
#include "vsc_internal.h"

#include <algorithm>
#include <type_traits>

namespace vsc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

static constexpr int CM_ROWS = 4;    // output rows per block (one per two waves)
static constexpr int CM_PX = 32;     // output pixels per row per block
static constexpr int CM_HALO = 4;    // f2 halo (max displacement supported)
static constexpr int CM_KC = 32;     // channels per chunk (one MFMA K step)

// element type traits: bytes per element, LDS pixel stride (elements)
template <int EB> struct CmLayout;
template <> struct CmLayout<2> { static constexpr int STRIDE = 40; };   // 80 B: 20 dwords
template <> struct CmLayout<1> { static constexpr int STRIDE = 40; };   // 40 B: 10 dwords

enum CmKind { CM_BF16 = 0, CM_F16 = 1, CM_FP8 = 2 };

template <int KIND>
__device__ inline f32x4 cm_mfma(const void* a, const void* b, f32x4 acc)
{
    if constexpr (KIND == CM_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(a),
                                                       *reinterpret_cast<const bf16x8*>(b), acc, 0, 0, 0);
    } else if constexpr (KIND == CM_F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const f16x8*>(a),
                                                      *reinterpret_cast<const f16x8*>(b), acc, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(*reinterpret_cast<const long*>(a),
                                                          *reinterpret_cast<const long*>(b), acc, 0, 0, 0);
    }
}

// One 8-byte LDS vector (GC = 8/EB channels of one pixel) for each of 4
// consecutive pixels, from GC channel-plane loads of those 4 pixels (NCHW):
// a register transpose with byte permutes.  raw[k] holds pixels 0..3 of
// channel k: 2 x 32 bits (16-bit elements) or 32 bits (FP8).
__device__ inline uint2 nchw_px16(const uint2 (&raw)[4], int j)
{
    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
    const bool hi = j >= 2;
    return make_uint2(__builtin_amdgcn_perm(hi ? raw[1].y : raw[1].x, hi ? raw[0].y : raw[0].x, sel),
                      __builtin_amdgcn_perm(hi ? raw[3].y : raw[3].x, hi ? raw[2].y : raw[2].x, sel));
}
__device__ inline uint2 nchw_px8(const uint32_t (&raw)[8], int j)
{
    const uint32_t sel = (uint32_t)j | ((uint32_t)(4 + j) << 8);
    const uint32_t t01 = __builtin_amdgcn_perm(raw[1], raw[0], sel), t23 = __builtin_amdgcn_perm(raw[3], raw[2], sel);
    const uint32_t t45 = __builtin_amdgcn_perm(raw[5], raw[4], sel), t67 = __builtin_amdgcn_perm(raw[7], raw[6], sel);
    return make_uint2(__builtin_amdgcn_perm(t23, t01, 0x05040100u), __builtin_amdgcn_perm(t67, t45, 0x05040100u));
}

template <int KIND, int MD, bool LEGACY, int DG, bool RUNS>
__device__ __forceinline__ void corr_mfma_tile(const void* __restrict__ f1v, const void* __restrict__ f2v,
                                               float* __restrict__ out, int C, int H, int W, const float* scale,
                                               int per_xcd, int blocks)
{
    constexpr int EB = (KIND == CM_FP8) ? 1 : 2;          // bytes per element
    constexpr int ST = CmLayout<EB>::STRIDE;              // LDS pixel stride in elements
    constexpr int P = 2 * MD + 1, G = P / DG;
    static_assert(P % DG == 0, "displacement groups of equal size");
    constexpr int BR = CM_ROWS + DG - 1, BC = CM_PX + 2 * CM_HALO;
    using E = typename std::conditional<EB == 2, uint16_t, uint8_t>::type;
    // LDS: the operand tiles during the channel loop, then the whole output
    // tile [row][plane][32 px] at a plane pitch of 36 floats (the operand
    // tiles are dead by then): the 16 lanes of a K group write 16 planes at
    // once, which a 32-float pitch puts on the same banks
    constexpr int SP = CM_PX + 4, PL = DG * P;
    constexpr int A_BYTES = CM_ROWS * CM_PX * ST * EB, B_BYTES = BR * BC * ST * EB;
    constexpr int OUT_BYTES = CM_ROWS * PL * SP * 4;
    constexpr int LDS_BYTES = (A_BYTES + B_BYTES) > OUT_BYTES ? (A_BYTES + B_BYTES) : OUT_BYTES;
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDS_BYTES];
    E (*sA)[CM_PX][ST] = reinterpret_cast<E (*)[CM_PX][ST]>(lds);
    E (*sB)[BC][ST] = reinterpret_cast<E (*)[BC][ST]>(lds + A_BYTES);
    float (*stage)[PL][SP] = reinterpret_cast<float (*)[PL][SP]>(lds);

    int dg, n, h0, w0;
    if constexpr (RUNS) {   // runs of neighbouring tiles on an XCD, a tile's groups together
        int t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
        if (t >= blocks) return;
        const int tiles = (W + CM_PX - 1) / CM_PX, rows = (H + CM_ROWS - 1) / CM_ROWS;
        dg = t % G;
        t /= G;
        w0 = t % tiles * CM_PX;
        t /= tiles;
        h0 = t % rows * CM_ROWS;
        n = t / rows;
    } else {
        const int tiles = gridDim.x / G;
        dg = blockIdx.x / tiles;
        w0 = blockIdx.x % tiles * CM_PX;
        h0 = blockIdx.y * CM_ROWS;
        n = blockIdx.z;
    }
    const long long HW = (long long)H * W;
    const E* f1 = static_cast<const E*>(f1v) + (long long)n * C * HW;
    const E* f2 = static_cast<const E*>(f2v) + (long long)n * C * HW;
    const int tid = threadIdx.x;
    const int q = tid / 64, lane = tid % 64;
    const int qr = q >> 1, seg = q & 1;         // output row in the block, 16-pixel segment
    const int lr = lane % 16, lg = lane / 16;   // operand row/column, K group

    f32x4 acc[DG][2];
#pragma unroll
    for (int d = 0; d < DG; ++d)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[d][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // Staging units: GC channels x 4 pixels of a row of one of the tiles.  A unit
    // loads its 4 pixels of GC channel planes, whatever their alignment, and
    // writes them channels-last into LDS.  One that hangs over the right edge is
    // read further left and shifted (zeros come in); images less than 4 pixels
    // wide are read pixel by pixel.
    constexpr int GC = 8 / EB, CG = CM_KC / GC;
    constexpr int NA4 = CG * CM_ROWS * (CM_PX / 4), NB4 = CG * BR * (BC / 4), NU4 = NA4 + NB4;
    constexpr int RU4 = (NU4 + 511) / 512;
    using Raw = typename std::conditional<EB == 2, uint2, uint32_t>::type;
    typedef uint32_t U2 __attribute__((ext_vector_type(2), aligned(2)));
    typedef uint32_t U1 __attribute__((aligned(1)));
    Raw raw[RU4][GC];
    const E* src[RU4];
    int cfirst[RU4], shift[RU4];
    E* dst[RU4];
#pragma unroll
    for (int k = 0; k < RU4; ++k) {
        const int u = tid + 512 * k;
        const bool inA = u < NA4;
        const int ul = inA ? u : u - NA4;
        const int rows = inA ? CM_ROWS : BR, groups = inA ? CM_PX / 4 : BC / 4;
        const int g = ul % groups, r = (ul / groups) % rows, cg = ul / (groups * rows);
        const int gh = inA ? h0 + r : h0 - MD + dg * DG + r;
        const int gw = inA ? w0 + 4 * g : w0 - CM_HALO + 4 * g;
        const bool ok = u < NU4 && gh >= 0 && gh < H && gw >= 0 && gw < W;
        const int xs = W >= 4 ? min(gw, W - 4) : gw;
        src[k] = (inA ? f1 : f2) + (ok ? (long long)cg * GC * HW + (long long)gh * W + xs : 0);
        shift[k] = W >= 4 ? gw - xs : W - gw;         // (narrow images: pixels left)
        cfirst[k] = ok ? cg * GC : 1 << 30;           // nothing to load
        dst[k] = u >= NU4 ? nullptr : inA ? &sA[r][4 * g][cg * GC] : &sB[r][4 * g][cg * GC];
    }
    auto fetch = [&](int c0) {
#pragma unroll
        for (int k = 0; k < RU4; ++k) {
            const E* s = src[k] + (long long)c0 * HW;
#pragma unroll
            for (int j = 0; j < GC; ++j) {
                Raw v{};
                if (c0 + j + cfirst[k] < C) {
                    const E* p = s + j * HW;
                    if (W >= 4) {
                        if constexpr (EB == 2) {
                            const U2 t = *reinterpret_cast<const U2*>(p);
                            v = make_uint2(t.x, t.y);
                        } else {
                            v = *reinterpret_cast<const U1*>(p);
                        }
                    } else {
                        if constexpr (EB == 2) {
                            v.x = p[0] | (shift[k] > 1 ? (uint32_t)p[1] << 16 : 0u);
                            v.y = shift[k] > 2 ? p[2] : 0u;
                        } else {
                            v = p[0] | (shift[k] > 1 ? (uint32_t)p[1] << 8 : 0u) | (shift[k] > 2 ? (uint32_t)p[2] << 16 : 0u);
                        }
                    }
                }
                raw[k][j] = v;
            }
        }
    };
    auto stage_chunk = [&]() {
#pragma unroll
        for (int k = 0; k < RU4; ++k) {
            if (!dst[k]) continue;
            if (W >= 4 && shift[k] > 0 && shift[k] < 4) {
#pragma unroll
                for (int j = 0; j < GC; ++j) {
                    if constexpr (EB == 2) {
                        const uint64_t t = ((uint64_t)raw[k][j].y << 32 | raw[k][j].x) >> (16 * shift[k]);
                        raw[k][j] = make_uint2((uint32_t)t, (uint32_t)(t >> 32));
                    } else {
                        raw[k][j] >>= 8 * shift[k];
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint2 v;
                if constexpr (EB == 2) v = nchw_px16(raw[k], j);
                else v = nchw_px8(raw[k], j);
                *reinterpret_cast<uint2*>(dst[k] + j * ST) = v;
            }
        }
    };

    fetch(0);
    for (int c0 = 0; c0 < C; c0 += CM_KC) {
        __syncthreads();
        stage_chunk();
        __syncthreads();
        if (c0 + CM_KC < C) fetch(c0 + CM_KC);
        // A operand: pixel lr of this wave's segment, channels 8*lg .. 8*lg+7
        const E* pa = &sA[qr][16 * seg + lr][8 * lg];
#pragma unroll
        for (int d = 0; d < DG; ++d) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const E* pb = &sB[qr + d][16 * seg + 8 * t + lr][8 * lg];
                acc[d][t] = cm_mfma<KIND>(pa, pb, acc[d][t]);
            }
        }
    }

    // FP8: one dequantisation factor s = s1*s2 (per-channel factors are folded
    // into the operands by the equalisation, see vsc_quantize_fp8_pair)
    const float sc = scale ? *scale : 1.0f;
    // diagonals -> stage[row][plane][pixel]: lane holds G[4*lg + r][lr + 8*t]
    __syncthreads();
#pragma unroll
    for (int d = 0; d < DG; ++d)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 4 * lg + r, j = lr + 8 * t;
                const int dx = j - i - CM_HALO;
                if (dx >= -MD && dx <= MD && !(t == 1 && j < 16)) {
                    float v = acc[d][t][r];
                    if (KIND == CM_FP8) v = v * sc;
                    if (LEGACY) v = v / (float)C;
                    stage[qr][d * P + dx + MD][16 * seg + i] = v;
                }
            }
    __syncthreads();
    // each group of 8 lanes writes one 128-byte row segment of one plane, 16
    // bytes a lane whatever the alignment (the tail of a row pixel by pixel); the
    // cost volume is not re-read by this kernel: non-temporal stores
    float* o0 = out + ((long long)n * P * P + dg * PL) * HW;
    for (int e = tid; e < CM_ROWS * PL * CM_PX / 4; e += 512) {
        const int x = 4 * (e % (CM_PX / 4)), pl = (e / (CM_PX / 4)) % PL, r = e / (CM_PX / 4 * PL);
        const int h = h0 + r, w = w0 + x;
        if (h >= H) continue;
        float* o = o0 + pl * HW + (long long)h * W + w;
        if (w + 3 < W) {
            typedef float F4U __attribute__((ext_vector_type(4), aligned(4)));
            __builtin_nontemporal_store(__builtin_bit_cast(F4U, *reinterpret_cast<const f32x4*>(&stage[r][pl][x])),
                                        reinterpret_cast<F4U*>(o));
        } else {
            for (int j = 0; j < 4; ++j)
                if (w + j < W) __builtin_nontemporal_store(stage[r][pl][x + j], o + j);
        }
    }
}

// Waves per SIMD the registers are capped for: three blocks per CU (four in
// FP8, whose staging holds less) with 3 or fewer vertical displacements a
// block, two with more (480x272x32, FP8: 24.6 us at 4, 21.2 at 6, 19.5 at 8;
// BF16: 32.6, 26.0, 35.0 with spills).
template <int KIND, int MD, bool LEGACY, int DG, bool RUNS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(DG > 3 ? 4 : KIND == CM_FP8 ? 8 : 6)))
void k_corr_mfma(const void* __restrict__ f1, const void* __restrict__ f2, float* __restrict__ out, int C, int H, int W,
                 const float* scale, int per_xcd, int blocks)
{
    corr_mfma_tile<KIND, MD, LEGACY, DG, RUNS>(f1, f2, out, C, H, W, scale, per_xcd, blocks);
}

template <int KIND, int MD, int DG, bool RUNS>
static void launch_mfma_dg(const void* f1, const void* f2, float* out, int N, int C, int H, int W, bool legacy,
                           const float* scale, hipStream_t s)
{
    dim3 grid((W + CM_PX - 1) / CM_PX * ((2 * MD + 1) / DG), (H + CM_ROWS - 1) / CM_ROWS, N);
    const int blocks = (int)(grid.x * grid.y * grid.z), per_xcd = (blocks + 7) / 8;
    if (RUNS) grid = dim3(8 * per_xcd);
    if (legacy)
        hipLaunchKernelGGL((k_corr_mfma<KIND, MD, true, DG, RUNS>), grid, dim3(512), 0, s, f1, f2, out, C, H, W, scale, per_xcd, blocks);
    else
        hipLaunchKernelGGL((k_corr_mfma<KIND, MD, false, DG, RUNS>), grid, dim3(512), 0, s, f1, f2, out, C, H, W, scale, per_xcd, blocks);
}

// Vertical displacements per block, and the blocks' order (md = 4; T: tiles of
// 32 x 4 pixels; us in BF16 | FP8 and pixels x channels).
//
// One a block while all of those still fit the chip at once: 30x17x196, T = 5,
// 10.6 with one, 13.1 with three, 25.1 with nine.
//
// Above that a block with all nine needs 72 sums a lane, so two stand on a CU,
// each a chain of loads, products, staging and stores; thirds stage half as much
// again but overlap three or four: 240x136x64, T = 272, 16.1 | 13.2 with nine, 14.7
// | 10.7 with three; 400x200x128, 650, 43.2 | 32.0 and 37.5 | 23.2.  Nine where they
// fill their rounds of 512: 320x180x128, 450, 25.4 and 28.9 (FP8, whose thirds stand
// four on a CU, 18.8 and 18.8); 480x272x64, 1020, 32.6 and 35.8 (FP8 25.2 and 24.8);
// FP8 only with one chunk: 480x272x32 19.2 and 20.7.
//
// Blocks go to the XCDs in runs of neighbouring tiles, a tile's thirds together,
// so that its f2 rows come from that XCD's L2 after the first, and the parts of a
// line of output at two tiles' border meet there: 320x180x128 38.0 | 24.0 in rows
// of blocks, 28.9 | 18.8 so; 213x119x64 14.3 and 11.9; 477x272x32 36.9 | 35.9 and 30.3
// | 27.0.  Rows of whole lines (W a multiple of 16) with up to 16 channels are bound
// by their stores and the faster in rows of blocks (320x192x8 with nine 12.3 | 11.1,
// 12.8 | 11.8 in runs; FP8's thirds up to 32, 384x200x32 14.0 and 14.6), and a grid of
// 8 or 16 tiles across keeps a column on an XCD in rows too (240x136x64 14.1 | 10.4 and
// 14.7 | 10.7; from T = 384 runs are no slower).  Rows that are not take thirds, whose
// stores meet sooner (476x272x32 26.0 | 21.6, with nine 35.1 | 27.9; 1916x1080x8 340 |
// 346 and 411 | 389), but for maps of one group of pixels (4x2000x32 13.0 | 11.9 in
// rows, 14.7 | 13.0 in runs of thirds; 3x2000x196, read pixel by pixel, 44.5 in runs with
// nine, 51.8 with three).
template <int KIND, int MD>
static void launch_mfma(const void* f1, const void* f2, float* out, int N, int C, int H, int W, bool legacy,
                        const float* scale, hipStream_t s)
{
    constexpr int P = 2 * MD + 1;
    const long long T = (long long)((W + CM_PX - 1) / CM_PX) * ((H + CM_ROWS - 1) / CM_ROWS) * N;
    auto go = [&](auto launch) { launch(f1, f2, out, N, C, H, W, legacy, scale, s); };
    if constexpr (MD != 4) {
        if (MD >= 2 && T * P <= 512) go(launch_mfma_dg<KIND, MD, 1, false>);
        else go(launch_mfma_dg<KIND, MD, P, false>);
    } else {
        const bool lines = W % 16 == 0 || W <= 4, nine = lines && T >= 0.85 * 512 * ((T + 511) / 512) && (KIND != CM_FP8 || C <= CM_KC);
        const bool near = W == 4 || (lines && (W + CM_PX - 1) / CM_PX % 8 == 0 && T < 384);
        // (the blocks' numbers and their threads fit 32 bits)
        const bool runs = (!lines || W < 4 || C > (nine || KIND != CM_FP8 ? 16 : CM_KC)) && !near && T < (1 << 20);
        if (T * P <= 256) go(launch_mfma_dg<KIND, MD, 1, false>);
        else if (nine) go(runs ? launch_mfma_dg<KIND, MD, P, true> : launch_mfma_dg<KIND, MD, P, false>);
        else go(runs ? launch_mfma_dg<KIND, MD, 3, true> : launch_mfma_dg<KIND, MD, 3, false>);
    }
}

template <int KIND>
static int dispatch_md(const void* f1, const void* f2, float* out, int N, int C, int H, int W, int md, bool legacy,
                       const float* scale, hipStream_t s)
{
    switch (md) {
        case 0: launch_mfma<KIND, 0>(f1, f2, out, N, C, H, W, legacy, scale, s); break;
        case 1: launch_mfma<KIND, 1>(f1, f2, out, N, C, H, W, legacy, scale, s); break;
        case 2: launch_mfma<KIND, 2>(f1, f2, out, N, C, H, W, legacy, scale, s); break;
        case 3: launch_mfma<KIND, 3>(f1, f2, out, N, C, H, W, legacy, scale, s); break;
        case 4: launch_mfma<KIND, 4>(f1, f2, out, N, C, H, W, legacy, scale, s); break;
        default:
            return set_error(VSC_E_UNSUPPORTED,
                             "vsc_correlation_forward: reduced-precision correlation supports max_displacement <= 4");
    }
    return check_launch("correlation mfma");
}

size_t corr_mfma_workspace_bytes(int N, int C, int H, int W, int in_dtype)
{
    if (in_dtype != VSC_BF16 && in_dtype != VSC_F16 && in_dtype != VSC_FP8E4M3) return 0;
    const size_t eb = in_dtype == VSC_FP8E4M3 ? 1 : 2;
    const size_t CP = (size_t)(C + CM_KC - 1) / CM_KC * CM_KC;
    const size_t one = ((size_t)N * H * W * CP * eb + 255) / 256 * 256;
    return 2 * one;
}

// Whether the entry points that take or hold a workspace ask for one.  The
// kernel reads its operands in place at any width and alignment; the requirement
// for other widths and alignments is the entry points' contract.
bool corr_mfma_asks_workspace(const void* f1, const void* f2, int W, int in_dtype)
{
    const uintptr_t align = in_dtype == VSC_FP8E4M3 ? 4 : 8;
    return W % 4 != 0 || reinterpret_cast<uintptr_t>(f1) % align != 0 || reinterpret_cast<uintptr_t>(f2) % align != 0;
}

int corr_mfma_dispatch(const void* f1, const void* f2, float* out, int N, int C, int H, int W, int md, int legacy,
                       int in_dtype, const float* chan_scale, hipStream_t s)
{
    if (md > 4)
        return set_error(VSC_E_UNSUPPORTED,
                         "vsc_correlation_forward: reduced-precision correlation supports max_displacement <= 4");
    if (in_dtype == VSC_BF16) return dispatch_md<CM_BF16>(f1, f2, out, N, C, H, W, md, legacy, nullptr, s);
    if (in_dtype == VSC_F16) return dispatch_md<CM_F16>(f1, f2, out, N, C, H, W, md, legacy, nullptr, s);
    if (in_dtype == VSC_FP8E4M3) return dispatch_md<CM_FP8>(f1, f2, out, N, C, H, W, md, legacy, chan_scale, s);
    return set_error(VSC_E_DTYPE, "vsc_correlation_forward: unsupported input type");
}

// ---------------------------------------------------------------------------
// conversions
// ---------------------------------------------------------------------------
// binary32 -> OCP FP8 E4M3 (bias 7, max 448, no infinities), round to nearest
// even, saturating to +-448; NaN -> 0x7F.
__host__ __device__ inline uint8_t f32_to_e4m3(float x)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const uint32_t sign = (u >> 24) & 0x80u;
    const uint32_t au = u & 0x7FFFFFFFu;
    if (au > 0x7F800000u) return 0x7F;
    const float a = __builtin_bit_cast(float, au);
    uint32_t code;
    if (a >= 448.0f) {
        code = 0x7E;
    } else if (a < 0.015625f) {                       // below 2^-6: subnormal grid of 2^-9
        code = (uint32_t)__builtin_rintf(a * 512.0f);  // exact scaling, RNE; 8 -> min normal 0x08
    } else {
        int e = (int)(au >> 23) - 127;                 // -6 .. 8
        uint32_t mant = au & 0x7FFFFFu;
        uint32_t keep = mant >> 20, rest = mant & 0xFFFFFu;
        if (rest > 0x80000u || (rest == 0x80000u && (keep & 1u))) ++keep;
        if (keep == 8u) { keep = 0; ++e; }
        if (e > 8 || (e == 8 && keep == 7u)) code = 0x7E;
        else code = ((uint32_t)(e + 7) << 3) | keep;
    }
    return (uint8_t)(sign | code);
}

__global__ void k_to_bf16(const float* in, uint16_t* out, long long n)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f32_to_bf16(in[i]);
}

__global__ void k_to_f16(const float* in, _Float16* out, long long n)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (_Float16)in[i];
}

__global__ void k_to_e4m3(const float* in, uint8_t* out, long long n)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f32_to_e4m3(in[i]);
}

// ---------------------------------------------------------------------------
// FP8 pair quantisation (SmoothQuant-style equalisation)
// ---------------------------------------------------------------------------
// per-channel max |f| over N, H, W, as ordered float bits (non-negative floats
// order like their bit patterns), accumulated with atomicMax
// mx[t*C + c] = largest magnitude of channel c of tensor t (0: f1, 1: f2);
// blockIdx.x = t * blocks of a plane + block.  4096 pixels and more a block and
// one atomic each: with 256 blocks' waves all updating a channel's word the
// updates alone took 60 us.
__global__ __launch_bounds__(256) void k_chan_absmax(const float* f1, const float* f2, uint32_t* mx, int C,
                                                     long long HW)
{
    const int gx = gridDim.x / 2, t = (int)blockIdx.x >= gx;
    const int c = blockIdx.y, n = blockIdx.z, bx = blockIdx.x - t * gx;
    const float* p = (t ? f2 : f1) + ((long long)n * C + c) * HW;
    typedef float F4U __attribute__((ext_vector_type(4), aligned(4)));
    float m = 0.0f;
    const long long step = (long long)gx * 1024;
    for (long long i = (long long)bx * 1024 + threadIdx.x * 4; i < HW; i += step) {
        if (i + 4 <= HW) {
            const F4U v = *reinterpret_cast<const F4U*>(p + i);
            m = fmaxf(fmaxf(fmaxf(m, fabsf(v.x)), fmaxf(fabsf(v.y), fabsf(v.z))), fabsf(v.w));
        } else {
            for (long long j = i; j < HW; ++j) m = fmaxf(m, fabsf(p[j]));
        }
    }
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    __shared__ float s_m[4];
    if ((threadIdx.x & 63) == 0) s_m[threadIdx.x / 64] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
        atomicMax(&mx[t * C + c], __builtin_bit_cast(uint32_t, m));
    }
}

__global__ void k_zero_u32(uint32_t* p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// r_c = sqrt(max2_c / max1_c) (1 when either is 0); s1 = max_c(max1_c r_c)/448,
// s2 = max_c(max2_c / r_c)/448; writes r[c], inv scales and scale = s1*s2.  A
// thread per channel (one thread for all took 40 us of 196 channels' divisions
// and roots in a row).
__global__ __launch_bounds__(256) void k_fp8_scales(const uint32_t* mx1, const uint32_t* mx2, float* r, float* sc,
                                                    float* scale, int C)
{
    __shared__ float s_m[2][4];
    float m1 = 0.0f, m2 = 0.0f;
    for (int c = threadIdx.x; c < C; c += 256) {
        const float a = __builtin_bit_cast(float, mx1[c]), b = __builtin_bit_cast(float, mx2[c]);
        const float rc = (a > 0.0f && b > 0.0f) ? sqrtf(b / a) : 1.0f;
        r[c] = rc;
        m1 = fmaxf(m1, a * rc);
        m2 = fmaxf(m2, b / rc);
    }
    for (int off = 32; off > 0; off >>= 1) {
        m1 = fmaxf(m1, __shfl_xor(m1, off));
        m2 = fmaxf(m2, __shfl_xor(m2, off));
    }
    if ((threadIdx.x & 63) == 0) {
        s_m[0][threadIdx.x / 64] = m1;
        s_m[1][threadIdx.x / 64] = m2;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < 4; ++w) {
        m1 = fmaxf(m1, s_m[0][w]);
        m2 = fmaxf(m2, s_m[1][w]);
    }
    const float s1 = m1 > 0.0f ? m1 / 448.0f : 1.0f;
    const float s2 = m2 > 0.0f ? m2 / 448.0f : 1.0f;
    sc[0] = s1 * s2;
    sc[1] = s1;
    sc[2] = s2;
    *scale = s1 * s2;
}

// Both tensors (blockIdx.y), 4 neighbouring pixels of a plane per thread, loaded
// and stored together whatever their alignment; blockIdx.x = (plane - first) * chunks + chunk
__global__ __launch_bounds__(256) void k_fp8_quant(const float* f1, const float* f2, uint8_t* q1, uint8_t* q2,
                                                   const float* r, const float* sc, int C, long long HW, int chunks,
                                                   long long first)
{
    typedef float F4U __attribute__((ext_vector_type(4), aligned(4)));
    typedef uint32_t U1 __attribute__((aligned(1)));
    const unsigned slot = blockIdx.x / chunks;
    const long long pl = first + slot;
    const long long i = ((long long)(blockIdx.x - slot * chunks) * 256 + threadIdx.x) * 4;
    if (i >= HW) return;
    const bool second = blockIdx.y != 0;
    const float rc = r[pl % C], s = sc[second ? 2 : 1];
    const float* f = (second ? f2 : f1) + pl * HW + i;
    uint8_t* q = (second ? q2 : q1) + pl * HW + i;
    const int n = (int)(HW - i < 4 ? HW - i : 4);
    float v[4];
    if (n == 4) {
        const F4U x = *reinterpret_cast<const F4U*>(f);
        for (int j = 0; j < 4; ++j) v[j] = x[j];
    } else {
        for (int j = 0; j < 4; ++j) v[j] = j < n ? f[j] : 0.0f;
    }
    uint32_t pk = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) pk |= (uint32_t)f32_to_e4m3((second ? v[j] / rc : v[j] * rc) / s) << (8 * j);
    if (n == 4) *reinterpret_cast<U1*>(q) = pk;
    else
        for (int j = 0; j < n; ++j) q[j] = (uint8_t)(pk >> (8 * j));
}

}  // namespace vsc

using namespace vsc;

extern "C" size_t vsc_quantize_fp8_pair_workspace_size(int C)
{
    return C < 1 ? 0 : (size_t)(3 * C + 4) * 4;
}

// workspace: vsc_quantize_fp8_pair_workspace_size(C) bytes, or NULL to
// allocate it stream-ordered for this call
static int quantize_fp8_pair(const float* f1, const float* f2, uint8_t* q1, uint8_t* q2, float* scale, int N, int C,
                             int H, int W, void* workspace, hipStream_t s)
{
    if (!f1 || !f2 || !q1 || !q2 || !scale) return set_error(VSC_E_INVALID, "vsc_quantize_fp8_pair: null pointer");
    if (N < 1 || C < 1 || H < 1 || W < 1) return set_error(VSC_E_INVALID, "vsc_quantize_fp8_pair: empty tensor");
    const long long HW = (long long)H * W, planes = (long long)N * C;
    // workspace: 2*C maxima + C equalisation factors + 3 scales
    void* ws = workspace;
    int rc;
    if (!ws && (rc = check_hip(hipMallocAsync(&ws, vsc_quantize_fp8_pair_workspace_size(C), s),
                               "vsc_quantize_fp8_pair workspace")))
        return rc;
    uint32_t* mx = static_cast<uint32_t*>(ws);
    float* r = reinterpret_cast<float*>(mx + 2 * C);
    float* sc = r + C;
    hipLaunchKernelGGL(k_zero_u32, dim3((2 * C + 255) / 256), dim3(256), 0, s, mx, 2 * C);
    const unsigned gx = (unsigned)std::min<long long>((HW + 4095) / 4096, 16);
    hipLaunchKernelGGL(k_chan_absmax, dim3(2 * gx, C, N), dim3(256), 0, s, f1, f2, mx, C, HW);
    hipLaunchKernelGGL(k_fp8_scales, dim3(1), dim3(256), 0, s, mx, mx + C, r, sc, scale, C);
    // (a launch holds fewer than 2^32 threads along a dimension: many small planes take several)
    const int chunks = (int)((HW + 1023) / 1024);
    const long long most = std::max(1LL, (1LL << 23) / chunks);
    for (long long first = 0; first < planes; first += most)
        hipLaunchKernelGGL(k_fp8_quant, dim3((unsigned)(std::min(most, planes - first) * chunks), 2), dim3(256), 0, s, f1, f2, q1, q2,
                           r, sc, C, HW, chunks, first);
    rc = check_launch("vsc_quantize_fp8_pair");
    if (workspace) return rc;
    const int rc2 = check_hip(hipFreeAsync(ws, s), "vsc_quantize_fp8_pair workspace free");
    return rc ? rc : rc2;
}

extern "C" int vsc_quantize_fp8_pair(const float* f1, const float* f2, uint8_t* q1, uint8_t* q2, float* scale, int N,
                                     int C, int H, int W, vsc_hip_stream stream)
{
    return quantize_fp8_pair(f1, f2, q1, q2, scale, N, C, H, W, nullptr, as_stream(stream));
}

extern "C" int vsc_quantize_fp8_pair_ws(const float* f1, const float* f2, uint8_t* q1, uint8_t* q2, float* scale,
                                        int N, int C, int H, int W, void* workspace, size_t workspace_bytes,
                                        vsc_hip_stream stream)
{
    if (!workspace || workspace_bytes < vsc_quantize_fp8_pair_workspace_size(C))
        return set_error(VSC_E_INVALID, "vsc_quantize_fp8_pair_ws: workspace missing or smaller than "
                                        "vsc_quantize_fp8_pair_workspace_size()");
    return quantize_fp8_pair(f1, f2, q1, q2, scale, N, C, H, W, workspace, as_stream(stream));
}

extern "C" int vsc_convert_f32(const float* in, void* out, size_t count, int out_dtype, vsc_hip_stream stream)
{
    if (!in || !out) return set_error(VSC_E_INVALID, "vsc_convert_f32: null pointer");
    if (count == 0) return VSC_OK;
    hipStream_t s = as_stream(stream);
    const long long n = (long long)count;
    const unsigned g = (unsigned)((n + 255) / 256);
    if (out_dtype == VSC_BF16)
        hipLaunchKernelGGL(k_to_bf16, dim3(g), dim3(256), 0, s, in, static_cast<uint16_t*>(out), n);
    else if (out_dtype == VSC_F16)
        hipLaunchKernelGGL(k_to_f16, dim3(g), dim3(256), 0, s, in, static_cast<_Float16*>(out), n);
    else if (out_dtype == VSC_FP8E4M3)
        hipLaunchKernelGGL(k_to_e4m3, dim3(g), dim3(256), 0, s, in, static_cast<uint8_t*>(out), n);
    else
        return set_error(VSC_E_DTYPE, "vsc_convert_f32: out_dtype must be BF16, F16 or FP8E4M3");
    return check_launch("vsc_convert_f32");
}
