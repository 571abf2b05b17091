// ORT custom-op kernels for gfx950: "Correlation" (9x9 cost volume) and
// "Warp" (bilinear backward warp), NCHW in / NCHW out, with the attribute and
// shape contract of src/ort_custom_ops.
#include "vsc_internal.h"

#include <algorithm>
#include <string>

namespace vsc {

// ---------------------------------------------------------------------------
// Correlation, FP32, sequential-in-c accumulation (the order of the reference
// CPU op, correlation.cc:163-177: *dst = 0; *dst += v1*v2 for c = 0..C-1).
//
// A block owns a tile of 8 rows x 8*QX pixels of one image and DG of the
// vertical displacements (blockIdx.z = item * (P / DG) + group).  A wave takes
// one vertical displacement and one of XS groups of horizontal ones; its lane
// (row, group of QX pixels) keeps QX x P/XS sums in registers (QX = 4: 12 f2
// values from LDS feed 36 multiply-adds).  Channels stream through LDS CC at a
// time: the f1 tile and the f2 rows that the block's displacements reach (a
// 4-pixel halo in x), zeros outside the image (acc + (+-0) == acc for the
// values that occur, so zero terms leave every bit unchanged).
//
// Staging.  A thread owns one 4-pixel slot of the tiles for the whole call and
// every CPT-th channel of it: its addresses are one pointer plus multiples of a
// plane, and all loads of the next chunk are in flight during this one's sums.
// The loads are 16 bytes wide whatever the alignment; a slot over the right edge
// is read further left and shifted.  (One pixel a load with its own index
// arithmetic took 4 us a chunk: 17x30x196 28.4 us, now 12.9; 480x272x32 34.9 us,
// now 24.1, its multiplications and additions alone 17.)  This staging
// replaces the reference's channels-last rearrange kernels and their per-call
// cudaMalloc (correlation_cuda.cu:32-95,365-370).  Output rows are written 4*QX
// bytes a lane, again whatever the alignment (479x271x32: 115 us with 4-byte
// stores where rows are not aligned, now 44).
// ---------------------------------------------------------------------------
static constexpr int CF_TH = 8, CF_HALO = 4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));

// CCT: channels of a chunk, rounded to what the threads take in whole passes.
// Needs W >= 4.
template <int MD, bool LEGACY, int QX, int DG, int XS, int CCT>
__global__ __launch_bounds__(64 * DG * XS) void k_corr_f32(const float* __restrict__ f1, const float* __restrict__ f2,
                                                           float* __restrict__ out, int C, int H, int W)
{
    constexpr int P = 2 * MD + 1, XG = P / XS, G = DG > P ? 1 : P / DG;
    static_assert(P % XS == 0 && (DG > P || P % DG == 0), "displacement groups of equal size");
    constexpr int TW = 8 * QX, NTH = 64 * DG * XS, SH = CF_TH + (DG > P ? P : DG) - 1;
    // f2 row pitch: the 1-pixel tile's lanes read 8 rows x 8 neighbouring
    // pixels at once; 24 floats put those rows on distinct banks (16 would not)
    constexpr int PITCH = QX == 1 ? 24 : TW + 2 * CF_HALO;
    constexpr int S1 = TW / 4, S2 = S1 + 2 * CF_HALO / 4;
    constexpr int N1 = CF_TH * S1, NS = N1 + S2 * SH;   // 4-pixel slots of a channel: f1 tile, both tiles
    static_assert(NS <= NTH, "a slot each");
    // channels of one pass of the threads, passes and channels of a chunk
    constexpr int CPT = NTH / NS, K = CCT / CPT > 1 ? CCT / CPT : 1, CC = CPT * K;
    __shared__ __attribute__((aligned(16))) float s1[CC][CF_TH * TW];
    __shared__ __attribute__((aligned(16))) float s2[CC][SH * PITCH];

    const int n = blockIdx.z / G, dg = blockIdx.z % G;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int dl = wave / XS, x0 = (wave % XS) * XG;
    const int d = dg * DG + dl;
    const int row = lane / 8, px = lane % 8 * QX;
    const int w0 = blockIdx.x * TW, h0 = blockIdx.y * CF_TH;
    const long long HW = (long long)H * W;

    const int slot = tid % NS, cl = tid / NS;
    const bool in1 = slot < N1;
    const int sr = in1 ? slot / S1 : (slot - N1) / S2, sq = in1 ? slot % S1 : (slot - N1) % S2;
    const int gy = in1 ? h0 + sr : h0 - MD + dg * DG + sr;
    const int gx = in1 ? w0 + 4 * sq : w0 - CF_HALO + 4 * sq;
    const bool ok = cl < CPT && gy >= 0 && gy < H && gx >= 0 && gx < W;
    const int xs = min(gx, W - 4), shift = gx - xs;     // a slot over the right edge is read further left and shifted
    const float* src = (in1 ? f1 : f2) + ((long long)n * C + cl) * HW + (ok ? (long long)gy * W + xs : 0);
    float* dst = in1 ? &s1[0][0] + cl * (CF_TH * TW) + sr * TW + 4 * sq
                     : &s2[0][0] + cl * (SH * PITCH) + sr * PITCH + 4 * sq;
    const int dpitch = CPT * (in1 ? CF_TH * TW : SH * PITCH);

    f32x4u_t rg[K];
    auto fetch = [&](int c0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            f32x4u_t v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (ok && c0 + cl + CPT * k < C)
                v = *reinterpret_cast<const f32x4u_t*>(src + (long long)(c0 + CPT * k) * HW);
            rg[k] = v;
        }
    };
    float acc[QX][XG];
#pragma unroll
    for (int x = 0; x < QX; ++x)
#pragma unroll
        for (int k = 0; k < XG; ++k) acc[x][k] = 0.0f;
    fetch(0);
    for (int c0 = 0; c0 < C; c0 += CC) {
        __syncthreads();
        if (cl < CPT) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                f32x4u_t v = rg[k];
                if (shift & 1) v = f32x4u_t{v.y, v.z, v.w, 0.0f};
                if (shift & 2) v = f32x4u_t{v.z, v.w, 0.0f, 0.0f};
                *reinterpret_cast<f32x4_t*>(dst + k * dpitch) = __builtin_bit_cast(f32x4_t, v);
            }
        }
        __syncthreads();
        if (c0 + CC < C) fetch(c0 + CC);
        if (DG > P && dl >= P) continue;   // a wave that only stages
        const int cn = min(CC, C - c0);
        const float* pa = &s1[0][row * TW + px];
        const float* pb = &s2[0][(row + dl) * PITCH + px + CF_HALO - MD + x0];
#pragma unroll 8
        for (int cc = 0; cc < cn; ++cc) {
            float va[QX], vb[QX + XG - 1];
#pragma unroll
            for (int x = 0; x < QX; ++x) va[x] = pa[cc * (CF_TH * TW) + x];
#pragma unroll
            for (int x = 0; x < QX + XG - 1; ++x) vb[x] = pb[cc * (SH * PITCH) + x];
#pragma unroll
            for (int x = 0; x < QX; ++x)
#pragma unroll
                for (int k = 0; k < XG; ++k) acc[x][k] += va[x] * vb[x + k];
        }
    }
    const int h = h0 + row, w = w0 + px;
    if (h >= H || (DG > P && dl >= P)) return;
    float* o = out + ((long long)n * P * P + (long long)d * P + x0) * HW + (long long)h * W + w;
    if (QX > 1 && w + QX <= W) {
        typedef float V __attribute__((ext_vector_type(QX), aligned(4)));
#pragma unroll
        for (int k = 0; k < XG; ++k) {
            V v;
#pragma unroll
            for (int x = 0; x < QX; ++x) v[x] = LEGACY ? acc[x][k] / (float)C : acc[x][k];
            __builtin_nontemporal_store(v, reinterpret_cast<V*>(o + k * HW));
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < XG; ++k)
#pragma unroll
        for (int x = 0; x < QX; ++x)
            if (w + x < W) __builtin_nontemporal_store(LEGACY ? acc[x][k] / (float)C : acc[x][k], o + k * HW + x);
}

// Any displacement, FP32 or FP64: one thread per output element, sequential
// in c (correlation.cc:147-182).  Used for max_displacement > 4, FP64 and
// images less than 4 pixels wide.
template <typename T, bool LEGACY>
__global__ __launch_bounds__(256) void k_corr_generic(const T* __restrict__ f1, const T* __restrict__ f2,
                                                      T* __restrict__ out, int N, int C, int H, int W, int md)
{
    const int P = 2 * md + 1;
    const long long HW = (long long)H * W;
    const long long total = (long long)N * P * P * HW;
    const long long i = ((long long)blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int w = (int)(i % W);
    const int h = (int)((i / W) % H);
    const long long nd = i / HW;
    const int d = (int)(nd % (P * P));
    const int n = (int)(nd / (P * P));
    const int dy = d / P - md, dx = d % P - md;
    const int h2 = h + dy, w2 = w + dx;
    T acc = 0;
    if (h2 >= 0 && h2 < H && w2 >= 0 && w2 < W) {
        const T* a = f1 + (long long)n * C * HW + (long long)h * W + w;
        const T* b = f2 + (long long)n * C * HW + (long long)h2 * W + w2;
        for (int c = 0; c < C; ++c) acc += a[c * HW] * b[c * HW];
    }
    out[i] = LEGACY ? acc / (T)C : acc;
}

template <typename T>
static void launch_corr_generic(const T* f1, const T* f2, T* out, int N, int C, int H, int W, int md, bool legacy, hipStream_t s)
{
    // (a launch holds fewer than 2^32 threads along a dimension)
    const long long blocks = ((long long)N * (2 * md + 1) * (2 * md + 1) * H * W + 255) / 256;
    const unsigned across = (unsigned)(blocks < (1 << 22) ? blocks : 1 << 22);
    const dim3 grid(across, (unsigned)((blocks + across - 1) / across));
    if (legacy) hipLaunchKernelGGL((k_corr_generic<T, true>), grid, dim3(256), 0, s, f1, f2, out, N, C, H, W, md);
    else hipLaunchKernelGGL((k_corr_generic<T, false>), grid, dim3(256), 0, s, f1, f2, out, N, C, H, W, md);
}

template <int MD, int QX, int DG, int XS, int CCT>
static void launch_corr_f32_q(const float* f1, const float* f2, float* out, int N, int C, int H, int W, bool legacy,
                              hipStream_t s)
{
    dim3 grid((W + 8 * QX - 1) / (8 * QX), (H + CF_TH - 1) / CF_TH, N * (DG > 2 * MD + 1 ? 1 : (2 * MD + 1) / DG));
    const dim3 block(64 * DG * XS);
    if (legacy)
        hipLaunchKernelGGL((k_corr_f32<MD, true, QX, DG, XS, CCT>), grid, block, 0, s, f1, f2, out, C, H, W);
    else
        hipLaunchKernelGGL((k_corr_f32<MD, false, QX, DG, XS, CCT>), grid, block, 0, s, f1, f2, out, C, H, W);
}

// The form by the number of 32x8 tiles, T.  Small levels are bound by the chain
// of their chunks, so they are cut into as many waves as there are CUs for, each
// with few sums and long chunks; large ones by LDS reads and the vector units,
// so a lane takes 4 pixels with all horizontal displacements and a block all
// vertical ones.  md = 4, us of the chosen form and of its two neighbours
// (pixels x channels, T):
//   30x17x196, 3      12.9 | 14.1 of the next
//   60x34x128, 10     10.9 of the one before | 10.9 | 11.9
//   120x68x96, 36     14.3 | 13.7 | 17.4
//   200x90x64, 84     25.1 | 16.3 | 20.0
//   240x150x32, 152   16.8 | 11.2 | 13.8
//   480x272x32, 510   39.4 | 24.1
// Other displacements: one small form and one large one (md = 0 with two waves
// that only stage).
template <int MD>
static void launch_corr_f32(const float* f1, const float* f2, float* out, int N, int C, int H, int W, bool legacy,
                            hipStream_t s)
{
    constexpr int P = 2 * MD + 1;
    const long long rows = (long long)((H + CF_TH - 1) / CF_TH) * N;
    long long T = (W + 31) / 32 * rows;
    // a map of one or two 8-pixel tiles across counts those, a quarter each (4x500x196, 63
    // tiles of 32 or 16 of 8: 32.8 us as the former, 14.0 as the latter)
    if (W <= 16 && T <= 120) T = ((W + 7) / 8 * rows + 3) / 4;
    if constexpr (MD == 4) {
        if (36 * T <= 256) launch_corr_f32_q<MD, 1, 1, 3, 64>(f1, f2, out, N, C, H, W, legacy, s);
        else if (12 * T <= 256) launch_corr_f32_q<MD, 1, 3, 3, 40>(f1, f2, out, N, C, H, W, legacy, s);
        else if (T <= 55) launch_corr_f32_q<MD, 1, 3, 3, 20>(f1, f2, out, N, C, H, W, legacy, s);
        else if (T <= 120) launch_corr_f32_q<MD, 2, 3, 1, 16>(f1, f2, out, N, C, H, W, legacy, s);
        else if (T < 256) launch_corr_f32_q<MD, 4, 3, 1, 16>(f1, f2, out, N, C, H, W, legacy, s);
        else launch_corr_f32_q<MD, 4, 9, 1, 4>(f1, f2, out, N, C, H, W, legacy, s);
    } else if constexpr (MD == 0) {
        if (T < 128) launch_corr_f32_q<MD, 1, 3, 1, 32>(f1, f2, out, N, C, H, W, legacy, s);
        else launch_corr_f32_q<MD, 4, 3, 1, 8>(f1, f2, out, N, C, H, W, legacy, s);
    } else {
        if (T < 128) launch_corr_f32_q<MD, 1, P % 3 == 0 ? 3 : P, 1, 32>(f1, f2, out, N, C, H, W, legacy, s);
        else launch_corr_f32_q<MD, 4, P, 1, 8>(f1, f2, out, N, C, H, W, legacy, s);
    }
}

// ---------------------------------------------------------------------------
// Warp (warp.cc:71-134 / warp_cuda.cu:28-84).  One thread per output pixel and
// group of WG_CH channels: the flow is read and the bilinear weights and in-bounds
// mask are computed once per group, then the planes are gathered with
// independent loads (the reference re-reads the flow once per channel,
// grid.y = C, and serialises nothing else).  FP32 weights; the reference evaluates
// weights in double for float tensors, so FP32 agrees to rounding, and the
// keep/zero decision (double)mask > 0.999 becomes mask >= 0.999f, the same
// threshold on the float grid (0.999f is the first float above 0.999).
// ---------------------------------------------------------------------------
static constexpr int WG_CH = 4;

// two neighbouring pixels of a plane row
template <typename T> struct Pair2;
template <> struct Pair2<float> { typedef float V __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct Pair2<double> { typedef double V __attribute__((ext_vector_type(2), aligned(8))); };

// A block takes 2^BITS columns, or 2^narrow of a map that is no wider (BITS = 0).
template <typename T, bool PAIR, int BITS>
__global__ __launch_bounds__(256) void k_warp(const T* __restrict__ in, const T* __restrict__ flow, T* __restrict__ out,
                                              int C, int H, int W, int narrow, int first)
{
    const int bits = BITS ? BITS : narrow;
    const int tiles = (W + (1 << bits) - 1) >> bits;
    const int x = (blockIdx.x % tiles << bits) + (threadIdx.x & ((1 << bits) - 1));
    const int y = blockIdx.y * (256 >> bits) + (threadIdx.x >> bits);
    const int n = blockIdx.z;
    const int c0 = first + blockIdx.x / tiles * WG_CH;
    const int c1 = min(C, c0 + WG_CH);
    if (x >= W || y >= H) return;
    const long long HW = (long long)H * W;
    const long long p = (long long)y * W + x;
    const T xf = (T)x + flow[(long long)n * 2 * HW + p];
    const T yf = (T)y + flow[(long long)n * 2 * HW + HW + p];
    const T xL = floor(xf), yT = floor(yf);
    const T alpha = xf - xL, beta = yf - yT;
    const T xR = xL + (T)1, yB = yT + (T)1;
    const bool mL = (T)0 <= xL && xL <= (T)(W - 1);
    const bool mR = (T)0 <= xR && xR <= (T)(W - 1);
    const bool mT = (T)0 <= yT && yT <= (T)(H - 1);
    const bool mB = (T)0 <= yB && yB <= (T)(H - 1);
    const T wTL = ((T)1 - alpha) * ((T)1 - beta);
    const T wTR = alpha * ((T)1 - beta);
    const T wBL = ((T)1 - alpha) * beta;
    const T wBR = alpha * beta;
    T mask = (T)0;
    mask = mask + (mT && mL ? wTL : (T)0);
    mask = mask + (mT && mR ? wTR : (T)0);
    mask = mask + (mB && mL ? wBL : (T)0);
    mask = mask + (mB && mR ? wBR : (T)0);
    bool keep;
    if constexpr (sizeof(T) == 4) keep = mask >= 0.999f;
    else keep = mask > 0.999;
    const long long base = (long long)n * C * HW;
    T* o = out + base + p;
    if (!keep) {
        for (int c = c0; c < c1; ++c) o[c * HW] = (T)0;
        return;
    }
    // All gathers are issued before any is used: from addresses
    // clamped into the image and into the group's channels, so every load is
    // valid; a corner outside the image is still left out of the sum below,
    // which keeps the reference's terms and order.  PAIR (W >= 2): the left and
    // right pixel of a row come with one 8-byte load, which halves what the
    // gathers cost; with that, groups of 4 channels beat 8 (480x272x32: 18.4 us
    // with single loads and 8 channels, 13.5 with pairs, 12.3 with 4 channels).
    const int iL = min(max((int)xL, 0), W - 1), iR = min(max((int)xR, 0), W - 1);
    const int iT = min(max((int)yT, 0), H - 1), iB = min(max((int)yB, 0), H - 1);
    const long long oTL = (long long)iT * W + iL, oTR = (long long)iT * W + iR;
    const long long oBL = (long long)iB * W + iL, oBR = (long long)iB * W + iR;
    const T* src = in + base;
    T vTL[WG_CH], vTR[WG_CH], vBL[WG_CH], vBR[WG_CH];
    if constexpr (PAIR) {
        using V = typename Pair2<T>::V;
        const int b = min(max(iL, 0), W - 2);
        const bool hiL = iL != b, hiR = iR != b;
        const long long oT = (long long)iT * W + b, oB = (long long)iB * W + b;
        V pT[WG_CH], pB[WG_CH];
#pragma unroll
        for (int j = 0; j < WG_CH; ++j) {
            const T* pl = src + (long long)min(c0 + j, c1 - 1) * HW;
            pT[j] = *reinterpret_cast<const V*>(pl + oT);
            pB[j] = *reinterpret_cast<const V*>(pl + oB);
        }
#pragma unroll
        for (int j = 0; j < WG_CH; ++j) {
            vTL[j] = hiL ? pT[j].y : pT[j].x;
            vTR[j] = hiR ? pT[j].y : pT[j].x;
            vBL[j] = hiL ? pB[j].y : pB[j].x;
            vBR[j] = hiR ? pB[j].y : pB[j].x;
        }
    } else {
#pragma unroll
        for (int j = 0; j < WG_CH; ++j) {
            const T* pl = src + (long long)min(c0 + j, c1 - 1) * HW;
            vTL[j] = pl[oTL];
            vTR[j] = pl[oTR];
            vBL[j] = pl[oBL];
            vBR[j] = pl[oBR];
        }
    }
#pragma unroll
    for (int j = 0; j < WG_CH; ++j) {
        if (c0 + j >= c1) break;
        T v = (T)0;
        if (mT && mL) v = v + wTL * vTL[j];
        if (mT && mR) v = v + wTR * vTR[j];
        if (mB && mL) v = v + wBL * vBL[j];
        if (mB && mR) v = v + wBR * vBR[j];
        o[(long long)(c0 + j) * HW] = v;
    }
}

template <typename T>
static void launch_warp(const T* in, const T* flow, T* out, int N, int C, int H, int W, hipStream_t s)
{
    // the least power of two that spans a narrow map, so that several rows share a
    // wave (3x20000x64 86.7 us with 64 columns, 11.6 with 4; 17x2000x196 40.2, 23.1)
    int bits = 2;
    while (bits < 6 && (1 << bits) < W) ++bits;
    const int cols = 1 << bits, rows = 256 >> bits;
    const int tiles = (W + cols - 1) / cols;
    // (a launch holds fewer than 2^32 threads along a dimension: the channels in several where they need more)
    const int most = std::max(1, (1 << 23) / tiles) * WG_CH;
    auto go = [&](auto kernel) {
        for (int first = 0; first < C; first += most)
            hipLaunchKernelGGL(kernel, dim3(tiles * ((std::min(most, C - first) + WG_CH - 1) / WG_CH), (H + rows - 1) / rows, N),
                               dim3(256), 0, s, in, flow, out, C, H, W, bits, first);
    };
    if (W > 32) go(k_warp<T, true, 6>);
    else if (W > 1) go(k_warp<T, true, 0>);
    else go(k_warp<T, false, 0>);
}

}  // namespace vsc

using namespace vsc;

namespace {

int correlation_forward(const void* f1, const void* f2, void* out, int N, int C, int H, int W, int max_displacement,
                        int legacy, int in_dtype, const float* chan_scale, vsc_hip_stream stream)
{
    if (!f1 || !f2 || !out) return set_error(VSC_E_INVALID, "vsc_correlation_forward: null pointer");
    if (N < 1 || C < 1 || H < 1 || W < 1) return set_error(VSC_E_INVALID, "vsc_correlation_forward: empty tensor");
    if (max_displacement < 0) return set_error(VSC_E_INVALID, "vsc_correlation_forward: max_displacement < 0");
    if (legacy && max_displacement > 4)
        return set_error(VSC_E_INVALID, "vsc_correlation_forward: legacy correlation pads by 4, max_displacement <= 4");
    const int md = max_displacement;
    hipStream_t s = as_stream(stream);
    if (in_dtype == VSC_F32) {
        const float* a = static_cast<const float*>(f1);
        const float* b = static_cast<const float*>(f2);
        float* o = static_cast<float*>(out);
        switch (W >= 4 ? md : -1) {   // (narrower images: one thread per output)
            case 0: launch_corr_f32<0>(a, b, o, N, C, H, W, legacy, s); break;
            case 1: launch_corr_f32<1>(a, b, o, N, C, H, W, legacy, s); break;
            case 2: launch_corr_f32<2>(a, b, o, N, C, H, W, legacy, s); break;
            case 3: launch_corr_f32<3>(a, b, o, N, C, H, W, legacy, s); break;
            case 4: launch_corr_f32<4>(a, b, o, N, C, H, W, legacy, s); break;
            default: launch_corr_generic(a, b, o, N, C, H, W, md, legacy, s);
        }
        return check_launch("correlation f32");
    }
    if (in_dtype == VSC_F64) {
        launch_corr_generic(static_cast<const double*>(f1), static_cast<const double*>(f2), static_cast<double*>(out), N, C, H, W, md,
                            legacy, s);
        return check_launch("correlation f64");
    }
    if (in_dtype == VSC_BF16 || in_dtype == VSC_F16 || in_dtype == VSC_FP8E4M3) {
        return corr_mfma_dispatch(f1, f2, static_cast<float*>(out), N, C, H, W, md, legacy, in_dtype, chan_scale, s);
    }
    return set_error(VSC_E_DTYPE, "vsc_correlation_forward: unsupported input type (float, double, bf16, f16, fp8e4m3)");
}

}  // namespace

extern "C" int vsc_correlation_forward(const void* f1, const void* f2, void* out, int N, int C, int H, int W,
                                       int max_displacement, int legacy, int in_dtype, const float* chan_scale,
                                       vsc_hip_stream stream)
{
    return correlation_forward(f1, f2, out, N, C, H, W, max_displacement, legacy, in_dtype, chan_scale, stream);
}

extern "C" int vsc_correlation_forward_noalloc(const void* f1, const void* f2, void* out, int N, int C, int H, int W,
                                               int max_displacement, int legacy, int in_dtype, const float* chan_scale,
                                               vsc_hip_stream stream)
{
    // the limit is the entry point's contract; no scratch is used
    const size_t need = (N < 1 || C < 1 || H < 1 || W < 1 || !corr_mfma_asks_workspace(f1, f2, W, in_dtype))
                            ? 0
                            : corr_mfma_workspace_bytes(N, C, H, W, in_dtype);
    if (need > VSC_CORRELATION_STATIC_SCRATCH)
        return set_error(VSC_E_INVALID,
                         "vsc_correlation_forward_noalloc: operands of a width that is no multiple of 4, or unaligned, are taken up "
                         "to a vsc_correlation_workspace_size() of " + std::to_string((size_t)VSC_CORRELATION_STATIC_SCRATCH) +
                         ", these have " + std::to_string(need) + " (no scratch is used: vsc_correlation_forward takes any)");
    return correlation_forward(f1, f2, out, N, C, H, W, max_displacement, legacy, in_dtype, chan_scale, stream);
}

extern "C" size_t vsc_correlation_workspace_size(int N, int C, int H, int W, int in_dtype)
{
    if (N < 1 || C < 1 || H < 1 || W < 1) return 0;
    return corr_mfma_workspace_bytes(N, C, H, W, in_dtype);
}

extern "C" int vsc_correlation_forward_ws(const void* f1, const void* f2, void* out, int N, int C, int H, int W,
                                          int max_displacement, int legacy, int in_dtype, const float* chan_scale,
                                          void* workspace, size_t workspace_bytes, vsc_hip_stream stream)
{
    const size_t need =
        corr_mfma_asks_workspace(f1, f2, W, in_dtype) ? vsc_correlation_workspace_size(N, C, H, W, in_dtype) : 0;
    if (need && (!workspace || workspace_bytes < need))
        return set_error(VSC_E_INVALID, "vsc_correlation_forward_ws: workspace missing or smaller than "
                                        "vsc_correlation_workspace_size() (vsc_correlation_forward takes the operands without one)");
    return correlation_forward(f1, f2, out, N, C, H, W, max_displacement, legacy, in_dtype, chan_scale, stream);
}

extern "C" int vsc_warp_forward(const void* in, const void* flow, void* out, int N, int C, int H, int W, int dtype,
                                vsc_hip_stream stream)
{
    if (!in || !flow || !out) return set_error(VSC_E_INVALID, "vsc_warp_forward: null pointer");
    if (N < 1 || C < 1 || H < 1 || W < 1) return set_error(VSC_E_INVALID, "vsc_warp_forward: empty tensor");
    hipStream_t s = as_stream(stream);
    if (dtype == VSC_F32) {
        launch_warp(static_cast<const float*>(in), static_cast<const float*>(flow), static_cast<float*>(out), N, C, H, W, s);
        return check_launch("warp f32");
    }
    if (dtype == VSC_F64) {
        launch_warp(static_cast<const double*>(in), static_cast<const double*>(flow), static_cast<double*>(out), N, C, H, W, s);
        return check_launch("warp f64");
    }
    return set_error(VSC_E_DTYPE, "vsc_warp_forward: unsupported input type (float or double)");
}
