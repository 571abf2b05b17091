// 3x3 convolution over channels-last (NHWC) tensors on MFMA (gfx950): the
// building block of the flow network (Conv2d layers of pwcnet.py:186-241,
// 511-535, 614-644; padding = dilation, stride 1 or 2; k_conv3x3w but for the
// layers of at most 16 channels) and of the learned flow upsampler (k_conv3x3).  FP32 (v_mfma_f32_16x16x4_f32), BF16 and FP16
// (v_mfma_f32_16x16x32_{bf16,f16}) operands, FP32 accumulation, bias,
// LeakyReLU(0.1) / ReLU and a residual add fused into the epilogue.
//
// GEMM form: D[cout][pixel] = sum_{tap, cin} W[cout][tap][cin] * X[tap(pixel)][cin].
// A block of NW waves owns TH = NW*MR output rows x 16 output columns and NT
// output channels; wave q computes rows q*MR .. q*MR+MR-1, i.e. MR pixel tiles
// of 16 against NT/16 channel tiles.  Input channels stream through LDS in chunks of
// KC (32 for 16-bit, 16 for FP32; 8 or 16 for 16-bit layers that narrow, whose
// MFMA K-steps then hold 4 or 2 taps): the input patch of the block (TH+2 x 18
// pixels at stride 1, 2*TH+1 x 33 at stride 2) and the weights of the chunk
// for all nine taps; the nine taps then read shifted windows of the patch.
// Dilated layers (dilation d > 1) are tiled on the d x d sub-grids of equal
// (y mod d, x mod d): on a sub-grid the dilated conv is a dense 3x3 conv, so
// the patch stays TH+2 x 18 whatever d is.
// Operand roles: A = weights (row = output channel), B = pixels (column), so
// each lane ends with 4 consecutive output channels of one pixel, stored as one
// 8- or 16-byte vector in NHWC.
#include "vsc_internal.h"

#include <algorithm>
#include <cstring>
#include <iterator>
#include <vector>

namespace vsc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 cv_bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 cv_f16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float cv_f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t cv_u32x4;

template <int EK> struct ConvK;
template <> struct ConvK<EK_F32> { static constexpr int KC = 16; };
template <> struct ConvK<EK_BF16> { static constexpr int KC = 32; };
template <> struct ConvK<EK_F16> { static constexpr int KC = 32; };

struct ConvArgs {
    const void* in; int in_cs, in_c0;
    int N, H, W, Cin;
    const void* wt; const void* wtp; const float* bias;
    void* out; int out_cs, out_c0;
    void* out2; int out2_cs, out2_c0;   // optional second copy of the result, in the input's element kind (Cout <= 16)
    const void* add; int add_cs, add_c0;
    const float* gate;
    const float* mask;                   // optional (FP32, the output's layout): the result is 0 where it is not above 0
    int Ho, Wo, Cout;
    int pad, pstep, act;
    int tiles_x, tiles_y;
    // packed weights: every `flush` chunks the accumulators are added to a total (0: never)
    int flush;
};

template <int EK>
__device__ inline cv_f32x4 conv_mfma(const cv_u32x4& a, const cv_u32x4& b, cv_f32x4 acc)
{
    if constexpr (EK == EK_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(cv_bf16x8, a),
                                                       __builtin_bit_cast(cv_bf16x8, b), acc, 0, 0, 0);
    } else if constexpr (EK == EK_F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(cv_f16x8, a),
                                                      __builtin_bit_cast(cv_f16x8, b), acc, 0, 0, 0);
    } else {
        // lane group g holds channels 4g .. 4g+3 of the 16-channel chunk; step t
        // feeds channel 4g+t as the instruction's k = g (same map for A and B)
        const cv_f32x4 fa = __builtin_bit_cast(cv_f32x4, a), fb = __builtin_bit_cast(cv_f32x4, b);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[t], fb[t], acc, 0, 0, 0);
        return acc;
    }
}

template <int EKO>
__device__ inline void conv_store4(void* out, long long off, const float v[4], int nvalid)
{
    using E = Elem<EKO>;
    typename E::T* p = static_cast<typename E::T*>(out) + off;
    if (nvalid >= 4) {
        if constexpr (EKO == EK_F32) {
            *reinterpret_cast<cv_f32x4*>(p) = cv_f32x4{v[0], v[1], v[2], v[3]};
        } else {
            const uint32_t lo = (uint32_t)E::st(v[0]) | ((uint32_t)E::st(v[1]) << 16);
            const uint32_t hi = (uint32_t)E::st(v[2]) | ((uint32_t)E::st(v[3]) << 16);
            *reinterpret_cast<uint2*>(p) = make_uint2(lo, hi);
        }
    } else {
        for (int r = 0; r < nvalid; ++r) p[r] = E::st(v[r]);
    }
}

template <int EKO>
__device__ inline void conv_load4(const void* src, long long off, float v[4], int nvalid)
{
    using E = Elem<EKO>;
    const typename E::T* p = static_cast<const typename E::T*>(src) + off;
    for (int r = 0; r < 4; ++r) v[r] += (r < nvalid) ? E::ld(p[r]) : 0.0f;
}

template <int EK, int EKO, int S, int NT, int MR, int NW, int KCX, bool EARLY>
__global__ __launch_bounds__(64 * NW) void k_conv3x3(ConvArgs a)
{
    using E = Elem<EK>;
    using T = typename E::T;
    constexpr int NTH = 64 * NW;
    constexpr int VEC = E::VEC, KC = KCX, KV = KC / VEC;
    constexpr int TH = NW * MR, TW = 16;
    constexpr int PR = (TH - 1) * S + 3, PC = (TW - 1) * S + 3;
    // LDS pixel stride: the chunk alone for FP32 (64 bytes: the plain form
    // 1.3% faster than with a 16-byte pad), the chunk and two 16-byte pads for
    // 16-bit operands (96 bytes for 32-channel chunks: 5% faster than 80 on the
    // 1080p level-3 layers, 64 and 112 no better, 144 slower)
    constexpr int ROW = KC + (EK == EK_F32 ? 0 : 2) * VEC;
    constexpr int NP = PR * PC * KV, NWU = NT * 9 * KV;
    constexpr int RP = (NP + NTH - 1) / NTH, RW = (NWU + NTH - 1) / NTH;
    __shared__ __attribute__((aligned(16))) T sP[PR * PC * ROW];
    __shared__ __attribute__((aligned(16))) T sW[NT * 9 * ROW];

    const int tid = threadIdx.x, q = tid / 64, lane = tid % 64;
    const int l16 = lane % 16, lg = lane / 16;
    const int n = blockIdx.z, nt0 = blockIdx.y * NT;
    int t = blockIdx.x;
    const int tx = t % a.tiles_x; t /= a.tiles_x;
    const int ty = t % a.tiles_y; t /= a.tiles_y;
    const int ps = a.pstep, py = t / ps, px = t % ps;
    const int base_y = py - a.pad + ps * ty * TH * S, base_x = px - a.pad + ps * tx * TW * S;
    const T* in = static_cast<const T*>(a.in) + (long long)n * a.H * a.W * a.in_cs + a.in_c0;
    const T* wt = static_cast<const T*>(a.wt);

    cv_f32x4 acc[NT / 16][MR];
#pragma unroll
    for (int i = 0; i < NT / 16; ++i)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[i][m] = cv_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // the epilogue's per-channel values, read before the products unless not EARLY
    // (after them the read is one more round trip to memory on every launch's tail:
    // 240x136x2, 64 -> 64, BF16, 17.0 us, 14.9 so)
    [[maybe_unused]] float bias[NT / 16][4];
    const float g = a.gate ? *a.gate : 1.0f;
    const bool with_bias = a.bias;
    if constexpr (EARLY) {
#pragma unroll
        for (int i = 0; i < NT / 16; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int co = nt0 + i * 16 + 4 * lg + r;
                bias[i][r] = with_bias ? a.bias[min(co, a.Cout - 1)] : 0.0f;
            }
    }

    // input channel chunks are staged through registers DEPTH chunks ahead of
    // the chunk in LDS, so the global loads of a chunk overlap the MFMAs of the
    // DEPTH chunks before it (deeper staging measured slower: with all of the flow
    // network on this kernel 2 and 3 chunks ahead cost its 1080p BF16 form 3% and 18%)
    constexpr int DEPTH = 1;
    cv_u32x4 rp[DEPTH][RP], rw[DEPTH][RW];
    auto fetch = [&](int c0, cv_u32x4 (&P)[RP], cv_u32x4 (&Wr)[RW]) {
#pragma unroll
        for (int k = 0; k < RP; ++k) {
            const int u = tid + NTH * k;
            const int p = u / KV, cv = u % KV;
            const int r = p / PC, c = p % PC;
            const int iy = base_y + ps * r, ix = base_x + ps * c, ch = c0 + cv * VEC;
            cv_u32x4 v = cv_u32x4{0u, 0u, 0u, 0u};
            if (u < NP && iy >= 0 && iy < a.H && ix >= 0 && ix < a.W && ch < a.Cin)
                v = *reinterpret_cast<const cv_u32x4*>(in + ((long long)iy * a.W + ix) * a.in_cs + ch);
            P[k] = v;
        }
#pragma unroll
        for (int k = 0; k < RW; ++k) {
            const int u = tid + NTH * k;
            const int row = u / KV, cv = u % KV;           // row = co_local*9 + tap
            const int co = nt0 + row / 9, ch = c0 + cv * VEC;
            cv_u32x4 v = cv_u32x4{0u, 0u, 0u, 0u};
            if (u < NWU && co < a.Cout && ch < a.Cin)
                v = *reinterpret_cast<const cv_u32x4*>(wt + ((long long)co * 9 + row % 9) * a.Cin + ch);
            Wr[k] = v;
        }
    };
    auto stage = [&](const cv_u32x4 (&P)[RP], const cv_u32x4 (&Wr)[RW]) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < RP; ++k) {
            const int u = tid + NTH * k;
            if (u < NP) *reinterpret_cast<cv_u32x4*>(&sP[(u / KV) * ROW + (u % KV) * VEC]) = P[k];
        }
#pragma unroll
        for (int k = 0; k < RW; ++k) {
            const int u = tid + NTH * k;
            if (u < NWU) *reinterpret_cast<cv_u32x4*>(&sW[(u / KV) * ROW + (u % KV) * VEC]) = Wr[k];
        }
        __syncthreads();
    };
    // The MFMA's K (32 for 16-bit, 16 for FP32: four lane groups of CPL
    // channels) covers TPK taps of a chunk narrower than K: lane group lg takes
    // tap step*TPK + lg/LPT, channels (lg % LPT)*CPL.. of it (a 16-bit layer
    // with 8 or 16 input channels runs 3 or 5 K-steps instead of 9 mostly
    // zero ones).  Each step's fragments are read from LDS while the previous
    // step's MFMAs issue (two register sets).
    constexpr int KK = EK == EK_F32 ? 16 : 32;
    constexpr int TPK = KK / KC, LPT = 4 / TPK, CPL = KC / LPT;
    constexpr int NSTEP = (9 + TPK - 1) / TPK;
    static_assert(KK % KC == 0 && CPL * (int)sizeof(T) == 16, "a lane group reads 16 bytes of one tap");
    auto compute = [&]() {
        cv_u32x4 wf[2][NT / 16], xf[2][MR];
        auto frag = [&](int step, cv_u32x4 (&w)[NT / 16], cv_u32x4 (&x)[MR]) {
            const int tap = step * TPK + lg / LPT, coff = (lg % LPT) * CPL;
            if (TPK > 1 && tap >= 9) {   // padding of the last K-step
#pragma unroll
                for (int i = 0; i < NT / 16; ++i) w[i] = cv_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int m = 0; m < MR; ++m) x[m] = cv_u32x4{0u, 0u, 0u, 0u};
                return;
            }
            const int ky = tap / 3, kx = tap % 3;
#pragma unroll
            for (int i = 0; i < NT / 16; ++i)
                w[i] = *reinterpret_cast<const cv_u32x4*>(&sW[((i * 16 + l16) * 9 + tap) * ROW + coff]);
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const int pr = (q * MR + m) * S + ky, pc = l16 * S + kx;
                x[m] = *reinterpret_cast<const cv_u32x4*>(&sP[(pr * PC + pc) * ROW + coff]);
            }
        };
        frag(0, wf[0], xf[0]);
#pragma unroll
        for (int step = 0; step < NSTEP; ++step) {
            if (step + 1 < NSTEP) frag(step + 1, wf[(step + 1) & 1], xf[(step + 1) & 1]);
            // keep the reads of the next step ahead of this step's MFMAs
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NT / 16; ++i)
#pragma unroll
                for (int m = 0; m < MR; ++m) acc[i][m] = conv_mfma<EK>(wf[step & 1][i], xf[step & 1][m], acc[i][m]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (d * KC < a.Cin) fetch(d * KC, rp[d], rw[d]);
    for (int c0 = 0; c0 < a.Cin; c0 += DEPTH * KC) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const int cc = c0 + d * KC;
            if (cc >= a.Cin) break;
            stage(rp[d], rw[d]);
            if (cc + DEPTH * KC < a.Cin) fetch(cc + DEPTH * KC, rp[d], rw[d]);
            compute();
        }
    }

    // epilogue: lane holds output channels nt0 + 16i + 4lg + r of pixel l16 of row q*MR+m
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        const int oy = py + ps * (ty * TH + q * MR + m), ox = px + ps * (tx * TW + l16);
        if (oy >= a.Ho || ox >= a.Wo) continue;
        const long long pix = ((long long)n * a.Ho + oy) * a.Wo + ox;
#pragma unroll
        for (int i = 0; i < NT / 16; ++i) {
            const int co = nt0 + i * 16 + 4 * lg;
            const int nv = min(4, a.Cout - co);
            if (nv <= 0) continue;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float x = acc[i][m][r];
                if (with_bias && r < nv) x += EARLY ? bias[i][r] : a.bias[co + r];
                if (a.act == 1) x = x > 0.0f ? x : x * 0.1f;
                else if (a.act == 2) x = x > 0.0f ? x : 0.0f;
                v[r] = a.gate ? x * g : x;
            }
            if constexpr (EKO == EK_F32) {
                if (a.mask) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (r < nv && !(a.mask[pix * a.out_cs + a.out_c0 + co + r] > 0.0f)) v[r] = 0.0f;
                }
            }
            if (a.add) conv_load4<EKO>(a.add, pix * a.add_cs + a.add_c0 + co, v, nv);
            conv_store4<EKO>(a.out, pix * a.out_cs + a.out_c0 + co, v, nv);
            // (compiled into the 16-channel tiles only: the flow heads use it)
            if constexpr (NT == 16)
                if (a.out2) conv_store4<EK>(a.out2, pix * a.out2_cs + a.out2_c0 + co, v, nv);
        }
    }
}

// The same layers with packed weights (conv_pack_weights), for chunks of a whole
// K step (32 channels, FP32 16): the flow network's layers.
//
// What bounded k_conv3x3 there is its weights' way from L2: a block's rows of 32
// channels lie 9*Cin elements apart, which falls on a few of the L2's channels
// (32 more input channels cost a 120x72x2 -> 128 layer 1.9 us at 17 MB), and
// every block passed them through LDS besides.  Packed, a tap's weights of 16
// output channels are 1 KB in the lanes' order: one coalesced load, straight to
// registers.  So a wave owns 16 output channels of MR rows of 16 pixels, its nine
// taps' weights stand in registers, and each is replaced by the next chunk's as
// soon as its products are issued.  Only the input patch goes through LDS, two
// buffers of it, so a chunk has one barrier, and a patch row's fragment is read
// once for the taps of all three rows.  The loads are buffer loads that give
// zeros past the end (the image's outside, the channels' tail) instead of
// branches, so that the waits count the loads behind them.
//
// FLUSH: every `flush` chunks the accumulators are added to a total and cleared:
// the order of sums of a channel loop split into parts, without the parts' way
// through memory and the launch that adds them (5 us).
//
// Measured, us a layer (k_conv3x3 -> this): BF16 120x72x2 pixels, 128 -> 128
// channels 16.9 -> 9.7, 256 -> 128 23.1 -> 13.3, 480x288 32 -> 32 24 -> 10.5;
// FP32 120x72x2 256 -> 128 120 -> 79 (its products alone are 69), 160 -> 64
// 55.8 -> 30.8, 15x9x2 256 -> 128 49 -> 12.6.  The network of a 1080p frame at
// half size in BF16 533 -> 386 us, of a 640x360 frame in FP32 786 -> 672 us.
template <int EK, int EKO, int S, int NT, int MR, bool FLUSH>
__global__ __launch_bounds__(256) void k_conv3x3w(ConvArgs a)
{
    using E = Elem<EK>;
    using T = typename E::T;
    constexpr int VEC = E::VEC, KC = ConvK<EK>::KC, KV = 4;
    static_assert(KC == KV * VEC, "four 16-byte vectors a pixel and chunk");
    constexpr int WC = NT / 16, RG = 4 / WC;            // channel groups and row groups of the waves
    constexpr int TH = RG * MR, TW = 16;
    constexpr int PR = (TH - 1) * S + 3, PC = (TW - 1) * S + 3;
    constexpr int ROW = KC + (EK == EK_F32 ? 0 : 2) * VEC;
    constexpr int NP = PR * PC * KV, RP = (NP + 255) / 256;
    constexpr int XR = (MR - 1) * S + 3;                // patch rows of a wave
    __shared__ __attribute__((aligned(16))) T sP[2][PR * PC * ROW];

    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int q = wave / WC, wc = wave % WC;
    const int l16 = lane % 16, lg = lane / 16;
    const int n = blockIdx.z, nt0 = blockIdx.y * NT + wc * 16;
    int t = blockIdx.x;
    const int tx = t % a.tiles_x; t /= a.tiles_x;
    const int ty = t % a.tiles_y; t /= a.tiles_y;
    const int ps = a.pstep, py = t / ps, px = t % ps;
    const int base_y = py - a.pad + ps * ty * TH * S, base_x = px - a.pad + ps * tx * TW * S;
    // buffer loads: one past the end (NOWHERE) gives zeros, so no load is in a branch
    // and the waits count the loads behind them
    constexpr unsigned NOWHERE = 0x80000000u;
    const __amdgpu_buffer_rsrc_t in = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(static_cast<const T*>(a.in) + (long long)n * a.H * a.W * a.in_cs + a.in_c0), 0,
        (int)((a.H * a.W * a.in_cs - a.in_c0) * sizeof(T)), 0x00020000);
    const int chunks = (a.Cin + KC - 1) / KC, c16 = (a.Cout + 15) / 16;
    const __amdgpu_buffer_rsrc_t wt = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.wtp), 0, c16 * chunks * 9 * 1024, 0x00020000);

    cv_f32x4 acc[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m] = cv_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const float g = a.gate ? *a.gate : 1.0f;
    const bool with_bias = a.bias;
    float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (with_bias) {
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[r] = a.bias[min(nt0 + 4 * lg + r, a.Cout - 1)];
    }

    const int cv = tid % KV * VEC;
    unsigned off[RP];
#pragma unroll
    for (int k = 0; k < RP; ++k) {
        const int p = (tid + 256 * k) / KV, r = p / PC, c = p % PC;
        const int iy = base_y + ps * r, ix = base_x + ps * c;
        off[k] = p < PR * PC && iy >= 0 && iy < a.H && ix >= 0 && ix < a.W ? ((iy * a.W + ix) * a.in_cs + cv) * sizeof(T) : NOWHERE;
    }
    cv_u32x4 rp[RP], w[9];
    auto fetch = [&](int c0) {
        const unsigned none = c0 + cv < a.Cin ? 0u : NOWHERE;
#pragma unroll
        for (int k = 0; k < RP; ++k)
            rp[k] = __builtin_bit_cast(cv_u32x4, __builtin_amdgcn_raw_buffer_load_b128(in, off[k] | none, c0 * sizeof(T), 0));
    };
    const unsigned wlane = nt0 < a.Cout ? lane * 16u : NOWHERE, wfirst = nt0 < a.Cout ? nt0 / 16 * chunks * 9 * 1024u : 0u;
    auto load_w = [&](int tap, int chunk) {
        w[tap] = __builtin_bit_cast(cv_u32x4, __builtin_amdgcn_raw_buffer_load_b128(wt, wlane, wfirst + (chunk * 9 + tap) * 1024, 0));
    };

    // (the loop's order, for the waits' counts)
    fetch(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) load_w(tap, 0);
    __builtin_amdgcn_sched_barrier(0);
    [[maybe_unused]] cv_f32x4 total[MR];
    [[maybe_unused]] int left = a.flush;
    if constexpr (FLUSH) {
#pragma unroll
        for (int m = 0; m < MR; ++m) total[m] = cv_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    int buf = 0;
    for (int c0 = 0; c0 < a.Cin; c0 += KC, buf ^= 1) {
        const bool more = c0 + KC < a.Cin;
#pragma unroll
        for (int k = 0; k < RP; ++k) {
            const int u = tid + 256 * k;
            if (u < NP) *reinterpret_cast<cv_u32x4*>(&sP[buf][(u / KV) * ROW + cv]) = rp[k];
        }
        // the LDS writes alone are waited for: the next chunk's loads stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        fetch(c0 + KC);
        const T* sp = &sP[buf][(q * MR * S * PC + l16 * S) * ROW + lg * VEC];
        cv_u32x4 x[3][XR];
        // rows of the tap's column that are not held yet
        auto frag = [&](int tap) {
            const int ky = tap / 3, kx = tap % 3;
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const int r = m * S + ky;
                if (ky >= S && m < MR - 1) continue;
                x[kx][r] = *reinterpret_cast<const cv_u32x4*>(sp + (r * PC + kx) * ROW);
            }
        };
        frag(0);
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            if (tap + 1 < 9) frag(tap + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MR; ++m) acc[m] = conv_mfma<EK>(w[tap], x[tap % 3][m * S + tap / 3], acc[m]);
            __builtin_amdgcn_sched_barrier(0);
            load_w(tap, more ? c0 / KC + 1 : c0 / KC);
        }
        if constexpr (FLUSH) {
            if (--left == 0 || !more) {
#pragma unroll
                for (int m = 0; m < MR; ++m) {
                    total[m] += acc[m];
                    acc[m] = cv_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }
                left = a.flush;
            }
        }
    }

    const int co = nt0 + 4 * lg, nv = min(4, a.Cout - co);
    if (nv <= 0) return;
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        const int oy = py + ps * (ty * TH + q * MR + m), ox = px + ps * (tx * TW + l16);
        if (oy >= a.Ho || ox >= a.Wo) continue;
        const long long pix = ((long long)n * a.Ho + oy) * a.Wo + ox;
        const cv_f32x4 s = FLUSH ? total[m] : acc[m];
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float y = with_bias ? s[r] + bias[r] : s[r];
            const float low = a.act == 1 ? y * 0.1f : a.act == 2 ? 0.0f : y;
            y = y > 0.0f ? y : low;
            v[r] = a.gate ? y * g : y;
        }
        if (a.add) conv_load4<EKO>(a.add, pix * a.add_cs + a.add_c0 + co, v, nv);
        conv_store4<EKO>(a.out, pix * a.out_cs + a.out_c0 + co, v, nv);
        if constexpr (NT == 16)
            if (a.out2) conv_store4<EK>(a.out2, pix * a.out2_cs + a.out2_c0 + co, v, nv);
    }
}

// The channel tile of k_conv3x3, and the rows of a wave of its pixel tile for
// `items` batch items (conv_pick says why).
template <int EK>
static int conv_nt(const ConvArgs& a)
{
    if (EK == EK_F32 && a.Cout > 32) return 64;
    return a.Cout > 16 ? 32 : 16;
}
template <int EK, int S>
static int conv_rows(const ConvArgs& a, int items)
{
    const int ps = a.pstep, nt = conv_nt<EK>(a);
    const long long px = (long long)((a.Ho + ps - 1) / ps) * ps * ((a.Wo + ps - 1) / ps) * ps * items;
    const long long ntiles = (a.Cout + nt - 1) / nt;
    auto blocks = [&](int mr) { return (px / (64LL * mr)) * ntiles; };
    const int mr = (S == 1 && blocks(4) >= 512) ? 4 : (blocks(2) >= (EK == EK_F32 ? 512 : 128) ? 2 : 1);
    return S == 2 && mr > 2 ? 2 : mr;
}

// Chunks whose sums a packed layer keeps apart (ConvArgs::flush): what a split of
// the channel loop over the CUs that one batch item's blocks of k_conv3x3 leave idle
// would give, bounded by kConvPartFloats of partial sums an item.  One item's
// geometry alone decides, the pixel tile's rows included, so an item's result has
// the same bits alone and in a batch of any size.
constexpr long long kConvPartFloats = 2LL << 20;
template <int EK, int S>
static int conv_flush(const ConvArgs& a)
{
    const int chunks = (a.Cin + ConvK<EK>::KC - 1) / ConvK<EK>::KC, ps = a.pstep, mr = conv_rows<EK, S>(a, 1), nt = conv_nt<EK>(a);
    const long long hs = (a.Ho + ps - 1) / ps, ws = (a.Wo + ps - 1) / ps;
    const long long item_blocks = (hs + 4 * mr - 1) / (4 * mr) * ((ws + 15) / 16) * ps * ps * ((a.Cout + nt - 1) / nt);
    if (chunks < 2 || item_blocks >= (EK == EK_F32 ? 128 : 32)) return 0;
    const long long item_stride = (long long)a.Ho * a.Wo * a.Cout;
    int parts = (int)std::min<long long>(chunks, (256 + item_blocks - 1) / item_blocks);
    parts = (int)std::min<long long>(parts, kConvPartFloats / std::max<long long>(item_stride, 1));
    if (parts < 2) return 0;
    return (chunks + parts - 1) / parts;
}

template <int EK, int EKO, int S, int NT, int MR, int NW, int KCX>
static void conv_go(const ConvArgs& a, hipStream_t s)
{
    const int ps = a.pstep;
    ConvArgs b = a;
    const int hs = (a.Ho + ps - 1) / ps, ws = (a.Wo + ps - 1) / ps;
    b.tiles_y = (hs + NW * MR - 1) / (NW * MR);
    b.tiles_x = (ws + 15) / 16;
    dim3 grid(b.tiles_x * b.tiles_y * ps * ps, (a.Cout + NT - 1) / NT, a.N);
    // The registers of an early bias cost several FP32 tiles a block of their CU: not
    // without a bias (400x200, stride 2, 32 -> 32, two items, 14.9 us, 14.0 without), nor
    // where three blocks a CU instead of four need a round more (480x272, 32 -> 32, 1020
    // blocks: 37.3 us with three, 31.3 with four; 320x256, 640 blocks: 20.8 and 22.1).
    if constexpr (EK == EK_F32 && NT <= 32) {
        const long long n = (long long)grid.x * grid.y * grid.z;
        if (!a.bias || (NT == 32 && MR == 3 - S && (n + 1023) / 1024 < (n + 767) / 768)) {
            hipLaunchKernelGGL((k_conv3x3<EK, EKO, S, NT, MR, NW, KCX, false>), grid, dim3(64 * NW), 0, s, b);
            return;
        }
    }
    hipLaunchKernelGGL((k_conv3x3<EK, EKO, S, NT, MR, NW, KCX, true>), grid, dim3(64 * NW), 0, s, b);
}

template <int EK, int EKO, int S, int NT, int MR>
static void conv_gow(const ConvArgs& a, hipStream_t s)
{
    constexpr int TH = 4 / (NT / 16) * MR;
    ConvArgs b = a;
    const int ps = a.pstep, hs = (a.Ho + ps - 1) / ps, ws = (a.Wo + ps - 1) / ps;
    b.tiles_y = (hs + TH - 1) / TH;
    b.tiles_x = (ws + 15) / 16;
    dim3 grid(b.tiles_x * b.tiles_y * ps * ps, (a.Cout + NT - 1) / NT, a.N);
    if (a.flush) {
        if constexpr (MR <= 3) hipLaunchKernelGGL((k_conv3x3w<EK, EKO, S, NT, MR, true>), grid, dim3(256), 0, s, b);
    } else {
        hipLaunchKernelGGL((k_conv3x3w<EK, EKO, S, NT, MR, false>), grid, dim3(256), 0, s, b);
    }
}

// Tile of a packed layer: the (channels, rows of a wave) of least modelled time a
// chunk, `full` blocks standing on the fullest CU.  FP32: the products bound it,
// 0.51 us a row and block and 0.06 a block.  16-bit: a block takes 0.26 + 0.045
// MR us (its loads and its barrier) but at least 0.1 MR beside others and 0.13
// MR alone.  (Fitted on 26 layers x 15 tiles, within 10% of the best tile on
// each; 120x72x2, 128 -> 128, BF16: 32 channels x 3 rows 11.0 us, 768 blocks, x 4
// 11.3, 576 blocks, 64 x 5 9.7, 480 blocks.)
template <int EK, int EKO, int S>
static void conv_packed(const ConvArgs& a, hipStream_t s)
{
    struct Tile {
        int nt, mr;
        void (*go)(const ConvArgs&, hipStream_t);
    };
    static const Tile narrow[] = {{16, 1, conv_gow<EK, EKO, S, 16, 1>}, {16, 2, conv_gow<EK, EKO, S, 16, 2>}};
    static const Tile wide[] = {
        {64, 1, conv_gow<EK, EK, S, 64, 1>}, {64, 2, conv_gow<EK, EK, S, 64, 2>}, {64, 3, conv_gow<EK, EK, S, 64, 3>},
        {32, 1, conv_gow<EK, EK, S, 32, 1>}, {32, 2, conv_gow<EK, EK, S, 32, 2>}, {32, 3, conv_gow<EK, EK, S, 32, 3>},
        {64, 4, conv_gow<EK, EK, S, 64, 4>}, {32, 4, conv_gow<EK, EK, S, 32, 4>}, {64, 5, conv_gow<EK, EK, S, 64, 5>},
        {64, 6, conv_gow<EK, EK, S, 64, 6>}};
    const int ps = a.pstep;
    const long long hs = (a.Ho + ps - 1) / ps, ws = (a.Wo + ps - 1) / ps;
    const Tile* first = a.Cout <= 16 ? narrow : wide;
    const Tile* last = a.Cout <= 16 ? std::end(narrow) : std::end(wide);
    const Tile* best = nullptr;
    double least = 1e300;
    for (const Tile* t = first; t != last; ++t) {
        if (a.flush && t->mr > 3) continue;
        if (a.Cout <= 32 && t->nt > 32) continue;
        const int th = 64 / t->nt * t->mr;
        const long long blocks = (hs + th - 1) / th * ((ws + 15) / 16) * ps * ps * ((a.Cout + t->nt - 1) / t->nt) * a.N;
        const double full = (double)((blocks + 255) / 256), m = t->mr;
        const double cost = EK == EK_F32 ? full * (0.51 * m + 0.06)
                                         : std::max(std::max(full * (0.26 + 0.045 * m), full * 0.1 * m), 0.13 * m);
        if (cost < least * 0.999) {
            least = cost;
            best = t;
        }
    }
    best->go(a, s);
}

template <int EK, int EKO, int S, int NT, int KCX>
static void conv_mr(const ConvArgs& a, int mr, hipStream_t s)
{
    if (mr == 4) conv_go<EK, EKO, S, NT, (S == 1 ? 4 : 2), 4, KCX>(a, s);
    else if (mr == 2) conv_go<EK, EKO, S, NT, 2, 4, KCX>(a, s);
    else conv_go<EK, EKO, S, NT, 1, 4, KCX>(a, s);
}

// Tile choice of k_conv3x3; packed layers choose theirs by modelled time
// (conv_packed) and take only the grouping of their sums from here (conv_flush).
// Channel tile: FP32 layers take the widest tile they fill (64, 32 or 16 output
// channels); 16-bit layers take 32 (16 when the layer has at most 16): twice the
// blocks of 64-channel tiles on small grids and half the weights staged per block
// (with all of the flow network on this kernel 1080p frames ran at 556 frames/s,
// with 64-channel tiles at 521).  Pixel tile:
// 256 pixels from two blocks per CU; 128 pixels from two blocks per CU (FP32)
// or from half a block per CU (16-bit: its MFMAs are 16x faster, so the weights
// every block re-reads dominate, and halving that traffic pays for the idle
// CUs of a smaller grid); else 64 pixels.
template <int EK, int EKO, int S>
static void conv_pick(const ConvArgs& a, hipStream_t s)
{
    const int ps = a.pstep, NTsel = conv_nt<EK>(a), mr = conv_rows<EK, S>(a, a.N);
    if constexpr (EK != EK_F16) {
        if (a.wtp) {
            ConvArgs b = a;
            b.flush = conv_flush<EK, S>(a);
            conv_packed<EK, EKO, S>(b, s);
            return;
        }
    }
    constexpr int KC = ConvK<EK>::KC;
    if constexpr (EK == EK_F32) {
        // Layers of 64-pixel tiles: the widest channel tiles are the cheapest a
        // channel, but on a grid of a few blocks per CU the fullest CU decides, and
        // 96 channels leave a quarter of two 64-channel tiles empty.  So the width of
        // least (blocks on the fullest CU) x (channels + 4).
        int nt = NTsel;
        if (mr == 1) {
            const long long item = (((a.Ho + ps - 1) / ps + 3) / 4) * (((a.Wo + ps - 1) / ps + 15) / 16) * (long long)ps * ps;
            long long best = 1LL << 62;
            for (int w = NTsel; w >= 16; w /= 2) {
                const long long cost = (item * ((a.Cout + w - 1) / w) * a.N + 255) / 256 * (w + 4);
                if (cost < best) {
                    best = cost;
                    nt = w;
                }
            }
        }
        if (nt == 64) conv_mr<EK, EKO, S, 64, KC>(a, mr, s);
        else if (nt == 32) conv_mr<EK, EKO, S, 32, KC>(a, mr, s);
        else conv_mr<EK, EKO, S, 16, KC>(a, mr, s);
    } else {
        // layers with 8 or 16 input channels (the image and the first feature
        // level) stage chunks of that width
        if (NTsel == 32) {
            if (a.Cin <= 8) conv_mr<EK, EKO, S, 32, 8>(a, mr, s);
            else if (a.Cin <= 16) conv_mr<EK, EKO, S, 32, 16>(a, mr, s);
            else conv_mr<EK, EKO, S, 32, KC>(a, mr, s);
        } else {
            if (a.Cin <= 8) conv_mr<EK, EKO, S, 16, 8>(a, mr, s);
            else if (a.Cin <= 16) conv_mr<EK, EKO, S, 16, 16>(a, mr, s);
            else conv_mr<EK, EKO, S, 16, KC>(a, mr, s);
        }
    }
}

template <int EK, int EKO>
static void conv_stride(const ConvArgs& a, int stride, hipStream_t s)
{
    if (stride == 2) conv_pick<EK, EKO, 2>(a, s);
    else conv_pick<EK, EKO, 1>(a, s);
}

// whole K steps of channels (16-bit layers of 8 or 16 channels put several taps
// into one instead), an item that a buffer descriptor spans
bool conv_takes_packed(int ek_in, int ek_out, int cin, int cout, long long item_elements)
{
    const int eb = ek_in == EK_F32 ? 4 : 2;
    return ek_in != EK_F16 && (ek_in == EK_F32 || cin > 16) && (ek_out == ek_in || cout <= 16) && item_elements * eb < (1LL << 31);
}

static int packed_chunks(int cin, int elem_bytes) { return (cin * elem_bytes + 63) / 64; }

size_t conv_packed_bytes(int cout, int cin, int elem_bytes)
{
    return (size_t)((cout + 15) / 16) * packed_chunks(cin, elem_bytes) * 9 * 1024;
}

void conv_pack_weights(const void* w, void* out, int cout, int cin, int elem_bytes)
{
    const int chunks = packed_chunks(cin, elem_bytes), vec = 16 / elem_bytes;
    char* o = static_cast<char*>(out);
    for (int ct = 0; ct < (cout + 15) / 16; ++ct)
        for (int ch = 0; ch < chunks; ++ch)
            for (int tap = 0; tap < 9; ++tap)
                for (int lane = 0; lane < 64; ++lane, o += 16) {
                    const int co = ct * 16 + lane % 16, ci = (ch * 4 + lane / 16) * vec;
                    const int n = co < cout ? std::max(0, std::min(vec, cin - ci)) : 0;
                    memset(o, 0, 16);
                    if (n) memcpy(o, static_cast<const char*>(w) + (((size_t)co * 9 + tap) * cin + ci) * elem_bytes, (size_t)n * elem_bytes);
                }
}

int launch_conv3x3(const ConvDesc& d, hipStream_t s)
{
    const int ek = d.ek_in, eko = d.ek_out;
    if (ek < 0 || eko < 0) return set_error(VSC_E_DTYPE, "conv3x3: unsupported element type");
    if (eko != ek && eko != EK_F32) return set_error(VSC_E_DTYPE, "conv3x3: output must be FP32 or the input type");
    const int vec = ek == EK_F32 ? 4 : 8;
    if (d.stride != 1 && d.stride != 2) return set_error(VSC_E_INVALID, "conv3x3: stride must be 1 or 2");
    if (d.dil < 1 || (d.stride == 2 && d.dil != 1)) return set_error(VSC_E_INVALID, "conv3x3: bad dilation");
    if (d.in.c <= 0 || d.in.c % vec || d.in.cs % vec || d.in.c0 % vec || d.in.c0 + d.in.c > d.in.cs)
        return set_error(VSC_E_INVALID, "conv3x3: input slice must be whole 16-byte vectors inside the pixel");
    const int Cout = d.out.c;
    if (Cout <= 0 || d.out.c0 + Cout > d.out.cs) return set_error(VSC_E_INVALID, "conv3x3: bad output slice");
    if ((d.out.c0 % 4 || d.out.cs % 4) && Cout >= 4)
        return set_error(VSC_E_INVALID, "conv3x3: output slice must be 4-channel aligned");
    if (d.add.p && (d.add.c0 % 4 || d.add.cs % 4) && Cout >= 4)
        return set_error(VSC_E_INVALID, "conv3x3: residual slice must be 4-channel aligned");
    const int Ho = (d.in.h + 2 * d.pad - 2 * d.dil - 1) / d.stride + 1;
    const int Wo = (d.in.w + 2 * d.pad - 2 * d.dil - 1) / d.stride + 1;
    if (Ho != d.out.h || Wo != d.out.w || d.out.n != d.in.n || (d.add.p && (d.add.h != Ho || d.add.w != Wo)))
        return set_error(VSC_E_INVALID, "conv3x3: output size does not match");
    if (d.out2.p && (Cout > 16 || d.out2.c != Cout || d.out2.c0 + Cout > d.out2.cs || d.out2.h != Ho ||
                     d.out2.w != Wo || d.out2.n != d.in.n || ((d.out2.c0 % 4 || d.out2.cs % 4) && Cout >= 4)))
        return set_error(VSC_E_INVALID, "conv3x3: bad second output slice (at most 16 channels)");
    if ((long long)d.in.n * d.in.h * d.in.w * d.in.cs >= (1LL << 31) ||
        (long long)d.out.n * Ho * Wo * d.out.cs >= (1LL << 31))
        return set_error(VSC_E_INVALID, "conv3x3: tensor too large");
    if (Ho <= 0 || Wo <= 0) return VSC_OK;
    ConvArgs a{};
    a.in = d.in.p; a.in_cs = d.in.cs; a.in_c0 = d.in.c0;
    a.N = d.in.n; a.H = d.in.h; a.W = d.in.w; a.Cin = d.in.c;
    a.wt = d.wt; a.wtp = d.wtp; a.bias = d.bias;
    if (d.wtp && !conv_takes_packed(ek, eko, d.in.c, Cout, (long long)d.in.h * d.in.w * d.in.cs))
        return set_error(VSC_E_INVALID, "conv3x3: packed weights for a layer that does not take them");
    a.out = d.out.p; a.out_cs = d.out.cs; a.out_c0 = d.out.c0;
    a.out2 = d.out2.p; a.out2_cs = d.out2.cs; a.out2_c0 = d.out2.c0;
    a.add = d.add.p; a.add_cs = d.add.cs; a.add_c0 = d.add.c0;
    a.gate = d.gate;
    a.mask = d.mask;
    if (d.mask && (eko != EK_F32 || d.wtp || d.add.p)) return set_error(VSC_E_INVALID, "conv3x3: a mask goes with FP32 outputs, plain weights and no residual");
    a.Ho = Ho; a.Wo = Wo; a.Cout = Cout;
    a.pad = d.pad; a.pstep = d.dil; a.act = d.act;
    if (ek == EK_F32) conv_stride<EK_F32, EK_F32>(a, d.stride, s);
    else if (ek == EK_BF16 && eko == EK_BF16) conv_stride<EK_BF16, EK_BF16>(a, d.stride, s);
    else if (ek == EK_BF16) conv_stride<EK_BF16, EK_F32>(a, d.stride, s);
    else if (eko == EK_F16) conv_stride<EK_F16, EK_F16>(a, d.stride, s);
    else conv_stride<EK_F16, EK_F32>(a, d.stride, s);
    return check_launch("conv3x3");
}

}  // namespace vsc

extern "C" int vsc_conv3x3_nhwc(const void* in, int in_cs, int in_c0, int N, int H, int W, int Cin, const void* wt,
                                const float* bias, void* out, int out_cs, int out_c0, int Cout, int stride,
                                int dilation, int pad, int act, const void* add, int add_cs, int add_c0, int dtype,
                                int out_dtype, vsc_hip_stream stream)
{
    using namespace vsc;
    if (!in || !wt || !out || N <= 0 || H <= 0 || W <= 0)
        return set_error(VSC_E_INVALID, "vsc_conv3x3_nhwc: null pointer or empty shape");
    if (stride != 1 && stride != 2) return set_error(VSC_E_INVALID, "vsc_conv3x3_nhwc: stride must be 1 or 2");
    if (act < 0 || act > 2) return set_error(VSC_E_INVALID, "vsc_conv3x3_nhwc: act must be 0, 1 or 2");
    ConvDesc d{};
    const int Ho = (H + 2 * pad - 2 * dilation - 1) / stride + 1, Wo = (W + 2 * pad - 2 * dilation - 1) / stride + 1;
    d.in = Nhwc{const_cast<void*>(in), N, H, W, Cin, in_cs, in_c0};
    d.out = Nhwc{out, N, Ho, Wo, Cout, out_cs, out_c0};
    d.add = Nhwc{const_cast<void*>(add), N, Ho, Wo, Cout, add_cs, add_c0};
    d.wt = wt; d.bias = bias;
    d.stride = stride; d.dil = dilation; d.pad = pad; d.act = act;
    d.ek_in = elem_kind(dtype); d.ek_out = elem_kind(out_dtype);
    return launch_conv3x3(d, as_stream(stream));
}

// Diagnostic (no declaration in vsc.h): a layer with packed weights.  wt: host
// [Cout][3][3][Cin] in the element type, packed and uploaded for the call;
// the output's pixel stride is its channels, input pixels hold Cin channels.
extern "C" int vsct_conv3x3_packed(const void* in, int N, int H, int W, int Cin, const void* wt, const float* bias,
                                   void* out, int Cout, int stride, int dilation, int act, int dtype, int out_dtype,
                                   vsc_hip_stream stream)
{
    using namespace vsc;
    const int eb = dtype == VSC_F32 ? 4 : 2;
    std::vector<char> pk(conv_packed_bytes(Cout, Cin, eb));
    conv_pack_weights(wt, pk.data(), Cout, Cin, eb);
    void* dev = nullptr;
    int rc = check_hip(hipMalloc(&dev, pk.size()), "vsct_conv3x3_packed");
    if (rc) return rc;
    if (!(rc = check_hip(hipMemcpy(dev, pk.data(), pk.size(), hipMemcpyHostToDevice), "vsct_conv3x3_packed"))) {
        ConvDesc d{};
        d.in = Nhwc{const_cast<void*>(in), N, H, W, Cin, Cin, 0};
        d.out = Nhwc{out, N, (H - 1) / stride + 1, (W - 1) / stride + 1, Cout, Cout, 0};
        d.wtp = dev; d.bias = bias;
        d.stride = stride; d.dil = dilation; d.pad = dilation; d.act = act;
        d.ek_in = elem_kind(dtype); d.ek_out = elem_kind(out_dtype);
        rc = launch_conv3x3(d, as_stream(stream));
    }
    (void)hipDeviceSynchronize();
    (void)hipFree(dev);
    return rc;
}

// Diagnostic (no declaration in vsc.h): the chunks whose sums a packed layer keeps
// apart, 0 when it has one sum.
extern "C" int vsct_conv_flush(int N, int H, int W, int Cin, int Cout, int stride, int dilation, int dtype)
{
    using namespace vsc;
    ConvArgs a{};
    a.N = N; a.H = H; a.W = W; a.Cin = Cin;
    a.Ho = (H - 1) / stride + 1; a.Wo = (W - 1) / stride + 1; a.Cout = Cout;
    a.pstep = dilation;
    if (dtype == VSC_F32) return stride == 2 ? conv_flush<EK_F32, 2>(a) : conv_flush<EK_F32, 1>(a);
    return stride == 2 ? conv_flush<EK_BF16, 2>(a) : conv_flush<EK_BF16, 1>(a);
}
