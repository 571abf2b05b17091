// One tile of the temporally blocked consistency solver, shared by the kernels
// that walk tiles (stab.hip, resident.hip).
#pragma once

#include "vsc_internal.h"

#include <type_traits>

namespace vsc {

// ---------------------------------------------------------------------------
// consistency solver, temporally blocked (planar state, one channel per block)
//
// A block of 128*STRIPS threads owns a TW x TH tile of one channel plane
// (TW = 128 columns, TH = STRIPS*R rows) that overlaps its neighbours by a halo of `halo`
// pixels.  Thread (tx, strip) keeps the R pixels of column tx in rows
// strip*R .. strip*R+R-1 in registers: O, U, lapP, A, w.  O and U are read
// with halo from the *in* planes and written to the *out* planes (neighbouring
// blocks read the pixels a block writes).  After `sweeps` <= halo sweeps the
// inner (TW-2*halo) x (TH-2*halo) pixels are exact and written back; halo
// pixels whose out-of-tile neighbours are missing never reach the output.
//
// Neighbour exchange goes through LDS, stored column-major: the R values of
// (strip, column) are contiguous with a padded stride RS = R+4 (RS/4 odd, so a
// 16-byte access of 8 consecutive lanes covers all 32 banks once).  A sweep
// reads the left and right columns of one plane with 16-byte loads issued one
// 4-row chunk ahead of their use and writes each chunk's new values into the
// other plane with a 16-byte store as soon as they are computed; the planes
// alternate, one barrier per sweep.  The up/down neighbours come from the
// thread's own registers (LDS only at the strip ends).
//
// Arithmetic per pixel and sweep is that of k_consist_sweep; lapP (the
// Laplacian of the processed frame, a constant of the level) is an input,
// computed once per level with the same operations, so the result is identical.
// The reference's neighbour conditions (flowconsistency.cu:215-236) cost no
// per-pixel work where they are uniform: a column whose left (right) neighbour
// is excluded reads a zero column from LDS instead (the neighbour sum gains a
// +0 term, which changes no nonzero sum), so only waves whose strip meets the
// image's top or bottom rows test rows per pixel, and waves wholly outside the
// image (never stored, never read by an image pixel) skip the arithmetic.
// ---------------------------------------------------------------------------
static constexpr int SB_TW = 128;
static constexpr int SB_R = 28;      // rows per thread, reference op order (5 values per pixel)
static constexpr int SB_R_FMA = 32;  // FMA form: 4 values per pixel in registers, taller strips
static constexpr int SB_STRIPS = 4;

// Tile placement along one axis of length L: tiles of T pixels whose outer
// `h` pixels on a side facing another tile are halo.  When L >= T the first
// tile starts at 0 and the last ends at L (flush with the image: an image
// edge needs no halo, its missing neighbours are the reference's boundary),
// the tiles between output T - 2h pixels each; otherwise tile i starts at
// i*(T - 2h) - h and pixels outside the image are padding.  A tile computes
// [start, start + T) and stores [lo, hi); the output ranges partition [0, L).
struct TileSpan {
    int start, lo, hi;
};

__host__ __device__ inline int tile_count(int L, int T, int h)
{
    const int O = T - 2 * h;
    if (L < T) return (L + O - 1) / O;
    if (L == T) return 1;
    const int rest = L - 2 * (T - h);
    return 2 + (rest > 0 ? (rest + O - 1) / O : 0);
}

__host__ __device__ inline TileSpan tile_span(int i, int n, int L, int T, int h)
{
    const int O = T - 2 * h;
    if (L < T) {
        const int s = i * O - h;
        return TileSpan{s, s + h, s + T - h < L ? s + T - h : L};
    }
    if (L == T) return TileSpan{0, 0, L};
    if (i == 0) return TileSpan{0, 0, T - h};
    const int lo = T - h + (i - 1) * O;
    if (i == n - 1) return TileSpan{L - T, lo, L};
    return TileSpan{lo - h, lo, lo + O};
}

// Rows of a strip are visited in ascending (REV false) or descending (REV
// true) order.  A row's old value is still needed by the next row visited
// after the row itself is updated, so a sweep leaves its O and U shifted by
// one register; the kernel alternates the two orders, and a descending sweep
// shifts them back, so a pair of sweeps needs no register copies.  Each
// pixel's arithmetic (and its operation order) is the same in both orders.
// colL / colR hold the left / right neighbours, or zeros where the column has
// none (cntc = number of horizontal neighbours).  EDGE says which rows lack
// a vertical neighbour: SE_NONE none, SE_TOP row 0 (the image's top row),
// SE_BOTTOM rows R-2 and R-1 (the image's last two rows), SE_ROWS any row,
// tested per pixel against rU / rD.
enum StripEdge { SE_NONE = 0, SE_TOP = 1, SE_BOTTOM = 2, SE_ROWS = 3 };

template <int R, bool MOM, int EDGE, bool REV>
__device__ __forceinline__ void sweep_strip(float (&o)[R], float (&u)[R], const float (&a)[R], const float (&w)[R],
                                            const float (&lp)[R], const float* colL, const float* colR,
                                            float* nxt, float up_edge, float dn_edge, float step, float mom, int cntc,
                                            int rU, int rD)
{
    constexpr int NK = R / 4;
    float4 l4 = *reinterpret_cast<const float4*>(colL + (REV ? R - 4 : 0));
    float4 r4 = *reinterpret_cast<const float4*>(colR + (REV ? R - 4 : 0));
    float prev = REV ? dn_edge : up_edge;  // old value of the row visited before
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int k = REV ? NK - 1 - i : i;
        float4 ln = l4, rn = r4;
        if (i + 1 < NK) {
            const int kn = REV ? k - 1 : k + 1;
            ln = *reinterpret_cast<const float4*>(colL + 4 * kn);
            rn = *reinterpret_cast<const float4*>(colR + 4 * kn);
        }
        const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
        const float rv[4] = {r4.x, r4.y, r4.z, r4.w};
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int j = REV ? 3 - jj : jj;
            const int r = 4 * k + j;
            const float cur = o[r];
            const float up = REV ? (r > 0 ? o[r - 1] : up_edge) : prev;
            const float dn = REV ? prev : (r < R - 1 ? o[r + 1] : dn_edge);
            float lo = rv[j] + lv[j];
            int cnt = cntc;
            if (EDGE == SE_ROWS) {
                if (r <= rD) { lo += dn; cnt += 1; }
                if (r >= rU) { lo += up; cnt += 1; }
            } else {
                if (!(EDGE == SE_BOTTOM && r >= R - 2)) { lo += dn; cnt += 1; }
                if (!(EDGE == SE_TOP && r == 0)) { lo += up; cnt += 1; }
            }
            lo -= (float)cnt * cur;
            const float t1 = w[r] * (cur - a[r]);
            const float t2 = lo - lp[r];
            const float g = t2 - t1;
            const float sg = step * g;
            o[r] = MOM ? (cur + sg) + mom * u[r] : cur + sg;
            u[r] = sg;
            prev = cur;
        }
        // publish the chunk's new values for the next sweep
        *reinterpret_cast<float4*>(nxt + 4 * k) = make_float4(o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]);
        l4 = ln;
        r4 = rn;
    }
}

// The same sweep in FMA form: q = cnt + w and kk = step*fma(-w, A, lapP) are
// per-pixel constants, and per pixel
//   X = fma(-q, O, sum of neighbours); U' = fma(step, X, -kk); O' = O + U' (+ mom*U)
// (7 VALU operations in the interior instead of 13).
template <int R, bool MOM, int EDGE, bool REV>
__device__ __forceinline__ void sweep_strip_fma(float (&o)[R], float (&u)[R], const float (&q)[R],
                                                const float (&kk)[R], const float* colL, const float* colR,
                                                float* nxt, float up_edge, float dn_edge, float step, float mom, int rU,
                                                int rD)
{
    constexpr int NK = R / 4;
    float4 l4 = *reinterpret_cast<const float4*>(colL + (REV ? R - 4 : 0));
    float4 r4 = *reinterpret_cast<const float4*>(colR + (REV ? R - 4 : 0));
    float prev = REV ? dn_edge : up_edge;  // old value of the row visited before
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int k = REV ? NK - 1 - i : i;
        float4 ln = l4, rn = r4;
        if (i + 1 < NK) {
            const int kn = REV ? k - 1 : k + 1;
            ln = *reinterpret_cast<const float4*>(colL + 4 * kn);
            rn = *reinterpret_cast<const float4*>(colR + 4 * kn);
        }
        const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
        const float rv[4] = {r4.x, r4.y, r4.z, r4.w};
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int j = REV ? 3 - jj : jj;
            const int r = 4 * k + j;
            const float cur = o[r];
            const float up = REV ? (r > 0 ? o[r - 1] : up_edge) : prev;
            const float dn = REV ? prev : (r < R - 1 ? o[r + 1] : dn_edge);
            float sum = rv[j] + lv[j];
            if (EDGE == SE_ROWS) {
                if (r <= rD) sum += dn;
                if (r >= rU) sum += up;
            } else {
                if (!(EDGE == SE_BOTTOM && r >= R - 2)) sum += dn;
                if (!(EDGE == SE_TOP && r == 0)) sum += up;
            }
            const float X = __builtin_fmaf(-q[r], cur, sum);
            const float sg = __builtin_fmaf(step, X, -kk[r]);
            const float on = cur + sg;
            o[r] = MOM ? __builtin_fmaf(mom, u[r], on) : on;
            u[r] = sg;
            prev = cur;
        }
        // publish the chunk's new values for the next sweep
        *reinterpret_cast<float4*>(nxt + 4 * k) = make_float4(o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]);
        l4 = ln;
        r4 = rn;
    }
}

// LDS row stride of a strip (floats): an odd number of 16-byte groups
template <int R> constexpr int sb_rs() { return ((R / 4) % 2 == 0) ? R + 4 : R + 8; }

// One tile of the temporally blocked solver: `sweeps` Jacobi sweeps of
// channel plane tile `tile` (tiles_x x tiles_y tiles per channel, channels
// one after the other) of a planar 3-channel level.  sO: the block's LDS
// exchange buffer.  Every thread of the block calls it with the same tile.
template <int R, int STRIPS, bool FMA>
__device__ __forceinline__ void consist_tile(
    const float* __restrict__ LapP, const float* __restrict__ A, const float* __restrict__ Wt, const float* Oin,
    float* Oout, const float* Uin, float* Uout, int W, int H, int sweeps, int first_sweep, float step, float mom,
    int halo, int tiles_x, int tiles_y, int store_u, int tile, float (*sO)[STRIPS][SB_TW + 1][sb_rs<R>()])
{
    constexpr int TW = SB_TW;
    constexpr int TH = STRIPS * R;
    constexpr int RS = sb_rs<R>();
    static_assert(R % 4 == 0 && (RS / 4) % 2 == 1, "strip stride must be an odd number of 16-byte groups");
    const int c = tile / (tiles_x * tiles_y);
    const int bxy = tile - c * tiles_x * tiles_y;
    const int bty = bxy / tiles_x, btx = bxy - bty * tiles_x;
    const long long plane = (long long)W * H;
    const float* __restrict__ Lc = LapP + c * plane;
    const float* __restrict__ Ac = A + c * plane;
    const float* __restrict__ Wc = Wt + c * plane;
    const float* __restrict__ Oi = Oin + c * plane;
    float* __restrict__ Oo = Oout + c * plane;
    const float* __restrict__ Ui = Uin + c * plane;
    float* __restrict__ Uo = Uout + c * plane;

    const int tx = threadIdx.x % TW;
    // TW is a multiple of the wave size, so a strip is wave-uniform: keep the
    // row bookkeeping in scalar registers.
    const int strip = __builtin_amdgcn_readfirstlane(threadIdx.x / TW);
    const int wave_tx0 = __builtin_amdgcn_readfirstlane((threadIdx.x % TW) & ~63);
    const int ty0 = strip * R;
    const TileSpan sx = tile_span(btx, tiles_x, W, TW, halo);
    const TileSpan sy = tile_span(bty, tiles_y, H, TH, halo);
    const int gx0 = sx.start, gy0 = sy.start;
    const int gx = gx0 + tx;
    const bool hr = (gx + 1) < (W - 1), hl = (gx - 1) >= 0;
    const int gys = gy0 + ty0;
    // no pixel of this wave (64 columns x R rows) lies in the image
    const bool wave_out = (gx0 + wave_tx0 >= W) || (gx0 + wave_tx0 + 63 < 0) || (gys >= H) || (gys + R - 1 < 0);
    // Which rows of this wave's strip lack a vertical neighbour.  With tiles
    // flush with the image (H >= TH), only the top tile's first strip (row 0)
    // and the bottom tile's last strip (rows R-2, R-1) hold such rows whose
    // values can reach a stored pixel: a tile's other rows with a missing
    // neighbour lie on its own edge towards a neighbouring tile, inside the
    // halo, whose values are not exact anyway.
    int edge;
    if (H >= TH)
        edge = gys == 0 ? SE_TOP : gys + R == H ? SE_BOTTOM : SE_NONE;
    else
        edge = (gys >= 1 && gys + R - 1 <= H - 3) ? SE_NONE : SE_ROWS;
    const int cntc = (hr ? 1 : 0) + (hl ? 1 : 0);

    // FMA: w holds q = cnt + w, lp holds kk; a is unused (and not loaded)
    float o[R], u[R], a[FMA ? 1 : R], w[R], lp[R];
    // Loads are unconditional, from clamped positions, so that all of them
    // issue back to back: a tile pixel outside the image holds some finite
    // in-image value that no in-image pixel ever reads (the neighbour sets
    // exclude out-of-image positions) and that is never stored.
    // 32-bit element offsets (a plane holds < 2^31 pixels).
    const int gxc = min(max(gx, 0), W - 1);
    const bool load_u = first_sweep > 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int gyc = min(max(gys + r, 0), H - 1);
        const int i = gyc * W + gxc;
        o[r] = Oi[i];
        if (!FMA) a[r] = Ac[i];
        w[r] = Wc[i];
        lp[r] = Lc[i];
    }
    if (load_u) {
#pragma unroll
        for (int r = 0; r < R; ++r) u[r] = Ui[min(max(gys + r, 0), H - 1) * W + gxc];
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) u[r] = 0.0f;
    }

    // zero columns, published by the first sweep's barrier
    for (int i = threadIdx.x; i < 2 * STRIPS * RS; i += TW * STRIPS) sO[i / (STRIPS * RS)][(i / RS) % STRIPS][TW][i % RS] = 0.0f;
    // neighbour columns (clamped at the tile edge, where the lane is halo)
    const int txl = !hl ? TW : tx > 0 ? tx - 1 : 0;
    const int txr = !hr ? TW : tx < TW - 1 ? tx + 1 : TW - 1;
    const int stU = strip > 0 ? strip - 1 : 0;
    const int stD = strip < STRIPS - 1 ? strip + 1 : STRIPS - 1;
    // row r has an up neighbour iff r >= rU and a down neighbour iff r <= rD
    const int rU0 = 1 - gys;
    const int rD0 = (H - 3) - gys;

    // One sweep: once every strip's values are in plane s&1, update this
    // strip from its neighbours there, writing each 4-row chunk's new values
    // into plane (s+1)&1 as soon as they are computed (the writes spread over
    // the sweep instead of bunching before its barrier).
    auto sweep = [&](int s, auto mom_c, auto rev_c, auto edge_c) {
        constexpr bool MOM = decltype(mom_c)::value, REV = decltype(rev_c)::value;
        constexpr int EDGE = decltype(edge_c)::value;
        float (*buf)[TW + 1][RS] = sO[s & 1];
        __syncthreads();
        const float up_edge = buf[stU][tx][R - 1];
        const float dn_edge = buf[stD][tx][0];
        const float* colL = buf[strip][txl];
        const float* colR = buf[strip][txr];
        float* nxt = sO[(s + 1) & 1][strip][tx];
        int rU = rU0, rD = rD0;
        // opaque per sweep: keeps the compiler from hoisting 2*R row
        // predicates out of the sweep loop into scalar registers
        asm volatile("" : "+s"(rU), "+s"(rD));
        if constexpr (FMA)
            sweep_strip_fma<R, MOM, EDGE, REV>(o, u, w, lp, colL, colR, nxt, up_edge, dn_edge, step, mom, rU, rD);
        else
            sweep_strip<R, MOM, EDGE, REV>(o, u, a, w, lp, colL, colR, nxt, up_edge, dn_edge, step, mom, cntc, rU,
                                           rD);
    };
    // The level's first sweep has no momentum term; after it, ascending and
    // descending sweeps alternate in pairs.  The initial values go to plane 0.
    auto run = [&](auto edge_c) {
        const std::true_type yes{};
        const std::false_type no{};
        {
            float* own = sO[0][strip][tx];
#pragma unroll
            for (int k = 0; k < R / 4; ++k)
                *reinterpret_cast<float4*>(own + 4 * k) =
                    make_float4(o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]);
        }
        int s = 0;
        if (first_sweep == 0) {
            sweep(0, no, no, edge_c);
            s = 1;
        }
        for (; s + 1 < sweeps; s += 2) {
            sweep(s, yes, no, edge_c);
            sweep(s + 1, yes, yes, edge_c);
        }
        if (s < sweeps) sweep(s, yes, no, edge_c);
    };
    // Every wave passes one barrier per sweep, whichever branch it takes.
    if (wave_out) {
        for (int s = 0; s < sweeps; ++s) __syncthreads();
    } else if (edge == SE_NONE) {
        run(std::integral_constant<int, SE_NONE>{});
    } else if (edge == SE_TOP) {
        run(std::integral_constant<int, SE_TOP>{});
    } else if (edge == SE_BOTTOM) {
        run(std::integral_constant<int, SE_BOTTOM>{});
    } else {
        run(std::integral_constant<int, SE_ROWS>{});
    }

    // each image pixel is stored by exactly one tile (its span's output range)
    if (gx >= sx.lo && gx < sx.hi) {
        const int wbase = gys * W + gx;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int gy = gys + r;
            if (gy >= sy.lo && gy < sy.hi) {
                Oo[wbase + r * W] = o[r];
                if (store_u) Uo[wbase + r * W] = u[r];
            }
        }
    }
}

}  // namespace vsc
