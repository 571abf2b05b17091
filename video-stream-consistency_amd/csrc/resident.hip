// Consistency solver with the level resident on the chip (FMA form): one
// launch runs every sweep of a pyramid level.
//
// The temporally blocked solver (stab.hip) reloads a tile for every halo's
// worth of sweeps and sweeps twice the level's area.  Here a block keeps its
// tile for the whole level and only the halo travels: every `h` sweeps a tile
// publishes the pixels its neighbours' halos need and takes its own halo from
// them.  A level fits when it has at most one tile per CU slot.
//
// Layout: a wave owns 64*PX columns x R rows, a lane PX neighbouring columns,
// NW waves stand on top of each other.  O, U and q stay in registers, k in LDS
// (one PX-wide read per row and sweep).  Left and right neighbours of a lane's
// outer pixels come from the next lane by a wave shift inside the addition
// (DPP), up and down neighbours from the lane's own registers, and from LDS at
// the waves' first and last rows: one barrier per sweep.
//
// Strips.  A level too large for the chip is swept in rounds of up to some tens
// of sweeps; in a round, strips of rows are resident one after the other, each
// with as many rows above its own as the round has sweeps, and one more below
// (their values go wrong from the cut inwards, a row a sweep, below two with the
// first: the row above the last has no lower neighbour; they are not kept).  O and U go
// through memory once a round.  A 3840x2160 frame of 150 and 75 sweeps: 2553 us
// against 3787 with the blocked solver on level 0, a 2560x1440 one 1211 against
// 1595, one of 2000x1125 898 against 985.
//
// The image's edges cost no branches: a wave shift brings 0 into lanes 0 and
// 63, so a tile flush with the image's left or right edge sees the missing
// neighbour as +0 (which changes no nonzero sum), the first wave's upper and
// the last wave's lower neighbours are zeros, and only the two exclusions
// inside a tile (column W-1 as column W-2's right neighbour, row H-1 as row
// H-2's lower one) are selects.  Tiles lie wholly inside the image.
//
// Waiting.  A block waits for its neighbours' publications, so all blocks of a
// launch have to run at once.  Resident launches of one process take turns on a
// device (an event orders each after the one before), and other kernels end,
// but nothing keeps another process' blocks from holding CUs.  So every wait is
// bounded: a launch whose wait exceeds RES_WAIT_TICKS raises its abort word,
// every block leaves, and k_consist_finish, launched behind it, computes the
// level from its initial state, which the resident launch does not write.
// k_consist_finish takes (phase, tile) items in ticket order and an item waits
// only for items of smaller tickets, so it needs no co-residency; it also tells
// the host, which keeps to the blocked solver for a while.
//
// Measured (FMA form, bit-identical to the blocked solver, whole level): 150
// sweeps of 1920x1080 372 us against 732, of 1571x784 260 against 489, of
// 640x360 130 to 139 against 220, 75 sweeps of 960x540 89 against 117; reference
// order: 640x360 151 against 378, 1281x719 312 against 489.  A sweep runs at
// 85% of the vector units' rate; an exchange costs 2 to 5 us, most of it the
// halo's way through memory (the flags alone cost 0.1 us).
#include "vsc_internal.h"
#include "stab_tile.h"

#include <algorithm>
#include <mutex>

namespace vsc {
namespace {

// control words of a stream (device memory, all zero at rest)
enum { CTL_ABORT = 0, CTL_EXIT = 16, CTL_TICKET = 32, CTL_FEXIT = 48, CTL_FLAGS = 64, CTL_STRIDE = 16, CTL_FSTRIDE = 4 };
constexpr int RES_MAX_TILES = 1024, FIN_MAX_TILES = 4096;
constexpr int RES_NW = 8;   // waves of a block
static_assert((CTL_FLAGS + RES_MAX_TILES * CTL_STRIDE) * 4 <= RESIDENT_CTL_BYTES &&
              (CTL_FLAGS + FIN_MAX_TILES * CTL_FSTRIDE) * 4 <= RESIDENT_CTL_BYTES, "control block size");
// 100 MHz ticks: 3 ms, several times the longest kernel of a frame
constexpr long long RES_WAIT_TICKS = 300000;

__device__ inline unsigned ld_agent(const unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void st_agent(unsigned* p, unsigned v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

struct ResArgs {
    const float* K;       // k (FMA form) or lapP (reference order)
    const float* Q;       // q or w
    const float* A;       // reference order: the adapted processed frame
    const float* Oin;
    float* Oout;
    const float* Uin;     // null: zero (the level's first sweeps)
    float* Uout;          // null: not kept (its last ones)
    float* X[2][2];       // exchange planes: [set][0] holds O, [set][1] holds U
    long long plane;      // elements of a channel's plane (of all but X)
    int own0, own1;       // rows that are the launch's to write
    int W, H, iters, h, nx, ny, per_xcd;   // H: rows of the region that the launch sweeps
    float step, mom;
    unsigned* ctl;
};

// start of tile i of n along an axis of length L (T <= L): spread evenly,
// rounded up to whole multiples of `q` (so that two neighbours are no further
// apart than the even distance rounded up) but for the last, which ends at L
__host__ __device__ inline int res_start(int i, int n, int L, int T, int q)
{
    if (i == 0) return 0;
    if (i == n - 1) return L - T;
    const unsigned at = ((unsigned)i * (unsigned)(L - T) + (unsigned)(n - 2)) / (unsigned)(n - 1);   // (launcher: below 2^32)
    return (int)((at + q - 1) / q * q);
}

template <int PX> struct Quad;
template <> struct Quad<4> {
    typedef float T __attribute__((ext_vector_type(4), aligned(4)));
    typedef uint32_t B __attribute__((ext_vector_type(4)));
};
template <> struct Quad<2> {
    typedef float T __attribute__((ext_vector_type(2), aligned(4)));
    typedef uint32_t B __attribute__((ext_vector_type(2)));
};
template <> struct Quad<1> {
    typedef float T __attribute__((ext_vector_type(1), aligned(4)));
    typedef uint32_t B;
};

// A lane's pixels to and from an exchange plane, coherent across the device
// (sc1: past the XCD's own L2).  NOWHERE lies past every
// plane's end, and a tile's rows further does not wrap.
constexpr int AUX_AGENT = 16, NOWHERE = 1 << 30;
template <int PX, int AUX = AUX_AGENT>
__device__ __forceinline__ void store_px(const typename Quad<PX>::T& v, const __amdgpu_buffer_rsrc_t& x, int at, int row)
{
    using B = typename Quad<PX>::B;
    if constexpr (PX == 4) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(B, v), x, at, row, AUX);
    else if constexpr (PX == 2) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(B, v), x, at, row, AUX);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(B, v), x, at, row, AUX);
}
template <int PX, int AUX = AUX_AGENT>
__device__ __forceinline__ typename Quad<PX>::T load_px(const __amdgpu_buffer_rsrc_t& x, int at, int row)
{
    using V = typename Quad<PX>::T;
    if constexpr (PX == 4) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(x, at, row, AUX));
    else if constexpr (PX == 2) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(x, at, row, AUX));
    else return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(x, at, row, AUX));
}

// buffer descriptor of a plane of `n` floats
__device__ inline __amdgpu_buffer_rsrc_t plane_rsrc(const float* p, long long n)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, (int)(n * 4), 0x00020000);
}

__device__ inline float from_left(float v)    // lane i-1's value, 0 in lane 0
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ inline float from_right(float v)   // lane i+1's value, 0 in lane 63
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}

template <int PX, int R, int NW, bool FMA>
__global__ __launch_bounds__(64 * NW, (8 / NW) * NW / 4) void k_consist_resident(ResArgs a)
{
    constexpr int TW = 64 * PX, TH = NW * R;
    using V = typename Quad<PX>::T;
    __shared__ __attribute__((aligned(16))) float sK[TH][TW];
    // [sweep parity]: the waves' first and last rows (wave w's first row at 2w - 1, its last at 2w; the tile's
    // outer two, which nobody reads, at DUMP)
    constexpr int DUMP = 2 * NW - 2;
    __shared__ __attribute__((aligned(16))) float sE[2][2 * NW - 1][TW];
    __shared__ int s_go;

    const int ntiles = a.nx * a.ny * 3;
    const int tile = (blockIdx.x % 8) * a.per_xcd + blockIdx.x / 8;   // XCD-contiguous runs of tiles
    if (tile >= ntiles) return;
    const int tid = threadIdx.x, lane = tid % 64;
    const int wv = __builtin_amdgcn_readfirstlane(tid / 64);
    const int c = tile / (a.nx * a.ny), bxy = tile - c * a.nx * a.ny;
    const int ty = bxy / a.nx, tx = bxy - ty * a.nx;
    const int gx0 = res_start(tx, a.nx, a.W, TW, 4), gy0 = res_start(ty, a.ny, a.H, TH, 1);
    unsigned* flags = a.ctl + CTL_FLAGS;

    if (tid == 0) s_go = ld_agent(a.ctl + CTL_ABORT) == 0u;   // given up already?
    const long long plane = (long long)a.W * a.H;              // of X; what a launch reaches of the other planes
    const int row0 = wv * R;                                   // the wave's first row in the tile
    const int base = (gy0 + row0) * a.W + gx0 + PX * lane;     // element offset of the lane's first pixel
    __syncthreads();
    bool go = s_go;
    if (go) {
        V o[R], u[R], q[R], ad[FMA ? 1 : R];   // FMA form: ad unused
        {
            // (buffer accesses: one offset register for all rows) k first, through registers that o, q and u take afterwards
            const __amdgpu_buffer_rsrc_t O_ = plane_rsrc(a.Oin + c * a.plane, plane), Q_ = plane_rsrc(a.Q + c * a.plane, plane);
            const __amdgpu_buffer_rsrc_t K_ = plane_rsrc(a.K + c * a.plane, plane), A_ = plane_rsrc(a.A + c * a.plane, plane);
#pragma unroll
            for (int r = 0; r < R; ++r)
                *reinterpret_cast<V*>(&sK[row0 + r][PX * lane]) = load_px<PX, 0>(K_, base * 4, r * a.W * 4);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                o[r] = load_px<PX, 0>(O_, base * 4, r * a.W * 4);
                q[r] = load_px<PX, 0>(Q_, base * 4, r * a.W * 4);
                if constexpr (!FMA) ad[r] = load_px<PX, 0>(A_, base * 4, r * a.W * 4);
                u[r] = V{};
            }
            if (a.Uin) {
                const __amdgpu_buffer_rsrc_t U_ = plane_rsrc(a.Uin + c * a.plane, plane);
#pragma unroll
                for (int r = 0; r < R; ++r) u[r] = load_px<PX, 0>(U_, base * 4, r * a.W * 4);
            }
        }
        // columns and rows whose values are exact after h sweeps
        const int xe0 = tx == 0 ? 0 : a.h, xe1 = tx == a.nx - 1 ? TW : TW - a.h;
        const int ye0 = ty == 0 ? 0 : a.h, ye1 = ty == a.ny - 1 ? TH : TH - a.h;
        const bool lane_exact = PX * lane >= xe0 && PX * lane < xe1;
        // the parts of them that the neighbours' halos take
        const int px0 = PX * lane, px1 = px0 + PX;
        bool col_pub = false;
        if (tx > 0) {
            const int e = res_start(tx - 1, a.nx, a.W, TW, 4) + TW - gx0;    // the left tile's right edge
            col_pub = px1 > e - a.h && px0 < e;
        }
        if (tx < a.nx - 1) {
            const int b = res_start(tx + 1, a.nx, a.W, TW, 4) - gx0;         // the right tile's left edge
            col_pub = col_pub || (px1 > b && px0 < b + a.h);
        }
        int up_e = 0, dn_b = TH;                                             // rows [up_e - h, up_e), [dn_b, dn_b + h)
        if (ty > 0) up_e = res_start(ty - 1, a.ny, a.H, TH, 1) + TH - gy0;
        if (ty < a.ny - 1) dn_b = res_start(ty + 1, a.ny, a.H, TH, 1) - gy0;
        const int at_row = lane_exact ? base * 4 : NOWHERE, at_col = lane_exact && col_pub ? base * 4 : NOWHERE;
        const bool bottom = ty == a.ny - 1 && wv == NW - 1;
        const bool right63 = tx == a.nx - 1 && lane == 63;
        // reference order: neighbour count of the lane's columns in a row with both vertical neighbours
        float cnt[PX];
#pragma unroll
        for (int p = 0; p < PX; ++p) {
            const int gx = gx0 + PX * lane + p;
            cnt[p] = 2.0f + (gx + 1 < a.W - 1 ? 1.0f : 0.0f) + (gx > 0 ? 1.0f : 0.0f);
        }
        const bool first_row = ty == 0 && wv == 0;
        const float step = a.step, mom = a.mom;

        const bool top = wv == 0, low = wv == NW - 1;               // no wave above / below
        const int e_up = top ? 0 : 2 * wv - 2, e_dn = low ? 0 : 2 * wv + 1;
        const int w_up = top ? DUMP : 2 * wv - 1, w_dn = low ? DUMP : 2 * wv;
        auto row_update = [&](int r, const V& vk, V& prev, const V& up, const V& dn) {
            const V cur = o[r];
            const float rm = right63 ? 0.0f : cur[PX - 1];
            const float lf = from_left(cur[PX - 1]), rt = from_right(PX == 1 ? rm : cur[0]);
#pragma unroll
            for (int p = 0; p < PX; ++p) {
                const float rv = p == PX - 1 ? rt : p == PX - 2 ? rm : cur[p + 1 < PX ? p + 1 : 0];
                const float lv = p == 0 ? lf : cur[p > 0 ? p - 1 : 0];
                float sum = rv + lv;
                sum += dn[p];
                sum += up[p];
                if constexpr (FMA) {
                    const float X = __builtin_fmaf(-q[r][p], cur[p], sum);
                    const float sg = __builtin_fmaf(step, X, -vk[p]);
                    const float on = cur[p] + sg;
                    o[r][p] = __builtin_fmaf(mom, u[r][p], on);
                    u[r][p] = sg;
                } else {
                    float n = cnt[p];
                    if (r == 0) n -= first_row ? 1.0f : 0.0f;
                    if (r >= R - 2) n -= bottom ? 1.0f : 0.0f;
                    sum -= n * cur[p];
                    const float t1 = q[r][p] * (cur[p] - ad[r][p]);
                    const float t2 = sum - vk[p];
                    const float g = t2 - t1;
                    const float sg = step * g;
                    o[r][p] = (cur[p] + sg) + mom * u[r][p];
                    u[r][p] = sg;
                }
            }
            prev = cur;
        };
        auto put_edge = [&](int par, int at, int r) { *reinterpret_cast<V*>(&sE[par][at][PX * lane]) = o[r]; };
        // One sweep.  Rows are visited in ascending and descending order on
        // alternate sweeps: a row's old value is needed by the next row after
        // the row is updated, so one order leaves the registers shifted by a
        // row and the other shifts them back (no copies in a pair of sweeps).
        // pub: the row's published pixels are stored as soon as they are computed,
        // under the rest of the sweep (lanes and rows that publish nothing are
        // sent past the plane's end, where the buffer store drops them).
        auto sweep = [&](int par, auto rev_c, bool pub, const __amdgpu_buffer_rsrc_t& XO, const __amdgpu_buffer_rsrc_t& XU) {
            constexpr bool REV = decltype(rev_c)::value;
            // opaque per sweep: keeps R rows' addresses and predicates from being hoisted into registers
            int yw = row0, pitch = a.W * 4;
            if constexpr (REV) asm volatile("" : "+s"(yw), "+s"(pitch));
            __syncthreads();
            V upe = *reinterpret_cast<const V*>(&sE[par][e_up][PX * lane]);
            V dne = *reinterpret_cast<const V*>(&sE[par][e_dn][PX * lane]);
#pragma unroll
            for (int p = 0; p < PX; ++p) {
                upe[p] = top ? 0.0f : upe[p];
                dne[p] = low ? 0.0f : dne[p];
            }
            V prev, kn = *reinterpret_cast<const V*>(&sK[row0 + (REV ? R - 1 : 0)][PX * lane]);
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int r = REV ? R - 1 - i : i;
                // k is read one row ahead and no further (the scheduler would read all rows' at once, into registers)
                const V vk = kn;
                if (i + 1 < R) kn = *reinterpret_cast<const V*>(&sK[row0 + (REV ? r - 1 : r + 1)][PX * lane]);
                V up, dn;
                if (REV) {
                    dn = i == 0 ? dne : prev;
                    up = r > 0 ? o[r > 0 ? r - 1 : 0] : upe;
                } else {
                    up = i == 0 ? upe : prev;
                    dn = r < R - 1 ? o[r < R - 1 ? r + 1 : 0] : dne;
                }
                if (r == R - 2) {
#pragma unroll
                    for (int p = 0; p < PX; ++p) dn[p] = bottom ? 0.0f : dn[p];
                }
                row_update(r, vk, prev, up, dn);
                if (r == 0) put_edge(par ^ 1, w_up, 0);
                if (r == R - 1) put_edge(par ^ 1, w_dn, R - 1);
                // the row is computed here, not sunk behind the next branch with its operands kept
#pragma unroll
                for (int p = 0; p < PX; ++p) asm volatile("" ::"v"(o[r][p]));
                if (REV && pub) {
                    const int y = yw + r;
                    const bool ex = (y >= ye0) & (y < ye1);
                    const bool all = ((y < up_e) & (y >= up_e - a.h)) | ((y >= dn_b) & (y < dn_b + a.h));
                    const int at = (all ? at_row : at_col) + r * pitch;
                    const int to = ex ? at : NOWHERE;
                    store_px<PX>(o[r], XO, to, 0);
                    store_px<PX>(u[r], XU, to, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };

        const int phases = (a.iters + a.h - 1) / a.h;
        for (int ph = 0; ph < phases; ++ph) {
            put_edge(0, w_up, 0);
            put_edge(0, w_dn, R - 1);
            // the set that leaves Oout's plane free for the end
            const int set = (phases - ph) & 1;
            const __amdgpu_buffer_rsrc_t XO = plane_rsrc(a.X[set][0] + c * plane, plane), XU = plane_rsrc(a.X[set][1] + c * plane, plane);
            const bool last = ph == phases - 1;
            // h is even: every phase but the last is whole pairs, and the last sweep of them publishes
            const int n = last ? a.iters - ph * a.h : a.h;
            int s = 0;
            for (; s + 1 < n; s += 2) {
                sweep(0, std::false_type{}, false, XO, XU);
                sweep(1, std::true_type{}, !last && s + 2 == n, XO, XU);
            }
            if (last) {
                if (s < n) sweep(0, std::false_type{}, false, XO, XU);
                break;
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's stores have reached memory
            __syncthreads();
            if (wv == 0) {
                if (lane == 0) st_agent(flags + tile * CTL_STRIDE, (unsigned)(ph + 1));
                // lanes 0 .. 8 watch the 3 x 3 tiles around this one, lane 9 the abort word
                const int dx = lane % 3 - 1, dy = lane / 3 - 1;
                const bool nb = lane < 9 && tx + dx >= 0 && tx + dx < a.nx && ty + dy >= 0 && ty + dy < a.ny;
                const unsigned* w = nb ? flags + (tile + dy * a.nx + dx) * CTL_STRIDE : a.ctl + CTL_ABORT;
                const long long t0 = wall_clock64();
                int ok = 0;
                for (;;) {
                    const unsigned v = ld_agent(w);
                    if (__any(!nb && v != 0u)) break;
                    if (__all(!nb || v >= (unsigned)(ph + 1))) {
                        ok = 1;
                        break;
                    }
                    if (wall_clock64() - t0 > RES_WAIT_TICKS) {
                        if (lane == 0) st_agent(a.ctl + CTL_ABORT, 1u);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                if (lane == 0) s_go = ok;
            }
            __syncthreads();
            if (!s_go) {
                go = false;
                break;
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int y = row0 + r;
                if (!lane_exact || y < ye0 || y >= ye1) {
                    o[r] = load_px<PX>(XO, base * 4, r * a.W * 4);
                    u[r] = load_px<PX>(XU, base * 4, r * a.W * 4);
                }
            }
        }
        if (go) {
            const __amdgpu_buffer_rsrc_t Oo = plane_rsrc(a.Oout + c * a.plane, plane);
            const __amdgpu_buffer_rsrc_t Uo = plane_rsrc(a.Uout + c * a.plane, plane);
            if (lane_exact) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int y = row0 + r;
                    if (y < ye0 || y >= ye1 || gy0 + y < a.own0 || gy0 + y >= a.own1) continue;
                    store_px<PX, 0>(o[r], Oo, base * 4, r * a.W * 4);
                    if (a.Uout) store_px<PX, 0>(u[r], Uo, base * 4, r * a.W * 4);
                }
            }
        }
    }
    // leave: the last block clears the control words
    __syncthreads();
    if (tid == 0) s_go = atomicAdd(a.ctl + CTL_EXIT, 1u) == (unsigned)ntiles - 1u;
    __syncthreads();
    if (s_go) {
        for (int i = tid; i < ntiles; i += 64 * NW) st_agent(flags + i * CTL_STRIDE, 0u);
        if (tid == 0) st_agent(a.ctl + CTL_EXIT, 0u);
    }
}

// The level computed by tickets, when a resident launch was given up: phase p
// of a tile reads planes p & 1 and writes planes (p + 1) & 1.
struct FinishArgs {
    const float* K;
    const float* Q;
    const float* A;
    float* O[2];
    float* U[2];
    int W, H, iters, halo, nx, ny, phases, base;   // base: the level's sweeps before these
    float step, mom;
    unsigned* ctl;
    unsigned* note;       // host word: a resident launch was given up
};

template <int R, bool FMA>
__global__ __launch_bounds__(SB_TW * SB_STRIPS) void k_consist_finish(FinishArgs a)
{
    __shared__ __attribute__((aligned(16))) float sO[2][SB_STRIPS][SB_TW + 1][sb_rs<R>()];
    __shared__ int s_t;
    if (ld_agent(a.ctl + CTL_ABORT) == 0u) return;
    const int tid = threadIdx.x, ntiles = a.nx * a.ny * 3;
    unsigned* flags = a.ctl + CTL_FLAGS;
    for (;;) {
        if (tid == 0) s_t = (int)atomicAdd(a.ctl + CTL_TICKET, 1u);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(s_t);
        if (t >= a.phases * ntiles) break;
        const int ph = t / ntiles, tile = t - ph * ntiles;
        if (ph > 0) {
            const int bxy = tile % (a.nx * a.ny), ty = bxy / a.nx, tx = bxy - ty * a.nx;
            if (tid < 25) {   // the 5 x 5 tiles around: the last tile of a row overlaps two before it
                const int dx = tid % 5 - 2, dy = tid / 5 - 2;
                if (tx + dx >= 0 && tx + dx < a.nx && ty + dy >= 0 && ty + dy < a.ny)
                    while (ld_agent(flags + (tile + dy * a.nx + dx) * CTL_FSTRIDE) < (unsigned)ph) __builtin_amdgcn_s_sleep(8);
            }
            __syncthreads();
            if (tid < 64) __threadfence();   // drops this CU's and this XCD's stale lines
            __syncthreads();
        }
        const int first = ph * a.halo, n = min(a.halo, a.iters - first);
        consist_tile<R, SB_STRIPS, FMA>(a.K, a.A, a.Q, a.O[ph & 1], a.O[(ph + 1) & 1], a.U[ph & 1], a.U[(ph + 1) & 1],
                                        a.W, a.H, n, a.base + first, a.step, a.mom, a.halo, a.nx, a.ny, 1, tile, sO);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid < 64) __threadfence();       // writes this XCD's lines back
        if (tid == 0) st_agent(flags + tile * CTL_FSTRIDE, (unsigned)(ph + 1));
        // keeps this branch apart from the next turn's: merged by the compiler, thread 0 would leave the others' loop
        __syncthreads();
    }
    __syncthreads();
    if (tid == 0) s_t = atomicAdd(a.ctl + CTL_FEXIT, 1u) == gridDim.x - 1u;
    __syncthreads();
    if (s_t) {
        for (int i = tid; i < ntiles; i += SB_TW * SB_STRIPS) st_agent(flags + i * CTL_FSTRIDE, 0u);
        if (tid == 0) {
            st_agent(a.ctl + CTL_TICKET, 0u);
            st_agent(a.ctl + CTL_FEXIT, 0u);
            st_agent(a.ctl + CTL_ABORT, 0u);
            __hip_atomic_store(a.note, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// ---------------------------------------------------------------------------
// plan and launch
// ---------------------------------------------------------------------------
template <int PX, int R, bool FMA>
void go_resident(const ResArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL((k_consist_resident<PX, R, RES_NW, FMA>), dim3(8 * a.per_xcd), dim3(64 * RES_NW), 0, s, a);
}

// tile shapes: 64*px x RES_NW*r pixels.  The FMA form holds three registers a
// pixel (o, u, q), the reference order four, so its tiles end at r = 12.  One
// pixel a lane is for small levels, whose sweeps are bound by their latency: more
// and smaller tiles (frames of 640x360 in reference order 250 us with two and
// more, 232 with one; 320x180 246 and 184; 200x113, FMA form, 251 and 192).
struct Variant {
    int px, r, fma;
    void (*go)(const ResArgs&, hipStream_t);
};
const Variant kVariants[] = {
    {2, 6, 1, go_resident<2, 6, true>},    {2, 8, 1, go_resident<2, 8, true>},   {2, 10, 1, go_resident<2, 10, true>},
    {2, 12, 1, go_resident<2, 12, true>},  {2, 16, 1, go_resident<2, 16, true>}, {4, 6, 1, go_resident<4, 6, true>},
    {4, 8, 1, go_resident<4, 8, true>},    {4, 10, 1, go_resident<4, 10, true>}, {4, 12, 1, go_resident<4, 12, true>},
    {4, 14, 1, go_resident<4, 14, true>},  {4, 16, 1, go_resident<4, 16, true>}, {2, 6, 0, go_resident<2, 6, false>},
    {2, 8, 0, go_resident<2, 8, false>},   {2, 10, 0, go_resident<2, 10, false>}, {2, 12, 0, go_resident<2, 12, false>},
    {2, 16, 0, go_resident<2, 16, false>}, {4, 6, 0, go_resident<4, 6, false>},  {4, 8, 0, go_resident<4, 8, false>},
    {4, 10, 0, go_resident<4, 10, false>}, {4, 12, 0, go_resident<4, 12, false>},
    {1, 4, 1, go_resident<1, 4, true>},    {1, 4, 0, go_resident<1, 4, false>},
    {1, 6, 1, go_resident<1, 6, true>},    {1, 8, 1, go_resident<1, 8, true>},   {1, 10, 1, go_resident<1, 10, true>},
    {1, 12, 1, go_resident<1, 12, true>},  {1, 6, 0, go_resident<1, 6, false>},  {1, 8, 0, go_resident<1, 8, false>},
    {1, 10, 0, go_resident<1, 10, false>}, {1, 12, 0, go_resident<1, 12, false>},
};

// the end of the last resident launch of each device
constexpr int RES_MAX_DEVICES = 64;
struct Turn {
    std::mutex m;
    hipEvent_t ev = nullptr;
};
Turn turns[RES_MAX_DEVICES];

// tiles along an axis, 0 if the axis does not take tiles of T pixels.  A tile
// waits for the tiles beside it and for no other, so no other's pixels may hold a
// part of its exact ones: it would publish or store them with nothing that orders
// this after that tile's loads of them.  Where the tiles overlap by much (three on
// an axis a little longer than two), h is refused.
int res_count(int L, int T, int h, int q)
{
    if (L < T || T < 4 * h + 4 * q) return 0;
    if (L == T) return 1;
    const int O = T - 2 * h;                    // the most two neighbours may be apart (a multiple of q)
    const int n = 1 + (L - T + O - 1) / O;
    for (int i = 0; i + 2 < n; ++i)
        if (res_start(i + 2, n, L, T, q) < res_start(i, n, L, T, q) + T - h) return 0;
    return n;
}

}  // namespace

// The tile shape and h of least cost, from a model fitted to 60 timings of the
// FMA form at 320x180 to 1920x1080 (4% rms): a phase costs 1.6 + 0.2 r us
// besides its sweeps and a sweep 0.25 us plus 0.0253 us per pixel of a lane
// (reference order 0.042).
bool plan_resident(int W, int H, int iters, int cus, int fma, ResidentPlan* out)
{
    if (iters < 1 || (long long)W * H >= (1LL << 28) || W > 65535 || H > 65535) return false;
    double best = 1e300;
    for (int v = 0; v < (int)(sizeof(kVariants) / sizeof(kVariants[0])); ++v) {
        const Variant& k = kVariants[v];
        if (k.fma != fma) continue;
        for (int h = 4; h <= 28; h += 4) {
            const int nx = res_count(W, 64 * k.px, h, 4), ny = res_count(H, RES_NW * k.r, h, 1);
            const long long tiles = 3LL * nx * ny;
            if (tiles == 0 || tiles > cus || tiles > RES_MAX_TILES) continue;
            const int phases = (iters + h - 1) / h;
            const double cost = phases * (1.6 + 0.2 * k.r) + iters * (0.25 + (fma ? 0.0253 : 0.042) * k.px * k.r);
            if (cost < best) {
                best = cost;
                *out = ResidentPlan{v, h, nx, ny, 1, 1, H};
            }
        }
    }
    return best < 1e299;
}

// halo and phases of the ticket form for a round of `iters` sweeps: odd, so that
// it ends in the planes that the resident form writes
static void finish_phases(int W, int H, int iters, int fma, int* halo, int* phases)
{
    const BlockedPlan bp = plan_consist_blocked(W, H, iters, fma);
    for (int k = (iters + bp.halo - 1) / bp.halo;; ++k) {
        *halo = (iters + k - 1) / k;
        *phases = (iters + *halo - 1) / *halo;
        if (*phases % 2 == 1) break;
    }
}
static int finish_tiles(int W, int H, int halo, int fma)
{
    return 3 * tile_count(W, SB_TW, halo) * tile_count(H, SB_STRIPS * (fma ? SB_R_FMA : SB_R), halo);
}

// The rounds, strips and tile shape of least modelled time for a level that does
// not fit at once.  A launch costs what plan_resident says and its way in and
// out, at 7.5 TB/s and 3 us; it has to beat the blocked solver's 0.88 us
// (reference order 1.15) a sweep and million values.  The exchange planes, four
// of a region's size, lie in A and P (reference order: P alone, A being read), or
// one in each of U, U, P and A when a single round leaves U alone.
bool plan_resident_strips(int W, int H, int iters, int cus, int fma, ResidentPlan* out)
{
    if (iters < 1 || W > 65535 || H > 65535) return false;
    const double px = 3.0 * W * H;
    double best = 0.95 * iters * px * (fma ? 0.88e-6 : 1.15e-6);
    bool found = false;
    for (int rounds = 1; rounds <= 8 && rounds <= iters; ++rounds) {
        const int sweeps = (iters + rounds - 1) / rounds;
        if ((iters + sweeps - 1) / sweeps != rounds) continue;
        for (int strips = 2; strips <= 12; ++strips) {
            const int own = (H + strips - 1) / strips, rows = std::min(H, own + 2 * sweeps + 1);
            if ((fma ? (rounds == 1 ? 1 : 2) : 4) * rows > H || (long long)W * rows >= (1LL << 28)) continue;
            for (int v = 0; v < (int)(sizeof(kVariants) / sizeof(kVariants[0])); ++v) {
                const Variant& k = kVariants[v];
                if (k.fma != fma || k.px < 4) continue;   // large levels fill the chip with large tiles
                for (int h = 4; h <= 16; h += 4) {
                    const int nx = res_count(W, 64 * k.px, h, 4), ny = res_count(rows, RES_NW * k.r, h, 1);
                    const long long tiles = 3LL * nx * ny;
                    if (tiles == 0 || tiles > cus || tiles > RES_MAX_TILES) continue;
                    const double io = (tiles * 512.0 * k.px * k.r * (fma ? 16 : 20) + 24.0 * W * own) / 7.5e6 + 3.0;
                    const double one = (sweeps + h - 1) / h * (1.6 + 0.2 * k.r) + sweeps * (0.25 + (fma ? 0.0253 : 0.042) * k.px * k.r);
                    if (rounds * strips * (one + io) < best) {
                        best = rounds * strips * (one + io);
                        *out = ResidentPlan{v, h, nx, ny, rounds, strips, rows};
                        found = true;
                    }
                }
            }
        }
    }
    if (!found) return false;
    for (int r = 0, first = 0; r < out->rounds; ++r) {   // the ticket form has room for every round
        const int n = std::min((iters + out->rounds - 1) / out->rounds, iters - first);
        int halo, phases;
        finish_phases(W, H, n, fma, &halo, &phases);
        if (finish_tiles(W, H, halo, fma) > FIN_MAX_TILES) return false;
        first += n;
    }
    return true;
}

int launch_resident(const ResidentLevel& l, const ResidentPlan& plan, hipStream_t s)
{
    const int fma = kVariants[plan.variant].fma;
    const long long plane = (long long)l.W * l.H;
    FinishArgs f{};
    f.K = l.K;
    f.Q = l.Q;
    f.A = l.A;
    f.W = l.W;
    f.H = l.H;
    f.step = l.step;
    f.mom = l.mom;
    f.ctl = l.ctl;
    f.note = l.note;
    ResArgs a{};
    a.A = l.A;
    a.plane = plane;
    a.W = l.W;
    a.H = plan.rows;
    a.h = plan.h;
    a.nx = plan.nx;
    a.ny = plan.ny;
    a.per_xcd = (3 * plan.nx * plan.ny + 7) / 8;
    a.step = l.step;
    a.mom = l.mom;
    a.ctl = l.ctl;
    if (plan.strips > 1) {
        const long long region = 3LL * l.W * plan.rows;
        const bool alone = fma && plan.rounds == 1;
        float* second = fma ? const_cast<float*>(l.A) : l.P + 2 * region;
        a.X[0][0] = l.P;
        a.X[0][1] = alone ? l.U[0] : l.P + region;
        a.X[1][0] = second;
        a.X[1][1] = alone ? l.U[1] : second + region;
    } else {
        a.X[0][0] = l.U[0];
        a.X[0][1] = l.U[1];
        a.X[1][0] = l.O[1];
        a.X[1][1] = l.P;
    }
    // after the resident launch before it on this device, whatever its stream
    int dev = 0, rc;
    if ((rc = check_hip(hipGetDevice(&dev), "resident solver"))) return rc;
    if (dev < 0 || dev >= RES_MAX_DEVICES) return set_error(VSC_E_INVALID, "resident solver: device number");
    Turn& turn = turns[dev];
    std::lock_guard<std::mutex> hold(turn.m);
    if (!turn.ev) {
        if ((rc = check_hip(hipEventCreateWithFlags(&turn.ev, hipEventDisableTiming), "resident solver"))) return rc;
    } else if ((rc = check_hip(hipStreamWaitEvent(s, turn.ev, 0), "resident solver"))) {
        return rc;
    }
    // algorithmic bytes: read O and the per-pixel constants and write O once
    const int slot = prof_start(PROF_CONSIST_BLOCKED, (fma ? 4.0 : 5.0) * 3 * 4 * (double)l.W * l.H, s);
    const int sweeps = (l.iters + plan.rounds - 1) / plan.rounds, own = (l.H + plan.strips - 1) / plan.strips;
    for (int r = 0, first = 0; r < plan.rounds; ++r, first += sweeps) {
        const int from = r & 1, n = std::min(sweeps, l.iters - first);
        a.iters = n;
        for (int k = 0; k < plan.strips; ++k) {
            const int y0 = std::min(k * own, l.H), y1 = std::min(y0 + own, l.H);
            if (y0 == y1) break;
            const int top = std::max(0, std::min(y0 - sweeps, l.H - plan.rows));   // the region's first row
            const long long at = (long long)top * l.W;
            a.K = l.K + at;
            a.Q = l.Q + at;
            if (!fma) a.A = l.A + at;
            a.Oin = l.O[from] + at;
            a.Oout = l.O[from ^ 1] + at;
            a.Uin = r > 0 ? l.U[from] + at : nullptr;
            a.Uout = r + 1 < plan.rounds ? l.U[from ^ 1] + at : nullptr;
            a.own0 = y0 - top;
            a.own1 = y1 - top;
            kVariants[plan.variant].go(a, s);
        }
        finish_phases(l.W, l.H, n, fma, &f.halo, &f.phases);
        f.nx = tile_count(l.W, SB_TW, f.halo);
        f.ny = tile_count(l.H, SB_STRIPS * (fma ? SB_R_FMA : SB_R), f.halo);
        f.iters = n;
        f.base = first;
        for (int i = 0; i < 2; ++i) {
            f.O[i] = l.O[from ^ i];
            f.U[i] = l.U[from ^ i];
        }
        if (fma) hipLaunchKernelGGL((k_consist_finish<SB_R_FMA, true>), dim3(256), dim3(SB_TW * SB_STRIPS), 0, s, f);
        else hipLaunchKernelGGL((k_consist_finish<SB_R, false>), dim3(256), dim3(SB_TW * SB_STRIPS), 0, s, f);
    }
    prof_stop(slot, s);
    if ((rc = check_launch("consist_resident"))) return rc;
    return check_hip(hipEventRecord(turn.ev, s), "resident solver");
}

}  // namespace vsc

// Diagnostic (no declaration in vsc.h): the resident tiling of a level, 0 when
// it has none.  out: tile width and height, h, tiles across and down; xs, ys:
// the tiles' first columns and rows (room for 1024 each).
extern "C" int vsct_resident_plan(int W, int H, int iters, int cus, int fma, int* out, int* xs, int* ys)
{
    using namespace vsc;
    ResidentPlan p;
    if (!plan_resident(W, H, iters, cus, fma, &p)) return 0;
    const int tw = 64 * kVariants[p.variant].px, th = RES_NW * kVariants[p.variant].r;
    const int v[5] = {tw, th, p.h, p.nx, p.ny};
    for (int i = 0; i < 5; ++i) out[i] = v[i];
    for (int i = 0; i < p.nx; ++i) xs[i] = res_start(i, p.nx, W, tw, 4);
    for (int i = 0; i < p.ny; ++i) ys[i] = res_start(i, p.ny, H, th, 1);
    return 1;
}

// Diagnostic (no declaration in vsc.h): the same for a level swept in strips;
// out also holds the rounds, the strips and a region's rows.
extern "C" int vsct_resident_strips(int W, int H, int iters, int cus, int fma, int* out, int* xs, int* ys)
{
    using namespace vsc;
    ResidentPlan p;
    if (!plan_resident_strips(W, H, iters, cus, fma, &p)) return 0;
    const int tw = 64 * kVariants[p.variant].px, th = RES_NW * kVariants[p.variant].r;
    const int v[8] = {tw, th, p.h, p.nx, p.ny, p.rounds, p.strips, p.rows};
    for (int i = 0; i < 8; ++i) out[i] = v[i];
    for (int i = 0; i < p.nx; ++i) xs[i] = res_start(i, p.nx, W, tw, 4);
    for (int i = 0; i < p.ny; ++i) ys[i] = res_start(i, p.ny, p.rows, th, 1);
    return 1;
}
