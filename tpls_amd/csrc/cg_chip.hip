// The plain conjugate-gradient solve (pressure.hip's iteration, ksp_pc none)
// of a grid whose vectors fit on the chip, as one cooperative launch.
//
// The streaming iteration (k_cg_p, k_cg_pf, k_cg_x, k_cg_xf) is four launches
// that read and write 64 B per unknown.  On the grids below it is bound by the
// launches and by re-reading vectors the chip could have kept: 22 us per
// iteration at 128x32x64 and 57 us at 256x64x128, against 0.7 and 6 us for
// the arithmetic.  Here every block owns a box of cells for the whole solve:
// x, r and w = A p in registers, p with a one-cell halo in LDS.  What
// crosses blocks per iteration is the box faces of w and two reductions.
//
//   p <- (r - mean r) + beta/beta_old p     own cells and halo cells alike
//   w = A p, p.w                            faces of w published
//   [reduction 1: alpha = beta / p.w]       faces of w loaded
//   r <- r - alpha w, sum r, sum r^2
//   [reduction 2: mean r, beta, test]       meanwhile x <- x + alpha p and the
//                                           halo's r <- r - alpha w
//
// A block keeps r of its halo cells too, so the one exchange per iteration
// (w) is off the path between the two reductions.  The arithmetic of a cell is
// the streaming kernels'; only the order of the sums differs.
//
// A reduction is an all-gather without atomics' read-modify-write: each block
// stores its partial as 8-byte words that carry the reduction's number in
// their upper half (so a word is valid by itself, with no ordering between
// words), and one wavefront of every block per 64 blocks polls the words of
// those 64; the sums are added in a fixed order.  All words that cross blocks
// are stored and loaded as relaxed agent-scope atomics, which bypass the
// caches that are not coherent between XCDs; a block's faces are complete
// (s_waitcnt, then the barrier) before the block stores its word.  The faces
// alternate between two buffers: one is written again only after every block
// has stored a word that follows its loads of it.
//
// Per iteration, before and after: 128x32x64 22 -> 6.9 us, 150x46x77 30 ->
// 8.3, 256x64x128 57 -> 11.8.  Of 150x46x77's (20,700 cycles) the two waits for
// the other blocks' sums take about 10,000, the stencil and the updates the
// rest: the latency of a word's way from one XCD to another bounds it.
//
// The launch is cooperative, so all blocks are resident; a wait that lasts
// longer than CHIP_LIMIT_S seconds all the same makes every block leave, and
// the solve report an error.
#include "reduce.hpp"
#include "tpls_kernels.hpp"

#include <algorithm>

namespace tpls {

namespace {

using u64 = unsigned long long;

// Most threads of a block, by cells per thread: 128 registers hold 8 cells'
// r, x and w, 256 hold 24.
constexpr int chip_threads(int cells) { return cells <= 8 ? 1024 : 512; }

// A halo cell: its place in p, and where the neighbour publishes its w.
struct HaloRef {
    int at, src;
};
constexpr int CHIP_LIMIT_S = 20;
constexpr long CHIP_CLOCK = 100000000;  // wall_clock64 ticks per second

// Pointers out of the case's table, as what they are: global memory.
template <typename V>
using gptr = __attribute__((address_space(1))) V*;
template <typename V>
__device__ __forceinline__ gptr<V> global(V* p)
{
    return (gptr<V>)p;
}

__device__ __forceinline__ void word_store(gptr<u64> p, u64 v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 word_load(gptr<u64> p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ double uniform(double v)
{
    const u64 b = (u64)__double_as_longlong(v);
    const u64 lo = unsigned(__builtin_amdgcn_readfirstlane(int(unsigned(b))));
    const u64 hi = unsigned(__builtin_amdgcn_readfirstlane(int(unsigned(b >> 32))));
    return __longlong_as_double((long long)(hi << 32 | lo));
}

template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    const u64 b = (u64)__double_as_longlong(v);
    const unsigned lo = unsigned(__builtin_amdgcn_mov_dpp(int(unsigned(b)), CTRL, 0xf, 0xf, true));
    const unsigned hi = unsigned(__builtin_amdgcn_mov_dpp(int(unsigned(b >> 32)), CTRL, 0xf, 0xf, true));
    return __longlong_as_double((long long)(u64(hi) << 32 | lo));
}

// Sum over each row of 16 lanes, in all of them (quad swaps, half-row and row
// mirrors), and over the wavefront.  Register moves: the shuffles of wave_sum
// pass LDS six times, 800 cycles of the 2 us a reduction takes.
__device__ __forceinline__ double row_sum(double v)
{
    v += dpp<0xb1>(v);   // quad_perm [1,0,3,2]
    v += dpp<0x4e>(v);   // quad_perm [2,3,0,1]
    v += dpp<0x141>(v);  // row_half_mirror
    v += dpp<0x140>(v);  // row_mirror
    return v;
}
__device__ __forceinline__ double lane_value(double v, int l)
{
    const u64 b = (u64)__double_as_longlong(v);
    const unsigned lo = unsigned(__builtin_amdgcn_readlane(int(unsigned(b)), l));
    const unsigned hi = unsigned(__builtin_amdgcn_readlane(int(unsigned(b >> 32)), l));
    return __longlong_as_double((long long)(u64(hi) << 32 | lo));
}
__device__ __forceinline__ double wavefront_sum(double v)
{
    v = row_sum(v);
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// Keeps what is computed from v inside the iteration: hoisted out of the loop,
// the addresses of every cell and face would take the registers of the cells.
__device__ __forceinline__ int here(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// One lane: block b's value q of reduction `epoch` as two tagged words.
__device__ __forceinline__ void put_value(gptr<u64> slots, int nblk, int b, int q, unsigned epoch, double v)
{
    const u64 bits = (u64)__double_as_longlong(v), tag = u64(epoch) << 32;
    word_store(slots + (2 * q) * nblk + b, tag | (bits >> 32));
    word_store(slots + (2 * q + 1) * nblk + b, tag | (bits & 0xffffffffu));
}

// Wavefront `wave` of a block: the sums over blocks 64 wave .. 64 wave + 63 of
// NV values of reduction `epoch`, in lane 0.  False if the wait ran out or
// another block's did.
template <int NV>
__device__ __forceinline__ bool gather_values(gptr<u64> slots, int nblk, int wave, unsigned epoch, gptr<int> failed,
                                              double (&sum)[NV])
{
    const unsigned b = unsigned(here((threadIdx.x & 63) + 64 * wave)), step = unsigned(nblk);
    u64 w[2 * NV];
    const long t0 = wall_clock64();
    for (int n = 0;; ++n) {
        if ((n & 255) == 255) {
            const bool late = long(wall_clock64()) - t0 > CHIP_CLOCK * CHIP_LIMIT_S;
            if (late || __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
        }
        bool mine = true;
#pragma unroll
        for (int e = 0; e < 2 * NV; ++e) w[e] = b < step ? word_load(slots + (e * step + b)) : u64(epoch) << 32;
#pragma unroll
        for (int e = 0; e < 2 * NV; ++e) mine = mine && unsigned(w[e] >> 32) == epoch;
        if (__all(mine)) break;
    }
#pragma unroll
    for (int v = 0; v < NV; ++v)
        sum[v] = wavefront_sum(__longlong_as_double((long long)((w[2 * v] << 32) | (w[2 * v + 1] & 0xffffffffu))));
    return true;
}

}  // namespace

// One thread holds a column segment of C cells (consecutive levels) of the
// box, C as long as the case's share of the grid asks for.
template <int C>
__global__ void __launch_bounds__(chip_threads(C)) k_cg_chip(CgChipArgs args)
{
    extern __shared__ double lds[];
    // cells whose loads are in flight together: all at once, the loads of a
    // long segment would spill the cells' own registers
    constexpr int GROUP = C == 8 ? 2 : 4;
    // the block's case (unrolled: with a search at run time the registers that
    // the solve's loop gets cost 256x64x128 1.5 % of its time)
    const CgChipCase* ap = args.c[0];
    unsigned epoch = args.epoch[0];
    int first = 0;
#pragma unroll
    for (int q = 1; q < CG_CHIP_MAX; ++q)
        if (q < args.n && int(blockIdx.x) >= args.b0[q]) {
            ap = args.c[q];
            epoch = args.epoch[q];
            first = args.b0[q];
        }
    const CgChipCase a = *ap;
    CgState* const st = a.st;
    if (st->done) return;
    const int b = int(blockIdx.x) - first, t = threadIdx.x, nthr = blockDim.x;
    const int gx = a.gx, gy = a.gy, gz = a.gz, bx = a.bx, by = a.by, bz = a.bz;
    const int nblk = gx * gy * gz;
    const int bX = b % gx, bY = (b / gx) % gy, bZ = b / (gx * gy);
    const int i0 = 1 + bX * bx, j0 = 1 + bY * by, k0 = 1 + bZ * bz;
    const int ex = min(bx, a.nx - i0 + 1), ey = min(by, a.ny - j0 + 1), ez = min(bz, a.nz - k0 + 1);
    const int SX = bx + 2, PL = SX * (by + 2), NP = PL * (a.nseg * C + 2);
    double* const p = lds;
    const int FX = by * bz, FY = bx * bz, FZ = bx * by, fst = 2 * (FX + FY + FZ);
    const int oYL = 2 * FX, oZL = oYL + 2 * FY;
    double* const hr = lds + NP;  // r of the halo cells
    HaloRef* const href = reinterpret_cast<HaloRef*>(hr + fst);
    double* const red = hr + 2 * fst;  // 2 x 16 wavefront sums
    double* const tot = red + 32;     // 4 + 2 x 4 sums over 64 blocks
    double* const cst = tot + 12;     // constants of the scalar recurrences
    int* const late = reinterpret_cast<int*>(cst + 4);
    const gptr<u64> slots = global(a.slots);
    const gptr<double> faces = global(a.faces);
    const gptr<int> failed = global(&st->pad);
    const double diag = a.diag, cx = a.cx, cy = a.cy, cz = a.cz;
    for (int e = t; e < NP; e += nthr) p[e] = 0.0;
    if (t == 0) *late = 0;
    for (int e = t; e < 12; e += nthr) tot[e] = 0.0;

    // the thread's cells: column (ci, cj), levels kk0 .. kk0+nk-1 of the box
    const int cols = bx * by, seg = t / cols, col = t - seg * cols, cj = col / bx, ci = col - cj * bx;
    const int kk0 = seg * C;
    const bool has = seg < a.nseg && ci < ex && cj < ey && kk0 < ez;
    const int nk = has ? min(C, ez - kk0) : 0;
    const int own = has ? (kk0 + 1) * PL + (cj + 1) * SX + ci + 1 : PL + SX + 1;
    // where its cells lie: at the grid's walls, and on published faces
    enum { WXL = 1, WXH = 2, WZL = 4, WZH = 8, FXL = 16, FXH = 32, FYL = 64, FYH = 128, FZL = 256, FZH = 512 };
    int where = 0;
    if (nk > 0) {
        where |= i0 + ci == 1 ? WXL : 0;
        where |= i0 + ci == a.nx ? WXH : 0;
        where |= k0 + kk0 == 1 ? WZL : 0;
        where |= k0 + kk0 + nk - 1 == a.nz ? WZH : 0;
        where |= ci == 0 && bX > 0 ? FXL : 0;
        where |= ci == ex - 1 && bX < gx - 1 ? FXH : 0;
        where |= cj == 0 ? FYL : 0;
        where |= cj == ey - 1 ? FYH : 0;
        where |= kk0 == 0 && bZ > 0 ? FZL : 0;
        where |= kk0 + nk == ez && bZ < gz - 1 ? FZH : 0;
    }
    double r[C], x[C], w[C];
    const gptr<double> gx0 = global(&a.x(i0, j0, k0)), gr0 = global(&a.r(i0, j0, k0));
    const int xo = has ? ci + cj * int(a.x.sy) + kk0 * int(a.x.sz) : 0, xz = int(a.x.sz);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        r[c] = c < nk ? gr0[xo + c * xz] : 0.0;
        x[c] = c < nk ? gx0[xo + c * xz] : 0.0;
    }
    // the block's halo cells, in a list shared by its threads: r, and HaloRef
    for (int h = t; h < fst; h += nthr) {
        int src, face, hi, hj, hk;  // source block and face; the halo cell in box coordinates
        bool ok;
        if (h < oYL) {
            const bool up = h >= FX;
            const int e = up ? h - FX : h;
            hj = e % by, hk = e / by;
            ok = (up ? bX < gx - 1 : bX > 0) && hj < ey && hk < ez;
            hi = up ? ex : -1;
            src = up ? b + 1 : b - 1;
            face = (up ? 0 : FX) + e;
        } else if (h < oZL) {
            const bool up = h >= oYL + FY;
            const int e = h - oYL - (up ? FY : 0);
            hi = e % bx, hk = e / bx;
            ok = hi < ex && hk < ez;
            hj = up ? ey : -1;
            src = up ? (bY < gy - 1 ? b + gx : b - (gy - 1) * gx) : (bY > 0 ? b - gx : b + (gy - 1) * gx);
            face = oYL + (up ? 0 : FY) + e;
        } else {
            const bool up = h >= oZL + FZ;
            const int e = h - oZL - (up ? FZ : 0);
            hi = e % bx, hj = e / bx;
            ok = (up ? bZ < gz - 1 : bZ > 0) && hi < ex && hj < ey;
            hk = up ? ez : -1;
            src = up ? b + gx * gy : b - gx * gy;
            face = oZL + (up ? 0 : FZ) + e;
        }
        // an entry without a cell keeps a place nothing reads and its own face
        href[h] = HaloRef{ok ? (hk + 1) * PL + (hj + 1) * SX + hi + 1 : 0, ok ? src * fst + face : b * fst + h};
        int j = j0 + hj;
        j = j < 1 ? j + a.ny : (j > a.ny ? j - a.ny : j);
        hr[h] = ok ? gr0[hi + (j - j0) * int(a.r.sy) + hk * int(a.r.sz)] : 0.0;
    }
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), nw = nthr >> 6;
    const int ng = (nblk + 63) / 64;  // wavefronts that gather
    if (t == 0) {
        const double ttol = st->ttol, dlim = st->dtol * st->rnorm0;
        cst[0] = 1.0 / (double(a.nx) * a.ny * a.nz);
        // |z|^2 strictly between these: no test can be met, and the square
        // root (on every wavefront, after the reduction) is left out
        cst[1] = ttol * ttol * (1.0 + 1e-14);
        cst[2] = dlim < 1e150 ? dlim * dlim * (1.0 - 1e-14) : 0.0;
        cst[3] = double(st->maxits);
    }
    double m = uniform(st->m), bt = 0.0, beta = uniform(st->beta), betaold = 0.0, sr = 0.0, alpha = 0.0, dpi = 0.0;
    int n = 0, reason = 0;
    bool moved = true;  // the last iteration changed x and r
    __syncthreads();
    for (;; ++n) {
        const int nc = here(nk);
        {
            // read all, then write, with no branch per cell (a cell past the
            // box goes to p[0], which nothing reads): one LDS latency
            const int o = here(own);
#pragma unroll
            for (int c = 0; c < C; ++c) w[c] = (r[c] - m) + bt * p[o + c * PL];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < C; ++c) p[c < nc ? o + c * PL : 0] = w[c];
        }
        for (int h0 = t; h0 < fst; h0 += 4 * nthr) {
            int at[4];
            double v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int h = min(h0 + e * nthr, fst - 1);
                at[e] = h0 + e * nthr < fst ? href[h].at : 0;
                v[e] = hr[h] - m;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += bt * p[at[e]];
#pragma unroll
            for (int e = 0; e < 4; ++e) p[at[e]] = v[e];
        }
        __syncthreads();
        double acc = 0.0;
        {
            const double* q = p + here(own);
            double zm = q[-PL], v = q[0];
            const int at = here(where);
            if (at & WZL) zm = v;
#pragma unroll
            for (int c = 0; c < C; ++c, q += PL) {
                double zp = q[PL];
                if (c + 1 == nc && (at & WZH)) zp = v;
                const double xm = at & WXL ? v : q[-1], xp = at & WXH ? v : q[1], ym = q[-SX], yp = q[SX];
                const double ww = diag * v - cz * zm - cx * xm - cy * ym - cy * yp - cx * xp - cz * zp;
                w[c] = c < nc ? ww : 0.0;
                acc += c < nc ? v * ww : 0.0;
                zm = v;
                v = zp;
                if ((c + 1) % GROUP == 0) __builtin_amdgcn_sched_barrier(0);
            }
        }
        const gptr<double> mine = faces + ((n & 1) * nblk + b) * fst;
        auto face = [&](int e, double f) { word_store((gptr<u64>)(mine + e), (u64)__double_as_longlong(f)); };
        auto side = [&](int e, int step) {
#pragma unroll
            for (int c = 0; c < C; ++c, e += step)
                if (c < nc) face(e, w[c]);
        };
        const int fx = here(cj + by * kk0), fy = here(ci + bx * kk0), fz = here(ci + bx * cj);
        const int out = here(where);
        if (out & FXL) side(fx, by);
        if (out & FXH) side(FX + fx, by);
        if (out & FYL) side(oYL + fy, bx);
        if (out & FYH) side(oYL + FY + fy, bx);
        if (out & FZL) face(oZL + fz, w[0]);
        if (out & FZH) {
            double last = w[0];
#pragma unroll
            for (int c = 1; c < C; ++c) last = c < nc ? w[c] : last;
            face(oZL + FZ + fz, last);
        }
        acc = wavefront_sum(acc);
        if (lane == 0) red[wave] = acc;
        __builtin_amdgcn_s_waitcnt(0);  // the faces are out before this block's word is
        __syncthreads();
        if (wave == 0) {
            const double s = row_sum(lane < nw ? red[lane] : 0.0);  // lane 0's row holds the nw <= 16 of them
            if (lane == 0) put_value(slots, nblk, b, 0, epoch + 2 * n, s);
        }
        if (wave < ng) {
            double g[1] = {0.0};
            if (!gather_values<1>(slots, nblk, wave, epoch + 2 * n, failed, g)) *late = 1;
            if (lane == 0) tot[wave] = g[0];
        }
        __syncthreads();
        dpi = uniform((tot[0] + tot[1]) + (tot[2] + tot[3]));
        if (*late) break;
        if (!(dpi > 0.0)) {
            reason = isnan(dpi) ? -9 : -10;
            moved = false;
            break;
        }
        alpha = uniform(beta / dpi);
        const gptr<double> halo = faces + (n & 1) * nblk * fst;
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            r[c] = r[c] - alpha * w[c];  // w = 0 and r = 0 past the box
            s0 += r[c];
            s1 += r[c] * r[c];
        }
        s0 = wavefront_sum(s0);
        s1 = wavefront_sum(s1);
        if (lane == 0) {
            red[wave] = s0;
            red[16 + wave] = s1;
        }
        __syncthreads();
        if (wave == 0) {
            const double u0 = row_sum(lane < nw ? red[lane] : 0.0), u1 = row_sum(lane < nw ? red[16 + lane] : 0.0);
            if (lane == 0) {
                put_value(slots + 2 * nblk, nblk, b, 0, epoch + 2 * n + 1, u0);
                put_value(slots + 2 * nblk, nblk, b, 1, epoch + 2 * n + 1, u1);
            }
        }
        {
            const double* q = p + here(own);
#pragma unroll
            for (int c = 0; c < C; ++c, q += PL) {  // x past the box is not stored
                x[c] = x[c] + alpha * *q;
                if ((c + 1) % GROUP == 0) __builtin_amdgcn_sched_barrier(0);
            }
        }
        for (int h0 = t; h0 < fst; h0 += 4 * nthr) {
            u64 v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = word_load((gptr<u64>)(halo + href[min(h0 + e * nthr, fst - 1)].src));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int h = h0 + e * nthr;
                if (h < fst) hr[h] = hr[h] - alpha * __longlong_as_double((long long)v[e]);
            }
        }
        if (wave < ng) {
            double g[2] = {0.0, 0.0};
            if (!gather_values<2>(slots + 2 * nblk, nblk, wave, epoch + 2 * n + 1, failed, g)) *late = 1;
            if (lane == 0) {
                tot[4 + wave] = g[0];
                tot[8 + wave] = g[1];
            }
        }
        __syncthreads();
        if (*late) break;
        sr = uniform((tot[4] + tot[5]) + (tot[6] + tot[7]));
        const double s2 = uniform((tot[8] + tot[9]) + (tot[10] + tot[11]));
        m = uniform(sr * cst[0]);
        betaold = beta;
        beta = uniform(s2 - sr * m);
        if (!(beta > uniform(cst[1]) && beta < uniform(cst[2]))) {
            const double dp = sqrt(beta > 0.0 ? beta : 0.0);
            if (isnan(beta))
                reason = -9;
            else if (dp <= st->ttol)
                reason = dp < st->abstol ? 3 : 2;
            else if (dp >= st->dtol * st->rnorm0)
                reason = -4;
        }
        reason = __builtin_amdgcn_readfirstlane(reason);
        if (!reason && double(n + 1) >= uniform(cst[3])) reason = -3;
        if (reason) break;
        bt = uniform(beta / betaold);
    }
    if (*late) {
        if (t == 0) __hip_atomic_store(failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
        if (c < nk) gx0[xo + c * xz] = x[c];
    if (b == 0 && t == 0) {
        st->dpi = dpi;
        st->alpha = alpha;
        st->its = n + 1;
        st->i = reason == -3 ? n + 1 : n;
        if (moved) {
            st->m = m;
            st->sr = sr;
            st->beta = beta;
            st->betaold = betaold;
            st->dp = sqrt(beta > 0.0 ? beta : 0.0);
        }
        st->reason = reason;
        st->done = 1;
    }
}

namespace {

template <typename F>
hipError_t with_cells(int cells, F&& f)
{
    switch (cells) {
    case 1: return f(k_cg_chip<1>);
    case 2: return f(k_cg_chip<2>);
    case 4: return f(k_cg_chip<4>);
    case 8: return f(k_cg_chip<8>);
    case 16: return f(k_cg_chip<16>);
    case 24: return f(k_cg_chip<24>);
    default: return hipErrorInvalidValue;
    }
}

size_t chip_lds(const CgChipPlan& p)
{
    return (size_t(p.bx + 2) * (p.by + 2) * (p.nseg * p.cells + 2) + 2 * p.fstride + 50) * sizeof(double);
}

}  // namespace

// The boxes of a grid: a function of its extents only, so that a case sums in
// the same order alone and in any batch.  Of all partitions into at most
// CG_CHIP_BLOCKS boxes that the registers and LDS of a block hold, the one
// with the least estimated ns per iteration beyond the fixed 4,000: 22 per
// wavefront and cell (LDS and FP64), 80 per wavefront, 100 per cell of a
// segment (the chain of its column), 100 per round of halo cells, 600 per 64
// blocks polled.  Fitted to 200 partitions of 17 grids, 6 % rms.  Measured us
// per iteration (cells per thread, blocks; the chosen one first): 64x16x32 5.0
// (2, 64), 5.3 (1, 64), 5.8 (4, 64), 6.0 (2, 128); 96x22x41 6.4 (2, 126), 6.8
// (2, 64), 6.8 (1, 192); 128x32x64 7.1 (4, 128), 7.6 (2, 128), 7.4 (4, 64), 8.0
// (8, 128); 150x46x77 8.3 (4, 192), 9.4 (8, 190), 10.2 (16, 192); 179x42x192
// 11.5 (8, 252), 12.0 (16, 252); 256x64x128 11.9 (16, 256), 12.9 (8, 256).
bool cg_chip_plan(int nx, int ny, int nz, CgChipPlan* out)
{
    if (long(nx) * ny * nz > long(CG_CHIP_BLOCKS) * chip_threads(24) * 24) return false;
    double best = -1.0;
    auto boxes = [](int n, int cap) {
        std::vector<int> v;  // distinct box extents, one per box count
        for (int g = 1; g <= std::min(n, cap); ++g) {
            const int b = (n + g - 1) / g;
            if (v.empty() || v.back() != b) v.push_back(b);
        }
        return v;
    };
    const std::vector<int> xs = boxes(nx, 64), ys = boxes(ny, 64), zs = boxes(nz, 64);
    for (int bx : xs)
        for (int by : ys) {
            const int gx = (nx + bx - 1) / bx, gy = (ny + by - 1) / by;
            if (long(gx) * gy > CG_CHIP_BLOCKS || long(bx) * by > 1024) continue;
            for (int bz : zs) {
                const int gz = (nz + bz - 1) / bz;
                if (long(gx) * gy * gz > CG_CHIP_BLOCKS) continue;
                for (int cells : {1, 2, 4, 8, 16, 24}) {
                    CgChipPlan p{};
                    p.cells = cells;
                    p.bx = bx, p.by = by, p.bz = bz, p.gx = gx, p.gy = gy, p.gz = gz;
                    p.nseg = (bz + cells - 1) / cells;
                    const long need = long(bx) * by * p.nseg;
                    p.fstride = 2 * (by * bz + bx * bz + bx * by);
                    if (need > chip_threads(cells)) continue;
                    p.nblk = gx * gy * gz;
                    p.threads = std::max(int(need + 63) / 64, (p.nblk + 63) / 64) * 64;  // a wavefront gathers 64 blocks
                    p.lds = chip_lds(p);
                    if (p.lds > CG_CHIP_LDS) continue;
                    const double waves = double((need + 63) / 64);
                    // registers: 8 cells spill a little, 24 a lot
                    const double spill = cells == 24 ? 4.0 : (cells == 8 ? 1.25 : 1.0);
                    const double cost = 22.0 * spill * waves * cells + 80.0 * waves + 100.0 * cells +
                                        100.0 * ((p.fstride + p.threads - 1) / p.threads) +
                                        600.0 * ((p.nblk + 63) / 64);
                    if (best < 0.0 || cost < best) {
                        best = cost;
                        *out = p;
                    }
                }
            }
        }
    return best >= 0.0;
}

// Whether the device runs the plan's blocks at once (cooperatively).
bool cg_chip_fits_device(const CgChipPlan& p)
{
    int dev = 0, cus = 0, coop = 0, lds = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess ||
        hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        return false;
    if (!coop || cus < CG_CHIP_BLOCKS || size_t(lds) < p.lds) return false;
    const hipError_t e = with_cells(p.cells, [&](auto k) {
        const void* f = reinterpret_cast<const void*>(k);
        const hipError_t rc = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, int(CG_CHIP_LDS));
        if (rc != hipSuccess) return rc;
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, p.threads, p.lds);
    });
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess && per >= 1;
}

size_t cg_chip_slot_bytes(const CgChipPlan& p) { return size_t(6) * p.nblk * sizeof(u64); }
size_t cg_chip_face_bytes(const CgChipPlan& p) { return size_t(2) * p.nblk * p.fstride * sizeof(double); }

// One launch per set of cases that fit on the device together (first fit in
// order, same segment length).  Beyond one block for each CU the set grows as
// long as the device holds the blocks at once: small grids have small blocks,
// and the launches of a large batch run one after another.  Grouped step of
// 64 cases of 64x16x32: 40.6 ms with at most 256 blocks a launch, 26.6 so, 30.5
// by streaming kernels that all cases share; of 16 such cases 11.8, 7.9 and
// 12.0.  An error leaves the cases of the launches before it solved.
hipError_t launch_cg_chip(hipStream_t s, const std::vector<CgChipLaunch>& cases)
{
    // the blocks of this shape that the device holds
    auto room = [](int cells, int threads, size_t lds) {
        int dev = 0, cus = 0, per = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        const hipError_t e = with_cells(cells, [&](auto k) {
            return hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, reinterpret_cast<const void*>(k), threads, lds);
        });
        return e == hipSuccess ? per * cus : 0;
    };
    std::vector<char> done(cases.size(), 0);
    for (size_t f = 0; f < cases.size(); ++f) {
        if (done[f]) continue;
        CgChipArgs a{};
        int blocks = 0, threads = 0;
        size_t lds = 0;
        bool refuse = false;
        for (size_t q = f; q < cases.size() && a.n < CG_CHIP_MAX; ++q) {
            const CgChipPlan& p = *cases[q].plan;
            if (done[q] || p.cells != cases[f].plan->cells) continue;
            const int t = std::max(threads, p.threads);
            const size_t l = std::max(lds, p.lds);
            if (blocks + p.nblk > CG_CHIP_BLOCKS && blocks + p.nblk > room(p.cells, t, l)) continue;
            a.c[a.n] = cases[q].dev;
            a.epoch[a.n] = cases[q].epoch;
            a.b0[a.n] = blocks;
            ++a.n;
            blocks += p.nblk;
            threads = t;
            lds = l;
            refuse = refuse || cases[q].refuse;
            done[q] = 1;
        }
        if (refuse) return hipErrorCooperativeLaunchTooLarge;
        void* argv[] = {&a};
        const hipError_t e = with_cells(cases[f].plan->cells, [&](auto k) {
            return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k), dim3(blocks), dim3(threads), argv,
                                              unsigned(lds), s);
        });
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace tpls
