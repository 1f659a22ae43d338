// The Helmholtz sweeps of u, v and w as one launch each.  The three
// components' loops are independent; on grids where one component's sweep
// does not fill the device (or is a march of a few blocks up k), running the
// three side by side takes about the time of one, and a third of the
// launches (the odd pass, 24 launches of 37 us a step at 128x32x64, marches up
// the column in 16 blocks of the chip's 256 CUs: three of them side by side
// take 38 us; a boundary kernel is 4.4 us of launch and drain for 1 us of
// loads).  Every cell computes what the component's own launch computes.
#include "helmholtz_ops.hpp"

#include <cstring>

namespace tpls {

// An op's family: the same kernel and launch shape for another component.
template <class Op>
struct Trio;
template <int Q, int RY, typename T>
struct Trio<OpJacobi<Q, RY, T>> {
    static constexpr int comp = Q;
    template <int C>
    using of = OpJacobi<C, RY, T>;
};
template <int Q, int RY, typename T>
struct Trio<OpSor3d<Q, RY, T>> {
    static constexpr int comp = Q;
    template <int C>
    using of = OpSor3d<C, RY, T>;
};
template <int Q, int RY, int D, typename T>
struct Trio<OpSor2d<Q, RY, D, T>> {
    static constexpr int comp = Q;
    template <int C>
    using of = OpSor2d<C, RY, D, T>;
};
template <int Q, int TX, int TY, int D, typename T>
struct Trio<OpRb2d<Q, TX, TY, D, T>> {
    static constexpr int comp = Q;
    template <int C>
    using of = OpRb2d<C, TX, TY, D, T>;
};
template <int Q, int TY, int D, bool ZERO, typename T>
struct Trio<OpJacobiSt<Q, TY, D, ZERO, T>> {
    static constexpr int comp = Q;
    template <int C>
    using of = OpJacobiSt<C, TY, D, ZERO, T>;
};
template <int Q, int TY, int D, typename T>
struct Trio<OpSor3dSt<Q, TY, D, T>> {
    static constexpr int comp = Q;
    template <int C>
    using of = OpSor3dSt<C, TY, D, T>;
};

// Blocks [0, b1) run u's, [b1, b2) v's and [b2, ..) w's launch, b1 and b2
// multiples of 8 so that the XCD-aware tile orders hold.
struct TrioBlocks {
    int b1, b2, n[3];
};

template <class O0, class O1, class O2>
__global__ void __launch_bounds__(O0::THREADS)
    k_three(typename O0::Args a0, typename O1::Args a1, typename O2::Args a2, TrioBlocks t)
{
    const int b = int(blockIdx.x);
    if (b < t.b1) {
        if (b < t.n[0]) O0::run(a0, Blk{b, 0, 0, t.n[0]});
    } else if (b < t.b2) {
        if (b - t.b1 < t.n[1]) O1::run(a1, Blk{b - t.b1, 0, 0, t.n[1]});
    } else {
        O2::run(a2, Blk{b - t.b2, 0, 0, t.n[2]});
    }
}

// Keeps u's and v's launch and sends the three with w's.
struct TrioEmit {
    static constexpr bool EVEN_PASS = false;
    hipStream_t s;
    int n = 0;
    const void* family = nullptr;
    alignas(16) char arg[2][256];
    int blocks[2];
    int slots(int dev_slots) const { return std::max(1, dev_slots / 3); }
    template <class Op>
    hipError_t go(const typename Op::Args& a, dim3 grid)
    {
        using F = Trio<Op>;
        using O0 = typename F::template of<0>;
        using O1 = typename F::template of<1>;
        using O2 = typename F::template of<2>;
        static_assert(sizeof(typename O0::Args) <= sizeof arg[0], "");
        if (F::comp != n || grid.y != 1 || grid.z != 1) return hipErrorInvalidValue;
        const void* fam = reinterpret_cast<const void*>(&k_three<O0, O1, O2>);
        if (n == 0) family = fam;
        if (family != fam) return hipErrorInvalidValue;
        if constexpr (F::comp < 2) {
            std::memcpy(arg[n], &a, sizeof a);
            blocks[n++] = int(grid.x);
            return hipSuccess;
        } else {
            typename O0::Args a0;
            typename O1::Args a1;
            std::memcpy(&a0, arg[0], sizeof a0);
            std::memcpy(&a1, arg[1], sizeof a1);
            auto up = [](int v) { return (v + GROUP_ALIGN - 1) / GROUP_ALIGN * GROUP_ALIGN; };
            TrioBlocks t{up(blocks[0]), up(blocks[0]) + up(blocks[1]), {blocks[0], blocks[1], int(grid.x)}};
            n = 0;
            hipLaunchKernelGGL((k_three<O0, O1, O2>), dim3(t.b2 + grid.x), O0::block(), 0, s, a0, a1, a, t);
            return hipGetLastError();
        }
    }
};

// The boundary conditions of the three components (OpBcUv, OpBcW): u's and
// v's columns, one thread per (k, j), then w's columns and walls.
template <typename T>
__global__ void __launch_bounds__(256) k_bc3(Grid g, T dtdx, FieldView<T> u, FieldView<T> v, FieldView<T> w,
                                             FieldView<T> pres)
{
    const int L = g.maxl, n = g.maxn, P = g.P;
    int q = int(blockIdx.x) * 256 + int(threadIdx.x);
    const int nuv = P * (n - 1), nw = P * (n - 2), nb = (L + 1) * P;
    if (q < nuv) {
        const int k = q % (n - 1), j = q / (n - 1) + 1;
        u(0, j, k) = u(1, j, k);
        u(L - 1, j, k) = u(L - 2, j, k) + dtdx * (pres(L, j, k + 1) + pres(L - 2, j, k + 1) - T(2) * pres(L - 1, j, k + 1));
        u(L, j, k) = T(0);
        return;
    }
    q -= nuv;
    if (q < nuv) {
        const int k = q % (n - 1), j = q / (n - 1) + 1;
        v(0, j, k) = v(1, j, k);
        v(L, j, k) = v(L - 1, j, k);
        return;
    }
    q -= nuv;
    if (q < nw) {
        const int k = q % (n - 2) + 1, j = q / (n - 2) + 1;
        w(0, j, k) = w(1, j, k);
        w(L, j, k) = w(L - 1, j, k);
        return;
    }
    q -= nw;
    if (q < nb) {
        const int i = q % (L + 1), j = q / (L + 1) + 1;
        w(i, j, 0) = T(0);
        w(i, j, n - 1) = T(0);
    }
}

template <typename T>
hipError_t launch_jacobi3(hipStream_t s, const Grid& g, const Phys& ph, const FieldView<T>* xold, const FieldView<T>* rhs,
                          FieldView<T> mu, const FieldView<T>* x, bool xold_is_zero, const Tiling& tl)
{
    TrioEmit e{};
    e.s = s;
    for (int q = 0; q < 3; ++q)
        if (hipError_t rc = jacobi_emit<T>(e, g, ph, q, xold[q], rhs[q], mu, x[q], xold_is_zero, tl)) return rc;
    return hipSuccess;
}

template <typename T>
hipError_t launch_sor3(hipStream_t s, const Grid& g, const Phys& ph, const FieldView<T>* x, const FieldView<T>* rhs,
                       FieldView<T> mu, int flg, int iteration_time, const Tiling& tl)
{
    TrioEmit e{};
    e.s = s;
    for (int q = 0; q < 3; ++q)
        if (hipError_t rc = sor_emit<T>(e, g, ph, q, x[q], rhs[q], mu, flg, iteration_time, tl)) return rc;
    return hipSuccess;
}

template <typename T>
hipError_t launch_sor_odd3(hipStream_t s, const Grid& g, const Phys& ph, const FieldView<T>* xin,
                           const FieldView<T>* xout, const FieldView<T>* rhs, FieldView<T> mu, const Tiling& tl)
{
    TrioEmit e{};
    e.s = s;
    for (int q = 0; q < 3; ++q)
        if (hipError_t rc = sor_pair_emit<T>(e, g, ph, q, xin[q], xout[q], rhs[q], mu, 1, tl)) return rc;
    return hipSuccess;
}

template <typename T>
hipError_t launch_helmholtz_bc3(hipStream_t s, const Grid& g, const Phys& ph, const FieldView<T>* x, FieldView<T> pres)
{
    const long n = 2L * g.P * (g.maxn - 1) + long(g.P) * (g.maxn - 2) + long(g.maxl + 1) * g.P;
    hipLaunchKernelGGL(k_bc3<T>, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, g, T(ph.dt / ph.dx), x[0], x[1], x[2],
                       pres);
    return hipGetLastError();
}

#define TPLS_INST_HH3(T)                                                                                            \
    template hipError_t launch_jacobi3<T>(hipStream_t, const Grid&, const Phys&, const FieldView<T>*,               \
                                          const FieldView<T>*, FieldView<T>, const FieldView<T>*, bool,             \
                                          const Tiling&);                                                           \
    template hipError_t launch_sor3<T>(hipStream_t, const Grid&, const Phys&, const FieldView<T>*,                  \
                                       const FieldView<T>*, FieldView<T>, int, int, const Tiling&);                 \
    template hipError_t launch_sor_odd3<T>(hipStream_t, const Grid&, const Phys&, const FieldView<T>*,              \
                                           const FieldView<T>*, const FieldView<T>*, FieldView<T>, const Tiling&);  \
    template hipError_t launch_helmholtz_bc3<T>(hipStream_t, const Grid&, const Phys&, const FieldView<T>*,         \
                                                FieldView<T>);

}  // namespace tpls
