// Launchers of the Helmholtz sweeps (helmholtz_ops.hpp), one component at a
// time and grouped over the cases of a batch; helmholtz3.hpp launches the
// three components together.
#include <memory>

#include "helmholtz_ops.hpp"

namespace tpls {

template <typename T>
hipError_t launch_jacobi(hipStream_t s, const Grid& g, const Phys& ph, int comp, FieldView<T> xold, FieldView<T> rhs,
                         FieldView<T> mu, FieldView<T> x, bool xold_is_zero, const Tiling& tl)
{
    DirectEmit e{s};
    return jacobi_emit<T>(e, g, ph, comp, xold, rhs, mu, x, xold_is_zero, tl);
}

template <typename T>
hipError_t launch_sor(hipStream_t s, const Grid& g, const Phys& ph, int comp, FieldView<T> x, FieldView<T> rhs,
                      FieldView<T> mu, int flg, int iteration_time, const Tiling& tl)
{
    DirectEmit e{s};
    return sor_emit<T>(e, g, ph, comp, x, rhs, mu, flg, iteration_time, tl);
}

template <typename T>
hipError_t launch_sor_pair(hipStream_t s, const Grid& g, const Phys& ph, int comp, FieldView<T> xin, FieldView<T> xout,
                           FieldView<T> rhs, FieldView<T> mu, int iteration_time, const Tiling& tl)
{
    DirectEmit e{s};
    return sor_pair_emit<T>(e, g, ph, comp, xin, xout, rhs, mu, iteration_time, tl);
}

// sor_pair_emit of u, v and w at one odd iteration_time as one launch
// (k_rb2d3).  8-row tiles only: hipErrorInvalidValue where sor_pair_emit
// would not take them (sor_pair3_fits).
template <typename T>
hipError_t launch_sor_pair3(hipStream_t s, const Grid& g, const Phys& ph, const FieldView<T>* xin,
                            const FieldView<T>* xout, const FieldView<T>* rhs, FieldView<T> mu, const Tiling& tl)
{
    if (!sor_pair3_fits(g, tl)) return hipErrorInvalidValue;
    const double ax = ph.dt / (ph.dx * ph.dx), ay = ph.dt / (ph.dy * ph.dy), az = ph.dt / (ph.dz * ph.dz);
    const T a2 = T(ax / 2.0), bb = T(ay / 2.0), c2 = T(az / 2.0);
    constexpr int TX = 32, TY = 8;
    const int nby = g.P / TY;
    const int n0 = (g.maxl - 2 + TX - 1) / TX * nby, n12 = (g.maxl - 1 + TX - 1) / TX * nby;
    const int b1 = (n0 + GROUP_ALIGN - 1) / GROUP_ALIGN * GROUP_ALIGN;
    const int b2 = b1 + (n12 + GROUP_ALIGN - 1) / GROUP_ALIGN * GROUP_ALIGN;
    const int nb0 = n0 / nby, nb12 = n12 / nby;
    auto go = [&](auto d_c, auto w_c) {
        constexpr int D = decltype(d_c)::value, W = decltype(w_c)::value;
        hipLaunchKernelGGL((k_rb2d3<TX, TY, D, W, T>), dim3(b2 + n12), dim3(RbLanes<TX, TY>::NT), 0, s,
                           typename OpRb2d<0, TX, TY, D, T>::Args{g, nb0, a2, bb, c2, xin[0], xout[0], rhs[0], mu},
                           typename OpRb2d<1, TX, TY, D, T>::Args{g, nb12, a2, bb, c2, xin[1], xout[1], rhs[1], mu},
                           typename OpRb2d<2, TX, TY, D, T>::Args{g, nb12, a2, bb, c2, xin[2], xout[2], rhs[2], mu},
                           b1, b2, n0, n12, n12);
        return hipGetLastError();
    };
    // 4 waves per SIMD (three 5-wave blocks per CU) with the deepest
    // prefetch that fits 128 registers unspilled: 2 levels in FP64, 4 in
    // FP32.  Measured at 512 x 128 x 256 (one launch against the three
    // one-component passes): FP64 500 against 520 us, FP32 step 17.3 against
    // 17.9 ms; 4 levels at 3 waves per SIMD, or 8 (FP32) / 4 (FP64) at 4
    // waves with spills, were slower.
    if (sizeof(T) == 8) return go(std::integral_constant<int, 2>{}, std::integral_constant<int, 4>{});
    return go(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
}

template <typename T>
hipError_t launch_jsor0(hipStream_t s, const Grid& g, const Phys& ph, int comp, FieldView<T> xs, FieldView<T> xd,
                        FieldView<T> rhs, FieldView<T> mu, FieldView<T> pres, const Tiling& tl)
{
    DirectEmit e{s};
    return jsor0_emit<T>(e, g, ph, comp, xs, xd, rhs, mu, pres, tl);
}

template <typename T>
hipError_t launch_helmholtz_bc(hipStream_t s, const Grid& g, const Phys& ph, int comp, FieldView<T> x,
                               FieldView<T> pres)
{
    DirectEmit e{s};
    return helmholtz_bc_emit<T>(e, g, ph, comp, x, pres);
}

// ---- the Helmholtz outer loops of many cases in lock-step (group.hpp) ----
// Each case's launches are the ones its own enqueue_pre makes (the same
// launchers, with the launch shapes below: every shape computes the same
// values); the emitter collects one sub-step of every case and appends it as
// one grouped launch per kernel variant.
namespace {

struct CollectEmit {
    struct Base {
        virtual ~Base() = default;
        virtual void flush(GroupPlan& P) = 0;
    };
    template <class Op>
    struct Table : Base {
        GroupItems<typename Op::Args> it;
        void flush(GroupPlan& P) override { P.add<Op>(it.v); }
    };
    static constexpr bool EVEN_PASS = true;
    int share = 1;
    std::vector<std::pair<const void*, std::unique_ptr<Base>>> tabs;
    int slots(int dev_slots) const { return std::max(1, dev_slots / share); }
    template <class Op>
    hipError_t go(const typename Op::Args& a, dim3 grid)
    {
        static const char key = 0;  // one address per kernel variant
        Table<Op>* t = nullptr;
        for (auto& e : tabs)
            if (e.first == &key) t = static_cast<Table<Op>*>(e.second.get());
        if (!t) {
            tabs.emplace_back(&key, std::make_unique<Table<Op>>());
            t = static_cast<Table<Op>*>(tabs.back().second.get());
        }
        t->it.add(a, grid);
        return hipSuccess;
    }
    void flush(GroupPlan& P)
    {
        for (auto& e : tabs) e.second->flush(P);
        tabs.clear();
    }
};

template <typename T>
int group_component(GroupPlan& P, const std::vector<HhGroupCase<T>>& cs, int q, bool diag)
{
    const size_t n = cs.size();
    std::vector<int> src(n), dst(n);
    int its = 0;
    for (size_t k = 0; k < n; ++k) {
        int others[2], m = 0;
        for (int b = 0; b < 3; ++b)
            if (b != cs[k].i2[q]) others[m++] = b;
        src[k] = others[0];
        dst[k] = others[1];
        its = std::max(its, cs[k].mom[q] / 2);
    }
    CollectEmit E;
    E.share = int(n);
    // The grouped launches use staged sweeps with long marches (chunks sized
    // for a share of the device) and the fused odd pass in 8-row tiles
    // wherever the period allows: measured on the 64-case FP32 batch, 94.5 ms
    // per step against 105.6 ms with each case's own (small-grid) shapes,
    // whose one-level blocks leave a grouped launch bound by block dispatch.
    std::vector<Tiling> tls(n);
    for (size_t k = 0; k < n; ++k) {
        Tiling t = cs[k].tl;
        const int P = cs[k].g.P;
        t.jst = P % 8 == 0 ? 8 : (P % 4 == 0 ? 4 : 2);
        t.fused = 1;  // odd iteration_time fused, even in two colour sweeps
        t.rb_rows_odd = 8;
        t.ks = 0;
        tls[k] = t;
    }
    for (int it = 1; it <= its; ++it) {
        std::vector<size_t> on;
        for (size_t k = 0; k < n; ++k)
            if (it <= cs[k].mom[q] / 2) on.push_back(k);
        auto fused = [&](size_t k) { return ((tls[k].fused >> (it % 2 ? 0 : 1)) & 1) != 0; };
        auto X = [&](size_t k, int b) { return cs[k].x[q][b]; };
        auto XJ = [&](size_t k) { return fused(k) ? X(k, cs[k].i2[q]) : X(k, dst[k]); };
        for (size_t k : on) {
            const HhGroupCase<T>& c = cs[k];
            if (int rc = jacobi_emit<T>(E, c.g, c.ph, q, X(k, src[k]), c.rhs[q], c.mu, XJ(k), it == 1, tls[k])) return rc;
        }
        E.flush(P);
        for (size_t k : on) helmholtz_bc_emit<T>(E, cs[k].g, cs[k].ph, q, XJ(k), cs[k].pres);
        E.flush(P);
        // the fused pass, or the first of the two colour sweeps
        for (size_t k : on) {
            const HhGroupCase<T>& c = cs[k];
            if (fused(k)) sor_pair_emit<T>(E, c.g, c.ph, q, XJ(k), X(k, dst[k]), c.rhs[q], c.mu, it, tls[k]);
            else sor_emit<T>(E, c.g, c.ph, q, X(k, dst[k]), c.rhs[q], c.mu, 0, it, tls[k]);
        }
        E.flush(P);
        for (size_t k : on)
            if (!fused(k)) sor_emit<T>(E, cs[k].g, cs[k].ph, q, X(k, dst[k]), cs[k].rhs[q], cs[k].mu, 1, it, tls[k]);
        E.flush(P);
        for (size_t k : on) helmholtz_bc_emit<T>(E, cs[k].g, cs[k].ph, q, X(k, dst[k]), cs[k].pres);
        E.flush(P);
        for (size_t k : on) std::swap(src[k], dst[k]);
    }
    if (diag) {
        // get_difference(x3, x3_old), as enqueue_pre
        std::vector<const HhGroupCase<T>*> on;
        std::vector<FieldView<T>> a, b;
        for (size_t k = 0; k < n; ++k)
            if (cs[k].mom[q] / 2 >= 2 && cs[k].part) {
                on.push_back(&cs[k]);
                a.push_back(cs[k].x[q][src[k]]);
                b.push_back(cs[k].x[q][dst[k]]);
            }
        group_difference<T>(P, on, a, b, q);
    }
    return 0;
}

}  // namespace

template <typename T>
int hh_group_loops(GroupPlan& P, const std::vector<HhGroupCase<T>>& cs, bool diag)
{
    if (cs.empty()) return 0;
    for (int q = 0; q < 3; ++q)
        if (int rc = group_component<T>(P, cs, q, diag)) return rc;
    return 0;
}
template int hh_group_loops<double>(GroupPlan&, const std::vector<HhGroupCase<double>>&, bool);
template int hh_group_loops<float>(GroupPlan&, const std::vector<HhGroupCase<float>>&, bool);

#define TPLS_INST_HH(T)                                                                                              \
    template hipError_t launch_jacobi<T>(hipStream_t, const Grid&, const Phys&, int, FieldView<T>, FieldView<T>,     \
                                         FieldView<T>, FieldView<T>, bool, const Tiling&);                           \
    template hipError_t launch_sor<T>(hipStream_t, const Grid&, const Phys&, int, FieldView<T>, FieldView<T>,        \
                                      FieldView<T>, int, int, const Tiling&);                                        \
    template hipError_t launch_sor_pair<T>(hipStream_t, const Grid&, const Phys&, int, FieldView<T>, FieldView<T>,   \
                                           FieldView<T>, FieldView<T>, int, const Tiling&);                          \
    template hipError_t launch_helmholtz_bc<T>(hipStream_t, const Grid&, const Phys&, int, FieldView<T>, FieldView<T>); \
    template hipError_t launch_sor_pair3<T>(hipStream_t, const Grid&, const Phys&, const FieldView<T>*,              \
                                            const FieldView<T>*, const FieldView<T>*, FieldView<T>, const Tiling&); \
    template hipError_t launch_jsor0<T>(hipStream_t, const Grid&, const Phys&, int, FieldView<T>, FieldView<T>,      \
                                        FieldView<T>, FieldView<T>, FieldView<T>, const Tiling&);
TPLS_INST_HH(double)
TPLS_INST_HH(float)

}  // namespace tpls

