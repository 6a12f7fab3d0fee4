// Fused vector update of multi-shift CG (SolverShifted::updateVectorQuantities,
// physics/algorithms/solver_shifted.cpp:174-198): for every active shift k
//   x_k <- beta_k p_k + x_k,   p_k <- zeta_k r + alpha_k p_k
// in one pass over the lattice, so r is read once and each x_k, p_k once, instead
// of two saxpy launches per shift that re-read r and p_k.
#include "cl2_device.hpp"
#include "cl2_internal.hpp"

namespace cl2 {

/* RX: precision of the solutions x_k (may be higher than R, the precision of r and p_k, so that a
 * reduced-precision recurrence still accumulates its solutions in FP64).  Bound by HBM: every active shift reads and
 * writes x_k and p_k once.  STREAM: x and p bypass the caches, for updates whose fields exceed the 256 MiB Infinity
 * Cache and could not be found there by the next one anyway: 281 us against 304 us cached for 16 shifts at 48^3x12
 * (510 MB of FP64 x, 255 MB of FP32 p; 1.55 GB per update, 5.5 TB/s).  Fields that fit stay cached: 74 us against
 * 82 streamed for 5 shifts there (239 MB), 7.6 against 15 for 10 shifts at 16^3x16.  Several shifts' loads in
 * flight per thread, or two elements per thread, gave nothing more. */
template<typename RX, typename R, bool STREAM>
__global__ __launch_bounds__(256) void k_multishift(void* const* __restrict__ xs, void* const* __restrict__ ps,
                                                    const vec2<R>* __restrict__ r, size_t n, int nshift,
                                                    const double* __restrict__ beta, const double* __restrict__ zeta,
                                                    const double* __restrict__ alpha, const double* __restrict__ active)
{
    const size_t step = (size_t)gridDim.x * 256;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += step) {
        const vec2<R> rv = r[e];
        for (int k = 0; k < nshift; ++k) {
            if (active[k] == 0.) continue;
            vec2<RX>* x      = reinterpret_cast<vec2<RX>*>(xs[k]);
            vec2<R>* p       = reinterpret_cast<vec2<R>*>(ps[k]);
            const RX b       = RX(beta[k]);
            const R z = R(zeta[k]), a = R(alpha[k]);
            const vec2<R> pv  = STREAM ? load_stream(p + e) : p[e];
            const vec2<RX> xv = STREAM ? load_stream(x + e) : x[e];
            const vec2<RX> xn = vec2<RX>{b * RX(pv.x) + xv.x, b * RX(pv.y) + xv.y};
            const vec2<R> pn  = vec2<R>{z * rv.x + a * pv.x, z * rv.y + a * pv.y};
            if constexpr (STREAM) {
                store_stream(x + e, xn);
                store_stream(p + e, pn);
            } else {
                x[e] = xn;
                p[e] = pn;
            }
        }
    }
}

hipError_t launch_multishift(cl2_ctx* c, void* const* xs_dev, int x_prec, void* const* ps_dev, const void* r, int prec,
                             size_t n, int nshift, const double* beta, const double* zeta, const double* alpha,
                             const double* active)
{
    const unsigned nb   = (unsigned)std::min<size_t>((n + 255) / 256, 16384);
    const size_t fields = n * (size_t)nshift * ((x_prec == CL2_F64 ? 16 : 8) + (prec == CL2_F64 ? 16 : 8));
    const bool stream   = fields > ((size_t)256 << 20);
    auto go             = [&](auto rx, auto rr) {
        using RX = decltype(rx);
        using R  = decltype(rr);
        const vec2<R>* rp = reinterpret_cast<const vec2<R>*>(r);
        if (stream)
            hipLaunchKernelGGL((k_multishift<RX, R, true>), dim3(nb), dim3(256), 0, c->stream, xs_dev, ps_dev, rp, n,
                               nshift, beta, zeta, alpha, active);
        else
            hipLaunchKernelGGL((k_multishift<RX, R, false>), dim3(nb), dim3(256), 0, c->stream, xs_dev, ps_dev, rp, n,
                               nshift, beta, zeta, alpha, active);
    };
    if (prec == CL2_F64)
        go(double{}, double{});
    else if (x_prec == CL2_F64)
        go(double{}, float{});
    else
        go(float{}, float{});
    return hipGetLastError();
}

}  // namespace cl2
