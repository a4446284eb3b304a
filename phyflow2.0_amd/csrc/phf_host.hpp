// phf_host.hpp -- the host side of a call: checking the caller's arrays,
// packing small inputs into one transfer, and bringing results back through
// pinned memory with several threads.
#pragma once

#include "phf_common.hpp"

#include <initializer_list>
#include <type_traits>

namespace phf {

// fn(0) .. fn(n - 1), taken in order by the calling thread and a few worker
// threads shared by the process; returns when all are done.  fn must not
// throw.  Several callers may be in it at once.
void host_parallel(int n, void (*fn)(void *, int), void *ctx);
template <class F>
void host_parallel(int n, F &&fn)
{
    using T = std::remove_reference_t<F>;
    host_parallel(
        n, [](void *c, int i) { (*static_cast<T *>(c))(i); }, &fn);
}

// n doubles of host memory into the device slice *dev each: one transfer
// through the lane's pinned staging when they are small, else one each.
struct HostIn {
    const double *host;
    int64_t n;
    double **dev;
};
int copy_in(Lane *L, std::initializer_list<HostIn> in);
// sources and targets; targets that are the sources' own arrays are not
// sent twice
int copy_points_in(Lane *L, const double *xb, const double *yb, const double *wb, int64_t nb,
                   const double *xt, const double *yt, int64_t nt, double **dxb, double **dyb,
                   double **dwb, double **dxt, double **dyt);

// bytes of device memory into the caller's (pageable) memory each, after the
// work enqueued on the lane's stream; complete when it returns.
struct HostOut {
    void *host;
    const void *dev;
    size_t bytes;
};
int copy_out(Lane *L, std::initializer_list<HostOut> out);

}  // namespace phf
