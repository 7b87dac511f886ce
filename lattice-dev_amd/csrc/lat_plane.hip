// lat_plane.hip -- plane sweeps of small lattices with nx = ny, one lattice size
// per launch: x R2C + y forward, and y inverse + x C2R + epilogue (planes.h).  The
// z pass between them is the column kernel of lat_fft.hip.
#include "planes.h"

namespace lat {

template <typename T, int N, bool DRIFT>
__global__ __launch_bounds__(plane_nt<N>()) void k_plane_fwd(T *__restrict__ f, const T *__restrict__ pi,
                                                             cpx<T> *__restrict__ Fk, const cpx<T> *__restrict__ tw,
                                                             int P, size_t nvol, size_t nk,
                                                             const DevScalars *__restrict__ dsc, int field0,
                                                             MemberStride ms)
{
    __shared__ __attribute__((aligned(16))) cpx<T> buf[plane_fwd_buf<T, N>()];
    __shared__ cpx<T> twl[N];
    const int l = blockIdx.z;
    plane_fwd_body<T, N, plane_nt<N>(), DRIFT>(f + l * nvol, DRIFT ? pi + l * nvol : f, Fk + l * nk, tw, P, dsc,
                                               field0 < 0 ? -1 : field0 + l, ms, hw_blk(), buf, twl);
}

template <typename T, int N, int NF, int EPI>
__global__ __launch_bounds__(plane_nt<N>()) void k_plane_inv(const cpx<T> *__restrict__ Fk,
                                                             const cpx<T> *__restrict__ tw, int P, size_t nk,
                                                             size_t nvol, const T *__restrict__ fld,
                                                             T *__restrict__ fldp, const DevScalars *__restrict__ dsc,
                                                             ModelDev md, double *__restrict__ partials,
                                                             MemberStride ms)
{
    __shared__ __attribute__((aligned(16))) cpx<T> buf[plane_inv_buf<T, N, NF>()];
    __shared__ cpx<T> twl[N];
    plane_inv_body<T, N, plane_nt<N>(), NF, EPI>(Fk, tw, P, nk, nvol, fld, fldp, dsc, md, partials, ms, hw_blk(), buf,
                                                 twl);
}

template <typename T>
bool plane_fwd_ok(const Ctx &c)
{
    if (c.nx != c.ny) return false;
    switch (c.nx) {
#define CASE(NN) \
    case NN: return plane_fwd_fits<T, NN>();
        LAT_FOR_PLANE_SIZES(CASE)
#undef CASE
    }
    return false;
}

template <typename T>
bool plane_inv_ok(const Ctx &c, int nf)
{
    if (c.nx != c.ny || nf < 1 || nf > 2) return false;
    switch (c.nx) {
#define CASE(NN) \
    case NN: return nf == 1 ? plane_inv_fits<T, NN, 1>() : plane_inv_fits<T, NN, 2>();
        LAT_FOR_PLANE_SIZES(CASE)
#undef CASE
    }
    return false;
}

template <typename T, int N>
static int fwd_go(Ctx &c, const cpx<T> *tw, T *f, const T *pi, cpx<T> *Fk, int nf, int drift, int field0)
{
    if constexpr (plane_fwd_fits<T, N>()) {
        const dim3 grid(c.nz, c.B, nf), blk(plane_nt<N>());
        if (drift)
            hipLaunchKernelGGL((k_plane_fwd<T, N, true>), grid, blk, 0, c.stream, f, pi, Fk, tw, c.P, c.nvol, c.nk,
                               c.dsc, field0, c.ms);
        else
            hipLaunchKernelGGL((k_plane_fwd<T, N, false>), grid, blk, 0, c.stream, f, pi, Fk, tw, c.P, c.nvol, c.nk,
                               c.dsc, field0, c.ms);
        LAT_HIP(&c, hipGetLastError());
        return 0;
    } else {
        c.last_error = "planes too large";
        return -2;
    }
}

template <typename T>
int launch_plane_fwd(Ctx &c, const cpx<T> *tw, T *f, const T *pi, cpx<T> *Fk, int nf, int drift, int field0)
{
    switch (c.nx) {
#define CASE(NN) \
    case NN: return fwd_go<T, NN>(c, tw, f, pi, Fk, nf, drift, field0);
        LAT_FOR_PLANE_SIZES(CASE)
#undef CASE
    }
    c.last_error = "unsupported plane size";
    return -2;
}

template <typename T, int N, int NF>
static int inv_go(Ctx &c, const cpx<T> *tw, const cpx<T> *Fk, int epi, const T *fld, T *fldp, int gwc0)
{
    if constexpr (plane_inv_fits<T, N, NF>()) {
        const ModelDev md = model_dev(c, gwc0);
        const dim3 grid(c.nz, c.B), blk(plane_nt<N>());
        if (epi == EPI_KICK)
            hipLaunchKernelGGL((k_plane_inv<T, N, NF, EPI_KICK>), grid, blk, 0, c.stream, Fk, tw, c.P, c.nk, c.nvol,
                               fld, fldp, c.dsc, md, c.partials, c.ms);
        else if (epi == EPI_REDUCE)
            hipLaunchKernelGGL((k_plane_inv<T, N, NF, EPI_REDUCE>), grid, blk, 0, c.stream, Fk, tw, c.P, c.nk, c.nvol,
                               fld, fldp, c.dsc, md, c.partials, c.ms);
        else if constexpr (NF == 2)
            hipLaunchKernelGGL((k_plane_inv<T, N, 2, EPI_GWKICK>), grid, blk, 0, c.stream, Fk, tw, c.P, c.nk, c.nvol,
                               fld, fldp, c.dsc, md, c.partials, c.ms);
        LAT_HIP(&c, hipGetLastError());
        return c.nz;
    } else {
        c.last_error = "planes too large";
        return -2;
    }
}

template <typename T>
int launch_plane_inv(Ctx &c, const cpx<T> *tw, const cpx<T> *Fk, int nf, int epi, const T *fld, T *fldp, int gwc0)
{
    switch (c.nx) {
#define CASE(NN) \
    case NN: return nf == 1 ? inv_go<T, NN, 1>(c, tw, Fk, epi, fld, fldp, gwc0) : inv_go<T, NN, 2>(c, tw, Fk, epi, fld, fldp, gwc0);
        LAT_FOR_PLANE_SIZES(CASE)
#undef CASE
    }
    c.last_error = "unsupported plane size";
    return -2;
}

template bool plane_fwd_ok<double>(const Ctx &);
template bool plane_fwd_ok<float>(const Ctx &);
template bool plane_inv_ok<double>(const Ctx &, int);
template bool plane_inv_ok<float>(const Ctx &, int);
template int launch_plane_fwd<double>(Ctx &, const cpx<double> *, double *, const double *, cpx<double> *, int, int,
                                      int);
template int launch_plane_fwd<float>(Ctx &, const cpx<float> *, float *, const float *, cpx<float> *, int, int, int);
template int launch_plane_inv<double>(Ctx &, const cpx<double> *, const cpx<double> *, int, int, const double *,
                                      double *, int);
template int launch_plane_inv<float>(Ctx &, const cpx<float> *, const cpx<float> *, int, int, const float *, float *,
                                     int);

} // namespace lat
