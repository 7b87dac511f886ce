// planes.h -- device bodies of the plane sweeps of small lattices with nx = ny:
// the x and y transforms of one (x, y) plane in one workgroup's LDS.
//
// Up to 128 sites per side a plane's half-complex array fits the 160 KB LDS
// of a CU (128 x 65 complex: 67 KB in FP32, 133 KB in FP64), so the x R2C and
// the y forward pass, and the y inverse pass and the x C2R + kick, run as one
// sweep each.  A force evaluation is then three launches instead of five or
// six, and moves 6 + 4 half-complex array passes per field instead of 6 + 8.  The
// two-field kick needs both fields' Laplacians at a site, i.e. two planes in
// LDS: FP64 at 128 per side does not fit and keeps the separate inverse sweeps.
// Per kick, one lattice / three in turn, against the separate sweeps: 16^3 FP64 two
// fields 41.5 -> 18.5 / 27.8 -> 15.9 us, 48^3 73 -> 28 / 27 -> 16, 64^3 FP64 one field
// 38.5 -> 27.3 / 21.9 -> 16.0, 96^3 mixed 83 -> 50 / 35 -> 23, 128^3 mixed 90 -> 66 /
// 57 -> 41, 128^3 FP64 one field 86 -> 70 / 56 -> 37, two fields (forward only)
// 137 -> 115 / 102 -> 91.  One workgroup per plane leaves CUs idle where nz is small, and
// is still the faster way: of the boxes nx = ny = 16 .. 128, nz = 8 .. 256, mixed and
// FP64, one and two fields, the least gain is 128 x 128 x 8 FP64 one field, 56.3 ->
// 47.2 / 26.1 -> 19.6 us; 128 x 128 x 256 mixed 154 -> 91 / 108 -> 75.
#pragma once
#include "sweeps.h"

namespace lat {

#define LAT_FOR_PLANE_SIZES(X) X(16) X(32) X(48) X(64) X(96) X(128)

// threads per plane (the larger planes' row passes are two or four
// butterflies per thread)
template <int N>
constexpr int plane_nt() { return N >= 48 ? 512 : 256; }
// radices: rows (N/2 points) up to 8, columns up to 16
constexpr int PLANE_MRX = 8, PLANE_MRY = 16;

constexpr int PLANE_LDS = 160 * 1024;
constexpr bool plane_size(int n)
{
    switch (n) {
#define CASE(NN) case NN:
        LAT_FOR_PLANE_SIZES(CASE)
#undef CASE
        return true;
    default:
        return false;
    }
}
template <typename T, int N>
constexpr int plane_fwd_buf() { return N * (N / 2 + 1); }
template <typename T, int N, int NF>
constexpr int plane_inv_buf() { return NF * N * (N / 2 + 2); }
// LDS bytes: planes, and the twiddle table of N entries (nx = ny = N)
template <typename T, int N>
constexpr int plane_fwd_lds() { return (int)sizeof(cpx<T>) * (plane_fwd_buf<T, N>() + N); }
template <typename T, int N, int NF>
constexpr int plane_inv_lds() { return (int)sizeof(cpx<T>) * (plane_inv_buf<T, N, NF>() + N) + 1024; } // + reduction
// Which sizes take the plane sweeps, for the host's choice (plane_fwd_ok,
// plane_inv_ok) and for what the shared launches compile alike: the size has
// plane kernels and its planes fit.  (The bytes alone would admit FP32 192, 147 KB.)
template <typename T, int N>
constexpr bool plane_fwd_fits() { return plane_size(N) && plane_fwd_lds<T, N>() <= PLANE_LDS; }
template <typename T, int N, int NF>
constexpr bool plane_inv_fits() { return plane_size(N) && plane_inv_lds<T, N, NF>() <= PLANE_LDS; }

// ---------------------------------------------------------------- x R2C + y forward
// Plane bk.x of the lattice, member bk.y; f, pi, Fk: the field's arrays.
// DRIFT as in x_r2c_body (same arithmetic).
template <typename T, int N, int NT, bool DRIFT>
__device__ __forceinline__ void plane_fwd_body(T *__restrict__ f, const T *__restrict__ pi, cpx<T> *__restrict__ Fk,
                                               const cpx<T> *__restrict__ tw, int P,
                                               const DevScalars *__restrict__ dsc, int field, MemberStride ms,
                                               const Blk bk, cpx<T> *__restrict__ buf, cpx<T> *__restrict__ twl)
{
    constexpr int M = N / 2, LS = M + 1;
    constexpr int VW = 16 / sizeof(T), NV = N * N / VW, IT = NV / NT;
    using VT = Vec16<T>;
    assume_blk(bk);
    f += bk.y * ms.f + (size_t)bk.x * N * N;
    pi += bk.y * ms.f + (size_t)bk.x * N * N;
    Fk += bk.y * ms.k + (size_t)bk.x * N * P;
    dsc += bk.y;
    int nd = 0;
    T dc0 = 0, dc1 = 0, nu = 0;
    if constexpr (DRIFT) {
        nd = dsc->nd;
        dc0 = T(dsc->dc[0]);
        dc1 = T(dsc->dc[1]);
        if (dsc->mixed && field >= 0) nu = T(dsc->nu[field]);
    }
    for (int i = threadIdx.x; i < N; i += NT) twl[i] = tw[i];
    // rows: four vectors of phi (and pi) in flight per thread
    constexpr int U = IT >= 4 ? 4 : (IT >= 2 ? 2 : 1);
    constexpr bool WHOLE = NV % (U * NT) == 0;
    for (int i0 = threadIdx.x; i0 < NV; i0 += U * NT) {
        VT v[U], p[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!WHOLE && i0 + u * NT >= NV) continue;
            v[u] = *reinterpret_cast<const VT *>(f + (size_t)(i0 + u * NT) * VW);
            if constexpr (DRIFT) p[u] = *reinterpret_cast<const VT *>(pi + (size_t)(i0 + u * NT) * VW);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = i0 + u * NT;
            if (!WHOLE && idx >= NV) continue;
            const int line = idx / (N / VW), e0 = (idx - line * (N / VW)) * VW;
            if constexpr (DRIFT) {
                if (nd > 0) {
#pragma unroll
                    for (int e = 0; e < VW; ++e) {
                        T x = v[u].e[e] + dc0 * p[u].e[e];
                        if (nd > 1) x = x + dc1 * p[u].e[e];
                        if constexpr (sizeof(T) == 4) x = x - nu;
                        v[u].e[e] = x;
                    }
                    *reinterpret_cast<VT *>(f + (size_t)idx * VW) = v[u];
                }
            }
#pragma unroll
            for (int e = 0; e < VW; e += 2) buf[line * LS + (e0 + e) / 2] = cpx<T>{v[u].e[e], v[u].e[e + 1]};
        }
    }
    lds_sync();
    lds_fft_range<T, M, -1, N, NT, false, 2, 0, num_passes(M, PLANE_MRX), PLANE_MRX>(buf, LS, 1, twl);
    // real-FFT split, as in x_r2c_body
    for (int idx = threadIdx.x; idx < N * (M / 2 + 1); idx += NT) {
        const int line = idx / (M / 2 + 1), k = idx - line * (M / 2 + 1);
        cpx<T> *z = buf + line * LS;
        const int km = (M - k) % M;
        const cpx<T> a = z[k], b = z[km];
        {
            const cpx<T> w = twl[k];
            const cpx<T> s = {T(0.5) * (a.x + b.x), T(0.5) * (a.y - b.y)};
            const cpx<T> d = {T(0.5) * (a.x - b.x), T(0.5) * (a.y + b.y)};
            const cpx<T> wd = cmul(w, d);
            z[k] = {s.x + wd.y, s.y - wd.x};
        }
        if (k != M - k) {
            const int k2 = M - k;
            const cpx<T> w = twl[k2];
            const cpx<T> s = {T(0.5) * (b.x + a.x), T(0.5) * (b.y - a.y)};
            const cpx<T> d = {T(0.5) * (b.x - a.x), T(0.5) * (b.y + a.y)};
            const cpx<T> wd = cmul(w, d);
            z[k2] = {s.x + wd.y, s.y - wd.x};
        }
    }
    lds_sync();
    // columns: M + 1 of them, elements LS apart; the last pass goes to memory
    constexpr int NP = num_passes(N, PLANE_MRY);
    lds_fft_range<T, N, -1, M + 1, NT, true, 1, 0, NP - 1, PLANE_MRY>(buf, 1, LS, twl);
    stockham_pass_out<T, N, NP - 1, -1, M + 1, NT, true, 1, PLANE_MRY>(
        buf, 1, LS, twl, [&](int line, int pos, cpx<T> a) { Fk[(size_t)pos * P + line] = a; });
}

// ---------------------------------------------------------------- y inverse + x C2R + epilogue
// EPI_KICK, EPI_REDUCE and EPI_GWKICK as in x_c2r_body; one reduction
// partial per plane.
template <typename T, int N, int NT, int NF, int EPI>
__device__ __forceinline__ void plane_inv_body(const cpx<T> *__restrict__ Fk, const cpx<T> *__restrict__ tw, int P,
                                               size_t nk, size_t nvol, const T *__restrict__ fld,
                                               T *__restrict__ fldp, const DevScalars *__restrict__ dsc, ModelDev md,
                                               double *__restrict__ partials, MemberStride ms, const Blk bk,
                                               cpx<T> *__restrict__ buf, cpx<T> *__restrict__ twl)
{
    constexpr int M = N / 2;
    constexpr int LS = M + 2; // even pitch: rows start 16-byte aligned
    constexpr int VW = 16 / sizeof(T), NV = N * N / VW;
    using VT = Vec16<T>;
    assume_blk(bk);
    Fk += bk.y * ms.k + (size_t)bk.x * N * P;
    fld += bk.y * ms.f;
    fldp += bk.y * ms.f;
    dsc += bk.y;
    partials += (size_t)bk.y * MAX_GRID * NRED;
    EpiEnv<T, EPI> env(dsc, md);
    for (int i = threadIdx.x; i < N; i += NT) twl[i] = tw[i];
    // first column pass straight from memory (radix R0, no twiddles)
    constexpr int NP = num_passes(N, PLANE_MRY);
    constexpr int R0 = radix_at(N, 0, PLANE_MRY), NR0 = N / R0, C0 = (M + 1) * NR0, TOT0 = NF * C0;
    constexpr int B0 = cdiv(TOT0, NT);
    {
        cpx<T> v[B0][R0];
#pragma unroll
        for (int b = 0; b < B0; ++b) {
            const int g = threadIdx.x + b * NT;
            if (TOT0 % NT == 0 || g < TOT0) {
                const int fi = g / C0, r = g - fi * C0, line = r % (M + 1), j = r / (M + 1);
#pragma unroll
                for (int q = 0; q < R0; ++q) v[b][q] = Fk[fi * nk + (size_t)(j + q * NR0) * P + line];
            }
        }
#pragma unroll
        for (int b = 0; b < B0; ++b) {
            const int g = threadIdx.x + b * NT;
            if (TOT0 % NT == 0 || g < TOT0) {
                const int fi = g / C0, r = g - fi * C0, line = r % (M + 1), j = r / (M + 1);
                dft_small<R0, +1>(v[b]);
#pragma unroll
                for (int q = 0; q < R0; ++q) buf[(fi * N + j * R0 + q) * LS + line] = v[b][q];
            }
        }
    }
    lds_sync();
#pragma unroll
    for (int fi = 0; fi < NF; ++fi)
        lds_fft_range<T, N, +1, M + 1, NT, true, 1, 1, NP, PLANE_MRY>(buf + fi * N * LS, 1, LS, twl);
    // Hermitian pre-split, as in x_c2r_body
    for (int idx = threadIdx.x; idx < NF * N * (M / 2 + 1); idx += NT) {
        const int fl = idx / (M / 2 + 1), k = idx - fl * (M / 2 + 1);
        cpx<T> *z = buf + fl * LS;
        cpx<T> a = z[k], b = z[M - k];
        if (k == 0) { a.y = 0; b.y = 0; }
        {
            cpx<T> w = twl[k];
            w.y = -w.y; // e^{+2 pi i k/N}
            const cpx<T> s = {a.x + b.x, a.y - b.y};
            const cpx<T> d = {a.x - b.x, a.y + b.y};
            const cpx<T> wd = cmul(w, d);
            z[k] = {s.x - wd.y, s.y + wd.x};
        }
        if (k != 0 && k != M - k) {
            const int k2 = M - k;
            cpx<T> w = twl[k2];
            w.y = -w.y;
            const cpx<T> s = {b.x + a.x, b.y - a.y};
            const cpx<T> d = {b.x - a.x, b.y + a.y};
            const cpx<T> wd = cmul(w, d);
            z[k2] = {s.x - wd.y, s.y + wd.x};
        }
    }
    lds_sync();
    lds_fft_range<T, M, +1, NF * N, NT, false, 2, 0, num_passes(M, PLANE_MRX), PLANE_MRX>(buf, LS, 1, twl);
    // epilogue: VW consecutive sites per thread, two vectors in flight
    double acc[NRED] = {0, 0, 0, 0, 0, 0, 0, 0};
    constexpr int U = NV / NT >= 2 ? 2 : 1;
    constexpr bool WHOLE = NV % (U * NT) == 0;
    for (int i0 = threadIdx.x; i0 < NV; i0 += U * NT) {
        VT ph[U][2], pv[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int fi = 0; fi < NF; ++fi) {
                if (!WHOLE && i0 + u * NT >= NV) continue;
                const size_t site = fi * nvol + (size_t)bk.x * N * N + (size_t)(i0 + u * NT) * VW;
                if constexpr (EPI != EPI_GWKICK) ph[u][fi] = *reinterpret_cast<const VT *>(fld + site);
                pv[u][fi] = *reinterpret_cast<const VT *>(fldp + site);
            }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = i0 + u * NT;
            if (!WHOLE && idx >= NV) continue;
            const int line = idx / (N / VW), e0 = (idx - line * (N / VW)) * VW;
            VT lap[2];
#pragma unroll
            for (int fi = 0; fi < NF; ++fi)
                lap[fi] = *reinterpret_cast<const VT *>(reinterpret_cast<const T *>(buf + (fi * N + line) * LS) + e0);
            if constexpr (EPI == EPI_GWKICK) gw_source_vec<T>(fld, md, nvol, N, line, bk.x, e0, ph[u]);
            env.sites(NF, lap, ph[u], pv[u], acc);
            if constexpr (EPI == EPI_KICK || EPI == EPI_GWKICK) {
#pragma unroll
                for (int fi = 0; fi < NF; ++fi)
                    *reinterpret_cast<VT *>(fldp + fi * nvol + (size_t)bk.x * N * N + (size_t)idx * VW) = pv[u][fi];
            }
        }
    }
    if constexpr (EPI == EPI_KICK || EPI == EPI_REDUCE)
        block_reduce_store<NRED, NT>(acc, partials + (size_t)bk.x * NRED);
}

} // namespace lat
