// lat_nn.hip -- the learned corrector: a 3-D convolutional network on MFMA.
//
// Network: 4 layers of 3x3x3 periodic convolutions, 8 -> W -> W -> W -> 4
// channels (W = 32), SiLU between layers, BF16 weights and activations, FP32
// accumulation on the matrix cores (gfx950's v_mfma_f32_16x16x32_bf16).  Input: the
// normalised (phi, chi, pi_phi, pi_chi) fluctuations after one coarse
// leapfrog step and four uniform channels that carry what the normalisation
// removes and the dynamics depend on (the homogeneous phi and pi_phi, the
// coupling, the chi fluctuation amplitude); output: the normalised residual
// to the fine Yoshida-4 trajectory.
//
// Layout: activations are site-major with channels fastest, X[site][C]
// (C a multiple of 4), so the four consecutive reduction indices an MFMA
// lane supplies are one 8-byte load.  A convolution is an implicit GEMM
//   Y[s][co] = sum_k W[co][k] X[nbr(s, tap(k))][ci(k)],  k = tap * CIN + ci,
// with M = output channels (16-row tiles), N = 16 sites per wave tile and
// K = 27 CIN padded to a multiple of 32, 32 reduction indices per MFMA (each
// lane supplies 8 consecutive ones: 8 channels of one tap, or 4 channels of
// two taps when CIN = 4).  The weight matrix of a layer is staged in LDS
// once per workgroup.
//
// Backward: the data gradient is the same convolution with the transposed,
// tap-reversed weights Wt[ci][t * COUT + co] = W[co][(26 - t) * CIN + ci];
// the weight gradient is a GEMM over sites (K = sites), staged through LDS
// per row segment and accumulated per workgroup into partials that are
// reduced in a fixed order (deterministic).
#include <cmath>

#include "lat_internal.h"

namespace lat {
namespace nn {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16;

// round-to-nearest-even FP32 -> BF16 (finite inputs).  The compiler's own
// conversion of this instruction set gives another result for about one in
// 1e4 activations, so host and device share the integer form.
__host__ __device__ inline bf16 to_bf16(float f)
{
    unsigned u = __builtin_bit_cast(unsigned, f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16)(u >> 16);
}
__host__ __device__ inline float from_bf16(bf16 h) { return __builtin_bit_cast(float, (unsigned)h << 16); }

__device__ inline float silu(float v) { return v / (1.0f + expf(-v)); }
__device__ inline float dsilu(float v)
{
    const float s = 1.0f / (1.0f + expf(-v));
    return s * (1.0f + v * (1.0f - s));
}

constexpr int KPAD(int cin) { return (27 * cin + 31) / 32 * 32; }

// D (16 x 16, FP32) += A (16 x 32) B (32 x 16) in BF16; lane l supplies
// A[l % 16][8 (l / 16) .. +7] and B[8 (l / 16) .. +7][l % 16] and holds
// D[4 (l / 16) + e][l % 16], e = 0..3
__device__ __forceinline__ f32x4 mfma32(s16x8 a, s16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

// epilogue modes of the convolution
enum { CONV_SILU = 0,  // Z = acc + b (BF16), Y = silu(Z) (BF16)
       CONV_LINEAR = 1, // Yf = acc + b (FP32)
       CONV_DSILU = 2 };  // Y = acc * silu'(Zin) (BF16): data gradient through the activation

// Epilogue of one 16-site x 16-channel tile: the lane holds D[co0 + e][site s],
// e = 0..3, co0 = 16 mt + 4 (lane / 16) < COUT.  Z may be null (inference: only the backward
// pass reads the pre-activations).
template <int COUT, int MODE>
__device__ __forceinline__ void conv_store(const f32x4 &acc, size_t s, int co0, const float *__restrict__ bias,
                                           bf16 *__restrict__ Y, float *__restrict__ Yf, bf16 *__restrict__ Z,
                                           const bf16x4 &zi)
{
    if constexpr (MODE == CONV_LINEAR) {
        float4 o;
        o.x = acc[0] + bias[co0];
        o.y = acc[1] + bias[co0 + 1];
        o.z = acc[2] + bias[co0 + 2];
        o.w = acc[3] + bias[co0 + 3];
        *reinterpret_cast<float4 *>(Yf + s * COUT + co0) = o;
    } else if constexpr (MODE == CONV_SILU) {
        bf16x4 zo, yo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = acc[e] + bias[co0 + e];
            const bf16 zb = to_bf16(v);
            zo[e] = (short)zb;
            yo[e] = (short)to_bf16(silu(from_bf16(zb)));
        }
        if (Z) *reinterpret_cast<bf16x4 *>(Z + s * COUT + co0) = zo;
        *reinterpret_cast<bf16x4 *>(Y + s * COUT + co0) = yo;
    } else {
        bf16x4 yo;
#pragma unroll
        for (int e = 0; e < 4; ++e) yo[e] = (short)to_bf16(acc[e] * dsilu(from_bf16((bf16)zi[e])));
        *reinterpret_cast<bf16x4 *>(Y + s * COUT + co0) = yo;
    }
}

// Convolution with 32 input channels: one K step of the MFMA is one tap.
// A wave owns 16 sites along x of T consecutive rows y.  Per dz it holds the
// nine taps' weight fragments in registers (from LDS, stored in fragment
// order: conflict-free 16-byte reads) and walks the T + 2 input rows; each
// row's three x-shifted fragments (1 KB contiguous per load, from L1 / L2)
// feed the output rows above, at and below it, i.e. up to 6 MFMAs per load
// instead of 2, and no address is computed per tap.  The loads of the next
// PF rows are in flight meanwhile.  Every output accumulates its taps in
// the order 0..26.  32 -> 32 channels at 128^3: 465 -> 162 us (716 TFLOP/s; the
// activations in and out take about 65 us at the copy rate), 32 -> 4: 265 -> 97 us.
constexpr int CONV32_WAVES = 4;
template <int COUT, int MODE, int T>
__global__ __launch_bounds__(64 * CONV32_WAVES, 2) void k_conv32(const bf16 *__restrict__ X, const bf16 *__restrict__ W,
                                                              const float *__restrict__ bias, bf16 *__restrict__ Y,
                                                              float *__restrict__ Yf, bf16 *__restrict__ Z,
                                                              const bf16 *__restrict__ Zin, int n)
{
    constexpr int CIN = 32, MT = (COUT + 15) / 16, KP = KPAD(CIN);
    __shared__ s16x8 ws[27 * MT * 64]; // [tap][mt][lane]
    for (int q = threadIdx.x; q < 27 * MT * 64; q += 64 * CONV32_WAVES) {
        const int l = q % 64, mt = q / 64 % MT, t = q / (64 * MT);
        ws[q] = *reinterpret_cast<const s16x8 *>(W + (mt * 16 + (l & 15)) * KP + t * CIN + 8 * (l >> 4));
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kg = lane >> 4;
    const int ntx = n / 16, nty = n / T, ntask = ntx * nty * n;
    // each XCD walks one contiguous eighth of the tasks (neighbouring rows and
    // planes in the same L2)
    const int G8 = gridDim.x >> 3, C = (ntask + 7) >> 3;
    const int t0 = (blockIdx.x & 7) * C, t1 = min(t0 + C, ntask);
    for (int task = t0 + (int)(blockIdx.x >> 3) * CONV32_WAVES + wave; task < t1; task += G8 * CONV32_WAVES) {
        const int x0 = task % ntx * 16, y0 = task / ntx % nty * T, z = task / (ntx * nty);
        int xo[3]; // element offset of the lane's fragment in a row, per dx
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
            int x = x0 + j + dx - 1;
            x = x < 0 ? x + n : (x >= n ? x - n : x);
            xo[dx] = x * CIN + 8 * kg;
        }
        constexpr int NR = T + 2, RING = NR % 5 == 0 ? 5 : 3, PF = RING - 1; // input rows per plane; fragments held
        static_assert(NR % RING == 0, "the ring starts anew with every plane");
        auto load_row = [&](int dz, int r, s16x8 (&b)[3]) {
            int zz = z + dz - 1, y = y0 + r - 1;
            zz = zz < 0 ? zz + n : (zz >= n ? zz - n : zz);
            y = y < 0 ? y + n : (y >= n ? y - n : y);
            const bf16 *row = X + ((size_t)zz * n + y) * n * CIN;
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) b[dx] = *reinterpret_cast<const s16x8 *>(row + xo[dx]);
        };
        f32x4 acc[T][MT];
#pragma unroll
        for (int r = 0; r < T; ++r)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[r][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        s16x8 b[RING][3];
#pragma unroll
        for (int r = 0; r < PF; ++r) load_row(0, r, b[r]);
        const size_t s0 = ((size_t)z * n + y0) * n + x0 + j;
        bf16x4 zi[T][MT];
#pragma unroll 1
        for (int dz = 0; dz < 3; ++dz) {
            s16x8 a[9][MT];
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) a[t][mt] = ws[((dz * 9 + t) * MT + mt) * 64 + lane];
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                // PF rows ahead, into the next plane at the end of this one
                if (r + PF < NR) load_row(dz, r + PF, b[(r + PF) % RING]);
                else if (dz < 2) load_row(dz + 1, r + PF - NR, b[(r + PF) % RING]);
                const s16x8(&c)[3] = b[r % RING];
#pragma unroll
                for (int dy = 0; dy < 3; ++dy) {
                    const int ro = r - dy; // output row that sees this input row as tap row dy
                    if (ro < 0 || ro >= T) continue;
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) acc[ro][mt] = mfma32(a[dy * 3 + dx][mt], c[dx], acc[ro][mt]);
                }
            }
        }
        if constexpr (MODE == CONV_DSILU) {
#pragma unroll
            for (int r = 0; r < T; ++r)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    zi[r][mt] =
                        *reinterpret_cast<const bf16x4 *>(Zin + (s0 + (size_t)r * n) * COUT + mt * 16 + 4 * kg);
        }
#pragma unroll
        for (int r = 0; r < T; ++r)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int co0 = mt * 16 + 4 * kg;
                if (co0 >= COUT) continue;
                conv_store<COUT, MODE>(acc[r][mt], s0 + (size_t)r * n, co0, bias, Y, Yf, Z, zi[r][mt]);
            }
    }
}

// Convolution with 4 or 8 input channels: a K step covers 8 or 4 taps, each lane
// supplying one tap's 8 channels or two taps' 4.  One wave per 16-site tile
// (within a row: n is a multiple of 16), CONV_WAVES waves per workgroup share
// the LDS copy of the weights; grid-stride over tiles.  The lane's tap offsets
// are the same for every tile and held in registers.  8 -> 32 at 128^3: 150 ->
// 129 us; bound by the vector instructions of addresses and activations.
// W: [MT*16][KP] BF16 (rows >= COUT and k >= 27*CIN are zero).
constexpr int CONV_WAVES = 8;
template <int CIN, int COUT, int MODE>
__global__ __launch_bounds__(64 * CONV_WAVES) void k_conv(const bf16 *__restrict__ X, const bf16 *__restrict__ W,
                                              const float *__restrict__ bias, bf16 *__restrict__ Y,
                                              float *__restrict__ Yf, bf16 *__restrict__ Z,
                                              const bf16 *__restrict__ Zin, int n)
{
    static_assert(CIN == 4 || CIN == 8, "narrow inputs; 32 channels: k_conv32");
    constexpr int MT = (COUT + 15) / 16;
    constexpr int KP = KPAD(CIN), KS = KP / 32;
    constexpr int TPL = 8 / CIN; // taps per lane and K step
    __shared__ s16x8 ws[KS * MT * 64]; // [K step][mt][lane]
    for (int q = threadIdx.x; q < KS * MT * 64; q += 64 * CONV_WAVES) {
        const int l = q % 64, mt = q / 64 % MT, ks = q / (64 * MT);
        ws[q] = *reinterpret_cast<const s16x8 *>(W + (mt * 16 + (l & 15)) * KP + ks * 32 + 8 * (l >> 4));
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kg = lane >> 4;
    int dx[KS][TPL], dy[KS][TPL], dz[KS][TPL]; // taps past the 27th: zeroed below
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int u = 0; u < TPL; ++u) {
            const int t = (ks * 32 + 8 * kg) / CIN + u;
            dx[ks][u] = t < 27 ? t % 3 - 1 : 0;
            dy[ks][u] = t < 27 ? (t / 3) % 3 - 1 : 0;
            dz[ks][u] = t < 27 ? t / 9 - 1 : 0;
        }
    const int ntx = n / 16;
    const int ntile = ntx * n * n; // n <= 1024: below 2^26
    for (int tile = (int)blockIdx.x * CONV_WAVES + wave; tile < ntile; tile += (int)gridDim.x * CONV_WAVES) {
        const int x = tile % ntx * 16 + j, y = tile / ntx % n, z = tile / (ntx * n);
        const size_t s = ((size_t)z * n + y) * n + x;
        bf16x4 zi[MT];
        if constexpr (MODE == CONV_DSILU) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                zi[mt] = *reinterpret_cast<const bf16x4 *>(Zin + s * COUT + mt * 16 + 4 * kg);
        }
        s16x8 b[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            auto at = [&](int u) {
                int xx = x + dx[ks][u], yy = y + dy[ks][u], zz = z + dz[ks][u];
                xx = xx < 0 ? xx + n : (xx >= n ? xx - n : xx);
                yy = yy < 0 ? yy + n : (yy >= n ? yy - n : yy);
                zz = zz < 0 ? zz + n : (zz >= n ? zz - n : zz);
                return X + ((size_t)(zz * n + yy) * n + xx) * CIN;
            };
            if constexpr (CIN == 8) {
                b[ks] = *reinterpret_cast<const s16x8 *>(at(0));
                if (4 * ks + 3 >= 27 && kg == 3) b[ks] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
            } else {
                const bf16x4 lo = *reinterpret_cast<const bf16x4 *>(at(0));
                const bf16x4 hi = *reinterpret_cast<const bf16x4 *>(at(1));
                b[ks] = s16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                if (8 * ks + 2 * kg + 1 >= 27) // the second tap (27, 29, 31), or both, do not exist
                    b[ks] = 8 * ks + 2 * kg < 27 ? s16x8{lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0}
                                                 : s16x8{0, 0, 0, 0, 0, 0, 0, 0};
            }
        }
        f32x4 acc[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma32(ws[(ks * MT + mt) * 64 + lane], b[ks], acc[mt]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int co0 = mt * 16 + 4 * kg;
            if (co0 >= COUT) continue;
            conv_store<COUT, MODE>(acc[mt], s, co0, bias, Y, Yf, Z, zi[mt]);
        }
    }
}

// Weight gradient dW[co][tap][ci] = sum_s G[s][co] X[s + tap][ci]: a GEMM over
// sites (32 per MFMA, A = G^T, B = X).  A task is a chunk of CL sites along x
// (64, 32 or 16, dividing n) of one plane z, marched over LY rows y.  Per step
// the block stages X row r of the planes z-1, z, z+1 (one site of halo in x)
// and G row r + 1 in LDS as they lie in memory (site-major, 16-byte copies,
// two buffers, the rows of the step after next in flight in registers) and
// reads them back transposed: ds_read_b64_tr_b16 gives a lane 4 consecutive
// sites of its channel, two of them the 8 reduction indices that it supplies.
// Wave (dz, nt) owns the nine (dy, dx) taps of plane dz and the input
// channels 16 nt ..: one X fragment per dx meets the G rows r + 1, r, r - 1
// (dy = 0, 1, 2; the older two kept in registers), so a step takes 6 + 4 LDS
// reads of 512 bytes per 32 sites for 18 MFMAs.  The block sums all its tasks
// in its accumulators and writes one partial dW (and db in column KP, from
// G times a matrix of ones) as [MT*16][KP + 16]; k_sum_chunks adds the partials
// in block order.  At 128^3: 32 x 32 channels 1078 -> 147 us (790 TFLOP/s),
// 32 x 4 767 -> 97 us, 8 x 32 369 -> 77 us (the form before wrote the tiles
// channel-major into LDS element by element and read X at odd offsets, one
// 2-byte read per element).
constexpr int DW_CLMAX = 64;
constexpr int DW_BLOCKS = 512; // most partials (2 blocks per CU)
typedef short s16x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline int dw_chunk(int n) { return n % 64 == 0 ? 64 : (n % 32 == 0 ? 32 : 16); }
// rows per task: as many as leave DW_BLOCKS tasks (each task recomputes two
// halo rows), at least 8
__host__ __device__ inline int dw_rows(int n)
{
    int ly = n;
    while (ly % 2 == 0 && ly > 8 && (long long)n * (n / dw_chunk(n)) * (n / ly) < DW_BLOCKS) ly /= 2;
    return ly;
}
__host__ __device__ inline int dw_tasks(int n) { return n * (n / dw_chunk(n)) * (n / dw_rows(n)); }
static int dw_blocks(int n) { return dw_tasks(n) < DW_BLOCKS ? dw_tasks(n) : DW_BLOCKS; }
template <int CIN>
constexpr int dw_waves() { return 3 * ((CIN + 15) / 16); }

// four reduction indices of this lane's channel: within a group of 16 lanes,
// lane 4 r + c points at channels 4 c .. 4 c + 3 of site r; lane i gets channel i of sites 0..3
__device__ __forceinline__ s16x4 lds_tr(const bf16 *p)
{
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(p));
}
__device__ __forceinline__ s16x8 join(s16x4 a, s16x4 b) { return s16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}; }

template <int CIN, int COUT, int CL>
__global__ __launch_bounds__(64 * dw_waves<CIN>(), 2) void k_conv_dw(const bf16 *__restrict__ G, const bf16 *__restrict__ X,
                                                                  float *__restrict__ part, int n, int LY, int ntask)
{
    constexpr int MT = (COUT + 15) / 16, NTL = (CIN + 15) / 16;
    constexpr int KP = KPAD(CIN), LD = KP + 16;
    constexpr int NT = 64 * dw_waves<CIN>();
    constexpr int KS = (CL + 31) / 32;
    // staged rows: X [3][CL + 2][CIN], then G [CL][COUT]; 16-byte copies
    constexpr int XE = 3 * (CL + 2) * CIN, GE = CL * COUT, BUF = XE + GE;
    constexpr int XI = XE / 8, GI = GE / 8, NI = cdiv(XI + GI, NT);
    static_assert(XE % 8 == 0 && GE % 8 == 0 && CL % 16 == 0, "16-byte items");
    __shared__ __attribute__((aligned(16))) bf16 lds[2 * BUF];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kg = lane >> 4;
    const int dz = wave % 3, nt = wave / 3;
    // the lane's part of a transposed read: site 8 kg + 4 h + lr, channels lc ..; a tensor
    // with fewer channels than 16 is read at its own (columns past the last are not used)
    const int lr = (lane & 15) >> 2, lc = (lane & 3) * 4;
    const int xc = CIN < 16 ? lc % CIN : nt * 16 + lc;
    const bool half = CL == 16 && kg >= 2; // a 16-site chunk fills half of a K step
    const int sk = half ? 8 * kg - 16 + lr : 8 * kg + lr;
    f32x4 acc[3][3][MT], accb[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        accb[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < 9; ++d) acc[d / 3][d % 3][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const s16x8 zero8 = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
    const short one = (short)0x3f80; // 1.0 in BF16
    const s16x8 ones = s16x8{one, one, one, one, one, one, one, one};
    const int ntx = n / CL, nly = n / LY;
    for (int task = blockIdx.x; task < ntask; task += gridDim.x) {
        const int x0 = task % ntx * CL, y0 = task / ntx % nly * LY, z = task / (ntx * nly);
        // the thread's staged items: row-independent element offsets
        size_t off[NI];
        auto isx = [&](int i) { return (int)threadIdx.x + i * NT < XI; };
        auto ok = [&](int i) { return (int)threadIdx.x + i * NT < XI + GI; };
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int q = threadIdx.x + i * NT;
            if (isx(i)) {
                constexpr int C8 = CIN / 8;
                const int c = q % C8, rest = q / C8, xi = rest % (CL + 2), p = rest / (CL + 2);
                int x = x0 + xi - 1, zz = z + p - 1;
                x = x < 0 ? x + n : (x >= n ? x - n : x);
                zz = zz < 0 ? zz + n : (zz >= n ? zz - n : zz);
                off[i] = ((size_t)zz * n * n + x) * CIN + 8 * c;
            } else {
                off[i] = ((size_t)z * n * n + x0) * COUT + 8 * (size_t)(q - XI);
            }
        }
        // step s: X row y0 - 1 + s, G row y0 + s (zero past the task's rows)
        s16x8 v[NI];
        auto fetch = [&](int s) {
            int yx = y0 - 1 + s;
            yx = yx < 0 ? yx + n : (yx >= n ? yx - n : yx);
            const size_t rx = (size_t)yx * n * CIN, rg = (size_t)(y0 + s) * n * COUT;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                v[i] = zero8;
                if (isx(i)) v[i] = *reinterpret_cast<const s16x8 *>(X + off[i] + rx);
                else if (ok(i) && s < LY) v[i] = *reinterpret_cast<const s16x8 *>(G + off[i] + rg);
            }
        };
        auto stage = [&](int s) {
            bf16 *b = lds + (s & 1) * BUF;
#pragma unroll
            for (int i = 0; i < NI; ++i)
                if (ok(i)) *reinterpret_cast<s16x8 *>(b + 8 * ((size_t)threadIdx.x + i * NT)) = v[i];
        };
        s16x8 g[3][KS][MT]; // G rows r + 1, r, r - 1 in rotation
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) g[u][ks][mt] = zero8;
        auto step = [&](int s, s16x8 (&gn)[KS][MT], const s16x8 (&g1)[KS][MT], const s16x8 (&g2)[KS][MT]) {
            if (s + 1 < LY + 2) stage(s + 1);
            if (s + 2 < LY + 2) fetch(s + 2);
            const bf16 *xb = lds + (s & 1) * BUF + dz * (CL + 2) * CIN, *gb = lds + (s & 1) * BUF + XE;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const bf16 *p = gb + (32 * ks + sk) * COUT + (COUT < 16 ? lc % COUT : mt * 16 + lc);
                    gn[ks][mt] = join(lds_tr(p), lds_tr(p + 4 * COUT));
                    if (half) gn[ks][mt] = zero8;
                    if (wave == 0) accb[mt] = mfma32(gn[ks][mt], ones, accb[mt]);
                }
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) {
                    const bf16 *p = xb + (32 * ks + sk + dx) * CIN + xc;
                    const s16x8 b = join(lds_tr(p), lds_tr(p + 4 * CIN));
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        acc[0][dx][mt] = mfma32(gn[ks][mt], b, acc[0][dx][mt]);
                        acc[1][dx][mt] = mfma32(g1[ks][mt], b, acc[1][dx][mt]);
                        acc[2][dx][mt] = mfma32(g2[ks][mt], b, acc[2][dx][mt]);
                    }
                }
            }
            __syncthreads();
        };
        fetch(0);
        stage(0);
        fetch(1);
        __syncthreads();
        int s = 0;
        for (; s + 2 < LY + 2; s += 3) {
            step(s, g[0], g[1], g[2]);
            step(s + 1, g[2], g[0], g[1]);
            step(s + 2, g[1], g[2], g[0]);
        }
        if (s < LY + 2) step(s, g[0], g[1], g[2]);
        if (s + 1 < LY + 2) step(s + 1, g[2], g[0], g[1]);
    }
    // D[row co = mt*16 + 4*kg + e][col ci = nt*16 + j] of tap t = dz*9 + dy*3 + dx
    float *dst = part + (size_t)blockIdx.x * (MT * 16) * LD;
    const int ci = nt * 16 + j;
    if (ci < CIN) {
#pragma unroll
        for (int d = 0; d < 9; ++d)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int co = mt * 16 + 4 * kg + e;
                    dst[(size_t)co * LD + (dz * 9 + d) * CIN + ci] = co < COUT ? acc[d / 3][d % 3][mt][e] : 0.f;
                }
    }
    // padding columns 27 CIN .. KP-1 and the bias block KP .. KP+15
    for (int q = threadIdx.x; q < MT * 16 * (LD - 27 * CIN); q += NT) {
        const int co = q / (LD - 27 * CIN), k = 27 * CIN + q % (LD - 27 * CIN);
        if (!(k == KP && co < COUT)) dst[(size_t)co * LD + k] = 0.f;
    }
    if (wave == 0 && j == 0) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int co = mt * 16 + 4 * kg + e;
                if (co < COUT) dst[(size_t)co * LD + KP] = accb[mt][e];
            }
    }
}

// out[q] = sum over chunks of part[chunk][q]: SUM_LANES threads per q take
// every SUM_LANES-th chunk, in order, and are added in order (512 chunks of a
// 32 x 32 layer: 129 us with one thread per q, 8.7 us).
constexpr int SUM_LANES = 8, SUM_Q = 32;
__global__ __launch_bounds__(SUM_LANES *SUM_Q) void k_sum_chunks(const float *__restrict__ part, int nchunk, int nq,
                                                                 float *__restrict__ out)
{
    __shared__ float red[SUM_LANES][SUM_Q];
    const int lq = threadIdx.x % SUM_Q, lane = threadIdx.x / SUM_Q;
    const int q = blockIdx.x * SUM_Q + lq;
    float s = 0.f;
    if (q < nq)
#pragma unroll 8
        for (int c = lane; c < nchunk; c += SUM_LANES) s += part[(size_t)c * nq + q];
    red[lane][lq] = s;
    __syncthreads();
    if (lane || q >= nq) return;
#pragma unroll
    for (int l = 1; l < SUM_LANES; ++l) s += red[l][lq];
    out[q] = s;
}

// Adam on the FP32 master weights of one layer; grad [MP][KP+16] (bias in
// column KP, row co).  Writes the BF16 copy W and the transposed, tap-reversed
// copy Wt[ci][t*COUT + co] (rows padded to a multiple of 16, K padded to KPt).
template <int CIN, int COUT>
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ w, float *__restrict__ b, float *__restrict__ mw,
                                              float *__restrict__ vw, float *__restrict__ mb,
                                              float *__restrict__ vb, const float *__restrict__ grad, float lr,
                                              float b1, float b2, float eps, float c1, float c2,
                                              bf16 *__restrict__ Wb, bf16 *__restrict__ Wt)
{
    constexpr int KP = KPAD(CIN), LD = KP + 16;
    constexpr int KPt = KPAD(COUT);
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q < COUT * 27 * CIN) {
        const int co = q / (27 * CIN), k = q - co * (27 * CIN);
        const float g = grad[(size_t)co * LD + k];
        const float m = b1 * mw[q] + (1.f - b1) * g;
        const float v = b2 * vw[q] + (1.f - b2) * g * g;
        mw[q] = m;
        vw[q] = v;
        const float wn = w[q] - lr * (m / c1) / (sqrtf(v / c2) + eps);
        w[q] = wn;
        const bf16 hb = to_bf16(wn);
        Wb[(size_t)co * KP + k] = hb;
        const int t = k / CIN, ci = k - t * CIN;
        Wt[(size_t)ci * KPt + (26 - t) * COUT + co] = hb;
    } else if (q < COUT * 27 * CIN + COUT) {
        const int co = q - COUT * 27 * CIN;
        const float g = grad[(size_t)co * LD + KP];
        const float m = b1 * mb[co] + (1.f - b1) * g;
        const float v = b2 * vb[co] + (1.f - b2) * g * g;
        mb[co] = m;
        vb[co] = v;
        b[co] = b[co] - lr * (m / c1) / (sqrtf(v / c2) + eps);
    }
}

} // namespace nn
} // namespace lat

// ======================================================================
// host side: network state, training on pairs from the plain integrator,
// corrected coarse stepping with the plain integrator as fallback
// ======================================================================
#include <cstring>
#include <random>
#include <vector>

namespace lat {
namespace nn {

constexpr int NL = 4;             // layers
constexpr int WID = 32;           // hidden channels
constexpr int NIN = 8;            // input channels: 4 fluctuations, 4 uniform
constexpr int CINS[NL] = {NIN, WID, WID, WID};
constexpr int COUTS[NL] = {WID, WID, WID, 4};
constexpr int CM_BLOCKS = 512;    // blocks of the channel-mean reduction
constexpr int CM_SLOTS = 40;      // doubles of Net::cm

struct Layer {
    int cin, cout, kp, mp, kpt, mpt; // padded shapes of W [mp][kp] and Wt [mpt][kpt]
    float *w = nullptr, *b = nullptr, *mw = nullptr, *vw = nullptr, *mb = nullptr, *vb = nullptr; // FP32 master
    bf16 *wb = nullptr, *wt = nullptr;                                                           // BF16 copies
    float *grad = nullptr;                                                                       // [mp][kp+16]
};

struct Net {
    Layer L[NL];
    int step = 0;
    // normalisation per channel, from the snapshot at hand (computed on the
    // GPU each time): input (v - <v>) / s_v, target (r - <r>) / (ratio s_v),
    // with <.> the spatial mean and s_v the spatial standard deviation of the
    // coarse state.  The network sees and corrects fluctuations only, at
    // unit scale, so neither the drift of the homogeneous mode nor the growth
    // of the fluctuations over a run leaves the range it was trained on.
    // ratio = RMS of the residual fluctuation / s_v, fixed at the first pair.
    double ratio[4] = {1, 1, 1, 1};
    bool stats = false;
    // activation buffers for lattice size n
    int n = 0;
    bf16 *x0 = nullptr, *a[3] = {nullptr, nullptr, nullptr}, *z[3] = {nullptr, nullptr, nullptr};
    bf16 *g4 = nullptr, *gA = nullptr, *gB = nullptr;
    float *y = nullptr, *tgt = nullptr, *part = nullptr, *lossp = nullptr;
    // channel statistics: [0,4) input mean, [4,8) residual mean, [8,12)
    // output mean, [12,16) input standard deviation, [16,20) residual
    // standard deviation (first training pair), [20,24) zeros, [24,28) RMS
    // of a judged step's difference from the plain step, [28,32) mean and
    // [32,36) standard deviation of the plain step, [36,40) RMS of the
    // leapfrog step's difference from it; block partials
    double *cm = nullptr, *cpart = nullptr;
    void *save_f = nullptr, *save_p = nullptr, *coarse_f = nullptr, *coarse_p = nullptr;
    void *leap_f = nullptr, *leap_p = nullptr; // judged steps: the leapfrog step alone
    DevScalars *save_s = nullptr;
    hipStream_t stream = nullptr;
    std::string err;
};

static size_t layer_wcount(const Layer &l) { return (size_t)l.cout * 27 * l.cin; }

} // namespace nn
} // namespace lat

struct lat_corrector {
    lat::nn::Net net;
};

namespace lat {
namespace nn {

template <typename T>
static int alloc(Net &net, T **p, size_t count, const char *what)
{
    if (hipMalloc((void **)p, sizeof(T) * count) != hipSuccess) {
        net.err = std::string("hipMalloc ") + what;
        return -3;
    }
    return 0;
}

static void free_buffers(Net &net)
{
    void *ps[] = {net.x0, net.a[0], net.a[1], net.a[2], net.z[0], net.z[1], net.z[2], net.g4, net.gA, net.gB,
                  net.y, net.tgt, net.part, net.lossp, net.save_f, net.save_p, net.coarse_f, net.coarse_p,
                  net.leap_f, net.leap_p, net.save_s, net.cm, net.cpart};
    for (void *p : ps)
        if (p) (void)hipFree(p);
    net.x0 = net.g4 = net.gA = net.gB = nullptr;
    for (int q = 0; q < 3; ++q) net.a[q] = net.z[q] = nullptr;
    net.y = net.tgt = net.part = net.lossp = nullptr;
    net.cm = net.cpart = nullptr;
    net.save_f = net.save_p = net.coarse_f = net.coarse_p = net.leap_f = net.leap_p = nullptr;
    net.save_s = nullptr;
    net.n = 0;
}

static int ensure_buffers(Net &net, const Ctx &c)
{
    if (net.n == c.nx) return 0;
    free_buffers(net);
    const size_t nv = c.nvol;
    int rc = 0;
    rc |= alloc(net, &net.x0, nv * NIN, "x0");
    for (int q = 0; q < 3; ++q) {
        rc |= alloc(net, &net.a[q], nv * WID, "act");
        rc |= alloc(net, &net.z[q], nv * WID, "preact");
    }
    rc |= alloc(net, &net.g4, nv * 4, "g4");
    rc |= alloc(net, &net.gA, nv * WID, "gradA");
    rc |= alloc(net, &net.gB, nv * WID, "gradB");
    rc |= alloc(net, &net.y, nv * 4, "out");
    rc |= alloc(net, &net.tgt, nv * 4, "target");
    size_t maxpart = 0;
    for (int l = 0; l < NL; ++l) {
        const size_t q = (size_t)net.L[l].mp * (net.L[l].kp + 16);
        maxpart = q > maxpart ? q : maxpart;
    }
    rc |= alloc(net, &net.part, maxpart * dw_blocks(c.nx), "dW partials");
    rc |= alloc(net, &net.lossp, 1024, "loss partials");
    rc |= alloc(net, &net.cm, CM_SLOTS, "channel statistics");
    rc |= alloc(net, &net.cpart, 4 * CM_BLOCKS, "channel-mean partials");
    const size_t es = elem_size(c);
    rc |= alloc(net, (char **)&net.save_f, es * c.ms.f, "saved fields");
    rc |= alloc(net, (char **)&net.save_p, es * c.ms.f, "saved momenta");
    rc |= alloc(net, (char **)&net.coarse_f, es * c.ms.f, "coarse fields");
    rc |= alloc(net, (char **)&net.coarse_p, es * c.ms.f, "coarse momenta");
    rc |= alloc(net, (char **)&net.leap_f, es * c.ms.f, "leapfrog fields");
    rc |= alloc(net, (char **)&net.leap_p, es * c.ms.f, "leapfrog momenta");
    rc |= alloc(net, &net.save_s, 1, "saved scalars");
    if (rc) {
        free_buffers(net);
        return rc;
    }
    const double zero[CM_SLOTS] = {};
    if (hipMemcpy(net.cm, zero, sizeof(zero), hipMemcpyHostToDevice) != hipSuccess) {
        free_buffers(net);
        net.err = "channel statistics upload failed";
        return -3;
    }
    net.n = c.nx;
    return 0;
}

// ---------------------------------------------------------------- data kernels
// Spatial channel sums, deterministic: CM_BLOCKS fixed blocks write partials,
// one block adds them in block order.  Source: the FP64 state (f, p), minus
// (cf, cp) when given, or the network output y [site][4]; with sub, the sums
// are of (v - sub)^2 instead (second pass of a standard deviation).
__global__ __launch_bounds__(256) void k_chsum(const double *__restrict__ f, const double *__restrict__ p,
                                               const double *__restrict__ cf, const double *__restrict__ cp,
                                               const float *__restrict__ y, const double *__restrict__ sub,
                                               size_t nvol, double *__restrict__ part)
{
    double a[4] = {0, 0, 0, 0};
    double m[4] = {0, 0, 0, 0};
    if (sub) {
#pragma unroll
        for (int q = 0; q < 4; ++q) m[q] = sub[q];
    }
    for (size_t s = blockIdx.x * (size_t)256 + threadIdx.x; s < nvol; s += (size_t)gridDim.x * 256) {
        double v[4];
        if (y) {
            const float4 t = *reinterpret_cast<const float4 *>(y + s * 4);
            v[0] = t.x;
            v[1] = t.y;
            v[2] = t.z;
            v[3] = t.w;
        } else {
            v[0] = cf ? f[s] - cf[s] : f[s];
            v[1] = cf ? f[nvol + s] - cf[nvol + s] : f[nvol + s];
            v[2] = cp ? p[s] - cp[s] : p[s];
            v[3] = cp ? p[nvol + s] - cp[nvol + s] : p[nvol + s];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] += sub ? (v[q] - m[q]) * (v[q] - m[q]) : v[q];
    }
    __shared__ double red[4][256];
#pragma unroll
    for (int q = 0; q < 4; ++q) red[q][threadIdx.x] = a[q];
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
#pragma unroll
            for (int q = 0; q < 4; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x < 4) part[blockIdx.x * 4 + threadIdx.x] = red[threadIdx.x][0];
}

// out[c] = sum / nvol, or with root the standard deviation sqrt(sum / nvol)
// (root 1: 1 where it is 0, so a channel without fluctuations is left
// unscaled; root 2: the RMS as it is).  One wave: lane 4 b + c takes every 16th partial of
// channel c, in order, and the 16 are added by shuffles (4 threads walking all
// 512 partials took 62 us of load latency; now 4.4 us).
__global__ __launch_bounds__(64) void k_chmean(const double *__restrict__ part, int nb, size_t nvol, int root,
                                               double *__restrict__ out)
{
    double t = 0;
#pragma unroll 8
    for (int q = threadIdx.x; q < 4 * nb; q += 64) t += part[q];
#pragma unroll
    for (int m = 4; m < 64; m <<= 1) t += __shfl_xor(t, m, 64);
    if (threadIdx.x < 4) {
        t /= (double)nvol;
        if (root) {
            t = sqrt(t);
            if (root == 1 && !(t > 0.0)) t = 1.0;
        }
        out[threadIdx.x] = t;
    }
}

// X0[s][c] = (v_c(s) - <v_c>) / s_c for (phi, chi, pi_phi, pi_chi), then
// the uniform channels <phi>, <pi_phi>, lg2 = log10(g^2/m^2) - 5 and
// log10(s_chi) / 10; st = channel statistics (means at 0, standard
// deviations at 12)
__global__ __launch_bounds__(256) void k_pack(const double *__restrict__ f, const double *__restrict__ p,
                                              size_t nvol, const double *__restrict__ st, float lg2,
                                              bf16 *__restrict__ X)
{
    const double4 mean = {st[0], st[1], st[2], st[3]};
    const double4 isd = {1.0 / st[12], 1.0 / st[13], 1.0 / st[14], 1.0 / st[15]};
    const short u0 = (short)to_bf16((float)st[0]), u1 = (short)to_bf16((float)st[2]);
    const short u2 = (short)to_bf16(lg2), u3 = (short)to_bf16((float)(log10(st[13]) / 10.0));
    for (size_t s = blockIdx.x * (size_t)256 + threadIdx.x; s < nvol; s += (size_t)gridDim.x * 256) {
        s16x8 o;
        o[0] = (short)to_bf16((float)((f[s] - mean.x) * isd.x));
        o[1] = (short)to_bf16((float)((f[nvol + s] - mean.y) * isd.y));
        o[2] = (short)to_bf16((float)((p[s] - mean.z) * isd.z));
        o[3] = (short)to_bf16((float)((p[nvol + s] - mean.w) * isd.w));
        o[4] = u0;
        o[5] = u1;
        o[6] = u2;
        o[7] = u3;
        *reinterpret_cast<s16x8 *>(X + s * NIN) = o;
    }
}

// tgt[s][c] = (r_c(s) - <r_c>) / (ratio_c s_c) with r = fine - coarse
__global__ __launch_bounds__(256) void k_target(const double *__restrict__ ff, const double *__restrict__ fp,
                                                const double *__restrict__ cf, const double *__restrict__ cp,
                                                size_t nvol, const double *__restrict__ st, double4 ratio,
                                                float *__restrict__ tgt)
{
    const double4 m = {st[4], st[5], st[6], st[7]};
    const double4 irsd = {1.0 / (ratio.x * st[12]), 1.0 / (ratio.y * st[13]), 1.0 / (ratio.z * st[14]),
                          1.0 / (ratio.w * st[15])};
    for (size_t s = blockIdx.x * (size_t)256 + threadIdx.x; s < nvol; s += (size_t)gridDim.x * 256) {
        float4 o;
        o.x = (float)((ff[s] - cf[s] - m.x) * irsd.x);
        o.y = (float)((ff[nvol + s] - cf[nvol + s] - m.y) * irsd.y);
        o.z = (float)((fp[s] - cp[s] - m.z) * irsd.z);
        o.w = (float)((fp[nvol + s] - cp[nvol + s] - m.w) * irsd.w);
        *reinterpret_cast<float4 *>(tgt + s * 4) = o;
    }
}

// G4 = 2 (y - tgt) / (4 nvol) in BF16; per-block partial sums of (y - tgt)^2
__global__ __launch_bounds__(256) void k_loss(const float *__restrict__ y, const float *__restrict__ tgt,
                                              size_t nvol, bf16 *__restrict__ g, float *__restrict__ part)
{
    __shared__ float red[256];
    const float scale = 2.0f / (4.0f * (float)nvol);
    float acc = 0.f;
    for (size_t q = blockIdx.x * (size_t)256 + threadIdx.x; q < nvol * 4; q += (size_t)gridDim.x * 256) {
        const float d = y[q] - tgt[q];
        acc += d * d;
        g[q] = to_bf16(d * scale);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// f_c += ratio_c s_c (y_c - <y_c>): the predicted residual fluctuation; the
// homogeneous mode keeps the coarse step's value
__global__ __launch_bounds__(256) void k_apply(double *__restrict__ f, double *__restrict__ p,
                                               const float *__restrict__ y, size_t nvol,
                                               const double *__restrict__ st, double4 ratio)
{
    const double4 m = {st[8], st[9], st[10], st[11]};
    const double4 rsd = {ratio.x * st[12], ratio.y * st[13], ratio.z * st[14], ratio.w * st[15]};
    for (size_t s = blockIdx.x * (size_t)256 + threadIdx.x; s < nvol; s += (size_t)gridDim.x * 256) {
        const float4 v = *reinterpret_cast<const float4 *>(y + s * 4);
        f[s] += rsd.x * (v.x - m.x);
        f[nvol + s] += rsd.y * (v.y - m.y);
        p[s] += rsd.z * (v.z - m.z);
        p[nvol + s] += rsd.w * (v.w - m.w);
    }
}

// ---------------------------------------------------------------- network passes
// Rows per wave of the 32-channel convolution: 8, or 4 where 8 would leave
// SIMDs idle (fewer wave tasks than the device's 4 x 256 SIMDs: n <= 48).
// Per launch, 32 -> 32, T = 8 / 4: 16^3 16.0 / 11.2 us, 32^3 16.7 / 12.2, 48^3
// 20.1 / 18.9; 64^3 and 96^3 together 67.7 / 75.2.
template <int CIN, int COUT, int MODE>
static void conv(Net &net, const bf16 *X, const bf16 *W, const float *bias, bf16 *Y, float *Yf, bf16 *Z,
                 const bf16 *Zin)
{
    const size_t ntile = (size_t)net.n * net.n * net.n / 16;
    if constexpr (CIN == 32) {
        const bool wide = ntile / 8 >= 1024;
        size_t g = (ntile / (wide ? 8 : 4) + CONV32_WAVES - 1) / CONV32_WAVES;
        g = g > 512 ? 512 : (g + 7) / 8 * 8;
        if (wide)
            hipLaunchKernelGGL((k_conv32<COUT, MODE, 8>), dim3((unsigned)g), dim3(64 * CONV32_WAVES), 0, net.stream,
                               X, W, bias, Y, Yf, Z, Zin, net.n);
        else
            hipLaunchKernelGGL((k_conv32<COUT, MODE, 4>), dim3((unsigned)g), dim3(64 * CONV32_WAVES), 0, net.stream,
                               X, W, bias, Y, Yf, Z, Zin, net.n);
    } else {
        size_t g = (ntile + CONV_WAVES - 1) / CONV_WAVES;
        if (g > 4096) g = 4096;
        hipLaunchKernelGGL((k_conv<CIN, COUT, MODE>), dim3((unsigned)g), dim3(64 * CONV_WAVES), 0, net.stream, X, W,
                           bias, Y, Yf, Z, Zin, net.n);
    }
}

// train: keep the pre-activations for the backward pass
static void forward(Net &net, bool train)
{
    bf16 *z[3];
    for (int q = 0; q < 3; ++q) z[q] = train ? net.z[q] : nullptr;
    conv<NIN, WID, CONV_SILU>(net, net.x0, net.L[0].wb, net.L[0].b, net.a[0], nullptr, z[0], nullptr);
    conv<WID, WID, CONV_SILU>(net, net.a[0], net.L[1].wb, net.L[1].b, net.a[1], nullptr, z[1], nullptr);
    conv<WID, WID, CONV_SILU>(net, net.a[1], net.L[2].wb, net.L[2].b, net.a[2], nullptr, z[2], nullptr);
    conv<WID, 4, CONV_LINEAR>(net, net.a[2], net.L[3].wb, net.L[3].b, nullptr, net.y, nullptr, nullptr);
}

template <int CIN, int COUT>
static void weight_grad(Net &net, Layer &l, const bf16 *G, const bf16 *X)
{
    const int nb = dw_blocks(net.n), ly = dw_rows(net.n), nt = dw_tasks(net.n);
    const dim3 blk(64 * dw_waves<CIN>());
    switch (dw_chunk(net.n)) {
    case 64:
        hipLaunchKernelGGL((k_conv_dw<CIN, COUT, 64>), dim3(nb), blk, 0, net.stream, G, X, net.part, net.n, ly, nt);
        break;
    case 32:
        hipLaunchKernelGGL((k_conv_dw<CIN, COUT, 32>), dim3(nb), blk, 0, net.stream, G, X, net.part, net.n, ly, nt);
        break;
    default:
        hipLaunchKernelGGL((k_conv_dw<CIN, COUT, 16>), dim3(nb), blk, 0, net.stream, G, X, net.part, net.n, ly, nt);
    }
    const int nq = l.mp * (l.kp + 16);
    hipLaunchKernelGGL(k_sum_chunks, dim3((nq + SUM_Q - 1) / SUM_Q), dim3(SUM_LANES * SUM_Q), 0, net.stream, net.part,
                       nb, nq, l.grad);
}

// output gradient G4 and the loss partials for the current y / tgt
static void loss_grad(Net &net)
{
    const size_t nv = (size_t)net.n * net.n * net.n;
    hipLaunchKernelGGL(k_loss, dim3(1024), dim3(256), 0, net.stream, net.y, net.tgt, nv, net.g4, net.lossp);
}

// gradients of all layers from G4; returns after launching
static void backward_layers(Net &net)
{
    weight_grad<WID, 4>(net, net.L[3], net.g4, net.a[2]);
    conv<4, WID, CONV_DSILU>(net, net.g4, net.L[3].wt, nullptr, net.gA, nullptr, nullptr, net.z[2]);
    weight_grad<WID, WID>(net, net.L[2], net.gA, net.a[1]);
    conv<WID, WID, CONV_DSILU>(net, net.gA, net.L[2].wt, nullptr, net.gB, nullptr, nullptr, net.z[1]);
    weight_grad<WID, WID>(net, net.L[1], net.gB, net.a[0]);
    conv<WID, WID, CONV_DSILU>(net, net.gB, net.L[1].wt, nullptr, net.gA, nullptr, nullptr, net.z[0]);
    weight_grad<NIN, WID>(net, net.L[0], net.gA, net.x0);
}

static void backward(Net &net)
{
    loss_grad(net);
    backward_layers(net);
}

template <int CIN, int COUT>
static void adam_layer(Net &net, Layer &l, float lr, float c1, float c2)
{
    const int nq = COUT * 27 * CIN + COUT;
    hipLaunchKernelGGL((k_adam<CIN, COUT>), dim3((nq + 255) / 256), dim3(256), 0, net.stream, l.w, l.b, l.mw, l.vw,
                       l.mb, l.vb, l.grad, lr, 0.9f, 0.999f, 1e-8f, c1, c2, l.wb, l.wt);
}

static void adam(Net &net, float lr)
{
    ++net.step;
    const float c1 = 1.f - powf(0.9f, (float)net.step), c2 = 1.f - powf(0.999f, (float)net.step);
    adam_layer<NIN, WID>(net, net.L[0], lr, c1, c2);
    adam_layer<WID, WID>(net, net.L[1], lr, c1, c2);
    adam_layer<WID, WID>(net, net.L[2], lr, c1, c2);
    adam_layer<WID, 4>(net, net.L[3], lr, c1, c2);
}

// Upload FP32 master weights (cout x 27 cin, k = tap*cin + ci) and biases of
// layer l, rebuilding the BF16 copies; the Adam moments are reset.
static int set_layer(Net &net, int li, const float *w, const float *b)
{
    Layer &l = net.L[li];
    const size_t nw = layer_wcount(l);
    std::vector<bf16> wb((size_t)l.mp * l.kp, 0), wt((size_t)l.mpt * l.kpt, 0);
    for (int co = 0; co < l.cout; ++co)
        for (int k = 0; k < 27 * l.cin; ++k) {
            const bf16 h = to_bf16(w[(size_t)co * 27 * l.cin + k]);
            wb[(size_t)co * l.kp + k] = h;
            const int t = k / l.cin, ci = k - t * l.cin;
            wt[(size_t)ci * l.kpt + (26 - t) * l.cout + co] = h;
        }
    std::vector<float> zeros(nw > (size_t)l.cout ? nw : l.cout, 0.f);
    bool ok = hipMemcpy(l.w, w, sizeof(float) * nw, hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(l.b, b, sizeof(float) * l.cout, hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(l.mw, zeros.data(), sizeof(float) * nw, hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(l.vw, zeros.data(), sizeof(float) * nw, hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(l.mb, zeros.data(), sizeof(float) * l.cout, hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(l.vb, zeros.data(), sizeof(float) * l.cout, hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(l.wb, wb.data(), sizeof(bf16) * wb.size(), hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(l.wt, wt.data(), sizeof(bf16) * wt.size(), hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
        net.err = "weight upload failed";
        return -3;
    }
    return 0;
}

} // namespace nn
} // namespace lat

// ---------------------------------------------------------------- C ABI
using namespace lat;
using namespace lat::nn;

static int corr_fail(Net &net, const char *msg)
{
    net.err = msg;
    return -2;
}

// A call borrows its context's stream: it ends with the stream drained and
// the borrow cleared, so the corrector never keeps the stream of a context
// that may be destroyed before it.
struct StreamLease {
    Net &net;
    ~StreamLease()
    {
        if (net.stream) (void)hipStreamSynchronize(net.stream);
        net.stream = nullptr;
    }
};

static int check_ctx(Net &net, Ctx &c)
{
    if (c.B != 1 || c.view) return corr_fail(net, "the corrector runs on single contexts");
    if (c.prec != LAT_F64 || c.nfld != 2) return corr_fail(net, "the corrector needs a two-field FP64 context");
    if (c.nx != c.ny || c.nx != c.nz || c.nx % 16) return corr_fail(net, "the corrector needs a cubic lattice, n % 16 == 0");
    net.stream = c.stream;
    return ensure_buffers(net, c);
}

static double4 d4(const double *v) { return double4{v[0], v[1], v[2], v[3]}; }

static int grid_sites(size_t nvol)
{
    size_t g = (nvol + 255) / 256;
    return (int)(g > 8192 ? 8192 : g);
}

// channel means into net.cm + 4 * slot (see Net::cm)
static void channel_means(Net &net, Ctx &c, const void *f, const void *p, const void *cf, const void *cp,
                          const float *y, int slot)
{
    hipLaunchKernelGGL(k_chsum, dim3(CM_BLOCKS), dim3(256), 0, c.stream, (const double *)f, (const double *)p,
                       (const double *)cf, (const double *)cp, y, (const double *)nullptr, c.nvol, net.cpart);
    hipLaunchKernelGGL(k_chmean, dim3(1), dim3(64), 0, c.stream, net.cpart, CM_BLOCKS, c.nvol, 0,
                       net.cm + 4 * slot);
}

// input means (slot 0) and standard deviations (slot 3) of the state (f, p), then X0
static void pack(Net &net, Ctx &c, const void *f, const void *p)
{
    channel_means(net, c, f, p, nullptr, nullptr, nullptr, 0);
    hipLaunchKernelGGL(k_chsum, dim3(CM_BLOCKS), dim3(256), 0, c.stream, (const double *)f, (const double *)p,
                       (const double *)nullptr, (const double *)nullptr, (const float *)nullptr,
                       (const double *)net.cm, c.nvol, net.cpart);
    hipLaunchKernelGGL(k_chmean, dim3(1), dim3(64), 0, c.stream, net.cpart, CM_BLOCKS, c.nvol, 1, net.cm + 12);
    const double g2 = c.cfg.model_params[1];
    const float lg2 = g2 > 0.0 ? (float)(std::log10(g2) - 5.0) : 0.0f;
    hipLaunchKernelGGL(k_pack, dim3(grid_sites(c.nvol)), dim3(256), 0, c.stream, (const double *)f,
                       (const double *)p, c.nvol, (const double *)net.cm, lg2, net.x0);
}

static int save_state(Net &net, Ctx &c)
{
    const size_t bytes = sizeof(double) * c.ms.f;
    LAT_HIP(&c, hipMemcpyAsync(net.save_f, c.fld, bytes, hipMemcpyDeviceToDevice, c.stream));
    LAT_HIP(&c, hipMemcpyAsync(net.save_p, c.fldp, bytes, hipMemcpyDeviceToDevice, c.stream));
    LAT_HIP(&c, hipMemcpyAsync(net.save_s, c.dsc, sizeof(DevScalars), hipMemcpyDeviceToDevice, c.stream));
    return 0;
}

static int restore_state(Net &net, Ctx &c)
{
    const size_t bytes = sizeof(double) * c.ms.f;
    LAT_HIP(&c, hipMemcpyAsync(c.fld, net.save_f, bytes, hipMemcpyDeviceToDevice, c.stream));
    LAT_HIP(&c, hipMemcpyAsync(c.fldp, net.save_p, bytes, hipMemcpyDeviceToDevice, c.stream));
    LAT_HIP(&c, hipMemcpyAsync(c.dsc, net.save_s, sizeof(DevScalars), hipMemcpyDeviceToDevice, c.stream));
    c.ke_valid = false;
    return 0;
}

extern "C" {

int lat_corrector_create(unsigned long long seed, lat_corrector **out)
{
    if (!out) return -1;
    *out = nullptr;
    lat_corrector *h = new lat_corrector();
    Net &net = h->net;
    std::mt19937_64 rng(seed);
    for (int li = 0; li < NL; ++li) {
        Layer &l = net.L[li];
        l.cin = CINS[li];
        l.cout = COUTS[li];
        l.kp = KPAD(l.cin);
        l.mp = (l.cout + 15) / 16 * 16;
        l.kpt = KPAD(l.cout);
        l.mpt = (l.cin + 15) / 16 * 16;
        const size_t nw = layer_wcount(l);
        int rc = 0;
        rc |= alloc(net, &l.w, nw, "w");
        rc |= alloc(net, &l.mw, nw, "adam m");
        rc |= alloc(net, &l.vw, nw, "adam v");
        rc |= alloc(net, &l.b, l.cout, "b");
        rc |= alloc(net, &l.mb, l.cout, "adam mb");
        rc |= alloc(net, &l.vb, l.cout, "adam vb");
        rc |= alloc(net, &l.wb, (size_t)l.mp * l.kp, "w bf16");
        rc |= alloc(net, &l.wt, (size_t)l.mpt * l.kpt, "wt bf16");
        rc |= alloc(net, &l.grad, (size_t)l.mp * (l.kp + 16), "grad");
        if (rc) {
            lat_corrector_destroy(h);
            return -3;
        }
        // He-normal initialisation; the last layer starts small so that the
        // untrained corrector is close to the plain coarse step
        const double sd = std::sqrt(2.0 / (27.0 * l.cin)) * (li == NL - 1 ? 0.1 : 1.0);
        std::normal_distribution<double> nd(0.0, sd);
        std::vector<float> w(nw), b(l.cout, 0.f);
        for (auto &x : w) x = (float)nd(rng);
        if (set_layer(net, li, w.data(), b.data())) {
            lat_corrector_destroy(h);
            return -3;
        }
    }
    *out = h;
    return 0;
}

void lat_corrector_destroy(lat_corrector *h)
{
    if (!h) return;
    Net &net = h->net;
    if (net.stream) (void)hipStreamSynchronize(net.stream);
    free_buffers(net);
    for (auto &l : net.L) {
        void *ps[] = {l.w, l.b, l.mw, l.vw, l.mb, l.vb, l.wb, l.wt, l.grad};
        for (void *p : ps)
            if (p) (void)hipFree(p);
    }
    delete h;
}

const char *lat_corrector_last_error(const lat_corrector *h) { return h ? h->net.err.c_str() : "null corrector"; }

int lat_corrector_set_layer(lat_corrector *h, int layer, const float *w, const float *b)
{
    if (!h || !w || !b || layer < 0 || layer >= NL) return -1;
    return set_layer(h->net, layer, w, b);
}

int lat_corrector_get_layer(lat_corrector *h, int layer, float *w, float *b)
{
    if (!h || !w || !b || layer < 0 || layer >= NL) return -1;
    Layer &l = h->net.L[layer];
    if (h->net.stream) (void)hipStreamSynchronize(h->net.stream);
    if (hipMemcpy(w, l.w, sizeof(float) * layer_wcount(l), hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(b, l.b, sizeof(float) * l.cout, hipMemcpyDeviceToHost) != hipSuccess)
        return -3;
    return 0;
}

int lat_corrector_set_norm(lat_corrector *h, const double *ratio)
{
    if (!h || !ratio) return -1;
    for (int q = 0; q < 4; ++q) {
        if (!(ratio[q] > 0.0)) return -1;
        h->net.ratio[q] = ratio[q];
    }
    h->net.stats = true;
    return 0;
}

int lat_corrector_get_norm(const lat_corrector *h, double *ratio)
{
    if (!h || !ratio) return -1;
    for (int q = 0; q < 4; ++q) {
        ratio[q] = h->net.ratio[q];
    }
    return 0;
}

// Network output (normalised residual, [site][4] FP32) for the current state of ctx.
int lat_corrector_infer(lat_corrector *h, lat_ctx *ctx, float *out)
{
    if (!h || !ctx || !out) return -1;
    Net &net = h->net;
    StreamLease lease{net};
    Ctx &c = ctx->c;
    int rc = check_ctx(net, c);
    if (rc) return rc;
    pack(net, c, c.fld, c.fldp);
    forward(net, false);
    return copy_to_host(c, out, net.y, sizeof(float) * 4 * c.nvol);
}

// Loss and gradients for the current state of ctx as input and `target`
// ([site][4] FP32, normalised residual): *loss = mean squared error; grads
// (nullable) receives, per layer, cout x 27 cin weight gradients then cout
// bias gradients.  No weight update.
int lat_corrector_gradients(lat_corrector *h, lat_ctx *ctx, const float *target, double *loss, float *grads)
{
    if (!h || !ctx || !target) return -1;
    Net &net = h->net;
    StreamLease lease{net};
    Ctx &c = ctx->c;
    int rc = check_ctx(net, c);
    if (rc) return rc;
    // the network's forward pass runs while the target is staged
    pack(net, c, c.fld, c.fldp);
    forward(net, true);
    if ((rc = copy_to_device(c, net.tgt, target, sizeof(float) * 4 * c.nvol))) return rc;
    backward(net);
    std::vector<float> lp(1024);
    LAT_HIP(&c, hipMemcpyAsync(lp.data(), net.lossp, sizeof(float) * 1024, hipMemcpyDeviceToHost, c.stream));
    LAT_HIP(&c, hipStreamSynchronize(c.stream));
    double s = 0;
    for (float v : lp) s += v;
    if (loss) *loss = s / (4.0 * (double)c.nvol);
    if (grads) {
        size_t off = 0;
        for (auto &l : net.L) {
            std::vector<float> g((size_t)l.mp * (l.kp + 16));
            LAT_HIP(&c, hipMemcpy(g.data(), l.grad, sizeof(float) * g.size(), hipMemcpyDeviceToHost));
            for (int co = 0; co < l.cout; ++co)
                for (int k = 0; k < 27 * l.cin; ++k) grads[off++] = g[(size_t)co * (l.kp + 16) + k];
            for (int co = 0; co < l.cout; ++co) grads[off++] = g[(size_t)co * (l.kp + 16) + l.kp];
        }
    }
    return 0;
}

// Train on npairs snapshot pairs generated along the trajectory of ctx by the
// plain integrator: from the current state S, coarse = one leapfrog step of
// coarse_factor * dt, fine = coarse_factor Yoshida-4 steps of dt; input =
// coarse, target = its residual fluctuation over (ratio x the coarse
// state's standard deviation), ratio fixed at the first pair of a fresh
// corrector; one Adam step per pair; the
// trajectory continues from the fine state.  losses (nullable): per pair,
// NaN for a pair whose coarse step was not finite (no update from it).
int lat_corrector_train(lat_corrector *h, lat_ctx *ctx, double dt, int coarse_factor, int npairs, double lr,
                        double *losses)
{
    if (!h || !ctx || coarse_factor < 1 || npairs < 0) return -1;
    Net &net = h->net;
    StreamLease lease{net};
    Ctx &c = ctx->c;
    int rc = check_ctx(net, c);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * c.ms.f;
    for (int it = 0; it < npairs; ++it) {
        if ((rc = save_state(net, c))) return rc;
        if ((rc = lat_symp(ctx, 2, coarse_factor * dt, 1))) return rc;
        LAT_HIP(&c, hipMemcpyAsync(net.coarse_f, c.fld, bytes, hipMemcpyDeviceToDevice, c.stream));
        LAT_HIP(&c, hipMemcpyAsync(net.coarse_p, c.fldp, bytes, hipMemcpyDeviceToDevice, c.stream));
        if ((rc = restore_state(net, c))) return rc;
        if ((rc = lat_symp(ctx, 4, dt, coarse_factor))) return rc;
        pack(net, c, net.coarse_f, net.coarse_p);
        channel_means(net, c, c.fld, c.fldp, net.coarse_f, net.coarse_p, nullptr, 1);
        bool usable = true;
        if (!net.stats) {
            // ratio = residual fluctuation RMS / input standard deviation
            hipLaunchKernelGGL(k_chsum, dim3(CM_BLOCKS), dim3(256), 0, c.stream, (const double *)c.fld,
                               (const double *)c.fldp, (const double *)net.coarse_f, (const double *)net.coarse_p,
                               (const float *)nullptr, (const double *)(net.cm + 4), c.nvol, net.cpart);
            hipLaunchKernelGGL(k_chmean, dim3(1), dim3(64), 0, c.stream, net.cpart, CM_BLOCKS, c.nvol, 1,
                               net.cm + 16);
            double st[20];
            LAT_HIP(&c, hipMemcpyAsync(st, net.cm, sizeof(st), hipMemcpyDeviceToHost, c.stream));
            LAT_HIP(&c, hipStreamSynchronize(c.stream));
            double r[4];
            for (int q = 0; q < 4; ++q) {
                r[q] = st[16 + q] / st[12 + q];
                // a non-finite coarse step (beyond the leapfrog's stability
                // limit) gives no usable scale: wait for a usable pair
                if (!std::isfinite(r[q]) || !std::isfinite(st[q]) || !std::isfinite(st[4 + q])) usable = false;
                if (!(r[q] > 0.0)) r[q] = 1.0;
            }
            if (usable) {
                for (int q = 0; q < 4; ++q) net.ratio[q] = r[q];
                net.stats = true;
            }
        }
        if (!usable) {
            if (losses) losses[it] = std::nan("");
            continue;
        }
        hipLaunchKernelGGL(k_target, dim3(grid_sites(c.nvol)), dim3(256), 0, c.stream, (const double *)c.fld,
                           (const double *)c.fldp, (const double *)net.coarse_f, (const double *)net.coarse_p,
                           c.nvol, (const double *)net.cm, d4(net.ratio), net.tgt);
        forward(net, true);
        loss_grad(net);
        std::vector<float> lp(1024);
        LAT_HIP(&c, hipMemcpyAsync(lp.data(), net.lossp, sizeof(float) * 1024, hipMemcpyDeviceToHost, c.stream));
        LAT_HIP(&c, hipStreamSynchronize(c.stream));
        double s = 0;
        for (float v : lp) s += v;
        const double loss = s / (4.0 * (double)c.nvol);
        if (losses) losses[it] = loss;
        // a pair whose coarse step left the stability region (non-finite
        // loss) would poison the weights: no update from it
        if (!std::isfinite(loss)) continue;
        backward_layers(net);
        adam(net, (float)lr);
    }
    LAT_HIP(&c, hipGetLastError());
    return 0;
}

// nsteps corrected coarse steps: save S, leapfrog(coarse_factor * dt), add
// the predicted residual, then check the Friedmann constraint: if
// |resid_after - resid_before| > threshold, restore S and take
// coarse_factor Yoshida-4 steps of dt instead (the plain integrator is the
// fallback).  stats (nullable, 3 doubles): fallbacks, max accepted
// constraint change, force evaluations used (a coarse step costs 1, a
// Yoshida-4 step 3).
int lat_corrector_step(lat_corrector *h, lat_ctx *ctx, double dt, int coarse_factor, int nsteps, double threshold,
                       double *stats)
{
    if (!h || !ctx || coarse_factor < 1 || nsteps < 0) return -1;
    Net &net = h->net;
    StreamLease lease{net};
    Ctx &c = ctx->c;
    if (!net.stats) return corr_fail(net, "the corrector has not been trained (no normalisation)");
    int rc = check_ctx(net, c);
    if (rc) return rc;
    double fb = 0, maxv = 0, forces = 0, e[LAT_NE];
    for (int it = 0; it < nsteps; ++it) {
        if ((rc = lat_energies(ctx, e))) return rc;
        const double r0 = e[LAT_E_RESID];
        if ((rc = save_state(net, c))) return rc;
        if ((rc = lat_symp(ctx, 2, coarse_factor * dt, 1))) return rc;
        pack(net, c, c.fld, c.fldp);
        forward(net, false);
        channel_means(net, c, nullptr, nullptr, nullptr, nullptr, net.y, 2);
        hipLaunchKernelGGL(k_apply, dim3(grid_sites(c.nvol)), dim3(256), 0, c.stream, (double *)c.fld,
                           (double *)c.fldp, net.y, c.nvol, (const double *)net.cm, d4(net.ratio));
        c.ke_valid = false;
        forces += 1;
        if ((rc = lat_energies(ctx, e))) return rc;
        const double v = std::fabs(e[LAT_E_RESID] - r0);
        if (!(v <= threshold)) {
            if ((rc = restore_state(net, c))) return rc;
            if ((rc = lat_symp(ctx, 4, dt, coarse_factor))) return rc;
            fb += 1;
            forces += 3.0 * coarse_factor;
        } else if (v > maxv) {
            maxv = v;
        }
    }
    if (stats) {
        stats[0] = fb;
        stats[1] = maxv;
        stats[2] = forces;
    }
    return 0;
}

// As lat_corrector_step, and every judge_every-th accepted corrected step is
// also taken by the plain integrator (coarse_factor Yoshida-4 steps of dt
// from the same start): the errors of the corrected step and of the leapfrog
// step alone against it, per channel (phi, chi, pi_phi, pi_chi) the RMS
// difference over the plain step's spatial standard deviation, the largest
// over the channels, are recorded and the plain step is kept.  Once a judged
// corrected step's error exceeds err_tol, or that of the leapfrog step
// alone, the corrector is switched off and every remaining step is the plain
// integrator's.  stats (nullable, 7 doubles): fallbacks (constraint), force
// evaluations, judged steps, largest judged error of the corrected step,
// step index at which the corrector was switched off (-1: never), largest
// accepted constraint change, largest judged error of the leapfrog step.
int lat_corrector_step_judged(lat_corrector *h, lat_ctx *ctx, double dt, int coarse_factor, int nsteps,
                              double threshold, int judge_every, double err_tol, double *stats)
{
    if (!h || !ctx || coarse_factor < 1 || nsteps < 0 || judge_every < 1) return -1;
    Net &net = h->net;
    StreamLease lease{net};
    Ctx &c = ctx->c;
    if (!net.stats) return corr_fail(net, "the corrector has not been trained (no normalisation)");
    int rc = check_ctx(net, c);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * c.ms.f;
    double fb = 0, forces = 0, judged = 0, maxerr = 0, maxleap = 0, off_at = -1, maxv = 0, e[LAT_NE];
    int accepted = 0;
    // largest over the channels of RMS(a - plain) / std(plain), the plain
    // step being the current state and its standard deviations at cm + 32
    auto judge_err = [&](const void *af, const void *ap, double *out) -> int {
        hipLaunchKernelGGL(k_chsum, dim3(CM_BLOCKS), dim3(256), 0, c.stream, (const double *)c.fld,
                           (const double *)c.fldp, (const double *)af, (const double *)ap, (const float *)nullptr,
                           (const double *)(net.cm + 20), c.nvol, net.cpart);
        hipLaunchKernelGGL(k_chmean, dim3(1), dim3(64), 0, c.stream, net.cpart, CM_BLOCKS, c.nvol, 2, net.cm + 24);
        double jd[12];
        LAT_HIP(&c, hipMemcpyAsync(jd, net.cm + 24, sizeof(jd), hipMemcpyDeviceToHost, c.stream));
        LAT_HIP(&c, hipStreamSynchronize(c.stream));
        double err = 0;
        for (int q = 0; q < 4; ++q) {
            const double r = jd[q] / jd[8 + q];
            err = (r > err || !(r == r)) ? r : err;
        }
        *out = err;
        return 0;
    };
    for (int it = 0; it < nsteps; ++it) {
        if (off_at >= 0) { // switched off: the plain integrator
            if ((rc = lat_symp(ctx, 4, dt, coarse_factor))) return rc;
            forces += 3.0 * coarse_factor;
            continue;
        }
        if ((rc = lat_energies(ctx, e))) return rc;
        const double r0 = e[LAT_E_RESID];
        if ((rc = save_state(net, c))) return rc;
        if ((rc = lat_symp(ctx, 2, coarse_factor * dt, 1))) return rc;
        const bool judge = accepted % judge_every == 0; // if this step is accepted
        if (judge) {
            LAT_HIP(&c, hipMemcpyAsync(net.leap_f, c.fld, bytes, hipMemcpyDeviceToDevice, c.stream));
            LAT_HIP(&c, hipMemcpyAsync(net.leap_p, c.fldp, bytes, hipMemcpyDeviceToDevice, c.stream));
        }
        pack(net, c, c.fld, c.fldp);
        forward(net, false);
        channel_means(net, c, nullptr, nullptr, nullptr, nullptr, net.y, 2);
        hipLaunchKernelGGL(k_apply, dim3(grid_sites(c.nvol)), dim3(256), 0, c.stream, (double *)c.fld,
                           (double *)c.fldp, net.y, c.nvol, (const double *)net.cm, d4(net.ratio));
        c.ke_valid = false;
        forces += 1;
        if ((rc = lat_energies(ctx, e))) return rc;
        const double v = std::fabs(e[LAT_E_RESID] - r0);
        if (!(v <= threshold)) {
            if ((rc = restore_state(net, c))) return rc;
            if ((rc = lat_symp(ctx, 4, dt, coarse_factor))) return rc;
            fb += 1;
            forces += 3.0 * coarse_factor;
            continue;
        }
        maxv = v > maxv ? v : maxv;
        ++accepted;
        if (!judge) continue;
        // judge: the plain step from the same start
        LAT_HIP(&c, hipMemcpyAsync(net.coarse_f, c.fld, bytes, hipMemcpyDeviceToDevice, c.stream));
        LAT_HIP(&c, hipMemcpyAsync(net.coarse_p, c.fldp, bytes, hipMemcpyDeviceToDevice, c.stream));
        if ((rc = restore_state(net, c))) return rc;
        if ((rc = lat_symp(ctx, 4, dt, coarse_factor))) return rc;
        forces += 3.0 * coarse_factor;
        judged += 1;
        channel_means(net, c, c.fld, c.fldp, nullptr, nullptr, nullptr, 7);
        hipLaunchKernelGGL(k_chsum, dim3(CM_BLOCKS), dim3(256), 0, c.stream, (const double *)c.fld,
                           (const double *)c.fldp, (const double *)nullptr, (const double *)nullptr,
                           (const float *)nullptr, (const double *)(net.cm + 28), c.nvol, net.cpart);
        hipLaunchKernelGGL(k_chmean, dim3(1), dim3(64), 0, c.stream, net.cpart, CM_BLOCKS, c.nvol, 1, net.cm + 32);
        double ec = 0, el = 0;
        if ((rc = judge_err(net.coarse_f, net.coarse_p, &ec))) return rc;
        if ((rc = judge_err(net.leap_f, net.leap_p, &el))) return rc;
        maxerr = (ec > maxerr || !(ec == ec)) ? ec : maxerr;
        maxleap = (el > maxleap || !(el == el)) ? el : maxleap;
        if (!(ec <= err_tol) || !(ec <= el)) off_at = it;
    }
    if (stats) {
        stats[0] = fb;
        stats[1] = forces;
        stats[2] = judged;
        stats[3] = maxerr;
        stats[4] = off_at;
        stats[5] = maxv;
        stats[6] = maxleap;
    }
    return 0;
}

} // extern "C"
