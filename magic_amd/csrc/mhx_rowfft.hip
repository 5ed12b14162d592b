// phi FFTs between Fourier rows and theta-fastest grids (Fortran f(n_theta,
// n_phi)) for n_phi = 64 P: one wave per pair of neighbouring theta rows of
// one component, both real rows in one complex FFT of length n_phi (a colatitude's
// north and south row, whose sums and differences are what the Legendre side takes
// and gives: each row's rounding error is relative to the larger of the two), 16-byte
// accesses of the pair throughout.  Other lengths run the generic kernels of mhx_fft.hip.
//
// Bound by HBM: n_theta n_phi 8 + n_theta n_m 16 bytes per component and
// level.  All components of a call run in one launch, 8 theta rows per
// workgroup (whole 128-byte lines of the Fourier arrays' blocks of 8 rows).
//
// Three components at n_phi = 512, l_max = 170 x 65 levels: 229 us by block-wide
// radix-4 passes and 16-byte gathers, one component per launch, 105 us so (341 MB:
// 3.2 TB/s; a large copy reaches 4.8).
#include "mhx_wavefft.h"

namespace mhx {

namespace {

// a pair of grid values; grids are aligned to 8 bytes only
struct __attribute__((packed, aligned(8))) Pair {
    double x, y;
};

template <int P> constexpr int row_waves() { return P <= 12 ? 4 : 2; }

// linear block -> (theta block, comp, level), neighbouring theta blocks on one
// XCD (they share the grid's cache lines)
__device__ __forceinline__ void row_block(const RowFFT &a, int ntb, int &tb, int &comp, int &lev)
{
    const int nx = 8, nb = gridDim.x, b = blockIdx.x;
    const int per = nb / nx, rem = nb % nx, x = b % nx, i = b / nx;
    const int lb = (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + i;
    tb = lb % ntb;
    comp = lb / ntb % a.ncomp;
    lev = lb / (ntb * a.ncomp);
}

template <int P> __global__ __launch_bounds__(64 * row_waves<P>()) void k_irow(RowFFT a)
{
    typedef WaveFFT<P> W;
    constexpr int NW = row_waves<P>(), N = W::N;
    __shared__ double2 sm[NW * W::BUF];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    int tb, comp, lev;
    row_block(a, (a.n_theta / 2 + NW - 1) / NW, tb, comp, lev);
    const int th = 2 * (tb * NW + wave);
    if (th >= a.n_theta) return;
    const double2 *X = reinterpret_cast<const double2 *>(a.F) + (size_t)lev * a.F_ld +
                       comp * f2_comp(a.n_m, a.n_theta) + (size_t)(th / 8) * a.n_m * 8 + th % 8;
    double2 x[P];
    // Y_k = X1_k + i X2_k, Y_{N-k} = conj X1_k + i conj X2_k (real parts of mode 0)
    const auto w64 = [&](int i) { return a.w64[8 * i + (lane & 7)]; };
    const auto wn = [&](int k1) { return a.wn[64 * k1 + lane]; };
    W::inverse(sm + wave * W::BUF, lane, w64, wn, [&](int, int, int k) {
        const int kk = k <= N / 2 ? k : N - k;
        const double2 *p = X + (size_t)min(kk, a.n_m - 1) * 8;
        const double2 u = p[0], v = p[1];
        double2 y = k <= N / 2 ? mk<double2>(u.x - v.y, u.y + v.x) : mk<double2>(u.x + v.y, v.x - u.y);
        if (k == 0) y = mk<double2>(u.x, v.x);
        return kk < a.n_m ? y : mk<double2>(0.0, 0.0);
    }, x);
    double *g = a.grid[comp] + (size_t)lev * a.grid_ld + th;
#pragma unroll
    for (int q = 0; q < P; ++q)
        *reinterpret_cast<Pair *>(g + (size_t)(lane + 64 * q) * a.n_theta) = Pair{x[q].x, x[q].y};
}

template <int P> __global__ __launch_bounds__(64 * row_waves<P>()) void k_frow(RowFFT a)
{
    typedef WaveFFT<P> W;
    constexpr int NW = row_waves<P>(), N = W::N;
    __shared__ double2 sm[NW * W::BUF];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    int tb, comp, lev;
    row_block(a, (a.n_theta / 2 + NW - 1) / NW, tb, comp, lev);
    const int th = 2 * (tb * NW + wave);
    if (th >= a.n_theta) return;
    const double *g = a.src[comp] + (size_t)lev * a.grid_ld + th;
    double2 x[P], *buf = sm + wave * W::BUF;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const Pair p = *reinterpret_cast<const Pair *>(g + (size_t)(lane + 64 * q) * a.n_theta);
        x[q] = mk<double2>(p.x, p.y);
    }
    W::forward(buf, lane, [&](int i) { return a.w64[8 * i + (lane & 7)]; }, [&](int k1) { return a.wn[64 * k1 + lane]; }, x);
    // X1_k = (Y_k + conj Y_{N-k}) / 2, X2_k = (Y_k - conj Y_{N-k}) / (2 i), scaled
    // by 1/N and, for the flagged comps, 1/sin^2(theta) (equal in the two rows)
    const double sc = (a.osin2_mask >> comp & 1u ? a.osin2[th] : 1.0) * (0.5 / (double)N);
    double2 *F = reinterpret_cast<double2 *>(a.F2) + (size_t)lev * a.F_ld + comp * f2_comp(a.n_m, a.n_theta) +
                 (size_t)(th / 8) * a.n_m * 8 + th % 8;
    for (int k = lane; k < a.n_m; k += 64) {
        const double2 u = buf[k], v = buf[k ? N - k : 0];
        double2 x1 = mk<double2>(sc * (u.x + v.x), sc * (u.y - v.y)), x2 = mk<double2>(sc * (u.y + v.y), sc * (v.x - u.x));
        if (k == 0) x1.y = x2.y = 0.0;
        F[(size_t)k * 8] = x1;
        F[(size_t)k * 8 + 1] = x2;
    }
}

template <int P> int launch_p(const RowFFT &a, int nlev, bool inverse, hipStream_t s)
{
    constexpr int NW = row_waves<P>();
    const dim3 grid((unsigned)((a.n_theta / 2 + NW - 1) / NW * a.ncomp * nlev));
    if (inverse)
        k_irow<P><<<grid, 64 * NW, 0, s>>>(a);
    else
        k_frow<P><<<grid, 64 * NW, 0, s>>>(a);
    MHX_HIP_CHECK(hipGetLastError());
    return MHX_OK;
}

}  // namespace

bool row_fft_supported(const Plan *p)
{
    if (!p->d_wn || p->n_phi % 64) return false;
    switch (p->n_phi / 64) {
    case 1: case 2: case 3: case 4: case 5: case 6: case 8: case 9: case 10: case 12: case 15: case 16: case 18:
    case 20: case 24: return true;
    default: return false;
    }
}

int launch_row_fft(const Plan *p, const RowFFT &args, int nlev, bool inverse, hipStream_t s)
{
    if (nlev <= 0) return MHX_OK;
    RowFFT a = args;
    a.w64 = reinterpret_cast<const double2 *>(p->d_w64);
    a.wn = reinterpret_cast<const double2 *>(p->d_wn);
    a.osin2 = p->d_osin2;
    a.n_m = p->n_m;
    a.n_theta = p->n_theta;
    switch (p->n_phi / 64) {
    case 1: return launch_p<1>(a, nlev, inverse, s);
    case 2: return launch_p<2>(a, nlev, inverse, s);
    case 3: return launch_p<3>(a, nlev, inverse, s);
    case 4: return launch_p<4>(a, nlev, inverse, s);
    case 5: return launch_p<5>(a, nlev, inverse, s);
    case 6: return launch_p<6>(a, nlev, inverse, s);
    case 8: return launch_p<8>(a, nlev, inverse, s);
    case 9: return launch_p<9>(a, nlev, inverse, s);
    case 10: return launch_p<10>(a, nlev, inverse, s);
    case 12: return launch_p<12>(a, nlev, inverse, s);
    case 15: return launch_p<15>(a, nlev, inverse, s);
    case 16: return launch_p<16>(a, nlev, inverse, s);
    case 18: return launch_p<18>(a, nlev, inverse, s);
    case 20: return launch_p<20>(a, nlev, inverse, s);
    case 24: return launch_p<24>(a, nlev, inverse, s);
    default: return fail(MHX_E_UNSUPPORTED, "row FFT length");
    }
}

}  // namespace mhx
