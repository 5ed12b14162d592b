// Grid stage of the FP64 nonlinear step on wave FFTs (n_phi = 128 P, P = 2, 4, 8,
// one wave per P): per radial level and theta row, the 18 inverse FFTs of the synthesised
// components, the grid products of src/get_nl.f90 (curl advection :262-273,
// Lorentz force :242-258 merged as src/rIter.f90:650-656, V s :320-325, V x B
// :376-388, u_h . grad_h s), the Courant maxima (src/courant.f90:209-275) and
// the 10 forward FFTs.
//
// One workgroup = one theta row, NW waves.  A real row of N = 128 P points is
// one complex FFT of M = 64 P points (mhx_wavefft.h) with the half-length pre-
// and post-step; in a round each wave transforms one component in its own LDS
// row, then every thread takes its M / (64 NW) complex points of the round's
// components and adds them to the products, which stay in registers.
//
// Bound by the row gathers (16 bytes of each 128-byte line per row, the line's
// other rows in neighbouring workgroups through the L2) and the LDS exchanges:
// n_phi = 512, l_max = 170 x 65 levels, 1.05 ms block-wide, 0.72 so, 0.68 with F
// theta-blocked (1.5 GB with the du/dr grids: 2.2 TB/s).
#include "mhx_wavefft.h"

namespace mhx {

namespace {

typedef double2 C;

struct GwArgs {
    const C *Fin;         // [lev][18][theta/8][m][theta%8]
    C *Fout;              // [lev][10][theta/8][m][theta%8]
    double *dgrid;        // [lev][3][theta][phi] du/dr grids; null: not computed
    double *full_grids;   // optional [lev][18][phi][theta]
    const C *w64, *wm;    // factors of the wave FFT
    const C *twr;         // exp(-2 pi i k / N), k <= M
    const double *osin2, *rad;
    double LFfac;
    int n_m, n_theta, nlev;
    CourArgs cour;
};

// components in the order they are absorbed, products in the order they are
// formed
enum GwIn { VR = 0, VT, VP, CVR, CVT, CVP, DVR, DVT, DVP, BR, BT, BP, CBR, CBT, CBP, SC, DST, DSP };
enum GwOut { ADVR = 0, ADVT, ADVP, VSR, VST, VSP, VXBR, VXBT, VXBP, UGS };
constexpr int NI = 18, NO = 10;

// waves per row: one complex point per thread.  P <= 8: the first pass of the
// wave FFT then has one round per lane and may read the row that it overwrites
template <int P> constexpr int gw_waves()
{
    static_assert(P <= 8, "in-place first pass");
    return P;
}

// LDS: one FFT row per wave, exp(-2 pi i k / N), k <= M, and the FFT's factors
template <int P> constexpr size_t gw_lds()
{
    return ((size_t)gw_waves<P>() * WaveFFT<P>::BUF + (64 * P + 1) + 64 + 64 * P) * sizeof(C);
}

// the real-row transforms of one wave: rows of M complex in `buf`
template <int P> struct RowReal {
    typedef WaveFFT<P> W;
    static constexpr int M = W::N, N = 2 * M;
    static constexpr int NK = M / 128 + 1;  // k = lane + 64 i <= M / 2
    C xa[NK], xc[NK];
    // X_k and X_{M-k} of this lane's k, zero past n_m
    __device__ __forceinline__ void load(const C *__restrict__ X, int n_m, int lane)
    {
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int k = lane + 64 * i, k2 = M - k;
            xa[i] = k < n_m ? X[k * 8] : mk<C>(0.0, 0.0);
            xc[i] = k2 < n_m && k <= M / 2 ? X[k2 * 8] : mk<C>(0.0, 0.0);
        }
    }
    // Z_k = (X_k + conj X_{M-k}) + i e^{+2 pi i k/N} (X_k - conj X_{M-k})
    __device__ __forceinline__ void pre(C *buf, const C *twr, int lane)
    {
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int k = lane + 64 * i, k2 = M - k;
            if (k > M / 2) continue;
            C a = xa[i];
            if (k == 0) a.y = 0.0;
            const C c = xc[i], s = mk<C>(a.x + c.x, a.y - c.y), d = cmul(cconj(twr[k]), mk<C>(a.x - c.x, a.y + c.y));
            buf[k] = mk<C>(s.x - d.y, s.y + d.x);
            // Z_{M-k} = conj of the sum with the odd part's sign turned
            if (k > 0) buf[k2] = mk<C>(s.x + d.y, d.x - s.y);
        }
    }
};

template <int P> __global__ __launch_bounds__(64 * gw_waves<P>(), P <= 6 ? 3 : 2) void k_grid_wave(GwArgs a)
{
    typedef WaveFFT<P> W;
    constexpr int M = W::N, N = 2 * M, NW = gw_waves<P>(), NPT = P / NW;
    extern __shared__ char smem_raw[];
    C *const rows = reinterpret_cast<C *>(smem_raw);
    C *const s_twr = rows + NW * W::BUF, *const s_w64 = s_twr + M + 1, *const s_wm = s_w64 + 64;
    // consecutive rows (eight share the 128-byte lines of F and F2) on one XCD
    int lb;
    {
        const int nx = 8, nb = gridDim.x, b = blockIdx.x;
        const int per = nb / nx, rem = nb % nx, x = b % nx, i = b / nx;
        lb = (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + i;
    }
    const int th = lb % a.n_theta, lev = lb / a.n_theta, n_m = a.n_m;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    C *const buf = rows + wave * W::BUF;
    const double o2 = a.osin2[th];
    const double or2 = a.rad[lev], or4 = a.rad[a.nlev + lev], orho1 = a.rad[2 * a.nlev + lev], LFfac = a.LFfac;
    const bool dudr = a.dgrid || a.full_grids;
    const int ni = dudr ? NI : NI - 3;
    // inverse order: u, curl u, (du/dr,) B, curl B, s, grad s
    auto in_comp = [&](int i) { return i >= 6 && !dudr ? i + 3 : i; };
    const size_t fcomp = f2_comp(n_m, a.n_theta), frow = (size_t)(th / 8) * n_m * 8 + th % 8;
    const C *const Fi = a.Fin + lev * NI * fcomp + frow;
    auto comp_of = [&](int i) { return Fi + in_comp(min(i, ni - 1)) * fcomp; };

    RowReal<P> rr;
    rr.load(comp_of(wave), n_m, lane);
    for (int k = tid; k <= M; k += 64 * NW) s_twr[k] = a.twr[k];
    for (int k = tid; k < 64; k += 64 * NW) s_w64[k] = a.w64[k];
    for (int k = tid; k < M; k += 64 * NW) s_wm[k] = a.wm[k];
    const auto w64 = [&](int i) { return s_w64[8 * i + (lane & 7)]; };
    const auto wn = [&](int k1) { return s_wm[64 * k1 + lane]; };
    __syncthreads();

    C u[3][NPT], b[3][NPT], adv[3][NPT], sc[NPT], ugs[NPT];
    auto fma2 = [](C &y, double f, C p, C v) {
        y.x += f * p.x * v.x;
        y.y += f * p.y * v.y;
    };
    auto mul2 = [](double f, C p, C v) { return mk<C>(f * p.x * v.x, f * p.y * v.y); };
#define GW_EACH(stmt) \
    _Pragma("unroll") for (int q = 0; q < NPT; ++q) { stmt; }
#pragma unroll 1
    for (int i0 = 0; i0 < ni; i0 += NW) {
        rr.pre(buf, s_twr, lane);
        wave_order();
        if (i0 + NW < ni) rr.load(comp_of(i0 + NW + wave), n_m, lane);
        C x[P];
        W::inverse(buf, lane, w64, wn, [&](int, int, int k) { return buf[k]; }, x);
#pragma unroll
        for (int q = 0; q < P; ++q) buf[lane + 64 * q] = x[q];
        __syncthreads();
        // absorb the round's components: thread tid owns complex points tid + 64 NW q
#pragma unroll 1
        for (int c = 0; c < NW && i0 + c < ni; ++c) {
            const int comp = in_comp(i0 + c);
            C v[NPT];
            GW_EACH(v[q] = rows[c * W::BUF + tid + 64 * NW * q])
            if (a.full_grids) {
                double *g = a.full_grids + ((size_t)lev * NI + comp) * N * a.n_theta + th;
                GW_EACH(g[(size_t)(2 * (tid + 64 * NW * q)) * a.n_theta] = v[q].x;
                        g[(size_t)(2 * (tid + 64 * NW * q) + 1) * a.n_theta] = v[q].y)
            }
            switch (comp) {
            case VR: GW_EACH(u[0][q] = v[q]) break;
            case VT: GW_EACH(u[1][q] = v[q]) break;
            case VP: GW_EACH(u[2][q] = v[q]) break;
            // -curl(u) x u (src/get_nl.f90:262-273)
            case CVR: GW_EACH(adv[1][q] = mul2(or4, u[2][q], v[q]); adv[2][q] = mul2(-or4, u[1][q], v[q])) break;
            case CVT: GW_EACH(adv[0][q] = mul2(-o2, u[2][q], v[q]); fma2(adv[2][q], or4, u[0][q], v[q])) break;
            case CVP: GW_EACH(fma2(adv[0][q], o2, u[1][q], v[q]); fma2(adv[1][q], -or4, u[0][q], v[q])) break;
            case DVR: case DVT: case DVP:
                if (a.dgrid) {
                    C *d = reinterpret_cast<C *>(a.dgrid + (((size_t)lev * 3 + comp - DVR) * a.n_theta + th) * N);
                    GW_EACH(d[tid + 64 * NW * q] = v[q])
                }
                break;
            case BR: GW_EACH(b[0][q] = v[q]) break;
            case BT: GW_EACH(b[1][q] = v[q]) break;
            case BP:
                GW_EACH(b[2][q] = v[q])
                if (a.cour.max)
                    courant_max<double, 2 * NPT>(a.cour, lev, a.nlev, o2, or2, or4, orho1, LFfac,
                                                 reinterpret_cast<const double(*)[2 * NPT]>(u),
                                                 reinterpret_cast<const double(*)[2 * NPT]>(b));
                break;
            // Lorentz force (src/get_nl.f90:242-258, src/rIter.f90:650-656)
            case CBR: GW_EACH(fma2(adv[1][q], -LFfac * or4, b[2][q], v[q]); fma2(adv[2][q], LFfac * or4, b[1][q], v[q])) break;
            case CBT: GW_EACH(fma2(adv[0][q], LFfac * o2, b[2][q], v[q]); fma2(adv[2][q], -LFfac * or4, b[0][q], v[q])) break;
            case CBP: GW_EACH(fma2(adv[0][q], -LFfac * o2, b[1][q], v[q]); fma2(adv[1][q], LFfac * or4, b[0][q], v[q])) break;
            // V s (src/get_nl.f90:320-325) and u_h . grad_h s
            case SC: GW_EACH(sc[q] = v[q]) break;
            case DST: GW_EACH(ugs[q] = mul2(or2 * o2, u[1][q], v[q])) break;
            case DSP: GW_EACH(fma2(ugs[q], or2 * o2, u[2][q], v[q])) break;
            default: break;
            }
        }
        __syncthreads();
    }

    C *const Fo = a.Fout + lev * NO * fcomp + frow;
#pragma unroll 1
    for (int o0 = 0; o0 < NO; o0 += NW) {
#pragma unroll 1
        for (int c = 0; c < NW && o0 + c < NO; ++c) {
            C v[NPT];
            auto cross = [&](int p1, int p2, double f) {
#pragma unroll
                for (int q = 0; q < NPT; ++q)
                    v[q] = mk<C>(f * (u[p1][q].x * b[p2][q].x - u[p2][q].x * b[p1][q].x),
                                 f * (u[p1][q].y * b[p2][q].y - u[p2][q].y * b[p1][q].y));
            };
            switch (o0 + c) {
            case ADVR: GW_EACH(v[q] = adv[0][q]) break;
            case ADVT: GW_EACH(v[q] = adv[1][q]) break;
            case ADVP: GW_EACH(v[q] = adv[2][q]) break;
            case VSR: GW_EACH(v[q] = mul2(1.0, u[0][q], sc[q])) break;
            case VST: GW_EACH(v[q] = mul2(or2, u[1][q], sc[q])) break;
            case VSP: GW_EACH(v[q] = mul2(or2, u[2][q], sc[q])) break;
            // V x B (src/get_nl.f90:376-388)
            case VXBR: cross(1, 2, orho1 * o2); break;
            case VXBT: cross(2, 0, orho1 * or4); break;
            case VXBP: cross(0, 1, orho1 * or4); break;
            default: GW_EACH(v[q] = ugs[q]) break;
            }
            GW_EACH(rows[c * W::BUF + tid + 64 * NW * q] = v[q])
        }
        __syncthreads();
        const int out = o0 + wave;
        if (out < NO) {
            C x[P];
#pragma unroll
            for (int q = 0; q < P; ++q) x[q] = buf[lane + 64 * q];
            wave_order();
            W::forward(buf, lane, w64, wn, x);
            // 1/N, and 1/sin^2 on the horizontal comps of the vector products
            const double f = 0.5 / (double)N * (out < UGS && out % 3 ? o2 : 1.0);
            C *fo = Fo + out * fcomp;
            for (int k = lane; k < n_m; k += 64) {
                const C zk = buf[k], zc = cconj(buf[k ? M - k : 0]);
                const C D = csub(zk, zc), X = cadd(cadd(zk, zc), cmul(s_twr[k], mk<C>(D.y, -D.x)));
                fo[(size_t)k * 8] = mk<C>(f * X.x, k ? f * X.y : 0.0);
            }
        }
        __syncthreads();
    }
#undef GW_EACH
}

template <int P> int launch_p(const GwArgs &a, hipStream_t s)
{
    constexpr size_t shm = gw_lds<P>();
    if (int rc = allow_lds((const void *)k_grid_wave<P>, shm)) return rc;
    k_grid_wave<P><<<dim3((unsigned)(a.n_theta * a.nlev)), 64 * gw_waves<P>(), shm, s>>>(a);
    MHX_HIP_CHECK(hipGetLastError());
    return MHX_OK;
}

}  // namespace

// powers of two, where the slot FFTs (M = 3 4^A 2^B) do not apply: per launch
// against the block-wide passes 402 -> 326 us (n_phi = 256 x 97 levels), 1050 ->
// 720 us (512 x 65) and 2481 -> 1154 us (1024 x 16); slower for 640 (858 -> 987
// us, five waves) and than the slots for 768 (2.2 -> 4.0 ms, registers)
bool grid_wave_supported(const Plan *p)
{
    if (!p->d_wm || p->n_phi % 128) return false;
    switch (p->n_phi / 128) {
    case 2: case 4: case 8: return true;
    default: return false;
    }
}

int launch_grid_wave(const Plan *p, int nlev, const void *Fin, void *Fout, const double *rad, double LFfac,
                     void *dgrid, void *full_grids, hipStream_t s)
{
    GwArgs a;
    a.Fin = static_cast<const C *>(Fin);
    a.Fout = static_cast<C *>(Fout);
    a.dgrid = static_cast<double *>(dgrid);
    a.full_grids = static_cast<double *>(full_grids);
    a.w64 = reinterpret_cast<const C *>(p->d_w64);
    a.wm = reinterpret_cast<const C *>(p->d_wm);
    a.twr = reinterpret_cast<const C *>(p->d_twr);
    a.osin2 = p->d_osin2;
    a.rad = rad;
    a.LFfac = LFfac;
    a.n_m = p->n_m;
    a.n_theta = p->n_theta;
    a.nlev = nlev;
    a.cour = p->cour;
    switch (p->n_phi / 128) {
    case 2: return launch_p<2>(a, s);
    case 4: return launch_p<4>(a, s);
    case 8: return launch_p<8>(a, s);
    default: return fail(MHX_E_UNSUPPORTED, "wave grid stage length");
    }
}

}  // namespace mhx
