// Legendre stage on FP64 MFMA (v_mfma_f64_16x16x4f64), batched over radial
// levels.
//
// Synthesis (src/shtransforms.f90:103-372,493-646): for one order m, the
// Fourier coefficient of every output component at every theta is a sum over
// l of P_lm(theta) or dP_lm(theta) times a complex column built from the input
// coefficients.  With theta rows as GEMM rows, l as K and (8 radial levels x
// re/im) as 16 GEMM columns this is a dense contraction per m.  The
// equatorial symmetry of the reference (ES/EA sums, :172-189) is kept: K runs
// over l of one parity at a time, and two accumulators per column gather
//     Sym  = sum over l - m even,   Anti = sum over l - m odd
// so that north = Sym + Anti and south = Sym - Anti (P is even under theta ->
// pi - theta for l - m even).
//
// Only P_lm is contracted: sin(theta) dP_l/dtheta = l c_{l+1} P_{l+1} -
// (l+1) c_l P_{l-1} (src/plms.f90:142-162) moves every dP product onto P,
//     sum_l dP_l x_l = sum_l P_l x'_l,  x'_l = (l-1) c_l x_{l-1} - (l+2) c_{l+1} x_{l+1}
// for l <= l_max + 1, so that a vector field takes three column products
// (Q, S' + i m T, i m S - T') instead of five.
//
// Analysis (src/shtransforms.f90:648-872): rows are l of one parity, K is the
// northern theta, columns as above; the ES/EA combinations of north/south
// Fourier rows are formed while staging B, Gauss weights are folded into the
// tables (wPlm, wdPlm).
#include "mhx_internal.h"

namespace mhx {

namespace {

constexpr int WG = 256;
constexpr int KQC = 8;          // quads (of 4 l or 4 theta) per staged chunk
constexpr int CHUNK = 4 * KQC;  // 32 rows of B per parity / per theta chunk

struct Prod {
    int acc, tab, col;  // tab 0: P, 1: dP
};

template <int KIND> struct AnaSpec;
template <> struct AnaSpec<ANA_SH> {      // cols: f
    static constexpr int NOUT = 1, NCOL = 1, NPROD = 1;
    static constexpr Prod prod[1] = {{0, 0, 0}};
    static constexpr bool divll[1] = {false};
};
template <> struct AnaSpec<ANA_SPHTOR> {  // cols: vt, -i m vp, -vp, -i m vt
    static constexpr int NOUT = 2, NCOL = 4, NPROD = 4;
    static constexpr Prod prod[4] = {{0, 1, 0}, {0, 0, 1}, {1, 1, 2}, {1, 0, 3}};
    static constexpr bool divll[2] = {true, true};
};
template <> struct AnaSpec<ANA_QST> {     // cols: f, vt, -i m vp, -vp, -i m vt
    static constexpr int NOUT = 3, NCOL = 5, NPROD = 5;
    static constexpr Prod prod[5] = {{0, 0, 0}, {1, 1, 1}, {1, 0, 2}, {2, 1, 3}, {2, 0, 4}};
    static constexpr bool divll[3] = {false, true, true};
};

struct SynArgs {
    SynJob job[MAX_SYN_JOBS];
    int njob, nlev, ng, gz;
    size_t src_ld, fout_ld;
    const int *lcut;
    const double *or2;
    const double *tab;     // P_lm, l <= l_max + 1 (layout: mhx_tables.hip)
    const size_t *off;
    const double *crec;
    const int *lstart;
    const double *osin2;
    int l_max, minc, n_m, nh, n_theta, nt16;
};

struct AnaArgs {
    AnaJob job;
    const double *aP, *adP;
    const size_t *off;
    const int *lstart;
    int l_max, m_max, minc, n_m, nh, n_theta, nq4;
};

// v_mfma_f64_16x16x4f64 operands: A lane l holds A[l % 16][l / 16], B lane l
// holds B[l / 16][l % 16]; D element j of lane l is D[l / 16 + 4 j][l % 16].
__device__ inline d4 mfma64(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Blocks are dispatched round-robin over the 8 XCDs (each with its own L2).
// Remap the linear block id so that each XCD works through a contiguous range
// of logical blocks; with the order index m fastest, the blocks resident on
// one XCD at a time cover neighbouring m, whose values share cache lines of
// the row-contiguous forward-side layout F2[lev][comp][theta][m].
__device__ inline int xcd_logical(int b, int nb)
{
    const int nx = 8;
    int per = nb / nx, rem = nb % nx;
    int x = b % nx, i = b / nx;
    return (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + i;
}

// i^ipow * m^mpow * scale applied to (re, im)
__device__ inline void apply_factor(double &re, double &im, int ipow, int mpow, double m,
                                    double scale)
{
    double f = scale;
    for (int k = 0; k < mpow; ++k) f *= m;
    re *= f;
    im *= f;
    for (int k = 0; k < (ipow & 3); ++k) {
        double t = re;
        re = -im;
        im = t;
    }
}

// ------------------------------------------------------------- synthesis
__device__ inline double2 czero() { return make_double2(0.0, 0.0); }
__device__ inline double2 cimul(double m, double2 z) { return make_double2(-m * z.y, m * z.x); }  // i m z

// B chunk in LDS: 32 consecutive l, [column][parity][pair of quads] blocks of
// 64 lanes x 2 quads; the blocks are padded so that the eight levels and the
// chunk's parities and pairs of one store fall on different banks (block
// strides 8, 16 modulo 32 doubles)
constexpr int SB_PAIR = 136, SB_PAR = 2 * SB_PAIR, SB_COL = 2 * SB_PAR;

template <int KIND> constexpr int syn_np() { return KIND == SYN_QST ? 3 : (KIND == SYN_SCAL ? 1 : 2); }

// One workgroup: one job, one order m (index mc), 8 radial levels from lev0,
// theta tiles of 16 rows dealt over the waves of gz workgroups, TPW per wave.
// Per chunk of 32 degrees a thread owns one (level, l): its coefficients are
// loaded a chunk ahead (consecutive l of a level by consecutive lanes), formed
// into the columns with the l -/+ 1 neighbours taken from the adjacent lanes,
// and written to the other half of the LDS buffer, so that one barrier per
// chunk is enough; the table fragments (16 bytes per lane: two quads) are
// loaded one step of 2 NP TPW products ahead.  Loads are unconditional at
// clamped addresses, the values masked at their use.
template <int TPW, int KIND>
__device__ __forceinline__ void syn_body(const SynArgs &a, const SynJob &job, int mc, int lev0, int gz, double *sB)
{
    constexpr int NP = syn_np<KIND>();
    constexpr bool QST = KIND == SYN_QST, TWO = KIND == SYN_QST || KIND == SYN_SPHTOR;
    constexpr int CS = QST ? 1 : 0, CT = QST ? 2 : 1;  // fields S (or x) and T
    const int m = mc * a.minc, L = a.l_max;
    const double dm = (double)m;
    const int tid = threadIdx.x, lane = tid & 63;
    const int tt0 = gz * 4 + __builtin_amdgcn_readfirstlane(tid >> 6), tstep = 4 * a.gz;
    const int l0 = a.lstart[mc];

    // the thread's (level, degree) of a chunk
    const int lv = tid >> 5, j = tid & 31, lev = lev0 + lv;
    const int lc = lev < a.nlev ? min(a.lcut[lev], L) : -1;
    int lcm = -1;  // largest cut-off of the level group
#pragma unroll
    for (int i = 0; i < LEV_GROUP; ++i) lcm = max(lcm, min(a.lcut[min(lev0 + i, a.nlev - 1)], L));
    const int nrow = max(lcm + 2 - m, 0);  // degrees m .. lcm + 1
    const int nch = (nrow + 31) >> 5;
    const int nquad[2] = {((nrow + 1) / 2 + 3) >> 2, (nrow / 2 + 3) >> 2};
    const int levc = min(lev, a.nlev - 1);
    const double or2 = a.or2 ? a.or2[levc] : 0.0;
    const size_t src0 = ((size_t)levc * a.src_ld + (size_t)(l0 - m)) * 2;

    const double *const q0 = job.col[0].x0, *const s0 = job.col[CS].x0;
    const double *const t0 = job.col[CT].x0, *const t1 = job.col[CT].x1;
    double2 xq, xs, xt0, xt1, hs, ht0, ht1;  // own degree; the chunk's outer neighbours (lanes 0, 31)
    auto ld = [&](const double *p, int l) { return *reinterpret_cast<const double2 *>(p + src0 + 2 * (size_t)l); };
    const int hd = j == 0 ? -1 : 1;
    auto load = [&](int c) {
        const int l = m + 32 * c + j;
        const int li = min(l, L), lh = max(min(l + hd, L), m);
        if constexpr (QST) xq = ld(q0, li);
        xs = ld(s0, li);
        if constexpr (KIND != SYN_SCAL) {
            if (j == 0 || j == 31) hs = ld(s0, lh);
        }
        if constexpr (TWO) {
            xt0 = ld(t0, li);
            if (j == 0 || j == 31) ht0 = ld(t0, lh);
            if (t1) {
                xt1 = ld(t1, li);
                if (j == 0 || j == 31) ht1 = ld(t1, lh);
            }
        }
    };
    // the field at (level, l), zero outside m <= l <= lcut
    auto field = [&](const ColOp &op, int l, double2 x0, double2 x1) {
        const double ll = (double)l * (double)(l + 1);
        const double g = op.gkind == G_ONE ? 1.0 : (op.gkind == G_LL ? ll : or2 * ll);
        double2 v = make_double2(g * x0.x, g * x0.y);
        if (op.x1) v = make_double2(v.x - x1.x, v.y - x1.y);
        if (op.im) v = cimul(dm, v);
        const bool ok = l >= m && l <= lc;
        return make_double2(ok ? v.x : 0.0, ok ? v.y : 0.0);
    };
    auto put = [&](int buf, int col, double2 v) {
        double *b = sB + buf * NP * SB_COL + col * SB_COL + (j & 1) * SB_PAR + (j >> 4) * SB_PAIR +
                    (((j >> 1) & 3) * 16 + 2 * lv) * 2 + ((j >> 3) & 1);
        b[0] = v.x;
        b[2] = v.y;
    };
    auto build = [&](int c, int buf) {
        const int l = m + 32 * c + j;
        if constexpr (QST) put(buf, 0, field(job.col[0], l, xq, czero()));
        const double2 s = field(job.col[CS], l, xs, czero());
        if constexpr (KIND == SYN_SCAL) {
            put(buf, 0, s);
        } else {
            const double *cr = a.crec + l0 + 2 * mc + min(l, L + 1) - m;
            const double fm = (double)(l - 1) * cr[0], fp = (double)(l + 2) * cr[1];
            // x' from the neighbours of x
            auto prime = [&](double2 x, double2 h) {
                double2 lo = make_double2(__shfl_up(x.x, 1, 32), __shfl_up(x.y, 1, 32));
                double2 hi = make_double2(__shfl_down(x.x, 1, 32), __shfl_down(x.y, 1, 32));
                if (j == 0) lo = h;
                if (j == 31) hi = h;
                return make_double2(fm * lo.x - fp * hi.x, fm * lo.y - fp * hi.y);
            };
            const double2 sp = prime(s, field(job.col[CS], l + hd, hs, czero()));
            if constexpr (TWO) {
                const double2 t = field(job.col[CT], l, xt0, xt1);
                const double2 tp = prime(t, field(job.col[CT], l + hd, ht0, ht1));
                put(buf, CS, make_double2(sp.x - dm * t.y, sp.y + dm * t.x));       // S' + i m T
                put(buf, CS + 1, make_double2(-dm * s.y - tp.x, dm * s.x - tp.y));  // i m S - T'
            } else {
                put(buf, 0, s);
                put(buf, 1, sp);
            }
        }
    };

    d4 acc[TPW][NP][2];
#pragma unroll
    for (int s = 0; s < TPW; ++s)
#pragma unroll
        for (int pr = 0; pr < NP; ++pr) acc[s][pr][0] = acc[s][pr][1] = d4{0.0, 0.0, 0.0, 0.0};

    // table fragments of (pair of quads kp, parity); past the last pair the
    // last one is loaded and not used
    const double2 *tab[2];
#pragma unroll
    for (int par = 0; par < 2; ++par)
        tab[par] = reinterpret_cast<const double2 *>(a.tab + a.off[2 * mc + par]) + lane;
    auto load_A = [&](double2 *f, int kp, int par) {
        const double2 *t = tab[par] + (size_t)max(min(kp, (nquad[par] - 1) >> 1), 0) * (a.nt16 * 64);
#pragma unroll
        for (int s = 0; s < TPW; ++s) f[s] = t[min(tt0 + s * tstep, a.nt16 - 1) * 64];
    };
    const bool act = tt0 < a.nt16;
    double2 fa[2][TPW];

    if (nch > 0) {
        load(0);
        if (nquad[0] > 0) load_A(fa[0], 0, 0);
        build(0, 0);
    }
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        const int buf = c & 1;
        if (c + 1 < nch) load(c + 1);
        if (act) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int par = k & 1, pair = k >> 1;
                // the next step's fragments
                if (nquad[1 - par] > 0) load_A(fa[1 - par], 2 * c + ((k + 1) >> 1), 1 - par);
                const int qq = 4 * c + 2 * pair;  // first quad of this step
                if (qq < nquad[par]) {
                    double2 b[NP];
                    const double *sb = sB + buf * NP * SB_COL + par * SB_PAR + pair * SB_PAIR + 2 * lane;
#pragma unroll
                    for (int pr = 0; pr < NP; ++pr) b[pr] = *reinterpret_cast<const double2 *>(sb + pr * SB_COL);
#pragma unroll
                    for (int pr = 0; pr < NP; ++pr)
#pragma unroll
                        for (int s = 0; s < TPW; ++s) acc[s][pr][par] = mfma64(fa[par][s].x, b[pr].x, acc[s][pr][par]);
                    if (qq + 1 < nquad[par]) {
#pragma unroll
                        for (int pr = 0; pr < NP; ++pr)
#pragma unroll
                            for (int s = 0; s < TPW; ++s)
                                acc[s][pr][par] = mfma64(fa[par][s].y, b[pr].y, acc[s][pr][par]);
                    }
                }
            }
        }
        if (c + 1 < nch) build(c + 1, buf ^ 1);
        __syncthreads();
    }

    // epilogue: north = Sym + Anti, south = Sym - Anti; adjacent lanes (re, im)
    // exchange, so that the even lane stores the northern complex value and
    // the odd lane the southern one: 128-byte runs of F[lev][comp][m][theta]
    const int col = lane & 15, elev = lev0 + (col >> 1), odd = col & 1;
    if (elev >= a.nlev) return;
    const size_t cstride = (size_t)a.n_m * a.n_theta;
    double2 *fo = reinterpret_cast<double2 *>(job.fout) + (size_t)elev * a.fout_ld + (size_t)mc * a.n_theta + odd;
#pragma unroll
    for (int s = 0; s < TPW; ++s) {
        const int tt = tt0 + s * tstep;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int th = tt * 16 + (lane >> 4) + 4 * jj;
            const bool ok = th < a.nh;
            const double sc = job.row_scale ? a.osin2[2 * min(th, a.nh - 1)] : 1.0;
#pragma unroll
            for (int pr = 0; pr < NP; ++pr) {
                const double n = acc[s][pr][0][jj] + acc[s][pr][1][jj];
                const double so = acc[s][pr][0][jj] - acc[s][pr][1][jj];
                const double other = __shfl_xor(odd ? n : so, 1, 64);
                double2 v = odd ? make_double2(other, so) : make_double2(n, other);
                if (job.row_scale) v = make_double2(sc * v.x, sc * v.y);
                auto store = [&](int o, double2 w) {
                    if (ok) fo[job.out_comp[o] * cstride + 2 * th] = w;
                };
                // columns: QST (Q, C1, C2), SPHTOR (C1, C2), SCAL x;
                // SG, GRAD: x, x' with d/dphi = i m (P x)
                if constexpr (KIND == SYN_SG) {
                    store(pr, v);
                    if (pr == 0) store(2, cimul(dm, v));
                } else if constexpr (KIND == SYN_GRAD) {
                    store(1 - pr, pr == 0 ? cimul(dm, v) : v);
                } else {
                    store(pr, v);
                }
            }
        }
    }
}

// the jobs of one launch: kinds of at most NP columns
template <int TPW, int NP>
__global__ __launch_bounds__(WG, 2) void k_syn(SynArgs a)
{
    __shared__ double sB[2 * NP * SB_COL];
    // block -> (order, level group, theta group, job): orders dealt to the 8
    // XCDs (blocks go round-robin over them) from the longest on, all blocks
    // of one order on one XCD, whose L2 then holds its table slice once, and
    // the jobs of a level group together, which share coefficients
    const int inner = a.njob * a.gz * a.ng;
    const int mc = (int)(blockIdx.x >> 3) / inner * 8 + (int)(blockIdx.x & 7);
    if (mc >= a.n_m) return;
    int r = (int)(blockIdx.x >> 3) % inner;
    const SynJob &job = a.job[r % a.njob];
    r /= a.njob;
    const int gz = r % a.gz, lev0 = r / a.gz * LEV_GROUP;
    switch (job.kind) {
    case SYN_SCAL: syn_body<TPW, SYN_SCAL>(a, job, mc, lev0, gz, sB); break;
    case SYN_GRAD: if constexpr (NP > 1) syn_body<TPW, SYN_GRAD>(a, job, mc, lev0, gz, sB); break;
    case SYN_SG: if constexpr (NP > 1) syn_body<TPW, SYN_SG>(a, job, mc, lev0, gz, sB); break;
    case SYN_SPHTOR: if constexpr (NP > 1) syn_body<TPW, SYN_SPHTOR>(a, job, mc, lev0, gz, sB); break;
    case SYN_QST: if constexpr (NP > 2) syn_body<TPW, SYN_QST>(a, job, mc, lev0, gz, sB); break;
    default: break;
    }
}

// -------------------------------------------------------------- analysis
template <int KIND>
__global__ __launch_bounds__(WG) void k_ana(AnaArgs a)
{
    using S = AnaSpec<KIND>;
    constexpr int NOUT = S::NOUT, NCOL = S::NCOL, NPROD = S::NPROD;
    constexpr int BS_DOUBLES = NCOL * 2 * CHUNK * 16;     // [col][sym/anti][32 th][16]
    constexpr int EP_DOUBLES = 4 * LEV_GROUP * 32 * 2;
    __shared__ double smem[BS_DOUBLES > EP_DOUBLES ? BS_DOUBLES : EP_DOUBLES];

    const AnaJob &job = a.job;
    const int lb = xcd_logical(blockIdx.x, gridDim.x);
    const int mc = lb % a.n_m;
    const int ng = (job.nlev + LEV_GROUP - 1) / LEV_GROUP;
    const int gy = (lb / a.n_m) % ng, gz = lb / (a.n_m * ng);
    const int m = mc * a.minc;
    const double dm = (double)m;
    const int lev0 = gy * LEV_GROUP;
    const int nlev_here = min(LEV_GROUP, job.nlev - lev0);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t = gz * 4 + wave;  // pair tile: l = m + 32 t + 0..31
    const int K0 = (a.l_max - m) / 2 + 1;
    const int ntile = (K0 + 15) / 16;
    const bool active = t < ntile;
    const int l0 = a.lstart[mc];

    // column definitions: source comp slot, i-power, m-power, scale
    // SH: f | SPHTOR: vt, -i m vp, -vp, -i m vt | QST: f + SPHTOR's
    int csrc[NCOL], cip[NCOL], cmp[NCOL];
    double csc[NCOL];
    if constexpr (KIND == ANA_SH) {
        csrc[0] = 0; cip[0] = 0; cmp[0] = 0; csc[0] = 1.0;
    } else {
        const int b = (KIND == ANA_QST) ? 1 : 0;
        if constexpr (KIND == ANA_QST) { csrc[0] = 0; cip[0] = 0; cmp[0] = 0; csc[0] = 1.0; }
        csrc[b + 0] = 1; cip[b + 0] = 0; cmp[b + 0] = 0; csc[b + 0] = 1.0;
        csrc[b + 1] = 2; cip[b + 1] = 1; cmp[b + 1] = 1; csc[b + 1] = -1.0;
        csrc[b + 2] = 2; cip[b + 2] = 0; cmp[b + 2] = 0; csc[b + 2] = -1.0;
        csrc[b + 3] = 1; cip[b + 3] = 1; cmp[b + 3] = 1; csc[b + 3] = -1.0;
    }

    d4 acc[NOUT][2];
#pragma unroll
    for (int o = 0; o < NOUT; ++o)
        for (int s = 0; s < 2; ++s) acc[o][s] = d4{0.0, 0.0, 0.0, 0.0};

    const int nchunk = (a.nq4 + KQC - 1) / KQC;
    for (int c = 0; c < nchunk; ++c) {
        __syncthreads();
        for (int idx = threadIdx.x; idx < CHUNK * LEV_GROUP; idx += WG) {
            int levl = idx % LEV_GROUP;
            int thl = idx / LEV_GROUP;
            int th = c * CHUNK + thl;
            int lev = lev0 + levl;
            bool valid = (levl < nlev_here) && (th < a.nh);
            if (valid) {
                int lc = job.lcut[lev];
                int mlim = lc < a.m_max ? lc : a.m_max;
                valid = m <= mlim;
            }
            double nr[3], ni[3], sr[3], si[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) { nr[k] = ni[k] = sr[k] = si[k] = 0.0; }
            if (valid) {
                int nsrc = (KIND == ANA_SH) ? 1 : 3;
                for (int k = 0; k < nsrc; ++k) {
                    int comp = job.in_comp[k];
                    if (comp < 0) continue;
                    size_t o = ((size_t)lev * job.fin_ld + ((size_t)comp * a.n_theta + 2 * th) * a.n_m + mc) * 2;
                    size_t o2 = o + (size_t)a.n_m * 2;
                    nr[k] = job.fin[o];
                    ni[k] = job.fin[o + 1];
                    sr[k] = job.fin[o2];
                    si[k] = job.fin[o2 + 1];
                }
            }
#pragma unroll
            for (int col = 0; col < NCOL; ++col) {
                int k = csrc[col];
                double syr = nr[k] + sr[k], syi = ni[k] + si[k];
                double anr = nr[k] - sr[k], ani = ni[k] - si[k];
                apply_factor(syr, syi, cip[col], cmp[col], dm, csc[col]);
                apply_factor(anr, ani, cip[col], cmp[col], dm, csc[col]);
                double *b0 = smem + (((col * 2 + 0) * CHUNK + thl) * 16 + levl * 2);
                double *b1 = smem + (((col * 2 + 1) * CHUNK + thl) * 16 + levl * 2);
                b0[0] = syr; b0[1] = syi;
                b1[0] = anr; b1[1] = ani;
            }
        }
        __syncthreads();
        if (active) {
            int nq = min(KQC, a.nq4 - c * KQC);
            for (int q = 0; q < nq; ++q) {
                size_t tq = (size_t)(c * KQC + q);
#pragma unroll
                for (int par = 0; par < 2; ++par) {
                    size_t o = a.off[2 * mc + par] + ((size_t)t * a.nq4 + tq) * 64 + lane;
                    double aP = a.aP[o];
                    double adP = a.adP[o];
#pragma unroll
                    for (int pr = 0; pr < NPROD; ++pr) {
                        const Prod P = S::prod[pr];
                        // even rows: P uses the symmetric combination, dP the antisymmetric
                        int use = (P.tab == 0) ? par : (1 - par);
                        double b = smem[((P.col * 2 + use) * CHUNK + q * 4 + (lane >> 4)) * 16 + (lane & 15)];
                        acc[P.acc][par] = mfma64(P.tab == 0 ? aP : adP, b, acc[P.acc][par]);
                    }
                }
            }
        }
    }

    // epilogue: rows r -> l = m + par + 2 (16 t + r); transpose to 32
    // consecutive l per level
    __syncthreads();
    double *ep = smem + wave * (LEV_GROUP * 32 * 2);
    const int col = lane & 15, levl_c = col >> 1, ri = col & 1;
#pragma unroll
    for (int o = 0; o < NOUT; ++o) {
        if (active) {
#pragma unroll
            for (int par = 0; par < 2; ++par)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    int r = (lane >> 4) + 4 * j;
                    int l = m + par + 2 * (16 * t + r);
                    double v = acc[o][par][j];
                    if (S::divll[o] && l > 0) v /= (double)l * (double)(l + 1);
                    ep[(levl_c * 32 + 2 * r + par) * 2 + ri] = v;
                }
        }
        __syncthreads();
        if (active) {
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                int e = rr * 64 + lane;
                int levl = e >> 5, ll = e & 31;
                int l = m + 32 * t + ll;
                if (levl < nlev_here && l <= a.l_max) {
                    int lev = lev0 + levl;
                    int lc = job.lcut[lev];
                    bool keep = (l <= lc) && (m <= (lc < a.m_max ? lc : a.m_max));
                    double2 v = keep ? make_double2(ep[(levl * 32 + ll) * 2], ep[(levl * 32 + ll) * 2 + 1])
                                     : make_double2(0.0, 0.0);
                    size_t o2 = ((size_t)lev * job.out_ld + (size_t)(l0 + l - m)) * 2;
                    *reinterpret_cast<double2 *>(job.out[o] + o2) = v;
                }
            }
        }
        __syncthreads();
    }
}

// theta tiles per wave and theta groups: 12 tiles per workgroup at most
// (three per wave: 144 accumulator registers of the 256 at two waves per SIMD)
template <int NP>
int launch_syn_np(const SynArgs &a, int tpw, unsigned grid, hipStream_t s)
{
    switch (tpw) {
    case 1: k_syn<1, NP><<<grid, WG, 0, s>>>(a); break;
    case 2: k_syn<2, NP><<<grid, WG, 0, s>>>(a); break;
    default: k_syn<3, NP><<<grid, WG, 0, s>>>(a); break;
    }
    MHX_HIP_CHECK(hipGetLastError());
    return MHX_OK;
}

}  // namespace

int launch_syn(const Plan *p, const SynJob *jobs, int njob, const SynBatch &b, hipStream_t s)
{
    if (b.nlev <= 0 || njob <= 0) return MHX_OK;
    if (njob > MAX_SYN_JOBS) return fail(MHX_E_INVALID, "too many synthesis jobs in one launch");
    if (int rc = ensure_p_tables(const_cast<Plan *>(p))) return rc;
    SynArgs a;
    int np = 0;
    for (int i = 0; i < njob; ++i) {
        a.job[i] = jobs[i];
        switch (jobs[i].kind) {
        case SYN_SCAL: np = np < 1 ? 1 : np; break;
        case SYN_GRAD: case SYN_SG: case SYN_SPHTOR: np = np < 2 ? 2 : np; break;
        case SYN_QST: np = 3; break;
        default: return fail(MHX_E_INVALID, "unknown synthesis kind");
        }
    }
    a.njob = njob;
    a.nlev = b.nlev;
    a.src_ld = b.src_ld;
    a.fout_ld = b.fout_ld;
    a.lcut = b.lcut;
    a.or2 = b.or2;
    a.tab = p->d_synx;
    a.off = p->d_synx_off;
    a.crec = p->d_crec64;
    a.lstart = p->d_lstart;
    a.osin2 = p->d_osin2;
    a.l_max = p->l_max;
    a.minc = p->minc;
    a.n_m = p->n_m;
    a.nh = p->nh;
    a.n_theta = p->n_theta;
    a.nt16 = p->nt16;
    a.ng = (b.nlev + LEV_GROUP - 1) / LEV_GROUP;
    a.gz = (p->nt16 + 11) / 12;
    const int tpw = (p->nt16 + 4 * a.gz - 1) / (4 * a.gz);
    const unsigned grid = (unsigned)((p->n_m + 7) / 8 * 8 * njob * a.ng * a.gz);
    switch (np) {
    case 1: return launch_syn_np<1>(a, tpw, grid, s);
    case 2: return launch_syn_np<2>(a, tpw, grid, s);
    default: return launch_syn_np<3>(a, tpw, grid, s);
    }
}

int launch_ana(const Plan *p, const AnaJob &job, hipStream_t s)
{
    if (int rc = ensure_fp64_tables(const_cast<Plan *>(p))) return rc;
    if (job.nlev <= 0) return MHX_OK;
    AnaArgs a;
    a.job = job;
    a.aP = p->d_ana_wP;
    a.adP = p->d_ana_wdP;
    a.off = p->d_ana_off;
    a.lstart = p->d_lstart;
    a.l_max = p->l_max;
    a.m_max = p->m_max;
    a.minc = p->minc;
    a.n_m = p->n_m;
    a.nh = p->nh;
    a.n_theta = p->n_theta;
    a.nq4 = p->nq4;
    int ntile0 = ((p->l_max) / 2 + 1 + 15) / 16;  // pair tiles at m = 0
    dim3 grid((unsigned)(p->n_m * ((job.nlev + LEV_GROUP - 1) / LEV_GROUP) * ((ntile0 + 3) / 4)));
    switch (job.kind) {
    case ANA_SH: k_ana<ANA_SH><<<grid, WG, 0, s>>>(a); break;
    case ANA_SPHTOR: k_ana<ANA_SPHTOR><<<grid, WG, 0, s>>>(a); break;
    case ANA_QST: k_ana<ANA_QST><<<grid, WG, 0, s>>>(a); break;
    default: return fail(MHX_E_INVALID, "unknown analysis kind");
    }
    MHX_HIP_CHECK(hipGetLastError());
    return MHX_OK;
}

}  // namespace mhx
