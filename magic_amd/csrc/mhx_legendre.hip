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
// table.  Again only wP is contracted, G_l = sum_theta wP_l v for l <= l_max +
// 1 and v = f, vt, vp; the dP products follow from the same identity,
//     sum_theta wdP_l v = l c_{l+1} G_{l+1} - (l+1) c_l G_{l-1}.
#include "mhx_internal.h"

#include <algorithm>

namespace mhx {

namespace {

constexpr int WG = 256;
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
    double or2_all;
    int l_max, minc, n_m, nh, n_theta, nt16;
    short lc_arg[LEV_ARG];  // lcut null: the levels' cut-offs
};

struct AnaArgs {
    AnaJob job[MAX_ANA_JOBS];
    int njob, nlev, ng, gz;
    size_t fin_ld, out_ld;
    const int *lcut;
    const double *tab;     // 2 pi w P_lm, l <= l_max + 1 (layout: mhx_tables.hip)
    const size_t *off;
    const double *crec;
    const int *lstart;
    int l_max, m_max, minc, n_m, nh, n_theta, nq8;
    int erows;             // rows of one epilogue area in LDS
    short lc_arg[LEV_ARG];
};

template <class Args> __device__ __forceinline__ int lcut_of(const Args &a, int lev)
{
    return a.lcut ? a.lcut[lev] : (int)a.lc_arg[lev];
}

// the cut-off (at most l_max) of level lev0 + lv, -1 past the levels, and the
// largest of the group of 8 levels from lev0: one load, lane i holding level i of
// eight, where eight scalar loads held up the head of every workgroup
template <class Args> __device__ __forceinline__ int group_cut(const Args &a, int lev0, int lv, int lane, int &lcm)
{
    const int v = min(lcut_of(a, min(lev0 + (lane & 7), a.nlev - 1)), a.l_max);
    const int own = __shfl(v, lv);
    int x = max(v, __shfl_xor(v, 1));
    x = max(x, __shfl_xor(x, 2));
    lcm = __builtin_amdgcn_readfirstlane(max(x, __shfl_xor(x, 4)));
    return lev0 + lv < a.nlev ? own : -1;
}

// a batch's cut-offs into the arguments
template <class Args, class Batch> int set_lcut(Args &a, const Batch &b)
{
    a.lcut = b.lcut;
    if (b.lcut) return MHX_OK;
    if (!b.lcut_host || b.nlev > LEV_ARG) return fail(MHX_E_INVALID, "levels of a Legendre launch without cut-offs");
    for (int i = 0; i < b.nlev; ++i) a.lc_arg[i] = (short)b.lcut_host[i];
    return MHX_OK;
}

// v_mfma_f64_16x16x4f64 operands: A lane l holds A[l % 16][l / 16], B lane l
// holds B[l / 16][l % 16]; D element j of lane l is D[l / 16 + 4 j][l % 16].
__device__ inline d4 mfma64(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// x of the lane before (wave_shr:1), after (wave_shl:1) and of the other lane of
// the pair (quad_perm 1 0 3 2), by data-parallel moves: no LDS permutation
template <int CTRL> __device__ __forceinline__ double dpp(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
constexpr int DPP_PREV = 0x138, DPP_NEXT = 0x130, DPP_PAIR = 0xb1;

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
//
// No unit is saturated: at l_max = 255 x 97 levels the matrix pipe is busy 42 % of
// the cycles, the vector-memory data path 68 % (53 % waiting for the cache), and at
// two waves per SIMD (144 accumulator registers) a chunk's loads, column forming and
// products add up more than they overlap (waves wait 39 % of their time, and 43 % on
// instructions in flight).  QST at that size: 0.65 ms with
// five products, one launch per field and 8-byte table loads; 0.31 on P alone;
// 0.28 with the neighbour exchange by data-parallel moves; 0.25 (29 of 72.8
// TFLOP/s) with every load unconditional and the cut-offs in one load (same box:
// 0.264 before).  Level groups in one workgroup one after the other, the next one's
// first chunk formed during the last, gave 0.5 % of a step more and cost the small
// ones (64 x 33 levels, fourfold symmetry) 5 %.
// Not faster: four fragments in flight, smaller theta groups; six waves of two
// tiles per workgroup at three waves per SIMD spill (0.65 ms).
template <int TPW, int KIND>
__device__ __forceinline__ void syn_body(const SynArgs &a, const SynJob &ajob, int mc, int lev0, int gz, double *sB)
{
    constexpr int NP = syn_np<KIND>();
    constexpr bool QST = KIND == SYN_QST, TWO = KIND == SYN_QST || KIND == SYN_SPHTOR;
    constexpr int CS = QST ? 1 : 0, CT = QST ? 2 : 1;  // fields S (or x) and T
    const SynJob job = ajob;  // in scalar registers, not read again at each use
    const int m = mc * a.minc, L = a.l_max;
    const double dm = (double)m;
    const int tid = threadIdx.x, lane = tid & 63;
    const int tt0 = gz * 4 + __builtin_amdgcn_readfirstlane(tid >> 6), tstep = 4 * a.gz;
    const int l0 = a.lstart[mc];

    // the thread's (level, degree) of a chunk
    const int lv = tid >> 5, j = tid & 31, lev = lev0 + lv;
    int lcm;  // largest cut-off of the level group
    const int lc = group_cut(a, lev0, lv, lane, lcm);
    const int nrow = max(lcm + 2 - m, 0);  // degrees m .. lcm + 1
    const int nch = (nrow + 31) >> 5;
    const int nquad[2] = {((nrow + 1) / 2 + 3) >> 2, (nrow / 2 + 3) >> 2};
    const int levc = min(lev, a.nlev - 1);
    const double or2 = a.or2 ? a.or2[levc] : a.or2_all;
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
                double2 lo = make_double2(dpp<DPP_PREV>(x.x), dpp<DPP_PREV>(x.y));
                double2 hi = make_double2(dpp<DPP_NEXT>(x.x), dpp<DPP_NEXT>(x.y));
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

    // no load of the sources or tables stands under a branch, here on the cut-offs
    // (whose own load it would wait for) or below on what is left to do: a load
    // under a branch makes the next wait cover every load in flight
    load(0);
    load_A(fa[0], 0, 0);
    if (nch > 0) build(0, 0);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        const int buf = c & 1;
        load(min(c + 1, nch - 1));
        if (act) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int par = k & 1, pair = k >> 1;
                // the next step's fragments
                load_A(fa[1 - par], 2 * c + ((k + 1) >> 1), 1 - par);
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
    // the odd lane the southern one: 128-byte lines of the theta-blocked F
    const int col = lane & 15, elev = lev0 + (col >> 1), odd = col & 1;
    if (elev >= a.nlev) return;
    const size_t cstride = f2_comp(a.n_m, a.n_theta);
    double2 *fo = reinterpret_cast<double2 *>(job.fout) + (size_t)elev * a.fout_ld + (size_t)mc * 8 + odd;
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
                const double other = dpp<DPP_PAIR>(odd ? n : so);
                double2 v = odd ? make_double2(other, so) : make_double2(n, other);
                if (job.row_scale) v = make_double2(sc * v.x, sc * v.y);
                auto store = [&](int o, double2 w) {
                    if (ok) fo[job.out_comp[o] * cstride + (size_t)(th >> 2) * (a.n_m * 8) + (2 * th & 7)] = w;
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
template <int KIND> constexpr int ana_np() { return KIND == ANA_QST ? 3 : (KIND == ANA_SH ? 1 : 2); }

// B chunk in LDS: 32 northern theta, [column][Sym/Anti][pair of quads] blocks
// of 64 lanes x 2 quads, padded as the synthesis' blocks
constexpr int AB_PAIR = 132, AB_SA = 4 * AB_PAIR, AB_COL = 2 * AB_SA;
// epilogue rows [l][8 levels x re/im], padded against the column reads
constexpr int AE_ROW = 18;

// One workgroup: one job, one order m (index mc), 8 radial levels from lev0,
// and up to 2 TPW pairs of l tiles (32 consecutive l: 16 of each parity);
// waves 0 and 1 take the even-parity tiles, 2 and 3 the odd ones.  Per chunk
// of 32 northern theta a thread owns one (level, theta): it loads the north
// and south rows (32 consecutive bytes of the theta-blocked F2) a chunk
// ahead, forms Sym and Anti and writes them to the other half of the LDS
// buffer; table fragments are loaded a step (8 theta) ahead.  Where the
// order's tiles need more than one workgroup they overlap by one tile pair,
// whose rows each workgroup's edge needs as neighbours.
//
// No unit is saturated: matrix pipe 41 % busy, data path 71 % (45 % waiting for the
// cache, for 3 n_theta n_m 16 bytes of F2 per level and component and the table), as in
// the synthesis.  QST at l_max = 255 x 97 levels: 0.72 ms with five sums, 16-byte gathers
// one per (theta, m) and 16-byte stores; 0.32 on wP alone with whole lines read and
// 512-byte runs stored; 0.28 (26 of 72.8 TFLOP/s) with every load unconditional.
template <int TPW, int KIND>
__device__ __forceinline__ void ana_body(const AnaArgs &a, const AnaJob &job, int mc, int lev0, int gz, double *sB)
{
    constexpr int NP = ana_np<KIND>();
    constexpr int BUF = NP * AB_COL;
    const int m = mc * a.minc, L = a.l_max;
    const double dm = (double)m;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int nt = (L + 2 - m + 31) >> 5;                // tile pairs of this order (l <= l_max + 1)
    const int zb = gz * (2 * TPW - 1);                   // first tile pair of this workgroup
    if (gz > 0 && zb + 1 >= nt) return;                  // covered by the workgroup before
    const int par = wave >> 1, t0 = zb + (wave & 1);     // this wave's tiles: t0 + 2 s
    const int l0 = a.lstart[mc];

    const int lv = tid >> 5, j = tid & 31, lev = lev0 + lv;
    int lcm;
    const int lc = group_cut(a, lev0, lv, lane, lcm);
    const bool lev_on = lev < a.nlev && m <= min(lc, a.m_max);
    const int nch = m <= min(lcm, a.m_max) ? (a.nh + 31) >> 5 : 0;

    // F2[lev][comp][theta/8][m][theta%8]
    const int levc = min(lev, a.nlev - 1);
    const double2 *fin = reinterpret_cast<const double2 *>(job.fin) + (size_t)levc * a.fin_ld;
    const size_t cstride = (size_t)((a.n_theta + 7) / 8) * a.n_m * 8;
    double2 xn[NP], xs[NP];
    auto load = [&](int c) {
        const int th = min(32 * c + j, a.nh - 1);
        const double2 *f = fin + ((size_t)(th >> 2) * a.n_m + mc) * 8 + (2 * th & 7);
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            xn[k] = f[(size_t)job.in_comp[k] * cstride];
            xs[k] = f[(size_t)job.in_comp[k] * cstride + 1];
        }
    };
    auto build = [&](int c, int buf) {
        const bool ok = lev_on && 32 * c + j < a.nh;
        double *b = sB + buf * BUF + (j >> 3) * AB_PAIR + ((j & 3) * 16 + 2 * lv) * 2 + ((j >> 2) & 1);
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            const double2 n = ok ? xn[k] : make_double2(0.0, 0.0), so = ok ? xs[k] : make_double2(0.0, 0.0);
            double *b0 = b + k * AB_COL, *b1 = b0 + AB_SA;
            b0[0] = n.x + so.x;
            b0[2] = n.y + so.y;
            b1[0] = n.x - so.x;
            b1[2] = n.y - so.y;
        }
    };

    d4 acc[TPW][NP];
#pragma unroll
    for (int s = 0; s < TPW; ++s)
#pragma unroll
        for (int k = 0; k < NP; ++k) acc[s][k] = d4{0.0, 0.0, 0.0, 0.0};
    const double2 *tab = reinterpret_cast<const double2 *>(a.tab + a.off[2 * mc + par]) + lane;
    const int nmine = t0 < nt ? min(TPW, (nt - t0 + 1) >> 1) : 0;  // tiles of this wave
    const int npair = a.nq8;
    auto load_A = [&](double2 *f, int p) {
        const double2 *t = tab + (size_t)min(p, npair - 1) * 64;
#pragma unroll
        for (int s = 0; s < TPW; ++s) f[s] = t[(size_t)min(t0 + 2 * s, nt - 1) * (npair * 64)];
    };
    double2 fa[2][TPW];

    load(0);
    load_A(fa[0], 0);
    if (nch > 0) build(0, 0);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        const int buf = c & 1;
        load(min(c + 1, nch - 1));
        if (nmine > 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int p = 4 * c + k;
                load_A(fa[(k + 1) & 1], p + 1);
                if (p < npair) {
                    double2 b[NP];
                    const double *sb = sB + buf * BUF + par * AB_SA + k * AB_PAIR + 2 * lane;
#pragma unroll
                    for (int q = 0; q < NP; ++q) b[q] = *reinterpret_cast<const double2 *>(sb + q * AB_COL);
#pragma unroll
                    for (int s = 0; s < TPW; ++s) {
                        if (s >= nmine) break;
#pragma unroll
                        for (int q = 0; q < NP; ++q) acc[s][q] = mfma64(fa[k & 1][s].x, b[q].x, acc[s][q]);
#pragma unroll
                        for (int q = 0; q < NP; ++q) acc[s][q] = mfma64(fa[k & 1][s].y, b[q].y, acc[s][q]);
                    }
                }
            }
        }
        if (c + 1 < nch) build(c + 1, buf ^ 1);
        __syncthreads();
    }

    // epilogue through LDS: rows of consecutive l (both parities), then one
    // (level, l) per thread and round, consecutive l by consecutive lanes
    const int nrow = min(32 * 2 * TPW, L + 2 - m - 32 * zb);  // rows held: l = m + 32 zb + row
    auto stage = [&](int area, int k) {
        const int col = lane & 15;
#pragma unroll
        for (int s = 0; s < TPW; ++s) {
            if (s >= nmine) break;
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const int row = 32 * (t0 + 2 * s - zb) + par + 2 * ((lane >> 4) + 4 * jj);
                if (row < nrow) sB[area * a.erows * AE_ROW + row * AE_ROW + col] = acc[s][k][jj];
            }
        }
    };
    auto at = [&](int area, int row) {
        return *reinterpret_cast<const double2 *>(sB + area * a.erows * AE_ROW + row * AE_ROW + 2 * lv);
    };
    const int lo = gz > 0 ? 31 : 0;  // rows written: the one before the edge belongs to the workgroup before
    const int zn = zb + 2 * TPW - 1;
    const int hi = nt > zn + 1 ? 32 * (zn + 1 - zb) - 1 : L + 1 - m - 32 * zb;
    double2 *const *outs = reinterpret_cast<double2 *const *>(job.out);
    const size_t o0 = (size_t)lev * a.out_ld + (size_t)(l0 + 32 * zb);
    auto kept = [&](int l) { return lev_on && l <= lc; };
    if constexpr (KIND != ANA_SH) {
        stage(0, NP - 2);  // G of vt
        stage(1, NP - 1);  // G of vp
        __syncthreads();
        double2 *oS = outs[NP - 2], *oT = outs[NP - 1];
        for (int row = lo + ((j - lo) & 31); row < hi; row += 32) {
            const int l = m + 32 * zb + row;
            const double dl = (double)l;
            const double *cr = a.crec + l0 + 2 * mc + l - m;
            const double fp = dl * cr[1], fm = (dl + 1.0) * cr[0];
            const double2 z = make_double2(0.0, 0.0);
            const double2 tm = row > 0 ? at(0, row - 1) : z, tp = at(0, row + 1), tc = at(0, row);
            const double2 pm = row > 0 ? at(1, row - 1) : z, pp = at(1, row + 1), pc = at(1, row);
            const double rl = dl * (dl + 1.0);
            // S = (dP vt - i m P vp) / l(l+1), T = (-dP vp - i m P vt) / l(l+1)
            double2 S = make_double2(fp * tp.x - fm * tm.x + dm * pc.y, fp * tp.y - fm * tm.y - dm * pc.x);
            double2 T = make_double2(fm * pm.x - fp * pp.x + dm * tc.y, fm * pm.y - fp * pp.y - dm * tc.x);
            if (l > 0) {
                S = make_double2(S.x / rl, S.y / rl);
                T = make_double2(T.x / rl, T.y / rl);
            }
            if (lev < a.nlev) {
                oS[o0 + row] = kept(l) ? S : z;
                oT[o0 + row] = kept(l) ? T : z;
            }
        }
        __syncthreads();
    }
    if constexpr (KIND != ANA_SPHTOR) {
        stage(0, 0);
        __syncthreads();
        for (int row = lo + ((j - lo) & 31); row < hi; row += 32)
            if (lev < a.nlev) outs[0][o0 + row] = kept(m + 32 * zb + row) ? at(0, row) : make_double2(0.0, 0.0);
    }
}

// the jobs of one launch: kinds of at most NP columns; blocks ordered as the
// synthesis'
template <int TPW, int NP>
__global__ __launch_bounds__(WG, 2) void k_ana(AnaArgs a)
{
    extern __shared__ __attribute__((aligned(16))) double sB[];
    const int inner = a.njob * a.gz * a.ng;
    const int mc = (int)(blockIdx.x >> 3) / inner * 8 + (int)(blockIdx.x & 7);
    if (mc >= a.n_m) return;
    int r = (int)(blockIdx.x >> 3) % inner;
    const AnaJob &job = a.job[r % a.njob];
    r /= a.njob;
    const int gz = r % a.gz, lev0 = r / a.gz * LEV_GROUP;
    switch (job.kind) {
    case ANA_SH: ana_body<TPW, ANA_SH>(a, job, mc, lev0, gz, sB); break;
    case ANA_SPHTOR: if constexpr (NP > 1) ana_body<TPW, ANA_SPHTOR>(a, job, mc, lev0, gz, sB); break;
    case ANA_QST: if constexpr (NP > 2) ana_body<TPW, ANA_QST>(a, job, mc, lev0, gz, sB); break;
    default: break;
    }
}

template <int TPW, int NP>
int launch_ana_t(const AnaArgs &a, unsigned grid, hipStream_t s)
{
    // the two B buffers, reused by the epilogue's areas (vt and vp; f alone
    // in a scalar launch)
    const size_t shm = std::max((size_t)2 * NP * AB_COL, (size_t)(NP > 1 ? 2 : 1) * a.erows * AE_ROW) * sizeof(double);
    if (int rc = allow_lds((const void *)k_ana<TPW, NP>, shm)) return rc;
    k_ana<TPW, NP><<<grid, WG, shm, s>>>(a);
    MHX_HIP_CHECK(hipGetLastError());
    return MHX_OK;
}

template <int NP>
int launch_ana_np(const AnaArgs &a, int tpw, unsigned grid, hipStream_t s)
{
    switch (tpw) {
    case 1: return launch_ana_t<1, NP>(a, grid, s);
    case 3: return launch_ana_t<3, NP>(a, grid, s);
    case 4: return launch_ana_t<4, NP>(a, grid, s);
    default: return launch_ana_t<5, NP>(a, grid, s);
    }
}

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
    if (int rc = set_lcut(a, b)) return rc;
    a.or2 = b.or2;
    a.or2_all = b.or2_all;
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
    // theta tiles: 12 per workgroup at most (three per wave: 144 accumulator
    // registers of the 256 at two waves per SIMD), spread evenly over the groups
    // and their waves
    a.gz = (p->nt16 + 11) / 12;
    const int tpw = (p->nt16 + 4 * a.gz - 1) / (4 * a.gz);
    const unsigned grid = (unsigned)((p->n_m + 7) / 8 * 8 * njob * a.ng * a.gz);
    switch (np) {
    case 1: return launch_syn_np<1>(a, tpw, grid, s);
    case 2: return launch_syn_np<2>(a, tpw, grid, s);
    default: return launch_syn_np<3>(a, tpw, grid, s);
    }
}

int launch_ana(const Plan *p, const AnaJob *jobs, int njob, const AnaBatch &b, hipStream_t s)
{
    if (b.nlev <= 0 || njob <= 0) return MHX_OK;
    if (njob > MAX_ANA_JOBS) return fail(MHX_E_INVALID, "too many analysis jobs in one launch");
    if (int rc = ensure_p_tables(const_cast<Plan *>(p))) return rc;
    AnaArgs a;
    int np = 0;
    for (int i = 0; i < njob; ++i) {
        a.job[i] = jobs[i];
        switch (jobs[i].kind) {
        case ANA_SH: np = np < 1 ? 1 : np; break;
        case ANA_SPHTOR: np = np < 2 ? 2 : np; break;
        case ANA_QST: np = 3; break;
        default: return fail(MHX_E_INVALID, "unknown analysis kind");
        }
    }
    a.njob = njob;
    a.nlev = b.nlev;
    a.fin_ld = b.fin_ld;
    a.out_ld = b.out_ld;
    if (int rc = set_lcut(a, b)) return rc;
    a.tab = p->d_anax;
    a.off = p->d_anax_off;
    a.crec = p->d_crec64;
    a.lstart = p->d_lstart;
    a.l_max = p->l_max;
    a.m_max = p->m_max;
    a.minc = p->minc;
    a.n_m = p->n_m;
    a.nh = p->nh;
    a.n_theta = p->n_theta;
    a.nq8 = (p->nh + 7) / 8;
    a.ng = (b.nlev + LEV_GROUP - 1) / LEV_GROUP;
    // tiles per wave: all of m = 0's tile pairs in one workgroup where five
    // per wave hold them (120 accumulator registers) and the epilogue's areas,
    // 288 (l_max + 2) bytes, leave room for a second workgroup on the CU; else
    // groups of eight pairs, 74 KB (groups of ten, 92 KB and one workgroup per CU,
    // took 5.37 / 6.92 / 4.57 ms per step at l_max = 341 x 40, 426 x 20, 511 x 12
    // levels, eight 5.17 / 6.70 / 4.33, six 5.22 / 6.75 / 4.41)
    const int nt = (p->l_max + 2 + 31) / 32;
    const int tpw = nt <= 2 ? 1 : (nt <= 6 ? 3 : (p->l_max + 2 <= 284 ? 5 : 4));
    a.erows = std::min(64 * tpw, p->l_max + 2);
    a.gz = nt <= 2 * tpw ? 1 : (nt - 1 + 2 * tpw - 2) / (2 * tpw - 1);
    const unsigned grid = (unsigned)((p->n_m + 7) / 8 * 8 * njob * a.ng * a.gz);
    switch (np) {
    case 1: return launch_ana_np<1>(a, tpw, grid, s);
    case 2: return launch_ana_np<2>(a, tpw, grid, s);
    default: return launch_ana_np<3>(a, tpw, grid, s);
    }
}

}  // namespace mhx
