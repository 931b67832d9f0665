// k_sweep16.hip -- LU-SGS hyperplane sweeps for nY > 1 on 16-row strips
// (the species-extended calc_next_step_implicit of LU-SGS/2d/
// time_lusgs_viscous.f90:24-63, NR/2d/time_NR_viscous.f90, precon/2d/ and
// preconLU-SGS/2d/time_precon_viscous.f90; dual time with its S scaling keeps
// the row-per-lane sweeps of k_implicit.hip).
//
// A workgroup owns 16 rows of a block and has C = ceil(dq/4) compute waves: the
// 16 x dq unknowns of a strip occupy one lane each.  The i-neighbour's
// contribution stays in the lane, the j-neighbour's comes from the row above or
// below by a 4-lane DPP shift or, at the edges of the four-row groups, through
// an LDS ring, and from the neighbouring strip through a hand-off row: the
// producer stores each column's value into a slot that holds a NaN sentinel, the
// consumer polls the slots (no flags, so no wave waits for its own stores).
// Two families: with the products A x in closed form (LU-SGS, NR), and over
// stored matrices (the preconditioned schemes).
#include "shcfd_device.h"
#include "shcfd_kernels.h"

namespace shcfd {

namespace {

constexpr int HO = 24; // hand-off column offset: entry (col + HO) dq + k, col >= -HO
constexpr unsigned long long SENT16 = 0x7FF4DEADBEEFCAFEULL;  // never produced by arithmetic

__device__ inline bool is_sent16(double x) { return (unsigned long long)__double_as_longlong(x) == SENT16; }

// workgroup barrier after this wave's LDS writes have completed; global
// loads in flight are not waited for (the prefetched operator rows)
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// per-lane inputs of one step of the sweeps over stored matrices: the lane's
// rows of the two matrices, the cell values of its row and the lane's
// component of the right-hand side
template <int DQ>
struct StepIn {
    double a[DQ], b[DQ];
    double al, fi, fj, r;
};

// the pair-interleaved operator rows and scalars of one step: `base` is the
// lane's pair 0 of that step
template <int DQ>
__device__ inline void load_ops(const double* __restrict__ base, StepIn<DQ>& in) {
    constexpr int dq2 = DQ + 2;
#pragma unroll
    for (int p = 0; p < dq2; p++) {
        const double2 v = *reinterpret_cast<const double2*>(base + 128LL * p);
        const int e0 = 2 * p, e1 = 2 * p + 1;
        double* dst0 = e0 < DQ ? &in.a[e0] : (e0 < 2 * DQ ? &in.b[e0 - DQ] : (e0 == 2 * DQ ? &in.al : &in.fj));
        *dst0 = v.x;
        if (e1 < DQ) in.a[e1] = v.y;
        else if (e1 < 2 * DQ) in.b[e1 - DQ] = v.y;
        else if (e1 == 2 * DQ + 1) in.fi = v.y;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Jacobian-free quad-row sweeps: LU-SGS and NR at nY > 1.
//
// The split Jacobians of these schemes are A+- = Atilde/2 +- (nuA/2) I with
// Atilde = n_x A + n_y B (LU-SGS/2d/sch_lusgs.raw.f90:112-129; NR likewise),
// A and B the species-extended Euler flux Jacobians of :39-110.  Their
// product with x = (x_k (k < nY), X, V, E) follows in closed form from those
// entries:
//     (Atilde x)_k    = U x_k + Y_k e                    (k < nY)
//     (Atilde x)_nY   = U X + u e + n_x dp
//     (Atilde x)_nY+1 = U V + v e + n_y dp
//     (Atilde x)_nY+2 = U E + H e + U dp
// with U = n_x u + n_y v, s = sum_k x_k, e = n_x (X - u s) + n_y (V - v s) and
// dp = sum_k DHi_k x_k + (gamma-1) ((u^2+v^2)/2 s - u X - v V + E).
// Each term is thus a diagonal part and three dot products with x: eA and eB
// (e with n = dsci alpha n_i / 2 and dscj alpha n_j / 2) and dp.  alpha is
// folded in as in k_fast.hip: the forward sweep computes
// v = R + GA v(i-1) + GB v(j-1) with GA = dsci alpha A+, the backward sweep
// z = v - (HA z(i+1) + HB z(j+1)), and dq = alpha z.  The record of a cell
// holds the coefficients of the dot products and of the terms per component.
//
// Layout and schedule.  Lane 4r + c of compute wave w holds component 4w + c
// of row r; the groups of four rows run one step apart (row r works on column
// t - r - floor(r/4) + 1 at step t), so that within a group the hop to the
// next row is one DPP row shift and between groups the value crosses through
// an LDS ring.  The records are stored by (strip, step, wave, lane): a step's
// loads and its store share one address, each is one run of consecutive bytes,
// and slots of no cell hold zeros (no masks); v and z replace R in place.  A
// step has one workgroup barrier: before it each quad puts its partial sums of
// the three dot products into LDS (lane c the c-th, from a transposing
// reduction), after it lane c adds the waves' and the quad exchanges the
// totals.  Two more waves move the hand-off: wave C polls the neighbour
// strip's row, wave C + 1 stores the strip's own, so a compute wave waits for
// no store and no other strip except at the barrier.
//
// Bound by the chain of one step, 240 ns: 17 FP64 operations (about 8 cycles
// each from one wave), the DPP moves and two LDS round trips, beside 5 loads of
// 64 x 16 bytes per wave; then by the hand-off, a strip running 18 steps plus
// about 4 us behind its neighbour.  Measured at nY = 9: 571 us forward and
// 542 us backward on 1024 x 512 (before 1285 and 986), 108 and 109 us on
// 223 x 99 (before 200 and 210); forming the records and the right-hand side
// in one pass, 195 us on 1024 x 512 (before, cell data 104 us and right-hand
// side 78 us in two), the update 56 us.  Before, dq was read and written in
// place: 64 lanes in 64 different cache lines per access, with the hand-off
// polls and stores in the same in-order vmcnt.  Looking at the hand-off more
// often than when a step needs it costs more than it gains, since a look waits
// for its load and the barrier for the look: 612 us forward with a look every
// second step.
// ---------------------------------------------------------------------------

namespace {
constexpr int JU = 8;          // steps per unrolled round; prefetch runs JU - 1 steps ahead
constexpr int JRS = 8;         // ring slots
constexpr int JRIN = 4;        // ring lanes of the neighbour strip's components

// Cell records by (strip, step, wave), in bytes: (c1, cP) and R per lane, the
// sweeps' diagonal pairs per row, (cA, cB) per row in waves of species alone,
// per lane in the others, which also hold (pA, pB); c1 = Y_k, u, v or H, cA,
// cB and cP the dot products' coefficients of the component, pA and pB the
// factors of dp
constexpr int JO_R = 1024, JO_LF = 1536, JO_LB = 1792, JO_E = 2048, JO_P = 3072;
template <int NY>
constexpr int jrec_step() { return jrec_off(NY, (NY + 6) / 4); }
static_assert(JO_E + 16 * 16 == JREC_S && JO_P + 16 * 64 == JREC_M && JU - 1 <= JPAD, "cell records");

template <int CTRL>
__device__ inline double quad_perm(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, true);
    hi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
constexpr int QP_X1 = 1 | (0 << 2) | (3 << 4) | (2 << 6), QP_X2 = 2 | (3 << 2) | (0 << 4) | (1 << 6);
// sums over the four lanes of each quad: of f0 in lane 0, f1 in lane 1, f2 in
// lanes 2 and 3; odd: lane 1 or 3, up: lane 2 or 3
__device__ inline double quad_sums(double f0, double f1, double f2, bool odd, bool up) {
    const double g01 = (odd ? f1 : f0) + quad_perm<QP_X1>(odd ? f0 : f1);
    const double g2 = f2 + quad_perm<QP_X1>(f2);
    return (up ? g2 : g01) + quad_perm<QP_X2>(up ? g01 : g2);
}

// Buffer views of the hand-off rows: the hardware's range check returns zero
// for loads beyond a row and drops stores there
typedef unsigned int jv_u32x2 __attribute__((ext_vector_type(2)));
constexpr int JV_DROP = 0x7FFFFF00;
constexpr int JV_AGENT = 16;   // sc1: device-coherent access
__device__ inline __amdgpu_buffer_rsrc_t jview(const void* base, long long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ inline double jv_ld(__amdgpu_buffer_rsrc_t r, int voff) {
    const jv_u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, JV_AGENT);
    return __longlong_as_double((long long)(((unsigned long long)v.y << 32) | v.x));
}
__device__ inline void jv_st(__amdgpu_buffer_rsrc_t r, double x, int voff) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(x);
    const jv_u32x2 v = {(unsigned)a, (unsigned)(a >> 32)};
    __builtin_amdgcn_raw_buffer_store_b64(v, r, voff, 0, JV_AGENT);
}
__device__ inline void jbarrier() { asm volatile("s_barrier" ::: "memory"); }

template <int NY>
struct JLds {
    static constexpr int C = (NY + 6) / 4;
    double ring[JRS][C * 64];  // slot t % JRS: the terms the edge rows take at step t
    double f[2][16][3][(C + 1) / 2 * 2];  // the waves' partial sums of each row's dot products
};

// hand-off rows of both sweeps: the sentinel for the columns 1..ni of the
// strip's block, zero elsewhere; over the whole grid
__device__ inline void refill_hand(const DevCtx& d, const Strip16* strips, int nstrips, double* hand, long long hstride,
                                   int dq) {
    const long long n = 2LL * (nstrips + 1) * hstride;
    const double sv = __longlong_as_double((long long)SENT16);
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256) {
        const int row = (int)((e / hstride) % (nstrips + 1));
        const long long col = (e % hstride) / dq - HO;
        const bool live = row < nstrips && col >= 1 && col <= d.blk[strips[row].b].ni;
        hand[e] = live ? sv : 0.0;
    }
}

// cell of (strip, step t, row r)
__device__ inline bool jslot_cell(const Strip16& S, const DevBlock& B, int t, int r, int& i, int& j) {
    i = t - r - JGD * (r >> 2) + 1;
    j = S.j0 + r;
    return i >= 1 && i <= B.ni && j <= B.nj;
}
}  // namespace

// The right-hand side of the update (k_rhs) and the cell data of the sweeps in
// one pass: workgroup = 16 steps x 16 rows of one strip, a wave taking 4 rows x
// 16 steps so that each load of a cell field reads four runs of 16 cells.
// Also stores alpha, as set_ABpm does, and refills the hand-off rows.
template <int NY>
__global__ void __launch_bounds__(256) k_rhs_jd16(DevCtx d, const Strip16* strips, int nstrips, int nsteps16,
                                                  int dqdt_inline, char* recs, double* hand, long long hstride) {
    using D = Dims<NY>;
    constexpr int dq = D::dq, C = (dq + 3) / 4, W0 = NY / 4;
    refill_hand(d, strips, nstrips, hand, hstride, D::dq);
    const int s = (int)blockIdx.x / nsteps16;
    const Strip16 S = strips[s];
    const int t = 16 * ((int)blockIdx.x % nsteps16) + (int)(threadIdx.x & 15), r = (int)(threadIdx.x >> 4);
    const DevBlock B = d.blk[S.b];
    int i, j;
    char* rec = recs + (JPAD + S.base + t) * jrec_step<NY>();
    if (!jslot_cell(S, B, t, r, i, j)) {
        if (t < (B.ni + JSPAN + JU - 1) / JU * JU) {  // the sweeps left their v and z here
#pragma unroll
            for (int w = 0; w < C; w++) {
                double2* R = reinterpret_cast<double2*>(rec + jrec_off(NY, w) + JO_R) + 2 * r;
                R[0] = R[1] = make_double2(0.0, 0.0);
            }
        }
        return;
    }
    const long long c = cidx(B, i, j);
    double bal[dq], x[dq];
    flux_balance<NY>(d, B, c, bal);
    rhs_of_cell<NY>(d, c, bal, dqdt_inline != 0, [](int) { return 0.0; }, [](int) { return 0.0; }, []() { return 0.0; }, x);
    // the scalars of cell_jacobian for the non-preconditioned schemes
    // (sch_lusgs.raw.f90:26-38, :131-133; sch_NR.raw.f90:134-136)
    const double rho = FLD(d, SHCFD_F_W, 0, c), u = FLD(d, SHCFD_F_W, IW_U, c), v = FLD(d, SHCFD_F_W, IW_V, c);
    const double p = FLD(d, SHCFD_F_W, IW_P, c), gamm = FLD(d, SHCFD_F_W, D::ig, c), H = FLD(d, SHCFD_F_W, D::ih, c);
    const double cs = sqrt((gamm * p) / rho);
    const double n1a = FLD(d, SHCFD_F_VNCI, 0, c), n2a = FLD(d, SHCFD_F_VNCI, 1, c);
    const double n1b = FLD(d, SHCFD_F_VNCJ, 0, c), n2b = FLD(d, SHCFD_F_VNCJ, 1, c);
    const double unA = (n1a * u) + (n2a * v), unB = (n1b * u) + (n2b * v);
    const double nuA = fabs(unA) + cs, nuB = fabs(unB) + cs;
    const double dsci = FLD(d, SHCFD_F_DSCI, 0, c), dscj = FLD(d, SHCFD_F_DSCJ, 0, c);
    const double vol = FLD(d, SHCFD_F_VOL, 0, c);
    const double dtv = (d.p.time_step == 0) ? d.scal[SCAL_DT_GRBL] : FLD(d, SHCFD_F_DT, 0, c);
    const double alpha = (d.p.scheme == SHCFD_SCHEME_NR)
                             ? 1.0 / ((((3.0 * vol) / (2.0 * dtv)) + (dsci * nuA)) + (dscj * nuB))
                             : 1.0 / (((vol / dtv) + (dsci * nuA)) + (dscj * nuB));
    FLD(d, SHCFD_F_ALPHA, 0, c) = alpha;
    const double fa = (0.5 * dsci) * alpha, fb = (0.5 * dscj) * alpha;
    const double g1 = gamm - 1.0, ke = 0.5 * ((u * u) + (v * v));
    const double2 lf = make_double2(fa * (unA + nuA), fb * (unB + nuB));
    const double2 lb = make_double2(fa * (unA - nuA), fb * (unB - nuB));
    const double2 es = make_double2(-(fa * unA), -(fb * unB));
#pragma unroll
    for (int w = 0; w < C; w++) {
        char* o = rec + jrec_off(NY, w);
        double2* o1 = reinterpret_cast<double2*>(o) + 4 * r;
        double2* oE = reinterpret_cast<double2*>(o + JO_E) + 4 * r;
        double2* oP = reinterpret_cast<double2*>(o + JO_P) + 4 * r;
        double rv[4];
#pragma unroll
        for (int cc = 0; cc < 4; cc++) {
            const int k = 4 * w + cc, m = k - NY;
            rv[cc] = k < dq ? x[k < dq ? k : 0] : 0.0;
            if (k < NY) o1[cc] = make_double2(FLD(d, SHCFD_F_W, 4 + k, c), FLD(d, SHCFD_F_DHI, k, c) + g1 * ke);
            else o1[cc] = m == 0 ? make_double2(u, -(g1 * u)) : m == 1 ? make_double2(v, -(g1 * v))
                        : m == 2 ? make_double2(H, g1) : make_double2(0.0, 0.0);
            if (w >= W0) {
                oE[cc] = m < 0 ? es : m == 0 ? make_double2(fa * n1a, fb * n1b)
                       : m == 1 ? make_double2(fa * n2a, fb * n2b) : make_double2(0.0, 0.0);
                oP[cc] = m == 0 ? make_double2(fa * n1a, fb * n1b) : m == 1 ? make_double2(fa * n2a, fb * n2b)
                       : m == 2 ? make_double2(fa * unA, fb * unB) : make_double2(0.0, 0.0);
            }
        }
        double2* oR = reinterpret_cast<double2*>(o + JO_R) + 2 * r;
        oR[0] = make_double2(rv[0], rv[1]);
        oR[1] = make_double2(rv[2], rv[3]);
        reinterpret_cast<double2*>(o + JO_LF)[r] = lf;
        reinterpret_cast<double2*>(o + JO_LB)[r] = lb;
        if (w < W0) reinterpret_cast<double2*>(o + JO_E)[r] = es;
    }
}

// the sweep's compute wave w, rec its record of the strip's step 0; BWD: stored
// steps descend
template <int NY, bool BWD, bool PURE>
__device__ inline void jsweep_compute(JLds<NY>& lds, char* rec, int nt, int w, int L) {
    constexpr int C = (NY + 6) / 4;
    constexpr long long STEP = BWD ? -jrec_step<NY>() : jrec_step<NY>();
    const int r = L >> 2, c = L & 3, gr = L >> 4;
    const bool odd = (c & 1) != 0, up = c >= 2;
    const int src = 64 * w + (BWD ? (gr == 3 ? JRIN + c : 16 * (gr + 1) + c)
                                  : (gr == 0 ? JRIN + c : 16 * (gr - 1) + 12 + c));
    const int dst = 64 * w + ((L & ~3) == JRIN ? L + 4 : L);
    const int fc = min(c, 2);
    const unsigned o16 = 16u * L, o8 = 8u * L + JO_R, ol = 16u * r + (BWD ? JO_LB : JO_LF),
                   oe = (PURE ? 16u * r : 16u * L) + JO_E;
    if (BWD) rec += (long long)(nt - 1) * jrec_step<NY>();
    auto ld16 = [](const char* u, unsigned o) { return *reinterpret_cast<const double2*>(u + o); };
    // a step's inputs, JU - 1 steps ahead
    double2 b1[JU], bE[JU], bP[JU], bL[JU];
    double bR[JU];
    const char* in = rec;
#define JLOAD(Q)                                                 \
    {                                                            \
        b1[Q] = ld16(in, o16);                                   \
        bE[Q] = ld16(in, oe);                                    \
        if constexpr (!PURE) bP[Q] = ld16(in + JO_P, o16);       \
        bL[Q] = ld16(in, ol);                                    \
        bR[Q] = *reinterpret_cast<const double*>(in + o8);       \
        in += STEP;                                              \
    }
#pragma unroll
    for (int q = 0; q < JU - 1; q++) JLOAD(q)
    wait_vmem();  // so that the waits in the loop follow its own accesses alone
    jbarrier();  // ring cleared, the neighbour's column of step 0 there
    double nb = lds.ring[0][src], a = bR[0], b = 0.0;
    for (int t0 = 0; t0 < nt; t0 += JU) {
#pragma unroll
        for (int q = 0; q < JU; q++) {
            JLOAD((q + JU - 1) % JU)
            const double bin = row_shift4<!BWD>(nb, b);
            const double v = BWD ? a - bin : a + bin;
            const double f = quad_sums(bE[q].x * v, bE[q].y * v, b1[q].y * v, odd, up);
            if (c < 3) lds.f[q & 1][r][c][w] = f;
            *reinterpret_cast<double*>(rec + o8) = v;
            rec += STEP;
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            double tot = lds.f[q & 1][r][fc][0];
#pragma unroll
            for (int m = 1; m < C; m++) tot = tot + lds.f[q & 1][r][fc][m];
            nb = lds.ring[(q + 1) & (JRS - 1)][src];
            const double eB = quad_perm<0x55>(tot), eA = quad_perm<0x00>(tot);
            const double rn = bR[(q + 1) % JU];
            b = fma(b1[q].x, eB, bL[q].y * v);
            a = BWD ? fma(-b1[q].x, eA, fma(-bL[q].x, v, rn)) : fma(b1[q].x, eA, fma(bL[q].x, v, rn));
            if constexpr (!PURE) {
                const double dp = quad_perm<0xAA>(tot);
                b = fma(bP[q].y, dp, b);
                a = fma(BWD ? -bP[q].x : bP[q].x, dp, a);
            }
            lds.ring[(q + 1 + JGD) & (JRS - 1)][dst] = b;
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#undef JLOAD
}

// the wave that takes the neighbour strip's columns: step e takes column
// col0 + e (forward) or col0 - e (backward), in the ring before the barrier of
// step e - 1.  Two loads cover 2 NQ steps; the next pair is issued, from the
// step then wanted, before the last is looked at.  Takes nt + 1 barriers.
template <int NY, bool BWD>
__device__ inline void jcourier_in(double (&ring)[JRS][(NY + 6) / 4 * 64], const DevCtx& d, const Strip16& S,
                                   const double* hand, long long hstride, long long spin_limit, int nt, int L) {
    constexpr int dq = NY + 3;
    constexpr int NQ = 64 / dq;
    const int from = BWD ? S.next : S.prev;
    if (from < 0) {
        for (int t = 0; t < nt + 1; t++) jbarrier();
        return;
    }
    const __amdgpu_buffer_rsrc_t rin = jview(hand + (long long)from * hstride, hstride * 8);
    const int col0 = BWD ? nt - JSPAN : 1;
    const int q0 = L / dq, k = L % dq;
    const bool used = q0 < NQ;
    auto poll = [&](int e, double& x0, double& x1) {
        asm volatile("" ::: "memory");  // a poll is a new load
        const int c0 = col0 + (BWD ? -(e + q0) : e + q0), c1 = c0 + (BWD ? -NQ : NQ);
        x0 = jv_ld(rin, ((HO + c0) * dq + k) * 8);
        x1 = jv_ld(rin, ((HO + c1) * dq + k) * 8);
    };
    int have = 0, f1 = 0;  // steps below `have` are in the ring
    double x0, x1;
    poll(0, x0, x1);
    long long it = 0;
    bool dead = false;
    // looks at the loads in flight; steps up to `last` may enter the ring
    auto look = [&](int last) {
        const double v0 = x0, v1 = x1;
        const int f = f1;
        f1 = have;
        poll(have, x0, x1);
        const unsigned long long m0 = __ballot(dead || !used || !is_sent16(v0));
        const unsigned long long m1 = __ballot(dead || !used || !is_sent16(v1));
        int ready = m0 == ~0ULL ? NQ : __builtin_ctzll(~m0) / dq;
        if (ready == NQ) ready += m1 == ~0ULL ? NQ : __builtin_ctzll(~m1) / dq;
        const int upto = min(f + ready - 1, last);
        const int e0 = f + q0, e1 = e0 + NQ;
        const int lane = 64 * (k >> 2) + JRIN + (k & 3);
        if (used && e0 >= have && e0 <= upto) ring[e0 & (JRS - 1)][lane] = is_sent16(v0) ? 0.0 : v0;
        if (used && e1 >= have && e1 <= upto) ring[e1 & (JRS - 1)][lane] = is_sent16(v1) ? 0.0 : v1;
        if (upto >= have) {
            have = upto + 1;
            it = 0;
        } else if (!dead && it++ >= spin_limit + 1) {
            atomicCAS(d.iflag + IFLAG_ERR, 0, SHCFD_E_SPIN);
            dead = true;  // no further waits in this sweep: it runs to its end with zeros
        }
    };
    while (have < 1) look(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    jbarrier();
    for (int t = 0; t < nt; t++) {
        while (have < t + 2) look(t + JRS - 1);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        jbarrier();
    }
}

// forward and backward sweeps: one workgroup of C compute waves and two
// hand-off waves per strip.  Backward, workgroup g handles strip nstrips-1-g,
// so the strip it waits on (the one above) has a lower workgroup id.
template <int NY, bool BWD>
__global__ void __launch_bounds__(64 * ((NY + 6) / 4 + 2)) __attribute__((amdgpu_waves_per_eu(1, 2)))
k_sweep16j(DevCtx d, const Strip16* strips, int nstrips, double* hand, long long hstride, long long spin_limit,
           char* recs) {
    constexpr int dq = NY + 3, C = (dq + 3) / 4;
    __shared__ __attribute__((aligned(16))) JLds<NY> lds;
    const int s = BWD ? nstrips - 1 - (int)blockIdx.x : (int)blockIdx.x;
    const int L = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const Strip16 S = strips[s];
    const int nt = (d.blk[S.b].ni + JSPAN + JU - 1) / JU * JU;  // steps, whole rounds
    for (int e = (int)threadIdx.x; e < JRS * C * 64; e += 64 * (C + 2)) lds.ring[e / (C * 64)][e % (C * 64)] = 0.0;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    jbarrier();
    if (wave < C) {
        char* rec = recs + (JPAD + S.base) * jrec_step<NY>() + jrec_off(NY, wave);
        if (wave < NY / 4) jsweep_compute<NY, BWD, true>(lds, rec, nt, wave, L);
        else jsweep_compute<NY, BWD, false>(lds, rec, nt, wave, L);
    } else if (wave == C) {
        jcourier_in<NY, BWD>(lds.ring, d, S, hand, hstride, spin_limit, nt, L);
        jbarrier();
    } else {
        // the strip's own columns: the terms of step t are in the ring after
        // the barrier of step t + 1.  Step e gives column col0 + e (forward)
        // or col0 - e (backward)
        const bool present = (BWD ? S.prev : S.next) >= 0 && L < dq;
        const __amdgpu_buffer_rsrc_t rout = jview(hand + (long long)s * hstride, hstride * 8);
        const int col0 = BWD ? nt : 1 - JSPAN;
        const int k = L < dq ? L : 0, lane = 64 * (k >> 2) + (BWD ? 0 : 60) + (k & 3);
        jbarrier();
        for (int t = 0; t <= nt; t++) {
            jbarrier();
            if (t == 0) continue;
            const double x = lds.ring[(t + JGD) & (JRS - 1)][lane];
            const int col = col0 + (BWD ? -(t - 1) : t - 1);
            jv_st(rout, x, present ? ((HO + col) * dq + k) * 8 : JV_DROP);
        }
    }
}

// ---------------------------------------------------------------------------
// Sweeps over the stored matrices (precon, preconLU-SGS; LU-SGS and NR with the
// closed form switched off), in the same layout and schedule, with the same
// hand-off in its own wave.  Every lane evaluates the reference's per-cell
// formula with the operation order of the row-per-lane sweeps, on the same
// inputs, in a topological order of the same dependency graph, so the results
// are identical:
//     x = alpha (R + (A+(i-1) x(i-1) dsci + B+(j-1) x(j-1) dscj))   forward
//     x = x* - alpha (A-(i+1) x(i+1) dsci + B-(j+1) x(j+1) dscj)    backward
// A lane reads its two matrix rows (2 dq doubles) and the cell's alpha, dsci,
// dscj of each step from the quad-row copy written by k_set_abpm16 as dq + 2
// pairs of doubles, pair p of global step g = base + t at
// ((((set NT + g) C + w) (dq+2) + p) 64 + lane) 2: every 16-byte load of a wave
// reads 1 KB of consecutive bytes.  The right-hand side and the results, R* in
// place, are stored by (strip, step, wave, lane).  Slots of no cell hold zeros.
//
// Bound by the matrix rows: 43 KB per step at nY = 9 through one CU's 64 bytes
// per cycle (280 ns of the 400 ns of a step), beside 48 dependent FP64
// operations; then by the hand-off.  Measured at nY = 9 on 223 x 99: 239 us
// forward and 243 us backward (before, dq and q read and written in place and
// the hand-off polled by the computing waves, 327 and 447 us); prefetching
// four steps instead of three 260 us, since the rows then pass through
// accumulation registers.
// ---------------------------------------------------------------------------
template <int NY>
__global__ void __launch_bounds__(256) k_rhs16m(DevCtx d, const Strip16* strips, int nstrips, int nsteps16,
                                                int dqdt_inline, double* Rs, double* hand, long long hstride) {
    using D = Dims<NY>;
    constexpr int dq = D::dq, C = (dq + 3) / 4;
    refill_hand(d, strips, nstrips, hand, hstride, dq);
    const int s = (int)blockIdx.x / nsteps16;
    const Strip16 S = strips[s];
    const int t = 16 * ((int)blockIdx.x % nsteps16) + (int)(threadIdx.x & 15), r = (int)(threadIdx.x >> 4);
    const DevBlock B = d.blk[S.b];
    if (t >= B.ni + JSPAN) return;
    int i, j;
    double x[dq];
    if (jslot_cell(S, B, t, r, i, j)) {
        const long long c = cidx(B, i, j);
        double bal[dq];
        flux_balance<NY>(d, B, c, bal);
        rhs_of_cell<NY>(
            d, c, bal, dqdt_inline != 0, [&](int k) { return FLD(d, SHCFD_F_PRE1, k, c); },
            [&](int k) { return FLD(d, SHCFD_F_PRE2, k, c); }, [&]() { return FLD(d, SHCFD_F_PRESCA, 1, c); }, x);
    } else {
#pragma unroll
        for (int k = 0; k < dq; k++) x[k] = 0.0;
    }
#pragma unroll
    for (int w = 0; w < C; w++) {
        double rv[4];
#pragma unroll
        for (int cc = 0; cc < 4; cc++) rv[cc] = 4 * w + cc < dq ? x[4 * w + cc < dq ? 4 * w + cc : 0] : 0.0;
        double2* o = reinterpret_cast<double2*>(Rs + ((S.base + t) * C + w) * 64) + 2 * r;
        o[0] = make_double2(rv[0], rv[1]);
        o[1] = make_double2(rv[2], rv[3]);
    }
}

template <int NY>
struct MLds {
    static constexpr int C = (NY + 6) / 4;
    double ring[JRS][C * 64];
    double x[2][16][4 * C];    // the unknowns of each row's cell
};

// prefetch distance, in steps, as far as the registers go without scratch: up
// to four waves have a SIMD's 512 registers each, more waves half of them.
// Eight steps of preconditioned LU-SGS on 223 x 99, in ms, one / two / three
// steps ahead: nY = 9 5.8 / 5.5 / 5.4, nY = 12 13.3 / 13.3 / 26.6, nY = 13 15.1 /
// 20.9 / 32.3 (from two on the rows spill), nY = 16 22.6 / 37.6 / 49.2
template <int NY>
constexpr int pdm() { return NY <= 9 ? 3 : NY <= 12 ? 2 : 1; }

template <int NY, bool BWD>
__global__ void __launch_bounds__(64 * ((NY + 6) / 4 + 1))
k_sweep16m(DevCtx d, const Strip16* strips, int nstrips, double* hand, long long hstride, long long spin_limit,
           const double* __restrict__ jac, long long nsl, double* Rs) {
    constexpr int dq = NY + 3, C = (dq + 3) / 4, dq2 = dq + 2, PD = pdm<NY>(), NB = PD + 1;
    __shared__ __attribute__((aligned(16))) MLds<NY> lds;
    const int s = BWD ? nstrips - 1 - (int)blockIdx.x : (int)blockIdx.x;
    const int L = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const Strip16 S = strips[s];
    // the loop below ends at any step: whole rounds would cost 200 blocks of 8 x 8
    // six steps of 32 (nine species, eight updates: 2.48 ms against 2.30)
    const int nt = d.blk[S.b].ni + JSPAN;
    for (int e = (int)threadIdx.x; e < JRS * C * 64; e += 64 * (C + 1)) lds.ring[e / (C * 64)][e % (C * 64)] = 0.0;
    lds_barrier();
    if (w == C) {
        jcourier_in<NY, BWD>(lds.ring, d, S, hand, hstride, spin_limit, nt, L);
        return;
    }
    const int r = L >> 2, c = L & 3, k = 4 * w + c, gr = L >> 4;
    const int src = 64 * w + (BWD ? (gr == 3 ? JRIN + c : 16 * (gr + 1) + c)
                                  : (gr == 0 ? JRIN + c : 16 * (gr - 1) + 12 + c));
    const int dst = 64 * w + ((L & ~3) == JRIN ? L + 4 : L);
    const double* jl = jac + ((((BWD ? nsl : 0) + S.base) * C + w) * dq2 * 64 + L) * 2;
    double* Rl = Rs + (S.base * C + w) * 64 + L;
    auto at = [&](int t) { return (long long)(BWD ? nt - 1 - t : t); };  // stored step of sweep step t
    auto load = [&](int t, StepIn<dq>& in) {
        const long long g = at(min(t, nt - 1));  // past the end: the last step again
        load_ops<dq>(jl + 128LL * C * dq2 * g, in);
        in.r = Rl[g * (C * 64)];
    };
    // the strip's own hand-off: row 15 (forward) or 0 (backward), column col at step t
    const bool out = (BWD ? S.prev : S.next) >= 0 && r == (BWD ? 0 : 15) && k < dq;
    const __amdgpu_buffer_rsrc_t rout = jview(hand + (long long)s * hstride, hstride * 8);
    StepIn<dq> buf[NB];
#pragma unroll
    for (int p = 0; p < PD; p++) load(p, buf[p]);
    wait_vmem();
    jbarrier();  // ring cleared, the neighbour's column of step 0 there
    double nb = lds.ring[0][src], a_in = 0.0, bo = 0.0;
    for (int t0 = 0; t0 < nt; t0 += NB) {
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const int t = t0 + u;
            if (t >= nt) break;
            load(t + PD, buf[(u + PD) % NB]);
            const StepIn<dq>& in = buf[u];
            const double b_in = row_shift4<!BWD>(nb, bo);
            const double x = BWD ? in.r - in.al * (a_in + b_in) : in.al * (in.r + (a_in + b_in));
            Rl[at(t) * (C * 64)] = x;
            lds.x[t & 1][r][k] = x;
            lds_barrier();
            double xa[dq];
#pragma unroll
            for (int l = 0; l < dq; l++) xa[l] = lds.x[t & 1][r][l];
            nb = lds.ring[(t + 1) & (JRS - 1)][src];
            double sa = 0.0, sb = 0.0;
#pragma unroll
            for (int l = 0; l < dq; l++) {
                sa = sa + in.a[l] * xa[l];
                sb = sb + in.b[l] * xa[l];
            }
            a_in = in.fi * sa;
            bo = in.fj * sb;
            lds.ring[(t + 1 + JGD) & (JRS - 1)][dst] = bo;
            const int col = BWD ? nt - t : t + 1 - JSPAN;
            jv_st(rout, bo, out ? ((HO + col) * dq + k) * 8 : JV_DROP);
        }
    }
}

// after the sweeps: dq (alpha z of the closed form; x of the matrix sweeps, MAT)
// into the natural field; LU-SGS and preconLU-SGS: q += dq over the active
// blocks; NR and precon: (res, omega) partials per workgroup
template <int NY, bool MAT>
__global__ void __launch_bounds__(256) k_post16j(DevCtx d, const Strip16* strips, int nsteps16, const char* recs,
                                                 double* part) {
    constexpr int dq = NY + 3, C = (dq + 3) / 4;
    __shared__ double shr[4], sho[4];
    const int s = (int)blockIdx.x / nsteps16;
    const Strip16 S = strips[s];
    const int t = 16 * ((int)blockIdx.x % nsteps16) + (int)(threadIdx.x & 15), r = (int)(threadIdx.x >> 4);
    const DevBlock B = d.blk[S.b];
    const bool inner = inner_loop_scheme(d.p.scheme);
    double res = 0.0, om = 1e300;
    int i, j;
    if (jslot_cell(S, B, t, r, i, j)) {
        const long long c = cidx(B, i, j);
        const char* rec = recs + (MAT ? (S.base + t) * (C * 512) : (JPAD + S.base + t) * jrec_step<NY>());
        const double al = MAT ? 1.0 : FLD(d, SHCFD_F_ALPHA, 0, c);
#pragma unroll
        for (int w = 0; w < C; w++) {
            const double2* z = reinterpret_cast<const double2*>(rec + (MAT ? w * 512 : jrec_off(NY, w) + JO_R)) + 2 * r;
            const double2 z0 = z[0], z1 = z[1];
            const double x[4] = {al * z0.x, al * z0.y, al * z1.x, al * z1.y};
#pragma unroll
            for (int cc = 0; cc < 4; cc++) {
                const int k = 4 * w + cc;
                if (k >= dq) continue;
                FLD(d, SHCFD_F_DQ, k, c) = x[cc];
                if (inner) {
                    if (k == NY + 2) res = x[cc] * x[cc];
                    if (k < NY && x[cc] < 0.0) om = dmin(om, (-FLD(d, SHCFD_F_Q, k, c) / x[cc]) * d.p.dqmax);
                } else if (B.active) {
                    FLD(d, SHCFD_F_Q, k, c) = FLD(d, SHCFD_F_Q, k, c) + x[cc];
                }
            }
        }
    }
    if (!inner) return;
    for (int off = 32; off >= 1; off >>= 1) {
        res = res + __shfl_xor(res, off);
        om = dmin(om, __shfl_xor(om, off));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { shr[w] = res; sho[w] = om; }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = (shr[0] + shr[1]) + (shr[2] + shr[3]);
        part[2 * blockIdx.x + 1] = dmin(dmin(sho[0], sho[1]), dmin(sho[2], sho[3]));
    }
}

#define INST(NY)                                                                                              \
    template __global__ void k_rhs16m<NY>(DevCtx, const Strip16*, int, int, int, double*, double*, long long);   \
    template __global__ void k_sweep16m<NY, false>(DevCtx, const Strip16*, int, double*, long long, long long,  \
                                                   const double*, long long, double*);                        \
    template __global__ void k_sweep16m<NY, true>(DevCtx, const Strip16*, int, double*, long long, long long,   \
                                                  const double*, long long, double*);                         \
    template __global__ void k_rhs_jd16<NY>(DevCtx, const Strip16*, int, int, int, char*, double*, long long);  \
    template __global__ void k_sweep16j<NY, false>(DevCtx, const Strip16*, int, double*, long long, long long,  \
                                                   char*);                                                    \
    template __global__ void k_sweep16j<NY, true>(DevCtx, const Strip16*, int, double*, long long, long long,   \
                                                  char*);                                                     \
    template __global__ void k_post16j<NY, false>(DevCtx, const Strip16*, int, const char*, double*);           \
    template __global__ void k_post16j<NY, true>(DevCtx, const Strip16*, int, const char*, double*);
SHCFD_FOR_EACH_NY(INST)
#undef INST

}  // namespace shcfd
