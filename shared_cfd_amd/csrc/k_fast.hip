// k_fast.hip -- the optimised implicit update (LU-SGS / preconditioned LU-SGS
// / dual time) for the single-species ideal gas (dimq = 4).
//
// Reformulation (exact algebra, different rounding from the plain path):
// with S = post-scaling of the dual-time sweeps, S y = (y + ps4 (pre2.y) pre1)/ps1
// (S = I for LU-SGS and preconditioned LU-SGS), the forward sweep of
// time_dual_viscous.f90:37-50 becomes
//     v(i,j) = R(i,j) + GA(i-1,j) v(i-1,j) + GB(i,j-1) v(i,j-1),
//     GA = dsci*alpha*Ap*S,  GB = dscj*alpha*Bp*S,  Dq* = alpha*S*v,
// and the backward sweep (:67-93), with z = y/alpha and x2 the second-stage
// result (:53-60),
//     z(i,j) = x2/alpha - (HA(i+1,j) z(i+1,j) + HB(i,j+1) z(i,j+1)),
//     HA = dsci*alpha*Am*S,  HB = dscj*alpha*Bm*S,  Dq = alpha*S*z.
// The dependency graph is the reference's: cell (i,j) still waits for
// (i-1,j) and (i,j-1) (forward) or (i+1,j) and (i,j+1) (backward).
//
// Layout: a "quad strip" is 16 rows of one block owned by one wavefront;
// lane L = 4r+c holds component c of row r.  Row r processes column
// i = d-r-floor(r/4)+1 at step d: the rows of a step lie on an anti-diagonal,
// with one extra step between the groups of four rows that share a 16-lane
// row of the wavefront (see the sweep schedule below).
// Per-cell coefficients are stored by (strip, d, lane) -- the "skewed
// layout" -- so every step of both sweeps reads 64 consecutive slots.
//
// Each strip's steps are padded to whole chunks of CH steps, with one chunk
// of guard steps on either side, so the sweeps prefetch and store without a
// bounds test.  Slots that hold no cell keep zero coefficients (the arrays
// are zeroed once and k_fast_rhs_prep writes only cells), which makes every
// contribution out of them exactly zero: the sweeps need no per-cell mask.
// Arrays with one double per lane and step (R, V, X, Z) interleave pairs of
// steps, (dd even, dd odd) per lane, so one 16-byte access covers two steps.
#include "shcfd_device.h"
#include "shcfd_kernels.h"

namespace shcfd {

constexpr int QR = 16;  // rows per quad strip
constexpr int CH = 16;  // steps a strip is padded to (padding unit)
constexpr int GD = 1;   // extra steps between the four-row groups of a strip
constexpr int SPAN = QR - 1 + 3 * GD;  // steps row 15 runs behind row 0

struct QStrip {
    int b, j0, prev, next;
    long long base;  // slot of (step 0, lane 0); multiple of 128
    int nch, pad;    // chunks of CH steps covering the ni + SPAN steps
};

// slot of the one-double arrays for (step dd, lane L): pair-interleaved
__device__ inline long long slot1(long long base, int dd, int L) {
    return base + 64LL * (dd & ~1) + 2 * L + (dd & 1);
}

// 4x4 helpers (column-major)
__device__ inline void mm4(const double* A, const double* B, double* C) {
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int l = 0; l < 4; l++) {
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < 4; m++) s = fma(A[k + 4 * m], B[m + 4 * l], s);
            C[k + 4 * l] = s;
        }
}

// post-scaling matrix S (dual) or identity
__device__ inline void post_matrix(const CellJac<1>& J, bool dual, double* S) {
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int l = 0; l < 4; l++) S[k + 4 * l] = (k == l) ? 1.0 : 0.0;
    if (dual) {
        const double ips1 = 1.0 / J.ps[0], ps4 = J.ps[3];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int l = 0; l < 4; l++) S[k + 4 * l] = ips1 * (S[k + 4 * l] + ps4 * J.pre1[k] * J.pre2[l]);
    }
}

// alpha and the dual-time vectors/scalars of a cell as set_ABpm stored them
// (ALPHA, PRE1, PRE2, PRESCA: the values cell_jacobian gives for the same
// state, which the stage kernels read instead of recomputing)
struct PostScal {
    double alpha, pre1[4], pre2[4], ps[4];
};
__device__ inline PostScal post_scal(const DevCtx& d, long long c) {
    PostScal J;
    J.alpha = FLD(d, SHCFD_F_ALPHA, 0, c);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        J.pre1[k] = FLD(d, SHCFD_F_PRE1, k, c);
        J.pre2[k] = FLD(d, SHCFD_F_PRE2, k, c);
        J.ps[k] = FLD(d, SHCFD_F_PRESCA, k, c);
    }
    return J;
}

// cell of slot (strip S, step d, row r)
__device__ inline bool slot_cell(const QStrip& S, const DevBlock& B, int d, int r, int& i, int& j) {
    i = d - r - GD * (r >> 2) + 1;
    j = S.j0 + r;
    return i >= 1 && i <= B.ni && j <= B.nj;
}

// ---------------------------------------------------------------------------
// prep: per cell, the folded sweep operators in the skewed layout.
// Workgroup = 16 steps x 16 rows of one quad strip; thread = one cell.
// ---------------------------------------------------------------------------
constexpr unsigned long long SENTINEL = 0x7FF4DEADBEEFCAFEULL;

// Hand-off rows: one per strip and sweep plus a final row of zeros (read by
// the strips with no neighbour); entry 4*(HOFF+i)+c holds component c of
// column i, for i from -HOFF on.
constexpr int HOFF = 48;

// Operator arrays G = (GA, GB) and H = (HA, HB): per step a 4 KB block of
// four 1 KB parts, part p holding elements (2p', 2p'+1) of every lane's row,
// p = 2*(0 for A, 1 for B) + p'; lane L's pair sits at 16 L in its part.
// Element m of lane 4r+k is that of column (k + m) mod 4: the lane's own
// component comes first and needs no broadcast, the others come by one DPP
// quad rotation each.
// Each 16-byte load of a sweep step then reads 1 KB of consecutive bytes.
__device__ inline long long op_index(const QStrip& S, int dd, int L, int p, int e) {
    return (S.base / 64 + dd) * 512 + p * 128 + 2 * L + e;
}

// the folded operators of one cell c (slot step dd, row r) in its skewed
// slots from its cell Jacobian J: (GA, GB) into G for the forward sweep when
// G is given, (HA, HB) into H for the backward sweep when H is given, and
// with S = I the backward sweep's diagonal terms into Dn when Dn is given:
// A- = A+ - nuA I and B- = B+ - nuB I, so HA = GA - dsci alpha nuA I and
// HB = GB - dscj alpha nuB I; Dn holds (-dsci alpha nuA, -dscj alpha nuB) per
// row and step, 256 bytes per step
__device__ inline void prep_ops(const DevCtx& d, const QStrip& S, int dd, int r, long long c, const CellJac<1>& J,
                                double* G, double* H, double* Dn) {
    const bool dual = d.p.scheme == SHCFD_SCHEME_DUAL;
    double Sm[16], T[16];
    post_matrix(J, dual, Sm);
    const double dsci = FLD(d, SHCFD_F_DSCI, 0, c), dscj = FLD(d, SHCFD_F_DSCJ, 0, c);
    const double fa = dsci * J.alpha, fb = dscj * J.alpha;
    if (Dn)
        *reinterpret_cast<double2*>(&Dn[(S.base / 64 + dd) * 32 + 2 * r]) =
            make_double2(-(fa * J.nuA), -(fb * J.nuB));
    // rows of the operators: lane 4r+k holds row k (4 doubles), element m the
    // one of column (k + m) mod 4
    const double* mats[4] = {J.Ap, J.Bp, J.Am, J.Bm};
    const double fs[2] = {fa, fb};
#pragma unroll
    for (int m = 0; m < 4; m++) {
        double* o = m < 2 ? G : H;
        if (!o) continue;
        mm4(mats[m], Sm, T);
        // elements (2p', 2p'+1) of a lane's row are adjacent: one 16-byte store
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int lp = 0; lp < 2; lp++)
                *reinterpret_cast<double2*>(&o[op_index(S, dd, 4 * r + k, 2 * (m & 1) + lp, 0)]) =
                    make_double2(fs[m & 1] * T[k + 4 * ((k + 2 * lp) & 3)], fs[m & 1] * T[k + 4 * ((k + 2 * lp + 1) & 3)]);
    }
}

// one cell's backward operators (HA, HB) from a new cell Jacobian
__device__ inline void prep_cell_h(const DevCtx& d, const QStrip& S, const DevBlock& B, int dd, int r, double* H) {
    int i, j;
    if (!slot_cell(S, B, dd, r, i, j)) return;
    const long long c = cidx(B, i, j);
    CellJac<1> J;
    cell_jacobian<1>(d, c, B.pitch, J);
    prep_ops(d, S, dd, r, c, J, nullptr, H, nullptr);
}

// XCD-aware work order.  The dispatcher hands a launch's workgroups to the
// 8 XCDs in turn (workgroup b runs on XCD b % 8).  Giving XCD x the
// contiguous work items x*per .. x*per + per - 1 keeps neighbouring items,
// which share cache lines at their edges, in one L2.  A launch then has
// 8*per workgroups; those past the last item do nothing but the refill.
constexpr int NXCD = 8;
__host__ __device__ inline int xcd_groups(int n) { return NXCD * ((n + NXCD - 1) / NXCD); }
__device__ inline int xcd_item(int b, int n) { return (b % NXCD) * ((n + NXCD - 1) / NXCD) + b / NXCD; }

// refill of the hand-off rows of both sweeps: the sentinel for the columns
// 1..ni of each strip's block, zero elsewhere (grid-stride over all rows)
__device__ inline void hand_refill(const DevCtx& d, const QStrip* strips, double* hand, int nstrips, long long hstride) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    const long long nhand = 2LL * (nstrips + 1) * hstride;
    const double sv = __longlong_as_double((long long)SENTINEL);
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < nhand; k += stride) {
        const int row = (int)((k / hstride) % (nstrips + 1));
        const long long col = (k % hstride) / 4 - HOFF;
        const bool live = row < nstrips && col >= 1 && col <= d.blk[strips[row].b].ni;
        hand[k] = live ? sv : 0.0;
    }
}

// The right-hand side and prep of the optimised update in one pass (k_rhs
// followed by the operators' prep): per cell one cell Jacobian gives
// set_ABpm's scalars (stored when abpm_inline, as k_rhs stores them), the
// right-hand side of the scheme goes straight into R, and the folded
// operators follow; the hand-off rows are refilled.  The natural DQ field is
// left to k_fast_post, which stores the update there.  (HA, HB) are formed
// here too when H is given, or their diagonal terms when Dn is given (S =
// I), else by the forward sweep's launch on the CUs its strips leave idle
// (k_fast_fwd).  Workgroup = one work item (16 steps x 16 rows of one quad
// strip, in XCD-aware order); a wave takes 4 rows x 16 steps, so each load of a cell field reads
// 4 runs of 16 consecutive cells.
__global__ void __launch_bounds__(256) k_fast_rhs_prep(DevCtx d, const QStrip* strips, const int2* work, int nwork,
                                                       int dqdt_inline, int abpm_inline, double* R_sl, double* G,
                                                       double* H, double* Dn, double* hand, int nstrips,
                                                       long long hstride) {
    hand_refill(d, strips, hand, nstrips, hstride);
    const int w = xcd_item((int)blockIdx.x, nwork);
    if (w >= nwork) return;
    const int2 wk = work[w];
    const QStrip S = strips[wk.x];
    const DevBlock B = d.blk[S.b];
    const int dd = wk.y + (int)(threadIdx.x & 15), r = (int)(threadIdx.x >> 4);
    int i, j;
    if (!slot_cell(S, B, dd, r, i, j)) return;
    const long long c = cidx(B, i, j);
    CellJac<1> J;
    cell_jacobian<1>(d, c, B.pitch, J);
    double s[4], x[4];
    if (abpm_inline) {
        store_abpm_scalars<1>(d, c, J);
        flux_balance<1>(d, B, c, s);
        rhs_of_cell<1>(
            d, c, s, dqdt_inline != 0, [&](int k) { return J.pre1[k]; }, [&](int k) { return J.pre2[k]; },
            [&]() { return J.ps[1]; }, x);
    } else {
        flux_balance<1>(d, B, c, s);
        rhs_of_cell<1>(
            d, c, s, dqdt_inline != 0, [&](int k) { return FLD(d, SHCFD_F_PRE1, k, c); },
            [&](int k) { return FLD(d, SHCFD_F_PRE2, k, c); }, [&]() { return FLD(d, SHCFD_F_PRESCA, 1, c); }, x);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) R_sl[slot1(S.base, dd, 4 * r + k)] = x[k];
    prep_ops(d, S, dd, r, c, J, G, H, Dn);
}

// ---------------------------------------------------------------------------
// Hand-off between quad strips.  The producer stores the outgoing
// contribution of its boundary row with agent-coherent 64-bit stores into a
// row whose slots hold a signalling-NaN sentinel (filled before every sweep);
// the consumer polls the slots until the sentinel is gone.  No flag and no
// store-completion wait is needed.  Arithmetic never produces this NaN
// payload.
// ---------------------------------------------------------------------------
__device__ inline bool is_sentinel(double x) { return (unsigned long long)__double_as_longlong(x) == SENTINEL; }

// Buffer views.  Each sweep addresses its strip through buffer resources
// (base in scalar registers, 32-bit lane offset, per-step offsets in scalar
// registers or the instruction's immediate), so a step spends one
// instruction per access instead of 64-bit address arithmetic per lane.
// Lanes that must not store give an offset beyond the view's size: the
// hardware's range check drops the access.
typedef unsigned int shcfd_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int shcfd_u32x2 __attribute__((ext_vector_type(2)));
constexpr int BUF_DROP = 0x7FFFFF00;     // lane offset beyond every view
constexpr int AUX_AGENT = 16;            // sc1: device-coherent access
__device__ inline __amdgpu_buffer_rsrc_t view(const double* base, long long ndoubles) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(base), 0, (int)(ndoubles * 8), 0x00020000);
}
__device__ inline double u2d(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline double2 ld_pair(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    const shcfd_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return make_double2(u2d(v.x, v.y), u2d(v.z, v.w));
}
__device__ inline void st_pair(__amdgpu_buffer_rsrc_t r, double2 x, int voff, int soff) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(x.x);
    const unsigned long long b = (unsigned long long)__double_as_longlong(x.y);
    const shcfd_u32x4 v = {(unsigned)a, (unsigned)(a >> 32), (unsigned)b, (unsigned)(b >> 32)};
    __builtin_amdgcn_raw_buffer_store_b128(v, r, voff, soff, 0);
}
__device__ inline double2 ld_agent2(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    const shcfd_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, AUX_AGENT);
    return make_double2(u2d(v.x, v.y), u2d(v.z, v.w));
}
__device__ inline void st_agent(__amdgpu_buffer_rsrc_t r, double x, int voff, int soff) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(x);
    const shcfd_u32x2 v = {(unsigned)a, (unsigned)(a >> 32)};
    __builtin_amdgcn_raw_buffer_store_b64(v, r, voff, soff, AUX_AGENT);
}
// byte offsets of step dd (dd >= -CH) inside a strip's views: operator
// blocks of 4 KB per step, step pairs of 1 KB (dd even), hand-off columns of
// 32 bytes
__device__ inline int op_off(int dd) { return (dd + CH) * 4096; }
__device__ inline int pair_off(int dd) { return (dd + CH) * 512; }
__device__ inline int dn_off(int dd) { return (dd + CH) * 256; }
__device__ inline int col_off(int col) { return (col + HOFF) * 32; }

// Sweep schedule.  A sweep workgroup has four wavefronts, one per SIMD of its
// CU, that meet at one s_barrier per chunk of CS steps:
//   * wave 0 computes.  It touches global memory only to store V/Z, so it
//     never waits for a vector-memory access: operators, right-hand sides and
//     hand-offs all come from LDS;
//   * wave 1 streams the strip's operator blocks and R/X pairs into LDS with
//     LDS-DMA loads (buffer_load ... lds), three chunk slots ahead.  A step
//     needs 4.5 KB of operators, and a CU's vector-memory path moves about 64
//     bytes per cycle;
//   * wave 2 takes the neighbour strip's hand-off row: it polls device memory
//     and puts each chunk's columns into an LDS ring;
//   * wave 3 stores the strip's own outgoing columns from that ring.
// In one wave the polling loads and the stores share the in-order vmcnt: each
// ring load then waits for the stores before it, which cost the compute wave
// a third of its time.
//
// What bounds the sweep is the issue of the compute wave: 9 FP64 operations
// (about 8 cycles each), 8 DPP moves and 7 LDS accesses per step, 148 cycles
// in isolation and 170 (74 ns) beside the loader, against 86 (35.8 ns) for the
// same step with all operands in registers and 78 for its dependent chain alone
// (v -> quad rotations -> four multiply-adds -> the neighbour row's lanes -> next
// v).  So the operator rows are stored rotated (own component first:
// 6 moves instead of 8 broadcasts), the next right-hand side opens the chain
// of a, and the neighbour value is read before the operators, which the step
// after next needs.  Within a 16-lane row of the wavefront (four grid rows)
// the hop to the next row is one DPP row shift.  Between those groups it would
// take a chain of whole-wave shifts, so the groups run GD = 1 step apart and
// the value crosses through LDS: 3 more steps per strip against 3 dependent
// DPP moves per step.
//
// Measured, forward / backward us per launch: 258,048-cell forward step 167 /
// 152 -> 133 to 140 / 124; 512x128 C-mesh 84 / 87 -> 64 / 67; 400x4 tube 47 / 47 ->
// 30 / 33 (one strip: 112 -> 75 ns per step).  A hop between strips costs 18
// steps of skew, up to 5 of chunk granularity and 1.3 us from the producer's
// store to the consumer's look.
constexpr int CS = 4;                                   // steps per LDS chunk
constexpr int SLOT_G = CS * 4096;                       // operator bytes per slot
constexpr int SLOT_DN = SLOT_G + (CS / 2) * 1024;       // + R/X step pairs
constexpr int SLOT_BYTES = SLOT_DN + CS * 256;          // + diagonal terms (backward sweep with S = I)
constexpr int LD_PER_CHUNK = 4 * CS + CS / 2;           // LDS-DMA loads per chunk, + 1 with Dn
static_assert(3 * CS <= CH, "chunks read past a strip's end fall in its guard steps");
static_assert(CS * 256 == 1024, "one LDS-DMA load carries a chunk's diagonal terms");

typedef __attribute__((address_space(3))) void lds_void;

__device__ inline void lds_dma(__amdgpu_buffer_rsrc_t r, char* lds, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voff, soff, 0, 0);
}
// the compiler keeps LDS accesses on their side of this point (everything
// else may cross)
__device__ inline void ds_order() { __builtin_amdgcn_sched_barrier(0x7F); }
// s_barrier that the compiler may not move memory accesses across; the second
// form first waits until the last LDS access of the wave alone is outstanding
__device__ inline void wg_barrier() { asm volatile("s_barrier" ::: "memory"); }
__device__ inline void chunk_barrier() { asm volatile("s_waitcnt lgkmcnt(1)\n\ts_barrier" ::: "memory"); }
// wait until at most N vector memory accesses of this wave are outstanding
template <int N>
__device__ inline void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}
__device__ inline void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// loader wave: chunk j = aligned block m of CS steps (steps CS*m .. CS*m+CS-1)
// into an LDS slot; the caller orders blocks (ascending or descending)
template <bool DN>
__device__ inline void load_block(__amdgpu_buffer_rsrc_t rop, __amdgpu_buffer_rsrc_t rpair, __amdgpu_buffer_rsrc_t rdn,
                                  char* slot, int m, int vl) {
#pragma unroll
    for (int t = 0; t < CS; t++)
#pragma unroll
        for (int p = 0; p < 4; p++) lds_dma(rop, slot + t * 4096 + p * 1024, vl, op_off(CS * m + t) + 1024 * p);
#pragma unroll
    for (int q = 0; q < CS / 2; q++) lds_dma(rpair, slot + SLOT_G + q * 1024, vl, pair_off(CS * m + 2 * q));
    if constexpr (DN) lds_dma(rdn, slot + SLOT_DN, vl, dn_off(CS * m));
}

// wave 1: NS chunk slots, block of chunk j = blk(j); DN: the chunks also carry
// the backward sweep's diagonal terms.  Chunk j's last operators are read
// during chunk j, the others during chunk j - 1, so chunk j + NS - 1 takes the
// slot of chunk j - 1 while chunk j is computed.
template <int NS, bool DN, typename BLK>
__device__ inline void sweep_loader(__amdgpu_buffer_rsrc_t rop, __amdgpu_buffer_rsrc_t rpair,
                                    __amdgpu_buffer_rsrc_t rdn, char* lds, int nck, int vl, BLK blk) {
    constexpr int LD = LD_PER_CHUNK + (DN ? 1 : 0);
    static_assert(NS >= 4 && (NS - 2) * LD < 64, "vmcnt range");
#pragma unroll
    for (int k = 0; k < NS - 1; k++) load_block<DN>(rop, rpair, rdn, lds + k * SLOT_BYTES, blk(k), vl);
    wait_vmcnt<(NS - 2) * LD>();  // chunk 0 in LDS
    wg_barrier();
    wait_vmcnt<(NS - 3) * LD>();  // chunk 1
    wg_barrier();
    int slot = (NS - 1) * SLOT_BYTES;
    for (int j = 0; j < nck; j++) {
        // the blocks past the strip's end fall in its guard steps
        load_block<DN>(rop, rpair, rdn, lds + slot, blk(j + NS - 1), vl);
        slot = slot == (NS - 1) * SLOT_BYTES ? 0 : slot + SLOT_BYTES;
        wait_vmcnt<(NS - 3) * LD>();  // chunk j + 2
        wg_barrier();
    }
    wg_barrier();
}

// ---- the LDS ring between the rows -----------------------------------------
// Slot e % RS belongs to sweep step e: the 64 lanes' outgoing terms of step
// e - 1 - GD (what the next group's edge row takes at step e) and, at RIN, the
// four components the strip's edge row takes from the neighbour strip (nothing
// reads the terms of those four lanes, which go four places further).  A lane
// reads the slot of step e + 1 during step e.
//
// With RS = 4 CS slots the outgoing courier may run one step behind the chunk
// barrier, so that the barrier need not wait for the last step's ring write
// (its own slot is rewritten two chunks later); with RS = 2 CS the barrier
// waits for it.
constexpr int RING = 64;                     // doubles per slot
constexpr int RIN = 4;
template <int RS>
constexpr bool late_out() { return RS >= 4 * CS; }

template <int NS, int RS>
struct SweepLds {
    char chunk[NS * SLOT_BYTES];
    double ring[RS * RING];
};

// lane 4r+c receives lane 4r + (c + K) mod 4
template <int K>
__device__ inline double quad_rot(double x) {
    constexpr int ctrl = (K & 3) | (((K + 1) & 3) << 2) | (((K + 2) & 3) << 4) | (((K + 3) & 3) << 6);
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), ctrl, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), ctrl, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// a step's operators (A and B rows of the lane) and, with DN, its diagonal
// terms
struct StepOps {
    double2 g[4], dn;
};
template <bool DN>
__device__ inline void read_ops(StepOps& o, const char* slot, int ts, int vl) {
    const char* p = slot + vl + ts * 4096;
#pragma unroll
    for (int k = 0; k < 4; k++) o.g[k] = *reinterpret_cast<const double2*>(p + k * 1024);
    // row r = lane/4: 16 bytes at 16 r (four lanes share it)
    if constexpr (DN) o.dn = *reinterpret_cast<const double2*>(slot + SLOT_DN + ts * 256 + 4 * (vl / 16 & ~3));
}
__device__ inline double2 read_pair(const char* slot, int q, int vl) {
    return *reinterpret_cast<const double2*>(slot + SLOT_G + q * 1024 + vl);
}

// wave 0: the sweep over nck chunks.  BWD: steps descend and v = R - (a + b);
// DN: the operators are (GA, GB) and the diagonal terms are subtracted from
// their diagonal elements (HA = GA - dsci alpha nuA I).  The next step's
// right-hand side opens the multiply-add chain of a.
template <int NS, int RS, bool BWD, bool DN>
__device__ inline void sweep_compute(SweepLds<NS, RS>& lds, __amdgpu_buffer_rsrc_t rv, int nck, int L) {
    const int vl = 16 * L;
    // where the lane's neighbour value comes from in a ring slot: the edge row
    // of its group takes the last row of the group before it in sweep order,
    // the strip's own edge row the neighbour strip's columns
    const int gr = L >> 4, c = L & 3;
    const int src = BWD ? (gr == 3 ? RIN + c : 16 * (gr + 1) + c) : (gr == 0 ? RIN + c : 16 * (gr - 1) + 12 + c);
    const double* rd = lds.ring + src;
    double* wr = lds.ring + ((L & ~3) == RIN ? L + 4 : L);
    StepOps o[CS];
    double2 r[CS / 2];
    auto pair_q = [](int q) { return BWD ? CS / 2 - 1 - q : q; };
    // R/X of step t of a chunk from its pairs
    auto rhs = [&](int t) { return ((BWD ? CS - 1 - t : t) & 1) ? r[t >> 1].y : r[t >> 1].x; };
    wg_barrier();  // chunk 0 and the neighbour's columns of steps 0..CS in LDS
#pragma unroll
    for (int t = 0; t < CS; t++) read_ops<DN>(o[t], lds.chunk, BWD ? CS - 1 - t : t, vl);
#pragma unroll
    for (int q = 0; q < CS / 2; q++) r[q] = read_pair(lds.chunk, pair_q(q), vl);
    double nb = rd[0];
    wait_lgkm0();
    wg_barrier();  // chunk 1 in LDS
    // a: the step's right-hand side with the term of the row's previous column
    double a = rhs(0), b = 0.0, keep = 0.0;
    const char* cur = lds.chunk;  // slot of chunk j
    for (int j = 0; j < nck; j += RS / CS) {
#pragma unroll
        for (int h = 0; h < RS / CS; h++) {
            const char* next = cur == lds.chunk + (NS - 1) * SLOT_BYTES ? lds.chunk : cur + SLOT_BYTES;
#pragma unroll
            for (int t = 0; t < CS; t++) {
                const int e = h * CS + t;                  // step modulo RS
                const int ts = BWD ? CS - 1 - t : t;       // step within the stored chunk
                const double bin = row_shift4<!BWD>(nb, b);
                // the neighbour value of the next step is read first, then the
                // operators that the step before has used: LDS returns in
                // order, so the next step waits for this value alone
                nb = rd[((e + 1) & (RS - 1)) * RING];
                ds_order();
                const double v = BWD ? a - bin : a + bin;
                const double v1 = quad_rot<1>(v), v2 = quad_rot<2>(v), v3 = quad_rot<3>(v);
                const double2 a01 = o[t].g[0], a23 = o[t].g[1], b01 = o[t].g[2], b23 = o[t].g[3];
                const double a0 = DN ? a01.x + o[t].dn.x : a01.x, b0 = DN ? b01.x + o[t].dn.y : b01.x;
                const double R = rhs((t + 1) & (CS - 1));
                if (t > 0)
                    read_ops<DN>(o[t - 1], next, BWD ? CS - t : t - 1, vl);
                else
                    read_ops<DN>(o[CS - 1], cur, BWD ? 0 : CS - 1, vl);
                b = fma(b23.y, v3, fma(b23.x, v2, fma(b01.y, v1, b0 * v)));
                a = BWD ? fma(-a23.y, v3, fma(-a23.x, v2, fma(-a01.y, v1, fma(-a0, v, R))))
                        : fma(a23.y, v3, fma(a23.x, v2, fma(a01.y, v1, fma(a0, v, R))));
                if (!(t & 1)) {
                    keep = v;
                    r[t >> 1] = read_pair(next, pair_q(t >> 1), vl);
                } else {
                    const int m = BWD ? nck - 1 - (j + h) : j + h;  // stored chunk
                    st_pair(rv, BWD ? make_double2(v, keep) : make_double2(keep, v), vl,
                            pair_off(CS * m + (ts & ~1)));
                }
                wr[((e + 1 + GD) & (RS - 1)) * RING] = b;
                ds_order();
            }
            cur = next;
            if (late_out<RS>()) {
                chunk_barrier();
            } else {
                wait_lgkm0();
                wg_barrier();
            }
        }
    }
    wait_lgkm0();
    wg_barrier();  // the last step's outgoing terms
}

// wave 2: columns of the neighbour strip's hand-off row (view rin) into the
// ring, those of steps CS j + 1 .. CS j + CS before chunk j is computed.  Step
// e takes column col0 + e (forward) or col0 - e (backward).  One load covers
// LK = 32 steps (lane l: components 2 (l & 1) and the next of step l/2).  The
// next one is issued, from the step then wanted, before the last is looked
// at: a look costs no more than the rest of its latency (about 0.7 us, since
// the loads queue behind the loader's), and a look that delivers several
// chunks lets the strip catch up.  More loads in flight slowed the loader by
// more than they saved.  Past spin_limit looks without progress it raises
// SHCFD_E_SPIN and goes on with zeros, so that the sweep still runs to its
// end.
constexpr int LK = 32;
template <int RS, bool BWD>
__device__ inline void courier_in(double* ring, __amdgpu_buffer_rsrc_t rin, bool present, int col0, int nck, int L,
                                  long long spin_limit, int* iflag) {
    if (!present) {
        for (int j = 0; j < nck + 3; j++) wg_barrier();
        return;
    }
    const int c = 2 * (L & 1), k = L >> 1;
    auto poll = [&](int e) {  // steps e .. e + LK - 1
        asm volatile("" ::: "memory");  // a poll is a new load
        return ld_agent2(rin, 8 * c + col_off(col0 + (BWD ? -1 : 1) * (e + k)), 0);
    };
    int e = 0, n = CS + 1, met = 0;  // steps e .. e + n - 1 are wanted; barriers met
    long long it = 0;
    bool dead = false;
    int f1 = 0;
    double2 x1 = poll(0);
    while (met < nck + 2) {
        const double2 x = x1;
        const int f = f1;
        f1 = e;
        x1 = poll(e);
        const unsigned long long got = __ballot(dead || !(is_sentinel(x.x) || is_sentinel(x.y)));
        while (met < nck + 2) {
            const unsigned long long want = (1ULL << (2 * n)) - 1;
            if (e + n - f > LK || (~(got >> (2 * (e - f))) & want) != 0ULL) break;
            const int q = k - (e - f);
            if (q >= 0 && q < n)
                *reinterpret_cast<double2*>(&ring[((e + q) & (RS - 1)) * RING + RIN + c]) =
                    make_double2(is_sentinel(x.x) ? 0.0 : x.x, is_sentinel(x.y) ? 0.0 : x.y);
            wait_lgkm0();
            wg_barrier();
            if (met == 0) {  // chunk 1 of the operators
                wg_barrier();
                met = 1;
            }
            met++;
            e += n;
            n = CS;
            it = -1;
        }
        if (!dead && it++ >= spin_limit + 1) {
            atomicCAS(iflag + IFLAG_ERR, 0, SHCFD_E_SPIN);
            dead = true;
        }
    }
    wg_barrier();
}

// wave 3: the strip's outgoing columns (lanes at `edge` of the ring) to its
// hand-off row after chunk j's barrier (late_out: up to the step before the
// chunk's last, whose terms follow with the next chunk's).  Step e gives column
// col0 + e (forward) or col0 - e (backward).
template <int RS, bool BWD>
__device__ inline void courier_out(const double* ring, __amdgpu_buffer_rsrc_t rout, bool present, int col0, int edge,
                                   int nck, int L) {
    constexpr int DIR = BWD ? -1 : 1;
    const int c = L & 3, k = L >> 2;
    wg_barrier();
    wg_barrier();
    for (int j = 0; j <= nck; j++) {
        wg_barrier();  // chunk j is computed (j = nck: nothing is left to compute)
        const int e = CS * j - (late_out<RS>() ? 1 : 0) + (k & (CS - 1));
        const double x = ring[((e + 1 + GD) & (RS - 1)) * RING + edge + c];
        const bool live = present && k < CS && e >= 0 && e < CS * nck;
        st_agent(rout, x, live ? 8 * c + col_off(col0 + DIR * e) : BUF_DROP, 0);
        wait_lgkm0();
    }
}

// clear the ring: the steps before the first values, and the columns of a
// strip that has no neighbour, are zero
template <int RS>
__device__ inline void clear_ring(double* ring) {
    for (int k = (int)threadIdx.x; k < RS * RING; k += 256) ring[k] = 0.0;
    wait_lgkm0();
    wg_barrier();
}

// ---------------------------------------------------------------------------
// forward sweep: one workgroup per quad strip
// ---------------------------------------------------------------------------
template <int NS, int RS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2)))
k_fast_fwd(DevCtx d, const QStrip* strips, int nstrips, const double* R_sl, const double* G, double* V_sl,
           double* hand, long long hstride, long long spin_limit, const int2* work, int nwork, double* H) {
    if ((int)blockIdx.x >= nstrips) {
        // workgroups past the strips form the backward operators (HA, HB) of
        // the work items, concurrently with the sweep: 16 steps x 16 rows per
        // item.  They wait on nothing, and the strips (lower workgroup ids)
        // are dispatched before them.
        const int nh = (int)gridDim.x - nstrips;
        for (int w = (int)blockIdx.x - nstrips; w < nwork; w += nh) {
            const int2 wk = work[w];
            const QStrip S = strips[wk.x];
            const DevBlock B = d.blk[S.b];
            prep_cell_h(d, S, B, wk.y + ((int)threadIdx.x & 15), (int)threadIdx.x >> 4, H);
        }
        return;
    }
    const int s = blockIdx.x;
    const int L = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const QStrip S = strips[s];
    const int nck = S.nch * (CH / CS);  // chunks, processed in ascending order
    const long long nstep = (long long)(S.nch + 2) * CH;
    __shared__ __attribute__((aligned(16))) SweepLds<NS, RS> lds;
    clear_ring<RS>(lds.ring);
    if (wave == 0) {
        sweep_compute<NS, RS, false, false>(lds, view(V_sl + S.base - 64 * CH, nstep * 64), nck, L);
    } else if (wave == 1) {
        const __amdgpu_buffer_rsrc_t rg = view(G + (S.base / 64 - CH) * 512, nstep * 512);
        const __amdgpu_buffer_rsrc_t rr = view(R_sl + S.base - 64 * CH, nstep * 64);
        sweep_loader<NS, false>(rg, rr, rr, lds.chunk, nck, 16 * L, [](int j) { return j; });
    } else if (wave == 2) {  // row 0 of step e is at column e + 1
        const long long prow = S.prev >= 0 ? S.prev : nstrips;
        courier_in<RS, false>(lds.ring, view(hand + prow * hstride, hstride), S.prev >= 0, 1, nck, L, spin_limit, d.iflag);
    } else {  // row 15 of step e is at column e - SPAN + 1
        courier_out<RS, false>(lds.ring, view(hand + (long long)s * hstride, hstride), S.next >= 0, 1 - SPAN, 60, nck, L);
    }
}

// ---------------------------------------------------------------------------
// between the sweeps (dual only): x2/alpha from v, in the skewed layout
// (time_dual_viscous.f90:44-60 applied to Dq* = alpha*S*v)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_fast_mid(DevCtx d, const QStrip* strips, const int2* work, int nwork,
                                                  const double* V_sl, double* X_sl) {
    // work items in XCD-aware order; a wave takes 4 rows x 16 steps
    const int w = xcd_item((int)blockIdx.x, nwork);
    if (w >= nwork) return;
    const int2 wk = work[w];
    const QStrip S = strips[wk.x];
    const DevBlock B = d.blk[S.b];
    const int r = (int)(threadIdx.x >> 4);
    const int dd = wk.y + (int)(threadIdx.x & 15);
    int i, j;
    if (!slot_cell(S, B, dd, r, i, j)) return;
    const long long c = cidx(B, i, j);
    // the dual-time scalars and vectors set_ABpm stored for this state
    const PostScal J = post_scal(d, c);
    double v[4], x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = V_sl[slot1(S.base, dd, 4 * r + k)];
    // Dq* = alpha * S v
    double dv = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) dv = fma(J.pre2[k], v[k], dv);
    const double ips1 = 1.0 / J.ps[0];
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = J.alpha * (ips1 * fma(J.ps[3] * dv, J.pre1[k], v[k]));
    // second stage: x2 = ps1*(x + ps3 (pre2.x) pre1); store x2/alpha
    double dx = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) dx = fma(J.pre2[k], x[k], dx);
#pragma unroll
    for (int k = 0; k < 4; k++)
        X_sl[slot1(S.base, dd, 4 * r + k)] = (J.ps[0] * fma(J.ps[2] * dx, J.pre1[k], x[k])) / J.alpha;
}

// ---------------------------------------------------------------------------
// backward sweep: workgroup g handles strip (n-1-g), so the strip it waits
// for (the one above) has a lower workgroup id
// ---------------------------------------------------------------------------
// DN: H holds (GA, GB) and Dn the diagonal terms (schemes with S = I)
template <int NS, int RS, bool DN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2)))
k_fast_bwd(DevCtx d, const QStrip* strips, int nstrips, const double* X_sl, const double* H, const double* Dn,
           double* Z_sl, double* hand, long long hstride, long long spin_limit) {
    const int s = nstrips - 1 - (int)blockIdx.x;
    const int L = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const QStrip S = strips[s];
    const int nck = S.nch * (CH / CS);  // chunk j holds block nck-1-j (steps descend)
    const long long nstep = (long long)(S.nch + 2) * CH;
    const int top = nck * CS - 1;  // stored step of sweep step 0
    __shared__ __attribute__((aligned(16))) SweepLds<NS, RS> lds;
    clear_ring<RS>(lds.ring);
    if (wave == 0) {
        sweep_compute<NS, RS, true, DN>(lds, view(Z_sl + S.base - 64 * CH, nstep * 64), nck, L);
    } else if (wave == 1) {
        const __amdgpu_buffer_rsrc_t rh = view(H + (S.base / 64 - CH) * 512, nstep * 512);
        const __amdgpu_buffer_rsrc_t rx = view(X_sl + S.base - 64 * CH, nstep * 64);
        const __amdgpu_buffer_rsrc_t rd = DN ? view(Dn + (S.base / 64 - CH) * 32, nstep * 32) : rx;
        sweep_loader<NS, DN>(rh, rx, rd, lds.chunk, nck, 16 * L, [nck](int j) { return nck - 1 - j; });
    } else if (wave == 2) {  // row 15 of stored step dd is at column dd - SPAN + 1
        const long long nrow = S.next >= 0 ? S.next : nstrips;
        courier_in<RS, true>(lds.ring, view(hand + nrow * hstride, hstride), S.next >= 0, top - SPAN + 1, nck, L, spin_limit,
                         d.iflag);
    } else {  // row 0 of stored step dd is at column dd + 1
        courier_out<RS, true>(lds.ring, view(hand + (long long)s * hstride, hstride), S.prev >= 0, top + 1, 0, nck, L);
    }
}

// ---------------------------------------------------------------------------
// post: Dq = alpha*S*z into the natural DQ field; inner-loop schemes: (res,
// omega) partials per workgroup; otherwise q += Dq
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_fast_post(DevCtx d, const QStrip* strips, const int2* work, int nwork,
                                                   const double* Z_sl, double* part) {
    __shared__ double shr[4], sho[4];
    // work items in XCD-aware order; the partials are stored per item, so
    // their summation order does not depend on it
    const int wi = xcd_item((int)blockIdx.x, nwork);
    if (wi >= nwork) return;
    const int2 wk = work[wi];
    const QStrip S = strips[wk.x];
    const DevBlock B = d.blk[S.b];
    const bool dual = d.p.scheme == SHCFD_SCHEME_DUAL;
    const bool inner = inner_loop_scheme(d.p.scheme);
    // without the (res, omega) partials a wave takes 4 rows x 16 steps, as in
    // k_fast_rhs_prep; with them it keeps 16 rows x 4 steps, the layout their
    // summation order follows
    const int r = inner ? (int)(threadIdx.x & 15) : (int)(threadIdx.x >> 4);
    const int dd = wk.y + (inner ? (int)(threadIdx.x >> 4) : (int)(threadIdx.x & 15));
    double res = 0.0, om = 1e300;
    int i, j;
    if (slot_cell(S, B, dd, r, i, j)) {
        const long long c = cidx(B, i, j);
        double z[4], x[4];
#pragma unroll
        for (int k = 0; k < 4; k++) z[k] = Z_sl[slot1(S.base, dd, 4 * r + k)];
        if (dual) {
            const PostScal J = post_scal(d, c);
            double dz = 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++) dz = fma(J.pre2[k], z[k], dz);
            const double ips1 = 1.0 / J.ps[0];
#pragma unroll
            for (int k = 0; k < 4; k++) x[k] = J.alpha * (ips1 * fma(J.ps[3] * dz, J.pre1[k], z[k]));
            res = x[3] * x[3];
            if (x[0] < 0.0) om = (-FLD(d, SHCFD_F_Q, 0, c) / x[0]) * d.p.dqmax;
#pragma unroll
            for (int k = 0; k < 4; k++) FLD(d, SHCFD_F_DQ, k, c) = x[k];
        } else {
            const double al = FLD(d, SHCFD_F_ALPHA, 0, c);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                x[k] = al * z[k];
                FLD(d, SHCFD_F_DQ, k, c) = x[k];
                if (B.active && !inner) FLD(d, SHCFD_F_Q, k, c) = FLD(d, SHCFD_F_Q, k, c) + x[k];
            }
            if (inner) {
                res = x[3] * x[3];
                if (x[0] < 0.0) om = (-FLD(d, SHCFD_F_Q, 0, c) / x[0]) * d.p.dqmax;
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
        part[2 * wi] = ((shr[0] + shr[1]) + (shr[2] + shr[3]));
        part[2 * wi + 1] = dmin(dmin(sho[0], sho[1]), dmin(sho[2], sho[3]));
    }
}

// ---------------------------------------------------------------------------
// Discrete adjoint: transposed LU-SGS.  With the folded operators above,
// one LU-SGS update is Dq = diag(alpha) (I + U)^-1 (I - L)^-1 R, where L holds
// GA, GB at the slots of the upwind neighbours and U holds HA, HB.  Its
// transpose applied to r is
//     y(c) = alpha(c) r(c) - HA(c)^T y(c - e_i) - HB(c)^T y(c - e_j)
//     x(c) = y(c) + GA(c)^T x(c + e_i) + GB(c)^T x(c + e_j),
// the same two sweeps with operators stored at the neighbour's slot:
//     GA'(c) = -HA(c + e_i)^T,  GB'(c) = -HB(c + e_j)^T,
//     HA'(c) = -GA(c - e_i)^T,  HB'(c) = -GB(c - e_j)^T,
// zero where the neighbour is outside the block.  LU-SGS and NR (S = I) only.
// ---------------------------------------------------------------------------
// one transposed operator of neighbour cn: -(fs * M)^T in lane rows
__device__ inline void put_transposed(double* o, const QStrip& S, int dd, int r, int pbase, const double* M, double fs,
                                      bool present) {
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int m = 0; m < 4; m++)
            o[op_index(S, dd, 4 * r + k, pbase + (m >> 1), m & 1)] = present ? -(fs * M[((k + m) & 3) + 4 * k]) : 0.0;
}

__global__ void __launch_bounds__(256) k_fast_adj_prep(DevCtx d, const QStrip* strips, const int2* work, int nwork,
                                                       double* G, double* H) {
    // work items in XCD-aware order; a wave takes 4 rows x 16 steps
    const int w = xcd_item((int)blockIdx.x, nwork);
    if (w >= nwork) return;
    const int2 wk = work[w];
    const QStrip S = strips[wk.x];
    const DevBlock B = d.blk[S.b];
    const int r = (int)(threadIdx.x >> 4);
    const int dd = wk.y + (int)(threadIdx.x & 15);
    int i, j;
    if (!slot_cell(S, B, dd, r, i, j)) return;
    const long long c = cidx(B, i, j), P = B.pitch;
    {
        CellJac<1> J;
        cell_jacobian<1>(d, c, P, J);
        FLD(d, SHCFD_F_ALPHA, 0, c) = J.alpha;
    }
    // GA' from HA(c+e_i): dsci alpha Am of the right neighbour
    {
        CellJac<1> J;
        const bool ok = i < B.ni;
        const long long cn = ok ? c + 1 : c;
        cell_jacobian<1>(d, cn, P, J);
        put_transposed(G, S, dd, r, 0, J.Am, FLD(d, SHCFD_F_DSCI, 0, cn) * J.alpha, ok);
        // HA' from GA(c-e_i)
    }
    {
        CellJac<1> J;
        const bool ok = j < B.nj;
        const long long cn = ok ? c + P : c;
        cell_jacobian<1>(d, cn, P, J);
        put_transposed(G, S, dd, r, 2, J.Bm, FLD(d, SHCFD_F_DSCJ, 0, cn) * J.alpha, ok);
    }
    {
        CellJac<1> J;
        const bool ok = i > 1;
        const long long cn = ok ? c - 1 : c;
        cell_jacobian<1>(d, cn, P, J);
        put_transposed(H, S, dd, r, 0, J.Ap, FLD(d, SHCFD_F_DSCI, 0, cn) * J.alpha, ok);
    }
    {
        CellJac<1> J;
        const bool ok = j > 1;
        const long long cn = ok ? c - P : c;
        cell_jacobian<1>(d, cn, P, J);
        put_transposed(H, S, dd, r, 2, J.Bp, FLD(d, SHCFD_F_DSCJ, 0, cn) * J.alpha, ok);
    }
}

// right-hand side of the transposed sweep: alpha r into the skewed layout
__global__ void __launch_bounds__(256) k_fast_adj_rhs(DevCtx d, const QStrip* strips, const int2* work, int nwork,
                                                      const double* r_cell, double* R_sl, double* hand, int nstrips,
                                                      long long hstride) {
    // the transposed sweeps' hand-off rows are refilled here too
    hand_refill(d, strips, hand, nstrips, hstride);
    // work items in XCD-aware order; a wave takes 4 rows x 16 steps
    const int w = xcd_item((int)blockIdx.x, nwork);
    if (w >= nwork) return;
    const int2 wk = work[w];
    const QStrip S = strips[wk.x];
    const DevBlock B = d.blk[S.b];
    const int r = (int)(threadIdx.x >> 4);
    const int dd = wk.y + (int)(threadIdx.x & 15);
    int i, j;
    if (!slot_cell(S, B, dd, r, i, j)) return;
    const long long c = cidx(B, i, j);
    const double al = FLD(d, SHCFD_F_ALPHA, 0, c);
#pragma unroll
    for (int k = 0; k < 4; k++) R_sl[slot1(S.base, dd, 4 * r + k)] = al * r_cell[k * d.NC + c];
}

// lambda += x (no alpha: the transposed product ends with the forward sweep's L^T)
__global__ void __launch_bounds__(256) k_fast_adj_post(DevCtx d, const QStrip* strips, const int2* work, int nwork,
                                                       const double* Z_sl, double* lam) {
    // work items in XCD-aware order; a wave takes 4 rows x 16 steps
    const int w = xcd_item((int)blockIdx.x, nwork);
    if (w >= nwork) return;
    const int2 wk = work[w];
    const QStrip S = strips[wk.x];
    const DevBlock B = d.blk[S.b];
    const int r = (int)(threadIdx.x >> 4);
    const int dd = wk.y + (int)(threadIdx.x & 15);
    int i, j;
    if (!slot_cell(S, B, dd, r, i, j)) return;
    const long long c = cidx(B, i, j);
#pragma unroll
    for (int k = 0; k < 4; k++) lam[k * d.NC + c] += Z_sl[slot1(S.base, dd, 4 * r + k)];
}

}  // namespace shcfd

// ---------------------------------------------------------------------------
// host driver
// ---------------------------------------------------------------------------
#include "shcfd_fast.h"

namespace shcfd {

int FastPath::init(Ctx& c) {
    if (c.ny != 1) return SHCFD_E_STATE;
    {
        int dev = 0;
        hipDeviceProp_t prop;
        ncu = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
                  ? prop.multiProcessorCount
                  : 0;
    }
    // strips (b, k) of every block; launch order: block by block, or, with
    // more strips than CUs, strip k of every block before strip k+1 of any,
    // so that a strip is launched well after the one it waits for instead
    // of holding a CU through the pipeline fill of its block.  Either way a
    // strip's neighbours in the sweep order have lower workgroup ids in the
    // sweep that waits for them.
    std::vector<int> nsb(c.nb), first(c.nb);
    int total = 0, maxns = 0;
    for (int b = 0; b < c.nb; b++) {
        nsb[b] = (c.hblk[b].nj + QR - 1) / QR;
        total += nsb[b];
        maxns = std::max(maxns, nsb[b]);
    }
    std::vector<int2> order;  // (b, k) in launch order
    if (ncu > 0 && total > ncu) {
        for (int k = 0; k < maxns; k++)
            for (int b = 0; b < c.nb; b++)
                if (k < nsb[b]) order.push_back(make_int2(b, k));
    } else {
        for (int b = 0; b < c.nb; b++)
            for (int k = 0; k < nsb[b]; k++) order.push_back(make_int2(b, k));
    }
    std::vector<int> idx(total);  // strip index of (b, k) at first[b] + k
    for (int b = 0, o = 0; b < c.nb; o += nsb[b], b++) first[b] = o;
    for (int s = 0; s < total; s++) idx[first[order[s].x] + order[s].y] = s;
    std::vector<QStrip> hs;
    std::vector<int2> hw;
    long long base = 0;
    int maxcols = 0;
    for (int s = 0; s < total; s++) {
        const int b = order[s].x, k = order[s].y;
        const DevBlock& B = c.hblk[b];
        const int nd = B.ni + SPAN;
        const int nch = (nd + CH - 1) / CH;
        maxcols = std::max(maxcols, nch * CH);
        QStrip S{};
        S.b = b;
        S.j0 = 1 + QR * k;
        S.prev = k > 0 ? idx[first[b] + k - 1] : -1;
        S.next = k < nsb[b] - 1 ? idx[first[b] + k + 1] : -1;
        S.nch = nch;
        // one chunk of guard steps before and after the padded steps
        S.base = base + 64LL * CH;
        for (int d0 = 0; d0 < nd; d0 += 16) hw.push_back(make_int2((int)hs.size(), d0));
        base += 64LL * CH * (nch + 2);
        hs.push_back(S);
    }
    nstrips = (int)hs.size();
    nwork = (int)hw.size();
    nslots = base;
    // columns -HOFF .. maxcols + 9 of every hand-off row (the views' range
    // check returns zero beyond, and drops stores)
    hstride = 4LL * (HOFF + maxcols + 10);
    auto al = [&](void** p, size_t bytes) {
        if (hipMalloc(p, bytes) != hipSuccess) return false;
        return hipMemset(*p, 0, bytes) == hipSuccess;
    };
    bool ok = al((void**)&strips, sizeof(QStrip) * hs.size()) && al((void**)&work, sizeof(int2) * hw.size()) &&
              al((void**)&R, sizeof(double) * nslots) && al((void**)&V, sizeof(double) * nslots) &&
              al((void**)&X, sizeof(double) * nslots) && al((void**)&Z, sizeof(double) * nslots) &&
              al((void**)&G, sizeof(double) * 8 * nslots) && al((void**)&H, sizeof(double) * 8 * nslots) &&
              al((void**)&Dn, sizeof(double) * (nslots / 2)) &&
              al((void**)&hand, sizeof(double) * 2 * hstride * (nstrips + 1)) &&
              al((void**)&part, sizeof(double) * 2 * nwork);
    if (!ok) return SHCFD_E_NOMEM;
    hipMemcpy(strips, hs.data(), sizeof(QStrip) * hs.size(), hipMemcpyHostToDevice);
    hipMemcpy(work, hw.data(), sizeof(int2) * hw.size(), hipMemcpyHostToDevice);
    ready = true;
    return SHCFD_OK;
}

void FastPath::release() {
    void* ptrs[] = {strips, work, R, V, X, Z, G, H, Dn, hand, part, aR, aV, aZ, aG, aH, ahand};
    for (void* p : ptrs)
        if (p) hipFree(p);
    *this = FastPath();
}

// With more strips than CUs a CU holds two strips: 80 KB of LDS each
static_assert(sizeof(SweepLds<4, 2 * CS>) <= 81920, "two sweep workgroups per CU");
constexpr int SWEEP_NS = 4, RS_ALONE = 4 * CS, RS_SHARED = 2 * CS;

void FastPath::sweep_fwd(Ctx& c, const DevCtx& d, int nhwg, const double* Rp, const double* Gp, double* Vp, double* hp,
                         double* Hp) {
    if (ncu > 0 && nstrips > ncu)
        hipLaunchKernelGGL((k_fast_fwd<SWEEP_NS, RS_SHARED>), dim3(nstrips + nhwg), dim3(256), 0, c.stream, d, strips,
                           nstrips, Rp, Gp, Vp, hp, hstride, c.spin_limit, work, nhwg ? nwork : 0, Hp);
    else
        hipLaunchKernelGGL((k_fast_fwd<SWEEP_NS, RS_ALONE>), dim3(nstrips + nhwg), dim3(256), 0, c.stream, d, strips,
                           nstrips, Rp, Gp, Vp, hp, hstride, c.spin_limit, work, nhwg ? nwork : 0, Hp);
}

void FastPath::sweep_bwd(Ctx& c, const DevCtx& d, bool diag, const double* Xp, const double* Hp, const double* Dp,
                         double* Zp, double* hp) {
#define SHCFD_BWD(RS, DN)                                                                                     \
    hipLaunchKernelGGL((k_fast_bwd<SWEEP_NS, RS, DN>), dim3(nstrips), dim3(256), 0, c.stream, d, strips, nstrips, Xp, Hp, \
                       Dp, Zp, hp, hstride, c.spin_limit)
    if (ncu > 0 && nstrips > ncu) {
        if (diag) SHCFD_BWD(RS_SHARED, true);
        else SHCFD_BWD(RS_SHARED, false);
    } else {
        if (diag) SHCFD_BWD(RS_ALONE, true);
        else SHCFD_BWD(RS_ALONE, false);
    }
#undef SHCFD_BWD
}

int FastPath::implicit(Ctx& c, int step_internal, int dqdt_inline, int abpm_inline, void (*pb)(Ctx*, int),
                       void (*pe)(Ctx*, int)) {
    DevCtx d = c.dev();
    const bool dual = c.p.scheme == SHCFD_SCHEME_DUAL;
    hipStream_t st = c.stream;
    double* hand_f = hand;
    double* hand_b = hand + hstride * (nstrips + 1);
    // Without the dual-time post-scaling (S = I) the backward operators are
    // the forward ones less diagonal terms: the backward sweep streams (GA,
    // GB) and the 16 bytes of those terms per cell that prep writes, instead
    // of 256 bytes of (HA, HB).  In dual time, when the strips leave CUs idle,
    // workgroups of the forward launch past the strips form (HA, HB) there.
    // The sweep's LDS (86 KB) keeps a CU to one of the launch's workgroups: an
    // operator workgroup next to a strip would take issue slots and
    // vector-memory bandwidth from the strip's waves.  128 of them spread the
    // work over the sweep's time; 512 finish sooner and slow the first strips
    // (258k-cell forward step, whole steps: 1 % slower).  With more
    // strips than CUs (batches of many blocks) no CU is idle: prep forms (HA,
    // HB) from the same cell Jacobians as (GA, GB), and the forward launch
    // holds the strips alone.
    const bool diag = !dual;
    const bool busy = ncu > 0 && nstrips > ncu;
    const int nhwg = (busy || diag) ? 0 : std::min(nwork, 128);
    pb(&c, PROF_PREP);
    hipLaunchKernelGGL(k_fast_rhs_prep, dim3(xcd_groups(nwork)), dim3(256), 0, st, d, strips, work, nwork, dqdt_inline,
                       abpm_inline, R, G,
                       (busy && !diag) ? H : nullptr, diag ? Dn : nullptr, hand, nstrips, hstride);
    pe(&c, PROF_PREP);
    pb(&c, PROF_SWEEP_FWD);
    sweep_fwd(c, d, nhwg, R, G, V, hand_f, H);
    pe(&c, PROF_SWEEP_FWD);
    const double* Xin = V;
    if (dual) {
        pb(&c, PROF_PREP);
        hipLaunchKernelGGL(k_fast_mid, dim3(xcd_groups(nwork)), dim3(256), 0, st, d, strips, work, nwork, V, X);
        pe(&c, PROF_PREP);
        Xin = X;
    }
    pb(&c, PROF_SWEEP_BWD);
    sweep_bwd(c, d, diag, Xin, diag ? G : H, diag ? Dn : nullptr, Z, hand_b);
    pe(&c, PROF_SWEEP_BWD);
    pb(&c, PROF_UPDATE);
    hipLaunchKernelGGL(k_fast_post, dim3(xcd_groups(nwork)), dim3(256), 0, st, d, strips, work, nwork, Z, part);
    if (inner_loop_scheme(c.p.scheme)) {
        hipLaunchKernelGGL(k_reduce_res_omega, dim3(1), dim3(256), 0, st, d, part, nwork);
        if (step_internal == 1) hipLaunchKernelGGL(k_copy_scal, dim3(1), dim3(1), 0, st, d, (int)SCAL_RES1, (int)SCAL_RES);
        if (c.defer_update)
            c.update_pending = 1;  // applied by the next primitive pass
        else
            hipLaunchKernelGGL(k_update<1>, dim3((unsigned)c.htiles.size()), dim3(64 * c.tile_rows), 0, st, d, c.dtiles);
    }
    pe(&c, PROF_UPDATE);
    return hipGetLastError() == hipSuccess ? SHCFD_OK : SHCFD_E_HIP;
}

int FastPath::adjoint_prep(Ctx& c) {
    const int sch = c.p.scheme;
    if (sch != SHCFD_SCHEME_LUSGS && sch != SHCFD_SCHEME_NR && sch != SHCFD_SCHEME_DUAL) return SHCFD_E_STATE;
    if (!aG) {
        auto al = [&](void** p, size_t bytes) {
            if (hipMalloc(p, bytes) != hipSuccess) return false;
            return hipMemset(*p, 0, bytes) == hipSuccess;
        };
        bool ok = al((void**)&aR, sizeof(double) * nslots) && al((void**)&aV, sizeof(double) * nslots) &&
                  al((void**)&aZ, sizeof(double) * nslots) && al((void**)&aG, sizeof(double) * 8 * nslots) &&
                  al((void**)&aH, sizeof(double) * 8 * nslots) &&
                  al((void**)&ahand, sizeof(double) * 2 * hstride * (nstrips + 1));
        if (!ok) return SHCFD_E_NOMEM;
    }
    // The transposed iteration is preconditioned with the LU-SGS operator of
    // the residual it solves: for the BDF2 steps of dual time that is the NR
    // operator (plain Jacobians, diagonal 3 Vol/(2 dt) + ...), whatever
    // pseudo-time preconditioning the primal inner loop used.
    DevCtx dp = c.dev();
    if (dp.p.scheme == SHCFD_SCHEME_DUAL) dp.p.scheme = SHCFD_SCHEME_NR;
    hipLaunchKernelGGL(k_fast_adj_prep, dim3(xcd_groups(nwork)), dim3(256), 0, c.stream, dp, strips, work, nwork, aG,
                       aH);
    return hipGetLastError() == hipSuccess ? SHCFD_OK : SHCFD_E_HIP;
}

int FastPath::adjoint_apply(Ctx& c, const double* r_cell, double* lam) {
    DevCtx d = c.dev();
    hipStream_t st = c.stream;
    hipLaunchKernelGGL(k_fast_adj_rhs, dim3(xcd_groups(nwork)), dim3(256), 0, st, d, strips, work, nwork, r_cell, aR,
                       ahand, nstrips, hstride);
    sweep_fwd(c, d, 0, aR, aG, aV, ahand, nullptr);
    sweep_bwd(c, d, false, aV, aH, nullptr, aZ, ahand + hstride * (nstrips + 1));
    hipLaunchKernelGGL(k_fast_adj_post, dim3(xcd_groups(nwork)), dim3(256), 0, st, d, strips, work, nwork, aZ, lam);
    return hipGetLastError() == hipSuccess ? SHCFD_OK : SHCFD_E_HIP;
}

}  // namespace shcfd
