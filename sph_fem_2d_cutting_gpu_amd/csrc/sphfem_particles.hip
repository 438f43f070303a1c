// Particle kernels: one kernel per reference function (actions_gpu.cu, leap_frog.cu,
// interactions_gpu.cu) for the drop-in entry points, and the fused FP64 step kernel that runs
// pair sums, Jaumann rate, continuity, momentum, advection, corrector, friction heat,
// plasticity, the far-from-tool contact reset, boundary conditions and NaN invalidation in one
// pass over the sorted particles.
#include "sphfem_physics.h"
#include "sphfem_rigid.h"

#pragma clang fp contract(off)

namespace sphfem {

// ---------------------------------------------------------------------------------------------
// pair sums of interactions_gpu.cu:143-379 for particle i, neighbours visited in the reference
// order: column ii, then row jj, then sorted index.  Within a column the occupied cells of
// rows [low_j, high_j) are one contiguous run of sorted indices, so each column is one loop.
// Pairs outside the kernel support contribute exact zeros in the reference and are skipped.
// ---------------------------------------------------------------------------------------------

__device__ __forceinline__ void column_range(const int *__restrict__ cs, const int *__restrict__ ce, int col0,
                                             int low_j, int high_j, int &first, int &last) {
    first = -1;
    last = -1;
    for (int jj = low_j; jj < high_j; jj++) {
        int s = cs[col0 + jj];
        if (s != -1) { first = s; break; }
    }
    if (first < 0) return;
    for (int jj = high_j - 1; jj >= low_j; jj--) {
        if (cs[col0 + jj] != -1) { last = ce[col0 + jj]; break; }
    }
}

// The neighbour fields come from pre (PreView), with the factors m/rho_j, (S_j - p_j)/rho_j^2,
// S_xy,j/rho_j^2 and sqrtf(K/rho_j) computed once per particle with the operations the reference repeats
// per pair, so the sums are bit-identical.  Bound by the L1's rate of cache lines: a wavefront's 64 lists
// drift apart, each load touches some 30 lines, and 2.3e8 of them filled 82 % of the cycles of the 1 M
// particle step's kernel while a pair's fields took 13 loads of 8 to 32 byte records, and a candidate's
// position and blanked flag two (503 us).  Eight loads of 16-byte records, and four candidates at a time:
// 417 us; all eight issued before the first is used: 358 us (371 with dividends outside 2^+-600 divided plainly;
// 145 M accesses, 69 % of the cycles, and 59 % of the VALU's).  Loading the next pair's fields ahead costs a
// third of the wavefronts (188 registers): 392 us.  The in-support neighbours go through a per-lane list
// of CHUNK entries in LDS (list = this lane's first entry, stride LIST_BS) before their terms are evaluated.
// WIN: every non-blanked particle of the 5x5 cells is evaluated, as the reference does, instead of
// the in-support ones only.  The kernel's zeros outside the support make the two the same sums for
// finite inputs; a neighbour with a non-finite input turns the sums NaN (0 * NaN) in the reference
// wherever it lies in the window, and only the WIN form reproduces that.
template <int LIST_BS, int CHUNK, bool WIN>
__device__ __forceinline__ PairSums pair_sums_fp64(const DevConsts &c, const sphfem_particles &P, int pidx,
                                                   double thermal_alpha, const int *__restrict__ cs,
                                                   const int *__restrict__ ce, const PreView &pre,
                                                   int *__restrict__ list) {
    const double mass = c.phys.mass;
    const double wdeltap = c.corr.wdeltap, alpha = c.corr.alpha, beta = c.corr.beta;
    const double eta = c.corr.eta, eps = c.corr.xspheps;
    const int nx = c.geom.nx, ny = c.geom.ny;
    const double rr2_min = c.rr2_min;
    const double is_tool_i = P.tool_particle[pidx];
    const sphfem_double2 pi = P.pos[pidx], vi = P.vel[pidx];
    const sphfem_double4 Si = P.S[pidx], Ri = P.R[pidx];
    const double hi = P.h[pidx], rhoi = P.rho[pidx], prsi = P.p[pidx];
    double Ti = 0.;
    if (thermal_alpha != 0.) Ti = P.T[pidx];
    const double rhoi21 = 1. / (rhoi * rhoi);
    const double fourh2 = 4 * hi * hi;
    const double h1 = 1 / hi;
    const bool unit_wdp = wdeltap == 1.;      // w / 1 == w exactly
    const double ci = pre.s2[pidx].y;
    const int hashi = P.hash[pidx];
    const int gi = hashi / ny;
    const int gj = hashi - gi * ny;
    const int low_i = gi - 2 < 0 ? 0 : gi - 2;
    const int low_j = gj - 2 < 0 ? 0 : gj - 2;
    const int high_i = gi + 3 > nx ? nx : gi + 3;
    const int high_j = gj + 3 > ny ? ny : gj + 3;
    PairSums r;
    r.v_der = {0., 0., 0., 0.};
    r.S_der = {0., 0., 0., 0.};
    r.vel_t = {0., 0.};
    r.pos_t = {0., 0.};
    r.T_lapl = 0.;
    // one in-support pair (xij, yij from the sorted positions); the order of the calls is the
    // reference's neighbour order, so the sums are the same whichever loop drives them
    auto pair = [&](int iter) {
        // every field of j is loaded before anything is computed from one
        const sphfem_double2 pj = pre.pos[iter], vr = pre.vr[iter], r2T = pre.r2[iter], vj = P.vel[iter];
        const sphfem_double2 s1 = pre.s1[iter], s2 = pre.s2[iter], Rj = pre.r1[iter];
        const double hj = P.h[iter];
        const double xij = pi.x - pj.x, yij = pi.y - pj.y;
        const bool heat = thermal_alpha != 0.;
        const double r2 = xij * xij + yij * yij;
        // the shared-reciprocal form (the 1M-particle step's k_pairs_fp64 529 -> 497 us) while the
        // single-precision radius and the quotients by it are normal numbers (in any length unit a case is
        // set up in), else, and in the window form, the plain one
        RadialTerms t;
        if (!WIN && r2 > 1e-36 && r2 < 1e36) t = radial_terms(xij, yij, r2, hi, h1, heat);
        else t = radial_terms_plain(pi.x, pi.y, pj.x, pj.y, xij, yij, r2, hi, rr2_min, heat);
        const double w = t.w, w_x = t.w_x, w_y = t.w_y;
        // the densities are positive where the window form is off (flag_nonfinite): the sign is free
        const double volj = vr.x, rhoj = WIN ? P.rho[iter] : fabs(vr.y);
        const bool tool_j = WIN ? P.tool_particle[iter] == 1. : vr.y < 0.;
        if (!(is_tool_i == 1.) && !tool_j) {
            const double sjx = s1.x, sjy = s1.y, sjz = s2.x, cj = s2.y, Rjz = r2T.x;
            r.v_der.x += (vj.x - vi.x) * w_x * volj;
            r.v_der.y += (vj.x - vi.x) * w_y * volj;
            r.v_der.z += (vj.y - vi.y) * w_x * volj;
            r.v_der.w += (vj.y - vi.y) * w_y * volj;
            double fab = unit_wdp ? w : w / wdeltap;
            fab *= fab;
            fab *= fab;
            double Rx = fab * (Ri.x + Rj.x);
            double Ry = fab * (Ri.y + Rj.y);
            double Rz = fab * (Ri.z + Rjz);
            r.S_der.x += mass * ((Si.x - prsi) * rhoi21 + sjx + Rx) * w_x;
            r.S_der.y += mass * (Si.y * rhoi21 + sjy + Ry) * w_y;
            r.S_der.z += mass * (Si.y * rhoi21 + sjy + Ry) * w_x;
            r.S_der.w += mass * ((Si.z - prsi) * rhoi21 + sjz + Rz) * w_y;
            double vijx = vi.x - vj.x;
            double vijy = vi.y - vj.y;
            double vijposij = vijx * xij + vijy * yij;
            double rhoij = 0.5 * (rhoi + rhoj);
            // both densities lie in the range that keeps the window form off (flag_nonfinite)
            Recip by_rhoij{};
            if constexpr (!WIN) by_rhoij = recip_from(rhoij, __builtin_amdgcn_rcp(rhoij));
            auto over_rhoij = [&](double a) {
                if constexpr (WIN) return a / rhoij;
                else return quot_holds(a) ? quot(a, by_rhoij) : a / rhoij;
            };
            if (vijposij < 0.) {
                double cij = 0.5 * (ci + cj);
                double hij = 0.5 * (hi + hj);
                double muij = (hij * vijposij) / (r2 + eta * eta * hij * hij);
                double piij = over_rhoij(-alpha * cij * muij + beta * muij * muij);
                r.vel_t.x += -mass * piij * w_x;
                r.vel_t.y += -mass * piij * w_y;
            }
            const double xsph = over_rhoij(-eps * w * mass);
            r.pos_t.x += xsph * vijx;
            r.pos_t.y += xsph * vijy;
        }
        if (heat && t.rij > 1e-8) {
            r.T_lapl += 2.0 * volj * (Ti - r2T.y) * t.rij1 * (t.ex * w_x + t.ey * w_y);
        }
    };
    // the in-support neighbours are listed first (in the same order) and the pair terms are
    // evaluated from the list, so the lanes of a wavefront evaluate pairs together instead of
    // idling on candidates outside the support
    int n = 0;
    auto run = [&]() {
        for (int k = 0; k < n; k++) {
            pair(list[k * LIST_BS]);
        }
        n = 0;
    };
    for (int ii = low_i; ii < high_i; ii++) {
        int first, last;
        column_range(cs, ce, ii * ny, low_j, high_j, first, last);
        if (first < 0 || last > (int)P.N) continue;
        for (int it4 = first; it4 < last; it4 += 4) {
            // four positions, loaded together; up to three past `last` are read and not used
            sphfem_double2 q[4];
#pragma unroll
            for (int k = 0; k < 4; k++) q[k] = pre.pos[it4 + k];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int iter = it4 + k;
                if (iter >= last) break;
                double xij = pi.x - q[k].x;
                double yij = pi.y - q[k].y;
                double rr2 = xij * xij + yij * yij;
                if (WIN ? P.blanked[iter] == 1. : (rr2 >= fourh2 || rr2 < rr2_min)) continue;
                list[n * LIST_BS] = iter;
                ++n;
            }
            // a full list empties every active lane's list at once: lanes that flushed at
            // their own points would each run their list with the rest of the wavefront idle
            if (__any(n > CHUNK - 4)) run();
        }
    }
    run();
    return r;
}

// ---------------------------------------------------------------------------------------------
// FP32-compensated form
// ---------------------------------------------------------------------------------------------

// the record at a 32-bit byte offset from a uniform base (one VGPR offset, no 64-bit address math)
__device__ __forceinline__ float4 ldrec(const float4 *__restrict__ base, unsigned byte_off) {
    return *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(base) + byte_off);
}
__device__ __forceinline__ int2 ldpos(const int2 *__restrict__ base, unsigned byte_off) {
    return *reinterpret_cast<const int2 *>(reinterpret_cast<const char *>(base) + byte_off);
}
// two position records from an 8-byte-aligned address
typedef int sphfem_v4i __attribute__((ext_vector_type(4), aligned(8)));

// Where the pair loops read the neighbours' positions from: HBM through L1 (the list kernel), or a
// wavefront's copy of its five columns' windows in LDS (the staged kernel).  Both give the same values,
// so the sums do not depend on the source.  A neighbour-list entry names where its records are.
struct GlobalPos {
    using Entry = int;                                      // sorted index
    const int2 *__restrict__ pos;
    // candidates j .. j + 3 of column d during the scan
    __device__ __forceinline__ void scan4(int, int j, int2 *b) const {
        const char *at = reinterpret_cast<const char *>(pos) + ((unsigned)j << 3);
        const sphfem_v4i u = *reinterpret_cast<const sphfem_v4i *>(at);
        const sphfem_v4i v = *reinterpret_cast<const sphfem_v4i *>(at + 16);
        b[0] = make_int2(u.x, u.y);
        b[1] = make_int2(u.z, u.w);
        b[2] = make_int2(v.x, v.y);
        b[3] = make_int2(v.z, v.w);
    }
    __device__ __forceinline__ Entry encode(int, int j) const { return j; }
    __device__ __forceinline__ unsigned index(Entry e) const { return (unsigned)e; }
    __device__ __forceinline__ int2 entry(Entry e) const { return ldpos(pos, (unsigned)e << 3); }
    // the range a lane scans in column d, limited to what the source holds (everything here)
    __device__ __forceinline__ bool clip(int, int &, int &) const { return true; }
};

struct StagedPos {
    using Entry = unsigned short;                           // LDS slot | column << 12
    const int2 *spos;         // LDS: the union windows of columns 0..4, one after the other
    const int *sdelta;        // LDS: per column, sorted index minus LDS slot
    int F[5], L[5], delta[5]; // per column: staged sorted range [F, L) and its delta (uniform)
    __device__ __forceinline__ void scan4(int d, int j, int2 *b) const {
        for (int u = 0; u < 4; u++) b[u] = spos[j + u - delta[d]];
    }
    __device__ __forceinline__ Entry encode(int d, int j) const { return (Entry)((j - delta[d]) | (d << 12)); }
    __device__ __forceinline__ unsigned index(Entry e) const { return (unsigned)((e & 0xfff) + sdelta[e >> 12]); }
    __device__ __forceinline__ int2 entry(Entry e) const { return spos[e & 0xfff]; }
    // a lane's window lies inside the wavefront's union by construction when the hashes are sorted;
    // otherwise the range is cut to the staged part (no access outside the LDS copy) and false
    // reports the inconsistent table
    __device__ __forceinline__ bool clip(int d, int &first, int &last) const {
        const bool inside = first >= F[d] && last <= L[d];
        first = first < F[d] ? F[d] : first;
        last = last > L[d] ? L[d] : last;
        if (last < first) last = first;
        return inside;
    }
};

// Particle i and the per-i kernel constants.  Distances D = x_i - x_j are in units u = cell / 2^28, with
// ku = u / h_i; the kernel's factors multiply the finished sums.
struct PairI {
    int xi, yi;
    float vxi, vyi, sxi, syi, szi, Rxi, Ryi, Rzi, rhoi, ci, Ti;
    float kf;                   // W to the artificial stress's w / wdeltap
    float D2max, D2min;         // the support test on |D|^2
    float beta2, eta2;          // 2 beta and eta^2 of the viscosity
    bool thermal;
    bool mech;                  // i is not a tool particle
    // general form only
    float ku, H, D2heat;        // u / h_i, h_i / u, the heat term's least |D|^2
    double xd, yd;              // the position where D is taken in FP64
};

struct PairAcc {                // FP32 block sums
    float v0, v1, v2, v3, ax, ay, p0, p1, T;
};

constexpr float KU = 1.f / (float)(1 << SPHFEM_POS_BITS);      // ku where the kernel width is the cell size

// one pair at distance D.  GEN: any kernel widths (h_j / u in Hj), else h_i = h_j = the cell size; win: window
// candidates outside the support are among the entries, with the kernel set to 0 as in the reference
template <bool GEN>
__device__ __forceinline__ void pair_term(const PairI &I, float dx, float dy, const float4 q1, const float4 q2,
                                          const float4 q3, float Hj, bool win, PairAcc &a) {
#pragma clang fp contract(fast)
    const float D2 = dx * dx + dy * dy;
    const float rinv = __builtin_amdgcn_rsqf(D2);
    const float ku = GEN ? I.ku : KU;
    const float r = D2 * rinv;
    const float u = 1.f - (0.5f * ku) * r;
    const float s = u * u;
    // W = kernel / (16 fac) and g: gradient = -3 fac / h_i * g * D
    const bool outer = r > (GEN ? I.H : 1.f / KU);
    float w = outer ? s * s * s : 0.0625f - (0.09375f * ku * ku) * D2 * u;
    float g = outer ? s * rinv : ku - (0.75f * ku * ku) * r;
    if constexpr (GEN) {
        if (win && (D2 >= I.D2max || D2 < I.D2min)) {        // a NaN distance keeps its NaN kernel
            w = 0.f;
            g = 0.f;
        }
    }
    const float volj = fabsf(q3.x);
    const float heat = volj * (I.Ti - q3.w) * g;
    // used only where the thermal block is set
    a.T += GEN && !(D2 > I.D2heat) ? 0.f : heat;
    if (I.mech && q3.x > 0.f) {                          // neither i nor j is a tool particle
        const float wx = g * dx, wy = g * dy;
        const float dvx = q1.x - I.vxi, dvy = q1.y - I.vyi;
        const float gx = dvx * volj, gy = dvy * volj;
        a.v0 += gx * wx;
        a.v1 += gx * wy;
        a.v2 += gy * wx;
        a.v3 += gy * wy;
        float f = w * I.kf;
        f *= f;
        f *= f;
        float Ax = (I.sxi + q1.z) + f * (I.Rxi + q2.y);
        const float Ay = (I.syi + q1.w) + f * (I.Ryi + q2.z);
        float Az = (I.szi + q2.x) + f * (I.Rzi + q2.w);
        const float half_inv_rhoij = __builtin_amdgcn_rcpf(I.rhoi + q3.y);
        const float vp = -(dvx * dx + dvy * dy);         // (v_i - v_j) . D
        if constexpr (GEN) {
            const float H = 0.5f * (I.H + Hj);
            const float mu = H * vp * __builtin_amdgcn_rcpf(D2 + I.eta2 * H * H);
            const float piij = vp < 0.f ? mu * (I.beta2 * mu - (I.ci + q3.z)) * half_inv_rhoij : 0.f;
            Ax -= piij;
            Az -= piij;
        } else {
            // receding pairs take mu = 0 and with it no viscous term
            const float mu = fminf(vp, 0.f) * __builtin_amdgcn_rcpf(D2 * KU + I.eta2);
            const float piij = mu * (I.beta2 * mu - (I.ci + q3.z)) * half_inv_rhoij;
            Ax -= piij;
            Az -= piij;
        }
        a.ax = Ay * wy + (Ax * wx + a.ax);
        a.ay = Az * wy + (Ay * wx + a.ay);
        const float wr = w * half_inv_rhoij;
        a.p0 -= wr * dvx;                                // sum W / (rho_i + rho_j) * (v_i - v_j)
        a.p1 -= wr * dvy;
    }
}

// the position, in units u from the grid's corner, of live record j of cell `hash` (general form)
__device__ __forceinline__ double2 wide_pos(const RecView &rv, int ny, int j, int hash) {
    const int2 p = rv.pos[j];
    const int ix = hash / ny, iy = hash - ix * ny;
    const int half = 1 << (SPHFEM_POS_BITS - 1);
    const int rx = (int)((unsigned)p.x - ((unsigned)ix << SPHFEM_POS_BITS) - half);
    const int ry = (int)((unsigned)p.y - ((unsigned)iy << SPHFEM_POS_BITS) - half);
    const unsigned two = 2u << SPHFEM_POS_BITS;
    if ((unsigned)rx + two > 2 * two || (unsigned)ry + two > 2 * two) return rv.away[j];   // not in its cell
    const double unit = (double)(1 << SPHFEM_POS_BITS);
    return make_double2((ix + 0.5) * unit + rx, (iy + 0.5) * unit + ry);
}

// FP32-compensated pair sums (same physics as pair_sums_fp64, different arithmetic), one lane per
// sorted particle:
//  * positions are 32-bit integers in units of cell / 2^28 that wrap every 16 cells: the difference of
//    any two particles near the cells of a 5x5 window is exact, and rounded once to FP32;
//  * one v_rsq per pair (the distance), one v_rcp (rho_i + rho_j) and one v_rcp for the viscosity
//    denominator; the kernel's dimensional factors and those of the equations multiply the finished sums
//    in FP64;
//  * the grad-T term uses e_ij . grad W / r_ij = the radial kernel-derivative factor: the reference's
//    algebra without its extra sqrt and divisions;
//  * each lane compacts its in-support candidates (columns in order, sorted index within a
//    column: the reference order) into an LDS list of CHUNK entries, loading candidates four
//    at a time, then evaluates the dense list with the records of the next entry in flight;
//  * summation: blocks of 8 pair terms in FP32, block sums accumulated in FP64, which bounds the
//    rounding of each sum by ~8 units of FP32 roundoff of the sum of |terms|; one final FP32
//    rounding on output.
// Outputs (FP32): psum[i] = velocity gradient (xx, xy, yx, yy); psum[N + i] = (mass * stress
// divergence - mass * viscous term) per axis, XSPH velocity per axis; psum_T[i] = Laplacian of T.
// Bound by VALU issue (70 - 80 % busy; 64 instructions a pair, 12 a candidate) and close behind by the
// L1's rate of cache lines per gather (a wavefront's 64 lists drift apart: some 30 lines per load).
// ROLL: the columns in a loop, which leaves the kernel with 128 registers and four wavefronts per SIMD
// where no update follows the sums (16 M particles: 3000 -> 2827 us); with the update's 166 registers there
// are three either way, and the unrolled columns are the faster (4 M: 779 us against 796).  Copying all
// records of 256-particle tiles to LDS cut the L1's accesses by five and cost as much in other issue.
// Positions of 16 bytes (cell-relative FP32 and the cell row, with the column in the list entry) and kernel
// factors applied per pair took 868 us (with the update) on 4 M particles and 3337 us (sums alone) on 16 M,
// against 779 and 2827 us.
// General form (GEN; the SPHFEM_FORM_ bits): kernel widths other than the cell size, at a fifth load per pair and
// the factors of h_i; and (SPECIAL), with a test of every candidate's record, widths that reach the place of
// blanked records, positions that the wrapped ones cannot tell apart, taken in FP64, and the window form, where
// every non-blanked record of the 5x5 cells is evaluated with the kernel set to 0 outside the support, as the
// reference does (see pair_sums_fp64).  With a third of the widths at 0.9 of the cell size the stage call takes
// 165 us at 204k and 580 us at 2M particles, a 1M-particle step 296 us; 178, 663 and 322 us with the 16-byte
// records, 302, 897 and 390 us while every state other than the first form's took the whole of the tests.
// The window form, met in the step after a value turns non-finite, takes 296 us at 204k and 980 us at 2M particles;
// 480 and 1627 us with every candidate's position taken in FP64, 239 and 883 us with the 16-byte records.
// Telling blanked records by their position instead of their sound speed: 284 and 900 us, but 168 registers.
__device__ __forceinline__ double interaction_alpha(const DevConsts &c, double is_tool) {
    // interactions_gpu.cu:164: the tool block (interactions_gpu.cu:19) is zero unless
    // interactions_setup_thermal_constants_tool set it (the rigid-tool setup does, benchmarks.cpp:518;
    // the FEM setups do not, benchmarks_NZ.cpp:354)
    return (is_tool == 0.) ? c.trml_wp.alpha : c.trml_itool.alpha;
}

// Arguments of the update (everything after the pair sums, leap_frog.cu:71-96 with the actions of
// the step), shared by the update kernel and the FP32C pair kernels that run it after their sums
struct UpdateArgs {
    sphfem_particles B, A;
    const sphfem_double2 *pos_init, *vel_init;
    const sphfem_double4 *S_init;
    const double *rho_init, *T_init;
    ToolView tv;
    int write_intermediates;
    const PairSums *psum64;
    const RigidTool *rt;
    RateView r_old, r_new;
    int skip_contact;
};

// the update of sorted particle i; g_sum, a_sum, T_lapl32 are its FP32C pair sums (the FP64 form
// reads psum64 instead).  NT: streaming stores, for the update run inside a pair kernel, whose
// neighbour records other wavefronts are still reading from L2 (plain stores would displace them)
template <bool F32C, bool RIGID, bool NT = false>
__device__ __forceinline__ void update_item(const DevConsts &c, const UpdateArgs &u, int i, float4 g_sum,
                                            float4 a_sum, float T_lapl32) {
    const sphfem_particles &B = u.B, &A = u.A;
    const sphfem_double2 *__restrict__ pos_init = u.pos_init;
    const sphfem_double2 *__restrict__ vel_init = u.vel_init;
    const sphfem_double4 *__restrict__ S_init = u.S_init;
    const double *__restrict__ rho_init = u.rho_init;
    const double *__restrict__ T_init = u.T_init;
    const ToolView &tv = u.tv;
    const int write_intermediates = u.write_intermediates;
    const PairSums *__restrict__ psum64 = u.psum64;
    const RigidTool *__restrict__ rt = u.rt;
    const RateView &r_old = u.r_old, &r_new = u.r_new;
    const int skip_contact = u.skip_contact;
    // FP32C: the reorder wrote only the neighbour records; every per-particle field is gathered here
    // from the unsorted arrays A through idx, and the sorted step result is written to B.  All loads
    // of the particle are issued before any branch on loaded values, so a wavefront waits for
    // memory once (the kernel holds 3 wavefronts per SIMD); the rates and pair sums of blanked
    // particles are read and not used.
    const int src = F32C ? B.idx[i] : i;
    sphfem_double2 pos, vel;
    sphfem_double4 S;
    double rho, T, eps_pl, eps_pl_dot, pr = 0.;
    sphfem_double2 fc0, ft0, nrm0;
    int on_seg0;
    sphfem_double2 v0 = {0., 0.};
    sphfem_double4 S0 = {0., 0., 0., 0.};
    double rho0 = 0.;
    double blanked0, tool, fixed, h_src = 0.;
    float2 vt_old = make_float2(0.f, 0.f);
    float4 St_old = make_float4(0.f, 0.f, 0.f, 0.f);
    float rt_old = 0.f, Tt_old = 0.f;
    if constexpr (F32C) {
        blanked0 = ld_stream(&A.blanked[src]);
        tool = ld_stream(&A.tool_particle[src]);
        fixed = ld_stream(&A.fixed[src]);
        pos = ld_stream(&A.pos[src]);
        v0 = ld_stream(&A.vel[src]);
        S0 = ld_stream(&A.S[src]);
        rho0 = ld_stream(&A.rho[src]);
        T = ld_stream(&A.T[src]);
        eps_pl = ld_stream(&A.eps_pl[src]);
        eps_pl_dot = ld_stream(&A.eps_pl_dot[src]);
        on_seg0 = ld_stream(&A.on_seg[src]);
        h_src = ld_stream(&A.h[src]);
        vt_old = ld_stream(&r_old.vel_t[src]);          // the FP32 derivative carry
        St_old = ld_stream(&r_old.S_t[src]);
        rt_old = ld_stream(&r_old.rho_t[src]);
        Tt_old = ld_stream(&r_old.T_t[src]);
    } else {
        blanked0 = B.blanked[i];
        tool = B.tool_particle[i];
        fixed = B.fixed[i];
    }
    const bool live = blanked0 != 1.;
    const double thermal_alpha = interaction_alpha(c, tool);
    PairSums r;
    if (live) {
        if constexpr (F32C) {
            // stress divergence and viscous acceleration come summed per axis
            r.v_der = {g_sum.x, g_sum.y, g_sum.z, g_sum.w};
            r.S_der = {a_sum.x, 0., a_sum.y, 0.};
            r.vel_t = {0., 0.};
            r.pos_t = {a_sum.z, a_sum.w};
            r.T_lapl = T_lapl32;
        } else {
            r = psum64[i];
        }
    }
    // FP32C: pos and T are the pre-step values (the corrector starts from them); velocity, stress and
    // density are predicted again from the pre-step state and rates (leap_frog.cu:45-69, the same
    // operations as in the reorder), as is the pressure (actions_gpu.cu:222-232)
    if constexpr (F32C) {
        vel = v0;
        S = S0;
        rho = rho0;
        if (live) {
            const double hdt = 0.5 * c.dt;
            vel.x = vel.x + hdt * vt_old.x;
            vel.y = vel.y + hdt * vt_old.y;
            S.x = S.x + hdt * St_old.x;
            S.y = S.y + hdt * St_old.y;
            S.z = S.z + hdt * St_old.z;
            S.w = S.w + hdt * St_old.w;
            rho = rho + hdt * (double)rt_old;
        }
        if (tool == 0.) pr = eos_pressure(c, rho);
        if (skip_contact && on_seg0 == -1) {
            // every writer of on_seg = -1 (contact s1, the far-from-tool reset) zeroes fc, ft and n
            // with it (actions_gpu.cu:455-491): nothing to read far from the tool
            const sphfem_double2 z = {0., 0.};
            fc0 = z;
            ft0 = z;
            nrm0 = z;
        } else {
            fc0 = ld_stream(&A.fc[src]);
            ft0 = ld_stream(&A.ft[src]);
            nrm0 = ld_stream(&A.n[src]);
        }
    } else {
        pos = B.pos[i];
        vel = B.vel[i];
        S = B.S[i];
        rho = B.rho[i];
        T = B.T[i];
        eps_pl = B.eps_pl[i];
        eps_pl_dot = B.eps_pl_dot[i];
        fc0 = B.fc[i];
        ft0 = B.ft[i];
        nrm0 = B.n[i];
        on_seg0 = B.on_seg[i];
    }
    double blanked = blanked0;
    sphfem_double2 fc = fc0, ft = ft0, nrm = nrm0;
    int on_seg = on_seg0;
    bool contact_written = false;
    bool near = false;
    sphfem_double2 pos_t = {0., 0.}, vel_t = {0., 0.};
    sphfem_double4 S_t = {0., 0., 0., 0.};
    double rho_t = 0., T_t = 0.;
    if (live) {
        pos_t = r.pos_t;
        vel_t = r.vel_t;
        if constexpr (F32C) T_t = thermal_alpha != 0. ? thermal_alpha * r.T_lapl : (double)Tt_old;
        else T_t = thermal_alpha != 0. ? thermal_alpha * r.T_lapl : A.T_t[A.idx[i]];
        if (tool == 0.) {
            S_t = jaumann_rate(c, r.v_der, S);        // actions_gpu.cu:280-314
            rho_t = -rho * (r.v_der.x + r.v_der.w);     // :626-639
            const double mass = c.phys.mass;            // :641-671
            // x / mass is x itself for x = +-0 (mass > 0): far from the tool the contact forces are
            // zero and their divisions are skipped, with the same sums
            sphfem_double2 fcm = fc, ftm = ft;
            if (fc.x != 0. || fc.y != 0. || ft.x != 0. || ft.y != 0.) {
                fcm = {fc.x / mass, fc.y / mass};
                ftm = {ft.x / mass, ft.y / mass};
            }
            vel_t.x += r.S_der.x + r.S_der.y + fcm.x + ftm.x;
            vel_t.y += r.S_der.z + r.S_der.w + fcm.y + ftm.y;
            pos_t.x = pos_t.x + vel.x;                  // :673-687
            pos_t.y = pos_t.y + vel.y;
        }
        if (write_intermediates) {
            A.S_der[i] = r.S_der;
            A.v_der[i] = r.v_der;
        }
        // leap_frog.cu:71-96
        const double dt = c.dt;
        const sphfem_double2 p0 = F32C ? pos : pos_init[i];
        if constexpr (!F32C) {
            v0 = vel_init[i];
            S0 = S_init[i];
            rho0 = rho_init[i];
        }
        const double T0 = F32C ? T : T_init[i];
        pos.x = p0.x + dt * pos_t.x;
        pos.y = p0.y + dt * pos_t.y;
        vel.x = v0.x + dt * vel_t.x;
        vel.y = v0.y + dt * vel_t.y;
        S.x = S0.x + dt * S_t.x;
        S.y = S0.y + dt * S_t.y;
        S.z = S0.z + dt * S_t.z;
        S.w = S0.w + dt * S_t.w;
        rho = rho0 + dt * rho_t;
        T = T0 + dt * T_t;
        if (tv.active) {
            if (!fric_heat_v21(c, tv, *tv.kin, i, eps_pl, ft, on_seg, nrm, vel, fc, rho, T)) blanked = 1.;
        }
        if constexpr (RIGID) {
            if (c.fric_heat && tool == 0.) T = rigid_fric_heat(c, rt->g.vel, vel, ft, nrm, T);
        }
        if (c.plastic && tool == 0. && blanked != 1.) {
            if (plasticity_jc(c, S, F32C ? pr : B.p[i], eps_pl, eps_pl_dot, T, rho)) blanked = 1.;
        }
        // contact s1 for particles outside the 1.05 ref_dist disc of the moved tool
        // (actions_gpu.cu:438-453); the others are finished by the near-tool pass
        if (tv.active && blanked != 1.) {
            ToolKin k = *tv.kin;
            k.tl_x += k.vel_x * dt;
            k.tl_y += k.vel_y * dt;
            if (near_tool(k, pos)) {
                near = true;
                int slot = atomicAdd(tv.near_count, 1);
                tv.near_list[slot] = i;
            } else {
                sphfem_double2 z = {0., 0.};
                fc = z; ft = z; nrm = z;
                on_seg = -1;
                contact_written = true;
            }
        }
    } else if constexpr (RIGID) {
        if (c.fric_heat && tool == 0.) T = rigid_fric_heat(c, rt->g.vel, vel, ft, nrm, T);
    }
    if constexpr (RIGID) {
        if (tool != 0.) {
            pos.x += c.dt * rt->g.vel.x;
            pos.y += c.dt * rt->g.vel.y;
        } else {
            rigid_contact(*rt, c.dt, pos, vel, ft0, fc, ft, nrm);
            contact_written = true;
        }
    }
    if (!near) {
        // actions_gpu.cu:765-781, 756-763, 787-824
        if (tool == 0. && fixed != 0.) {
            sphfem_double2 z = {0., 0.};
            vel = z;
            fc = z;
            pos_t = z;
            vel_t = z;
            contact_written = true;
        }
        if (c.thermal_bc && fixed == 1.) T = c.trml_wp.T_init;
        if (blanked != 1. && live) {
            bool bad = isnaninf(pos_t.x) || isnaninf(pos_t.y) || isnaninf(vel_t.x) || isnaninf(vel_t.y) ||
                       isnaninf(S_t.x) || isnaninf(S_t.y) || isnaninf(S_t.z) || isnaninf(S_t.w) ||
                       isnaninf(rho_t) || isnaninf(T_t);
            if (bad) blanked = 1.;
        }
    }
    if constexpr (F32C) {
        // the new rates in sorted order, FP32 (the pair sums they come from are FP32)
        st_maybe_stream<NT>(&r_new.pos_t[i], make_float2((float)pos_t.x, (float)pos_t.y));
        st_maybe_stream<NT>(&r_new.vel_t[i], make_float2((float)vel_t.x, (float)vel_t.y));
        st_maybe_stream<NT>(&r_new.S_t[i], make_float4((float)S_t.x, (float)S_t.y, (float)S_t.z, (float)S_t.w));
        st_maybe_stream<NT>(&r_new.rho_t[i], (float)rho_t);
        st_maybe_stream<NT>(&r_new.T_t[i], (float)T_t);
    } else {
        B.pos_t[i] = pos_t;
        B.vel_t[i] = vel_t;
        B.S_t[i] = S_t;
        B.rho_t[i] = rho_t;
        B.T_t[i] = T_t;
    }
    const sphfem_particles &O = F32C ? B : A;
    st_maybe_stream<NT>(&O.pos[i], pos);
    st_maybe_stream<NT>(&O.vel[i], vel);
    st_maybe_stream<NT>(&O.S[i], S);
    st_maybe_stream<NT>(&O.rho[i], rho);
    st_maybe_stream<NT>(&O.T[i], T);
    st_maybe_stream<NT>(&O.eps_pl[i], eps_pl);
    st_maybe_stream<NT>(&O.eps_pl_dot[i], eps_pl_dot);
    st_maybe_stream<NT>(&O.blanked[i], blanked);
    if constexpr (F32C) {
        // the sorted copy of every remaining field; p of tool particles stays at its array position,
        // as the reference neither gathers p nor computes it for them
        st_maybe_stream<NT>(&B.fc[i], fc);
        st_maybe_stream<NT>(&B.ft[i], ft);
        st_maybe_stream<NT>(&B.n[i], nrm);
        st_maybe_stream<NT>(&B.on_seg[i], on_seg);
        st_maybe_stream<NT>(&B.h[i], h_src);
        st_maybe_stream<NT>(&B.fixed[i], fixed);
        st_maybe_stream<NT>(&B.tool_particle[i], tool);
        st_maybe_stream<NT>(&B.p[i], tool == 0. ? pr : A.p[i]);
    } else if (contact_written && (fc.x != fc0.x || fc.y != fc0.y || ft.x != ft0.x || ft.y != ft0.y ||
                                   nrm.x != nrm0.x || nrm.y != nrm0.y || on_seg != on_seg0)) {
        // contact fields in place, written only when they change (far from the tool they stay zero)
        B.fc[i] = fc;
        B.ft[i] = ft;
        B.n[i] = nrm;
        B.on_seg[i] = on_seg;
    }
}

struct PairOut {           // one particle's FP32C sums: psum[i], psum[N + i], psum_T[i]
    float4 g, a;
    float T;
};

template <int BS, int CHUNK, bool GEN, bool SPECIAL, bool ROLL, class Pos = GlobalPos>
__device__ __forceinline__ PairOut pairs_fp32c_one(const DevConsts &c, const int *__restrict__ hash, int N,
                                                   const RecView &rv,
                                                   const int *__restrict__ cs, const int *__restrict__ ce, int i,
                                                   typename Pos::Entry *__restrict__ list, const Pos &pos,
                                                   int *__restrict__ flags, int form) {
#pragma clang fp contract(fast)
    // of a window's candidates the blanked ones are left out by their records; a finite position near its cell
    // (one that is not sets AWAY) lies where the wrapped one says
    const bool win = SPECIAL && (form & SPHFEM_FORM_WINDOW), tests = SPECIAL && (form & ~SPHFEM_FORM_WIDTH);
    const bool wide = SPECIAL && (form & (SPHFEM_FORM_AWAY | SPHFEM_FORM_REACH));
    double d_v0 = 0., d_v1 = 0., d_v2 = 0., d_v3 = 0.;
    double d_ax = 0., d_ay = 0., d_p0 = 0., d_p1 = 0., d_T = 0.;
    const float4 a3 = rv.r3[i];
    // tool particles (negative volume) sum only the Laplacian of T, and only when the tool's
    // thermal block of the pair sums is set (interactions_gpu.cu:157-164, 260-262); blanked
    // particles are skipped
    const bool tool_i = a3.x < 0.f;
    const double alpha_i = tool_i ? c.trml_itool.alpha : c.trml_wp.alpha;
    const double dxc = c.geom.dx;
    const double hi = GEN ? (double)rv.h[i] * (dxc / (double)(1 << SPHFEM_POS_BITS)) : dxc;
    // nor does one whose key names no cell (the records' kernel reported it): its window's entries are read
    // before their columns are known to exist
    const int nx = c.geom.nx, ny = c.geom.ny;
    const int hashi = hash[i];
    if (a3.z != -INFINITY && (!tool_i || alpha_i != 0.) && (unsigned)hashi < (unsigned)(nx * ny)) {
        const int gi = hashi / ny;
        const int gj = hashi - gi * ny;
        const int low_j = gj - 2 < 0 ? 0 : gj - 2;
        const int high_j = gj + 3 > ny ? ny : gj + 3;
        // cell-table entries of a column's window: its lowest and highest row decide the sorted range
        // unless those cells are empty.  A column's are loaded while the one before it is scanned.
        auto cells = [&](int col, int &lo_s, int &hi_s, int &hi_e) {
            const bool ok = col >= 0 && col < nx;
            const int c0 = (ok ? col : gi) * ny;
            lo_s = cs[c0 + low_j];
            hi_s = cs[c0 + high_j - 1];
            hi_e = ce[c0 + high_j - 1];
            if (!ok) lo_s = hi_s = -1;
        };
        int lo_s, hi_s, hi_e;
        cells(gi - 2, lo_s, hi_s, hi_e);
        const int2 a0 = rv.pos[i];
        const float4 a1 = rv.r1[i], a2 = rv.r2[i];
        PairI I;
        I.xi = a0.x; I.yi = a0.y;
        I.vxi = a1.x; I.vyi = a1.y; I.sxi = a1.z; I.syi = a1.w;
        I.szi = a2.x; I.Rxi = a2.y; I.Ryi = a2.z; I.Rzi = a2.w;
        I.rhoi = a3.y; I.ci = a3.z; I.Ti = a3.w;
        I.thermal = alpha_i != 0.;
        I.mech = !tool_i;
        I.kf = (float)(16. * SPHFEM_PI_FAC / (hi * hi * c.corr.wdeltap));
        const double inv_u = (double)(1 << SPHFEM_POS_BITS) / dxc;
        I.D2min = (float)(c.rr2_min * inv_u * inv_u);
        I.beta2 = (float)(2. * c.corr.beta);
        if constexpr (GEN) {
            I.H = rv.h[i];
            I.ku = 1.f / I.H;
            I.D2max = 4.f * I.H * I.H;
            I.D2heat = (float)(1e-16 * inv_u * inv_u);
            I.eta2 = (float)(c.corr.eta * c.corr.eta);
            if (wide) {
                const double2 x = wide_pos(rv, ny, i, hashi);
                I.xd = x.x;
                I.yd = x.y;
            }
        } else {
            I.D2max = 4.f / (KU * KU);
            I.eta2 = (float)(c.corr.eta * c.corr.eta / (double)KU);      // on the scale of D2 * KU
        }

        auto flush = [&](PairAcc &a) {
            d_v0 += a.v0; d_v1 += a.v1; d_v2 += a.v2; d_v3 += a.v3;
            d_ax += a.ax; d_ay += a.ay; d_p0 += a.p0; d_p1 += a.p1; d_T += a.T;
            a = PairAcc{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        };
        auto distance = [&](unsigned j, int2 p, float &dx, float &dy) {
            if (SPECIAL && wide) {
                const double2 x = wide_pos(rv, ny, (int)j, hash[j]);
                dx = (float)(I.xd - x.x);
                dy = (float)(I.yd - x.y);
            } else {
                dx = (float)(int)((unsigned)I.xi - (unsigned)p.x);       // modulo 2^32
                dy = (float)(int)((unsigned)I.yi - (unsigned)p.y);
            }
        };
        auto term = [&](typename Pos::Entry e, const int2 q0, const float4 q1, const float4 q2, const float4 q3,
                        float Hj, PairAcc &acc) {
            float dx, dy;
            distance(pos.index(e), q0, dx, dy);
            pair_term<GEN>(I, dx, dy, q1, q2, q3, Hj, win, acc);
        };
        auto width = [&](unsigned byte_off) {      // of the record at this offset of a block of 16-byte ones
            if constexpr (!GEN) return 0.f;
            else return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(rv.h) + (byte_off >> 2));
        };
        // dense list of the entries in front of list[end]: two per iteration, the records of the next
        // entry loaded before the current one is evaluated (ping-pong registers, no copies); each list
        // entry is read from LDS one pair term before its records are loaded, so the LDS latency passes
        // under that term.  The two entries past the end, which are loaded and not evaluated, repeat the
        // last one (i itself need not be among the records that Pos holds, if the cell table leaves it out).
        auto run_list = [&](int end) {
            if (end <= 0) return;
            PairAcc acc{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            list[end] = list[end + BS] = list[end - BS];
            typename Pos::Entry eA = list[0];
            typename Pos::Entry eB = list[BS];
            unsigned oA = pos.index(eA) << 4;
            int2 A0 = pos.entry(eA);
            float4 A1 = ldrec(rv.r1, oA), A2 = ldrec(rv.r2, oA), A3 = ldrec(rv.r3, oA);
            float Ah = width(oA);
            for (int k = 0; k < end; k += 2 * BS) {
                const typename Pos::Entry eA_next = list[k + 2 * BS];
                const unsigned oB = pos.index(eB) << 4;
                const int2 B0 = pos.entry(eB);
                const float4 B1 = ldrec(rv.r1, oB), B2 = ldrec(rv.r2, oB), B3 = ldrec(rv.r3, oB);
                const float Bh = width(oB);
                term(eA, A0, A1, A2, A3, Ah, acc);
                if (k + BS < end) {
                    const typename Pos::Entry eB_next = list[k + 3 * BS];
                    eA = eA_next;
                    oA = pos.index(eA) << 4;
                    A0 = pos.entry(eA);
                    A1 = ldrec(rv.r1, oA); A2 = ldrec(rv.r2, oA); A3 = ldrec(rv.r3, oA);
                    Ah = width(oA);
                    term(eB, B0, B1, B2, B3, Bh, acc);
                    eB = eB_next;
                }
                if (((k + 2 * BS) & (8 * BS - 1)) == 0) flush(acc);
            }
            flush(acc);
        };

        int end = 0;               // BS times the number of entries
#pragma unroll ROLL ? 1 : 5
        for (int d = 0; d < 5; d++) {
            const int col = gi - 2 + d;
            int first = lo_s, last = hi_s != -1 ? hi_e : -1;
            if (d < 4) cells(col + 1, lo_s, hi_s, hi_e);
            if (col < 0 || col >= nx) continue;
            const int c0 = col * ny;
            for (int jr = low_j + 1; first == -1 && jr < high_j; jr++) first = cs[c0 + jr];
            if (first == -1) continue;                                   // empty window
            for (int jr = high_j - 2; last == -1 && jr >= low_j; jr--)
                if (cs[c0 + jr] != -1) last = ce[c0 + jr];
            if (last > N || first < 0) continue;                        // inconsistent cell table
            if (!pos.clip(d, first, last)) atomicOr(&flags[0], 4);
            for (int j = first; j < last; j += 4) {
                // four positions; up to three past `last` are read (both sources are padded)
                int2 b[4];
                pos.scan4(d, j, b);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (SPECIAL && tests && (j + u >= last || rv.r3[j + u].z == -INFINITY)) continue;
                    float dx, dy;
                    distance((unsigned)(j + u), b[u], dx, dy);
                    const float D2 = dx * dx + dy * dy;
                    if (j + u < last && (win || (D2 < I.D2max && D2 >= I.D2min))) {
                        list[end] = pos.encode(d, j + u);
                        end += BS;
                    }
                }
                // dense region: every active lane empties its list at once (a lane emptying its
                // list alone runs it with the rest of the wavefront idle)
                if (__any(end > (CHUNK - 4) * BS)) {
                    run_list(end);
                    end = 0;
                }
            }
        }
        run_list(end);
    }
    // the factors of the kernel gradient, -3 fac / h, and of its value, 16 fac; the heat term holds the
    // gradient over the distance, in units of u
    const double mass = c.phys.mass;
    const double h1 = 1. / hi, fac = SPHFEM_PI_FAC * h1 * h1, grad = -3. * fac * h1;
    const double ma = mass * grad, xs = -32. * c.corr.xspheps * mass * fac;
    const double heat = 2. * grad * (double)(1 << SPHFEM_POS_BITS) / dxc;
    PairOut o;
    o.g = make_float4((float)(grad * d_v0), (float)(grad * d_v1), (float)(grad * d_v2), (float)(grad * d_v3));
    o.a = make_float4((float)(ma * d_ax), (float)(ma * d_ay), (float)(xs * d_p0), (float)(xs * d_p1));
    o.T = (float)(heat * d_T);
    return o;
}

// Where a pair kernel's sums go: psum / psum_T, read by the update kernel; straight into the particle's
// update (the update needs no other particle's sums); or the reference's interaction outputs
// (interactions_gpu.cu:370-378): v_der; the stress-divergence plus viscous acceleration per axis as
// S_der = {ax, 0, ay, 0} with vel_t = 0 (the momentum equation only uses S_der.x + S_der.y + vel_t.x and
// S_der.z + S_der.w + vel_t.y); XSPH in pos_t; alpha times the Laplacian in T_t where the thermal block
// is set.  Those of blanked particles are left untouched, as by the reference.
enum PairsTo { TO_PSUM, TO_UPDATE, TO_OUTPUTS };
template <int TO, bool RIGID>
__device__ __forceinline__ void emit_pairs(const DevConsts &c, const UpdateArgs &u, float4 *__restrict__ psum,
                                           float *__restrict__ psum_T, int N, int i, const PairOut &o) {
    if constexpr (TO == TO_UPDATE) {
        update_item<true, RIGID, true>(c, u, i, o.g, o.a, o.T);
    } else if constexpr (TO == TO_OUTPUTS) {
        const sphfem_particles &P = u.B;
        if (P.blanked[i] == 1.) return;
        const double alpha = interaction_alpha(c, P.tool_particle[i]);
        // streaming, as the update's stores: the records other wavefronts still read stay in L2
        st_maybe_stream<true>(&P.v_der[i], sphfem_double4{o.g.x, o.g.y, o.g.z, o.g.w});
        st_maybe_stream<true>(&P.S_der[i], sphfem_double4{o.a.x, 0., o.a.y, 0.});
        st_maybe_stream<true>(&P.vel_t[i], sphfem_double2{0., 0.});
        st_maybe_stream<true>(&P.pos_t[i], sphfem_double2{o.a.z, o.a.w});
        if (alpha != 0.) P.T_t[i] = alpha * (double)o.T;
    } else {
        psum[i] = o.g;
        psum[(size_t)N + i] = o.a;
        psum_T[i] = o.T;
    }
}

// in-support pair sums, one lane per sorted particle, in the form that the form words ask for.  TO: what
// each lane does with its particle's sums (emit_pairs).
__device__ __forceinline__ int pairs_form(const DevConsts &c, const int *__restrict__ form) {
    // a support that reaches below the heat term's least distance needs the test of the general form
    int f = c.rr2_min > 1e-16 ? 0 : SPHFEM_FORM_WIDTH;
    for (int k = 0; k < SPHFEM_FORM_WORDS; k++) f |= form[k] != 0 ? 1 << k : 0;
    return f;
}

// the list kernel's sums of particle i, in the given form.  Fused with the update there are two forms in the
// kernel, the tests switched by uniform branches: a third one takes it from 166 to 168 registers and costs the
// first form 3 % (1 M particles: 260 -> 269 us a step)
template <int BS, int CHUNK, int TO>
__device__ __forceinline__ PairOut pairs_fp32c_list(const DevConsts &c, const int *__restrict__ hash, int N,
                                                    const RecView &rv, const int *__restrict__ cs,
                                                    const int *__restrict__ ce, int i, int *__restrict__ list,
                                                    int form) {
    const GlobalPos pos{rv.pos};
    if (form == 0)
        return pairs_fp32c_one<BS, CHUNK, false, false, TO != TO_UPDATE>(c, hash, N, rv, cs, ce, i, list, pos, nullptr,
                                                                         0);
    if (TO != TO_UPDATE && form == SPHFEM_FORM_WIDTH)
        return pairs_fp32c_one<BS, CHUNK, true, false, true>(c, hash, N, rv, cs, ce, i, list, pos, nullptr, form);
    return pairs_fp32c_one<BS, CHUNK, true, true, true>(c, hash, N, rv, cs, ce, i, list, pos, nullptr, form);
}

template <int BS, int CHUNK, int TO = TO_PSUM, bool RIGID = false>
__global__ void __launch_bounds__(BS) k_pairs_fp32c(DevConsts c, const int *__restrict__ hash, int N, RecView rv,
                                                         const int *__restrict__ cs, const int *__restrict__ ce,
                                                         float4 *__restrict__ psum, float *__restrict__ psum_T,
                                                         const int *__restrict__ form_words, UpdateArgs u) {
    __shared__ int nb_list[(CHUNK + 2) * BS];
    const int form = pairs_form(c, form_words);
    const int i = xcd_logical_block() * BS + threadIdx.x;
    if (i >= N) return;
    const PairOut o = pairs_fp32c_list<BS, CHUNK, TO>(c, hash, N, rv, cs, ce, i, nb_list + threadIdx.x, form);
    emit_pairs<TO, RIGID>(c, u, psum, psum_T, N, i, o);
}

// LDS-staged form of k_pairs_fp32c, one wavefront per workgroup.  When the wavefront's 64
// particles lie in one cell column and the union of their 5x5-cell windows holds at most CAP
// records, the wavefront first copies the position records of that union -- five sorted ranges,
// one per neighbour column, rows [first row - 2, last row + 2] -- into LDS with coalesced loads;
// the candidate scan and the pair terms then read positions from LDS and only the three other
// records of each pair from L2/HBM.  Otherwise (a wavefront across two columns, a larger union, or
// a long run of empty cells) it runs the list kernel's path.  The per-lane loops, votes and FP32
// summation blocks are those of k_pairs_fp32c and both kernels group particles into wavefronts
// alike, so the two give the same sums bit for bit.  All 64 lanes take part in the staging (lanes
// past N copy records but sum nothing); the union comes from the hashes of the wavefront's first and
// last particles, read by every lane from memory, so no lane depends on another lane's registers.
#define SPHFEM_STAGE_ROW_SCAN 64
template <int CHUNK, int CAP, int TO = TO_PSUM, bool RIGID = false>
__global__ void __launch_bounds__(64) k_pairs_fp32c_staged(DevConsts c, const int *__restrict__ hash, int N, RecView rv,
                                                           const int *__restrict__ cs, const int *__restrict__ ce,
                                                           float4 *__restrict__ psum, float *__restrict__ psum_T,
                                                           const int *__restrict__ form_words, int *__restrict__ flags,
                                                           UpdateArgs u) {
    // LDS: staged -- positions [CAP + 4] (+4: the scan reads up to three records past a range) and
    // 16-bit list entries; list path -- 32-bit list entries in the same bytes
    constexpr int POS_BYTES = (CAP + 4) * 8, LIST16 = (CHUNK + 2) * 64 * 2, LIST32 = (CHUNK + 2) * 64 * 4;
    constexpr int LDS_BYTES = POS_BYTES + LIST16 > LIST32 ? POS_BYTES + LIST16 : LIST32;
    __shared__ __align__(16) unsigned char lds[LDS_BYTES];
    __shared__ int sdelta[8];
    int2 *spos = reinterpret_cast<int2 *>(lds);
    unsigned short *list16 = reinterpret_cast<unsigned short *>(lds + POS_BYTES);
    int *list32 = reinterpret_cast<int *>(lds);
    const int form = pairs_form(c, form_words);
    const int base = xcd_logical_block() * 64;
    if (base >= N) return;                              // the whole wavefront
    const int lane = (int)threadIdx.x;
    const int i = base + lane;
    const int last_i = base + 63 < N ? base + 63 : N - 1;
    const int nx = c.geom.nx, ny = c.geom.ny;
    const int h0 = hash[base], h1 = hash[last_i];
    const int col0 = h0 / ny;
    StagedPos sp;
    sp.spos = spos;
    sp.sdelta = sdelta;
    bool staged = form == 0 && h0 >= 0 && h1 >= h0 && h1 / ny == col0 && col0 < nx;
    int total = 0;
    if (staged) {
        const int r_lo = h0 - col0 * ny - 2 < 0 ? 0 : h0 - col0 * ny - 2;
        const int r_hi = h1 - col0 * ny + 2 > ny - 1 ? ny - 1 : h1 - col0 * ny + 2;
        // the end cells of the five row ranges, loaded together; runs of empty cells are scanned
        // only where an end cell is empty
        int lo_s[5], hi_s[5], hi_e[5];
#pragma unroll
        for (int d = 0; d < 5; d++) {
            const int col = col0 - 2 + d;
            const bool ok = col >= 0 && col < nx;
            const int c0 = (ok ? col : col0) * ny;
            lo_s[d] = ok ? cs[c0 + r_lo] : -1;
            hi_s[d] = ok ? cs[c0 + r_hi] : -1;
            hi_e[d] = ok ? ce[c0 + r_hi] : -1;
        }
#pragma unroll
        for (int d = 0; d < 5; d++) {
            const int col = col0 - 2 + d;
            int F = 0, L = 0;
            if (col >= 0 && col < nx) {
                const int c0 = col * ny;
                // first and last non-empty cell of the rows [r_lo, r_hi] (empty cells hold -1)
                int r = r_lo, f = lo_s[d];
                while (f == -1 && r < r_hi && r - r_lo < SPHFEM_STAGE_ROW_SCAN) f = cs[c0 + ++r];
                if (f != -1) {
                    int l = hi_s[d] != -1 ? hi_e[d] : -1, r2 = r_hi;
                    while (l == -1 && r2 > r && r_hi - r2 < SPHFEM_STAGE_ROW_SCAN)
                        if (cs[c0 + --r2] != -1) l = ce[c0 + r2];
                    if (l == -1) staged = false;                 // the downward scan gave up
                    F = f;
                    L = l;
                } else if (r < r_hi) {
                    staged = false;                              // the upward scan gave up
                }
                if (F < 0 || L > N || L < F) staged = false;     // inconsistent cell table
            }
            sp.F[d] = F;
            sp.L[d] = L;
            sp.delta[d] = F - total;
            total += L - F;
        }
        if (total > CAP) staged = false;
    }
    if (staged) {
#pragma unroll
        for (int d = 0; d < 5; d++) {
            if (lane == d) sdelta[d] = sp.delta[d];
            const int n = sp.L[d] - sp.F[d], off = sp.F[d] - sp.delta[d];
            for (int k = lane; k < n; k += 64) spos[off + k] = rv.pos[sp.F[d] + k];
        }
        __syncthreads();
    }
    if (i >= N) return;
    PairOut o;
    if (staged)
        o = pairs_fp32c_one<64, CHUNK, false, false, false, StagedPos>(c, hash, N, rv, cs, ce, i, list16 + lane, sp,
                                                                       flags, 0);
    else
        o = pairs_fp32c_list<64, CHUNK, TO>(c, hash, N, rv, cs, ce, i, list32 + lane, form);
    emit_pairs<TO, RIGID>(c, u, psum, psum_T, N, i, o);
}

// interactions_gpu.cu:143-379 for the drop-in entry point, first kernel: the neighbour factors of
// k_pairs_fp64's pair loop from the arrays as they stand (the same operations the reference repeats
// per pair), and the switch to the reference's full window: a live particle with a non-finite input
// or factor, or out of the range of pair_inputs_in_range (a zero kernel value times such a factor is not
// zero).
__global__ void __launch_bounds__(256) k_pre_state(DevConsts c, const sphfem_particles P, const PreView pre,
                                                   int *__restrict__ window, int *__restrict__ next_window) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *next_window = 0;         // the first form word; this call knows no others
    if (i >= (int)P.N) return;
    const double rho = P.rho[i], pr = P.p[i];
    const sphfem_double4 S = P.S[i], R = P.R[i];
    const sphfem_double2 pos = P.pos[i], vel = P.vel[i];
    const double blanked = P.blanked[i], T = P.T[i], h = P.h[i];
    const double vol = c.phys.mass / rho;
    const double rho21 = 1. / (rho * rho);
    const sphfem_double4 f = {(S.x - pr) * rho21, S.y * rho21, (S.z - pr) * rho21, sqrtf_d(c.phys.K / rho)};
    pre.pos[i] = scan_pos(blanked, pos);
    pre.vr[i] = {vol, P.tool_particle[i] == 1. ? -rho : rho};
    pre.s1[i] = {f.x, f.y};
    pre.s2[i] = {f.z, f.w};
    pre.r1[i] = {R.x, R.y};
    pre.r2[i] = {R.z, T};
    const double s = ((pos.x + pos.y) + (vel.x + vel.y)) + ((T + h) + (R.x + R.y)) + (R.z + vol) +
                     ((f.x + f.y) + (f.z + f.w));
    if (blanked != 1. && !(isfinite(s) && pair_inputs_in_range(rho, vel))) *window = 1;
}

// second kernel: the pair sums in the reference's arithmetic and neighbour order.  With finite inputs
// the candidates outside the support add exact zeros and are skipped; otherwise (`window`) every
// particle of the 5x5 cells is evaluated, as the reference visits them.  Bound by the neighbour gathers
// and the FP64 arithmetic of the in-support pairs: evaluating the whole window instead (about twice
// the pairs, with each neighbour's factors divided out again per pair) took 3106 us per launch at
// 2.07M particles of the chip domain, this and k_pre_state 2140 us, 2010 us with the shared reciprocals,
// 1320 us with the fields in 16-byte records, 1360 us with extreme dividends divided plainly (pair_sums_fp64).
__global__ void __launch_bounds__(256) k_interactions_ref(DevConsts c, sphfem_particles P, const int *__restrict__ cs,
                                                          const int *__restrict__ ce,
                                                          const PreView pre,
                                                          const int *__restrict__ window) {
    __shared__ int nb_list[48 * 256];
    const int pidx = xcd_logical_block() * 256 + (int)threadIdx.x;
    if (pidx >= (int)P.N) return;
    if (P.blanked[pidx] == 1.) return;
    const double thermal_alpha = interaction_alpha(c, P.tool_particle[pidx]);
    PairSums r;
    if (*window != 0)
        r = pair_sums_fp64<256, 48, true>(c, P, pidx, thermal_alpha, cs, ce, pre,
                                                nb_list + threadIdx.x);
    else
        r = pair_sums_fp64<256, 48, false>(c, P, pidx, thermal_alpha, cs, ce, pre,
                                                 nb_list + threadIdx.x);
    P.S_der[pidx] = r.S_der;
    P.v_der[pidx] = r.v_der;
    P.pos_t[pidx] = r.pos_t;
    P.vel_t[pidx] = r.vel_t;
    if (thermal_alpha != 0.) P.T_t[pidx] = thermal_alpha * r.T_lapl;
}

// interactions_gpu.cu:84-140 with lapl_pse (kernels.cuh:67-84): particle strength exchange heat
// conduction over every particle of the 5x5 cells (no support cut-off; blanked neighbours count),
// the column-run order being the reference's cell order
__global__ void __launch_bounds__(256) k_interactions_pse(DevConsts c, sphfem_particles P, const int *__restrict__ cs,
                                                          const int *__restrict__ ce) {
    const int pidx = blockIdx.x * blockDim.x + threadIdx.x;
    if (pidx >= (int)P.N) return;
    if (P.blanked[pidx] == 1.) return;
    const double mass = c.phys.mass;
    const int nx = c.geom.nx, ny = c.geom.ny;
    const sphfem_double2 pi = P.pos[pidx];
    const double hi = P.h[pidx], Ti = P.T[pidx];
    // the host copies of interactions_gpu.cu:453 (the tool's is zero unless
    // interactions_setup_thermal_constants_tool was called)
    const double alpha = (P.tool_particle[pidx] == 1.) ? c.itool_alpha_pse : c.trml_wp.alpha;
    const int hashi = P.hash[pidx];
    const int gi = hashi / ny;
    const int gj = hashi - gi * ny;
    const int low_i = gi - 2 < 0 ? 0 : gi - 2;
    const int low_j = gj - 2 < 0 ? 0 : gj - 2;
    const int high_i = gi + 3 > nx ? nx : gi + 3;
    const int high_j = gj + 3 > ny ? ny : gj + 3;
    double T_ti = 0.;
    for (int ii = low_i; ii < high_i; ii++) {
        int first, last;
        column_range(cs, ce, ii * ny, low_j, high_j, first, last);
        if (first < 0 || last > (int)P.N) continue;
        for (int iter = first; iter < last; iter++) {
            const sphfem_double2 pj = P.pos[iter];
            const double Tj = P.T[iter], rhoj = P.rho[iter];
            const double xij = pi.x - pj.x, yij = pi.y - pj.y;
            const double xx = sqrt(xij * xij + yij * yij);
            const double h2 = hi * hi;
            const double h4 = h2 * h2;
            const double w2 = +4. / (h4 * 3.14159265358979323846) * exp(-xx * xx / (h2));
            T_ti += (Tj - Ti) * w2 * mass / rhoj;
        }
    }
    P.T_t[pidx] = alpha * T_ti;
}

void launch_interactions_pse(sphfem_ctx *ctx, const sphfem_particles &p, const int *cs, const int *ce) {
    KTimer t(ctx, "interactions_pse");
    k_interactions_pse<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(ctx->c, p, cs, ce);
}

void launch_interactions_ref(sphfem_ctx *ctx, const sphfem_particles &p, const int *cs, const int *ce) {
    int *window = ctx->d_flags + SPHFEM_FLAG_MONAGHAN + ctx->monaghan_turn * SPHFEM_FORM_WORDS;
    ctx->monaghan_turn ^= 1;
    int *next_window = ctx->d_flags + SPHFEM_FLAG_MONAGHAN + ctx->monaghan_turn * SPHFEM_FORM_WORDS;
    {
        KTimer t(ctx, "interactions_pre");
        k_pre_state<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(ctx->c, p, pre_view(ctx->pre, p.N), window, next_window);
    }
    KTimer t(ctx, "interactions_ref");
    k_interactions_ref<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(ctx->c, p, cs, ce, pre_view(ctx->pre, p.N),
                                                                window);
}

// ---------------------------------------------------------------------------------------------
// per-reference-function kernels (actions_gpu.cu)
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_action(DevConsts c, sphfem_particles P, int which) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int)P.N) return;
    switch (which) {
    case ACT_EOS:   // :222-232
        if (P.tool_particle[i] != 0.) return;
        P.p[i] = eos_pressure(c, P.rho[i]);
        break;
    case ACT_ARTSTRESS:   // :234-278
        if (P.tool_particle[i] != 0.) return;
        P.R[i] = artificial_stress(c, P.rho[i], P.p[i], P.S[i]);
        break;
    case ACT_JAUMANN:   // :280-314
        if (P.tool_particle[i] == 1.) return;
        P.S_t[i] = jaumann_rate(c, P.v_der[i], P.S[i]);
        break;
    case ACT_CONTINUITY:   // :626-639
        if (P.tool_particle[i] != 0.) return;
        P.rho_t[i] = -P.rho[i] * (P.v_der[i].x + P.v_der[i].w);
        break;
    case ACT_MOMENTUM: {   // :641-671
        if (P.tool_particle[i] != 0.) return;
        const double mass = c.phys.mass;
        sphfem_double4 sd = P.S_der[i];
        sphfem_double2 fc = P.fc[i], ft = P.ft[i], vt = P.vel_t[i];
        vt.x += sd.x + sd.y + fc.x / mass + ft.x / mass;
        vt.y += sd.z + sd.w + fc.y / mass + ft.y / mass;
        P.vel_t[i] = vt;
        break;
    }
    case ACT_ADVECTION: {   // :673-687
        if (P.tool_particle[i] != 0.) return;
        sphfem_double2 pt = P.pos_t[i], v = P.vel[i];
        pt.x = pt.x + v.x;
        pt.y = pt.y + v.y;
        P.pos_t[i] = pt;
        break;
    }
    case ACT_PLASTICITY: {   // :689-754
        if (P.tool_particle[i] != 0.) return;
        if (P.blanked[i] == 1.) return;
        sphfem_double4 S = P.S[i];
        double eps = P.eps_pl[i], epsd = P.eps_pl_dot[i], T = P.T[i];
        double S_in[4] = {S.x, S.y, S.z, S.w};
        bool melt = plasticity_jc(c, S, P.p[i], eps, epsd, T, P.rho[i]);
        P.eps_pl_dot[i] = epsd;
        if (S.x != S_in[0] || S.y != S_in[1] || S.z != S_in[2] || S.w != S_in[3] || eps != P.eps_pl[i]) {
            P.eps_pl[i] = eps;
            P.S[i] = S;
        }
        P.T[i] = T;
        if (melt) P.blanked[i] = 1.;
        break;
    }
    case ACT_BC:   // :765-781
        if (P.tool_particle[i] != 0.) return;
        if (P.fixed[i] != 0.) {
            sphfem_double2 z = {0., 0.};
            P.vel[i] = z;
            P.fc[i] = z;
            P.pos_t[i] = z;
            P.vel_t[i] = z;
        }
        break;
    case ACT_BC_THERMAL:   // :756-763
        if (P.fixed[i] == 1.) P.T[i] = c.trml_wp.T_init;
        break;
    case ACT_INVALIDATE: {   // :787-824
        if (P.blanked[i] == 1.) return;
        sphfem_double2 pt = P.pos_t[i], vt = P.vel_t[i];
        sphfem_double4 st = P.S_t[i];
        bool bad = isnaninf(pt.x) || isnaninf(pt.y) || isnaninf(vt.x) || isnaninf(vt.y) || isnaninf(st.x) ||
                   isnaninf(st.y) || isnaninf(st.z) || isnaninf(st.w) || isnaninf(P.rho_t[i]) || isnaninf(P.T_t[i]);
        if (bad) P.blanked[i] = 1.;
        break;
    }
    }
}

void launch_actions(sphfem_ctx *ctx, int which, const sphfem_particles &p) {
    static const char *names[] = {"eos", "artificial_stress", "jaumann", "continuity", "momentum", "advection",
                                  "plasticity", "bc", "bc_thermal", "invalidate"};
    KTimer t(ctx, names[which]);
    k_action<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(ctx->c, p, which);
}

// leap_frog.cu:25-96
__global__ void __launch_bounds__(256) k_leapfrog(sphfem_particles P, int which, double dt,
                                                  sphfem_double2 *pos_init, sphfem_double2 *vel_init,
                                                  sphfem_double4 *S_init, double *rho_init, double *T_init) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int)P.N) return;
    if (P.blanked[i] == 1.) return;
    if (which == LF_INIT) {
        pos_init[i] = P.pos[i];
        vel_init[i] = P.vel[i];
        S_init[i] = P.S[i];
        rho_init[i] = P.rho[i];
        T_init[i] = P.T[i];
        return;
    }
    double f = which == LF_PREDICT ? 0.5 * dt : dt;
    sphfem_double2 pt = P.pos_t[i], vt = P.vel_t[i], p0 = pos_init[i], v0 = vel_init[i];
    sphfem_double4 St = P.S_t[i], S0 = S_init[i];
    // predict: x0 + 0.5*dt*x_t, correct: x0 + dt*x_t (same products as the reference)
    P.pos[i] = {p0.x + f * pt.x, p0.y + f * pt.y};
    P.vel[i] = {v0.x + f * vt.x, v0.y + f * vt.y};
    P.S[i] = {S0.x + f * St.x, S0.y + f * St.y, S0.z + f * St.z, S0.w + f * St.w};
    P.rho[i] = rho_init[i] + f * P.rho_t[i];
    P.T[i] = T_init[i] + f * P.T_t[i];
}

void launch_leapfrog(sphfem_ctx *ctx, int which, const sphfem_particles &p, sphfem_leap_frog *lf, double dt) {
    static const char *names[] = {"lf_init", "lf_predict", "lf_correct"};
    KTimer t(ctx, names[which]);
    k_leapfrog<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(p, which, dt, lf->pos_init, lf->vel_init, lf->S_init,
                                                        lf->rho_init, lf->T_init);
}

// ---------------------------------------------------------------------------------------------
// fused step kernel (FP64 form).  B: sorted predicted state (read), A: corrected state (write).
// Fields: A.pos/vel/S/rho/T/eps_pl/eps_pl_dot/blanked are outputs; B.fc/ft/n/on_seg are updated
// in place (own particle only); derivatives go to A.pos_t/vel_t/rho_t/S_t/T_t.
// ---------------------------------------------------------------------------------------------

// B = sorted predicted state (the grid buffer); A = the caller's arrays, whose unsorted content
// is dead after the reorder except the previous derivatives.  Outputs: corrected state into
// A.pos/vel/S/rho/T/eps_pl/eps_pl_dot/blanked, derivatives into B.pos_t/vel_t/rho_t/S_t/T_t,
// contact fields in place in B.fc/ft/n/on_seg; S_der/v_der into A when requested.
// FP64 pair sums of the sorted predicted state (interactions_gpu.cu:143-379) into psum64, for the
// update kernel; a kernel of its own so that the pair loop keeps 3 waves per SIMD instead of the
// update's 2
// nonfinite[0] is set by the reorder when a live particle carries a non-finite pair input: then
// every particle is evaluated with the reference's full window.
template <int BS>
__global__ void __launch_bounds__(BS) k_pairs_fp64(DevConsts c, sphfem_particles B, const int *__restrict__ cs,
                                                   const int *__restrict__ ce, const PreView pre,
                                                   PairSums *__restrict__ psum64, const int *__restrict__ nonfinite) {
    constexpr int CHUNK = 48;
    __shared__ int nb_list[CHUNK * BS];
    const int N = (int)B.N;
    const int i = xcd_logical_block() * BS + (int)threadIdx.x;
    if (i >= N || B.blanked[i] == 1.) return;
    const double thermal_alpha = interaction_alpha(c, B.tool_particle[i]);
    // the window form when a live particle carries a non-finite input (see pair_sums_fp64)
    if (*nonfinite != 0)
        psum64[i] = pair_sums_fp64<BS, CHUNK, true>(c, B, i, thermal_alpha, cs, ce, pre,
                                                          nb_list + threadIdx.x);
    else
        psum64[i] = pair_sums_fp64<BS, CHUNK, false>(c, B, i, thermal_alpha, cs, ce, pre,
                                                           nb_list + threadIdx.x);
}

// RIGID: the rigid-tool step (leap_frog.cu:99-160): friction heat after the corrector
// (actions_gpu.cu:316-343), tool particles moved and contact against the moved tool
// (tool_gpu.cu:146-216) after plasticity, for blanked particles too as in the reference.
// the update as its own kernel, after k_pairs_fp64 or a k_pairs_fp32c that wrote psum
template <bool F32C, int BS, bool RIGID>
__global__ void __launch_bounds__(BS) k_fused_update(DevConsts c, UpdateArgs u, const float4 *__restrict__ psum,
                                                     const float *__restrict__ psum_T, int *__restrict__ nonfinite) {
    const int i = xcd_logical_block() * BS + threadIdx.x;
    if (i == 0) *nonfinite = 0;      // the pair kernels of this step have read it
    if (i >= (int)u.B.N) return;
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f), a = g;
    float tl = 0.f;
    if constexpr (F32C) {
        g = psum[i];                 // sums of k_pairs_fp32c
        a = psum[(size_t)u.B.N + i];
        tl = psum_T[i];
    }
    update_item<F32C, RIGID>(c, u, i, g, a, tl);
}

template <int BSZ, int CH, int TO, bool RIGID>
static void launch_pairs_fp32c(sphfem_ctx *ctx, const sphfem_particles &B, sphfem_leap_frog *lf, const int *cs,
                               const int *ce, const int *form, const UpdateArgs &u) {
    const size_t n = B.N;
    const RecView rv = rec_view(lf->rec, n);
    k_pairs_fp32c<BSZ, CH, TO, RIGID><<<nblk(B.N, BSZ), BSZ, 0, ctx->stream>>>(
        ctx->c, B.hash, (int)B.N, rv, cs, ce, lf->psum, lf->psum_T, form, u);
}

template <int CH, int TO, bool RIGID>
static void launch_pairs_fp32c_staged(sphfem_ctx *ctx, const sphfem_particles &B, sphfem_leap_frog *lf, const int *cs,
                                      const int *ce, const int *form, const UpdateArgs &u) {
    const size_t n = B.N;
    const RecView rv = rec_view(lf->rec, n);
    k_pairs_fp32c_staged<CH, SPHFEM_STAGE_CAP, TO, RIGID><<<nblk(B.N, 64), 64, 0, ctx->stream>>>(
        ctx->c, B.hash, (int)B.N, rv, cs, ce, lf->psum, lf->psum_T, form, ctx->d_flags, u);
}

template <int TO, bool RIGID>
static void launch_pairs_fp32c_shape(sphfem_ctx *ctx, const sphfem_particles &B, sphfem_leap_frog *lf, const int *cs,
                                     const int *ce, const int *form, const UpdateArgs &u) {
    const int pb = lf->tuning.pair_block, pc = lf->tuning.pair_chunk;
    const int k = lf->tuning.pair_kernel;
    if (k == SPHFEM_PAIRS_STAGED || k == SPHFEM_PAIRS_STAGED_FUSED) {
        if (pc == 16) launch_pairs_fp32c_staged<16, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
        else if (pc == 48) launch_pairs_fp32c_staged<48, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
        else launch_pairs_fp32c_staged<32, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
    } else if (pb == 128 && pc == 16) launch_pairs_fp32c<128, 16, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
    else if (pb == 128 && pc == 32) launch_pairs_fp32c<128, 32, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
    else if (pb == 128 && pc == 48) launch_pairs_fp32c<128, 48, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
    else if (pb == 256 && pc == 16) launch_pairs_fp32c<256, 16, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
    else if (pb == 256 && pc == 48) launch_pairs_fp32c<256, 48, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
    else launch_pairs_fp32c<256, 32, TO, RIGID>(ctx, B, lf, cs, ce, form, u);
}

// the tuned FP32C pair kernel of the step; fuse: it also runs every particle's update, with these
// arguments (the rigid-tool update when fuse->rt is set)
static void launch_pairs_fp32c_tuned(sphfem_ctx *ctx, const sphfem_particles &B, sphfem_leap_frog *lf, const int *cs,
                                     const int *ce, const UpdateArgs *fuse = nullptr) {
    const int *form = ctx->d_flags + SPHFEM_FLAG_FORM;
    if (fuse) {
        KTimer tm(ctx, "pairs_update_fp32c");
        if (fuse->rt) launch_pairs_fp32c_shape<TO_UPDATE, true>(ctx, B, lf, cs, ce, form, *fuse);
        else launch_pairs_fp32c_shape<TO_UPDATE, false>(ctx, B, lf, cs, ce, form, *fuse);
    } else {
        KTimer tm(ctx, "pairs_fp32c");
        launch_pairs_fp32c_shape<TO_PSUM, false>(ctx, B, lf, cs, ce, form, UpdateArgs{});
    }
}

// The pair kernel writes the outputs itself: 3121 us on 16 M particles, against 2827 us for the sums and
// 442 us for a second kernel that read them back and spread them into the outputs.
void launch_interactions_fp32c(sphfem_ctx *ctx, const sphfem_particles &p, sphfem_leap_frog *lf, const int *cs,
                               const int *ce, int num_cell) {
    int *form = ctx->d_flags + SPHFEM_FLAG_MONAGHAN_FP32C + ctx->fp32c_turn * SPHFEM_FORM_WORDS;
    ctx->fp32c_turn ^= 1;
    int *next_form = ctx->d_flags + SPHFEM_FLAG_MONAGHAN_FP32C + ctx->fp32c_turn * SPHFEM_FORM_WORDS;
    launch_records_state(ctx, p, num_cell, rec_view(lf->rec, p.N), form, next_form);
    KTimer tm(ctx, "pairs_fp32c");
    UpdateArgs u{};
    u.B = p;
    launch_pairs_fp32c_shape<TO_OUTPUTS, false>(ctx, p, lf, cs, ce, form, u);
}

void launch_fused_update(sphfem_ctx *ctx, const sphfem_particles &B, const sphfem_particles &A, sphfem_leap_frog *lf,
                         const int *cs, const int *ce, sphfem_tool *t, sphfem_rigid_tool *rt,
                         const RateView *rates_old, const RateView *rates_new, bool skip_contact) {
    const RateView none{};
    const RateView r_old = rates_old ? *rates_old : none, r_new = rates_new ? *rates_new : none;
    const int skip = skip_contact ? 1 : 0;
    ToolView tv{};
    if (t) {
        tv.T_nodes = t->T_half;
        tv.marks = t->marks;
        tv.fric_heat = t->fric_heat;
        tv.physical_para = t->physical_para;
        tv.sliding_force = t->sliding_force;
        tv.kin = t->kin;
        tv.near_list = lf->near_list;
        tv.near_count = ctx->d_flags + 1;
        tv.active = 1;
        tv.sink = SegSink{ctx->d_flags + SPHFEM_FLAG_SINK_FRIC, t->sink_keys, t->sink_vals, SPHFEM_SEG_SINK_CAP};
    }
    const RigidTool *rtd = rt ? rt->dev : nullptr;
    UpdateArgs u{};
    u.B = B;
    u.A = A;
    u.pos_init = lf->pos_init;
    u.vel_init = lf->vel_init;
    u.S_init = lf->S_init;
    u.rho_init = lf->rho_init;
    u.T_init = lf->T_init;
    u.tv = tv;
    u.write_intermediates = lf->intermediates ? 1 : 0;
    u.rt = rtd;
    u.r_old = r_old;
    u.r_new = r_new;
    int *nf = ctx->d_flags + SPHFEM_FLAG_FORM;      // the WINDOW word
    if (lf->precision == SPHFEM_FP32C) {
        u.skip_contact = skip;
        // the fused pair kernels run the update themselves
        const int pk = lf->tuning.pair_kernel;
        if (pk == SPHFEM_PAIRS_LIST_FUSED || pk == SPHFEM_PAIRS_STAGED_FUSED) {
            launch_pairs_fp32c_tuned(ctx, B, lf, cs, ce, &u);
            return;
        }
        launch_pairs_fp32c_tuned(ctx, B, lf, cs, ce);
        KTimer tm(ctx, "update_fp32c");
#define SPHFEM_UPDATE(BSZ, RG)                                                                              \
    k_fused_update<true, BSZ, RG><<<nblk(B.N, BSZ), BSZ, 0, ctx->stream>>>(ctx->c, u, lf->psum, lf->psum_T, nf)
        if (lf->tuning.update_block == 128) {
            if (rtd) SPHFEM_UPDATE(128, true);
            else SPHFEM_UPDATE(128, false);
        } else {
            if (rtd) SPHFEM_UPDATE(256, true);
            else SPHFEM_UPDATE(256, false);
        }
#undef SPHFEM_UPDATE
    } else {
        u.psum64 = lf->psum64;
        {
            KTimer tp(ctx, "pairs_fp64");
            if (lf->tuning.pair_block == 128)
                k_pairs_fp64<128><<<nblk(B.N, 128), 128, 0, ctx->stream>>>(ctx->c, B, cs, ce, pre_view(lf->pre, B.N),
                                                                            lf->psum64, nf);
            else
                k_pairs_fp64<256><<<nblk(B.N, 256), 256, 0, ctx->stream>>>(ctx->c, B, cs, ce, pre_view(lf->pre, B.N),
                                                                            lf->psum64, nf);
        }
        KTimer tm(ctx, "fused_update");
#define SPHFEM_UPDATE(BSZ, RG)                                                                              \
    k_fused_update<false, BSZ, RG><<<nblk(B.N, BSZ), BSZ, 0, ctx->stream>>>(ctx->c, u, nullptr, nullptr, nf)
        if (lf->tuning.update_block == 128) {
            if (rtd) SPHFEM_UPDATE(128, true);
            else SPHFEM_UPDATE(128, false);
        } else {
            if (rtd) SPHFEM_UPDATE(256, true);
            else SPHFEM_UPDATE(256, false);
        }
#undef SPHFEM_UPDATE
    }
}

// FP32C derivative carry <-> the particle arrays' FP64 rates, and its gather by a permutation
__global__ void __launch_bounds__(256) k_rates_import(sphfem_particles P, RateView d) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int)P.N) return;
    const sphfem_double2 pt = P.pos_t[i], vt = P.vel_t[i];
    const sphfem_double4 St = P.S_t[i];
    d.pos_t[i] = make_float2((float)pt.x, (float)pt.y);
    d.vel_t[i] = make_float2((float)vt.x, (float)vt.y);
    d.S_t[i] = make_float4((float)St.x, (float)St.y, (float)St.z, (float)St.w);
    d.rho_t[i] = (float)P.rho_t[i];
    d.T_t[i] = (float)P.T_t[i];
}

__global__ void __launch_bounds__(256) k_rates_export(RateView r, sphfem_particles P) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int)P.N) return;
    const float2 pt = r.pos_t[i], vt = r.vel_t[i];
    const float4 St = r.S_t[i];
    P.pos_t[i] = {pt.x, pt.y};
    P.vel_t[i] = {vt.x, vt.y};
    P.S_t[i] = {St.x, St.y, St.z, St.w};
    P.rho_t[i] = r.rho_t[i];
    P.T_t[i] = r.T_t[i];
}

__global__ void __launch_bounds__(256) k_rates_gather(RateView a, RateView b, const int *__restrict__ perm, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int s = perm[i];
    if ((unsigned)s >= (unsigned)n) return;
    b.pos_t[i] = a.pos_t[s];
    b.vel_t[i] = a.vel_t[s];
    b.S_t[i] = a.S_t[s];
    b.rho_t[i] = a.rho_t[s];
    b.T_t[i] = a.T_t[s];
}

void launch_rates_import(sphfem_ctx *ctx, const sphfem_particles &p, const RateView &dst) {
    KTimer t(ctx, "rates_import");
    k_rates_import<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(p, dst);
}

void launch_rates_export(sphfem_ctx *ctx, const RateView &src, const sphfem_particles &p) {
    KTimer t(ctx, "rates_export");
    k_rates_export<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(src, p);
}

void launch_rates_gather(sphfem_ctx *ctx, const RateView &src, const RateView &dst, const int *perm, int n) {
    KTimer t(ctx, "rates_gather");
    k_rates_gather<<<nblk(n, 256), 256, 0, ctx->stream>>>(src, dst, perm, n);
}

// ---------------------------------------------------------------------------------------------
// output.cu:22-30: sum of fc and ft over all particles (deterministic two-level reduction)
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_force_partial(sphfem_particles P, double *part) {
    __shared__ double sx[256], sy[256];
    double x = 0., y = 0.;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < (int)P.N; i += gridDim.x * 256) {
        sphfem_double2 a = P.fc[i], b = P.ft[i];
        x += a.x + b.x;
        y += a.y + b.y;
    }
    sx[threadIdx.x] = x;
    sy[threadIdx.x] = y;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            sx[threadIdx.x] += sx[threadIdx.x + s];
            sy[threadIdx.x] += sy[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sx[0];
        part[2 * blockIdx.x + 1] = sy[0];
    }
}

__global__ void k_force_final(const double *part, int n, double *out) {
    if (threadIdx.x != 0) return;
    double x = 0., y = 0.;
    for (int b = 0; b < n; b++) {
        x += part[2 * b];
        y += part[2 * b + 1];
    }
    out[0] = x;
    out[1] = y;
}

void launch_report_force(sphfem_ctx *ctx, const sphfem_particles &p, double *part, double *out) {
    KTimer t(ctx, "report_force");
    k_force_partial<<<SPHFEM_FORCE_BLOCKS, 256, 0, ctx->stream>>>(p, part);
    k_force_final<<<1, 64, 0, ctx->stream>>>(part, SPHFEM_FORCE_BLOCKS, out);
}

}  // namespace sphfem
