// nbabfs_force.hip -- per-call kernels of the ABFS energy/gradient on gfx950.
//
// Replaces PairwiseInteractionABFS_MMMMEnergy (analytic branch,
// pMolecule-1.9.0/extensions/csource/PairwiseInteraction.c:292-429) and the
// OpenMP gradient reduction (NBModelABFSState.c:19-38).
//
// Tiled (default, "mixed") path: one wavefront per work item (a super-cluster
// of 8 i-clusters against a run of j-clusters).  Lane l = 8a + b pairs i-atom
// a of cluster c with j-atom b.  1/r comes from the FP32 v_rsq seed refined by
// one FP64 Newton step; force vectors are summed in FP32 registers; i-forces
// stay in registers for the whole item, j-forces are reduced across the 8
// lanes that share b and added once per j-cluster.  All gradient sums land in
// 64-bit fixed point, so the result does not depend on the order in which
// items finish.
//
// Periodic images (MMMMImageEnergy, pMolecule-1.9.0/extensions/csource/
// NBModelABFS.c:1161-1290): an image item's j-clusters are transformed to the
// image on the fly (x' = R x + T, FP64), its energies and forces carry the
// image scale, its j-gradients are rotated back by R^T before they are added,
// and it sums the image-side gradients and their moments for dE/dM.
#include "nbabfs_internal.h"
#include "nbabfs_kernels.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <type_traits>

static inline int nblk(size_t m, int b) { return (int)((m + b - 1) / b); }

// ------------------------------------------------------------------------------------------------
// Per-pair terms.
// ------------------------------------------------------------------------------------------------
// FP64, reference expression order (pMolecule-1.9.0/extensions/cinclude/PairwiseInteraction.h:72-119).
__device__ __forceinline__ bool pair_fp64(const AbfsFactors &F, double r2, double qij, double A, double B,
                                          double &eel, double &elj, double &dF)
{
#pragma clang fp contract(off)
    if (r2 > F.r2Off) return false;
    double s, s2;
    if (r2 < F.r2Damp) { s2 = 0.0; s = 0.0; }
    else { s2 = 1.0 / r2; s = sqrt(s2); }
    double d = 0.0;
    if (r2 > F.r2On) {
        eel = qij * (s * (F.a - r2 * (F.b + r2 * (F.c + F.d * r2))) + F.qShift2);
        d += -qij * 0.5 * s * (F.a + r2 * (F.b + r2 * (3.0 * F.c + 5.0 * F.d * r2))) / r2;
    } else if (r2 > F.r2Damp) {
        eel = qij * (s + F.qShift1);
        d += -qij * 0.5 * s / r2;
    } else {
        eel = qij * (F.qF0 - F.qAlpha * r2);
        d += -qij * F.qAlpha;
    }
    double s6 = s2 * s2 * s2;
    if (r2 > F.r2On) {
        double l1 = s6 - F.aF6, l2 = (s / r2) - F.bF3;
        elj = A * F.aK12 * (l1 * l1) - B * F.bK6 * (l2 * l2);
        d += -3.0 * s6 * (2.0 * A * F.aK12 * l1 / r2 - B * F.bK6 * l2 / s);
    } else if (r2 > F.r2Damp) {
        elj = A * (s6 * s6 - F.aShift12) - B * (s6 - F.bShift6);
        d += -3.0 * s6 * (2.0 * A * s6 - B) / r2;
    } else {
        elj = A * (F.aF0 - F.aAlpha * r2) - B * (F.bF0 - F.bAlpha * r2);
        d += -A * F.aAlpha + B * F.bAlpha;
    }
    dF = d;
    return true;
}

// Tiled path: one pair with 1/r from the FP32 v_rsq seed refined by one
// Newton step in FP64 (relative error ~1e-14; no FP64 divide or square root).
// The kernel is bound by VALU issue, and every instruction here but the FP32
// multiply-adds, moves and 32-bit adds takes a full issue slot (measured: 1.9 ns
// per wave instruction and SIMD for FP64 arithmetic, compares, selects, shifts
// and conversions alike, 1.05 ns for v_fma/add/mul_f32, v_add_u32, v_mov_b32 and
// v_and_b32, 3.6 ns for v_rsq_f32), so the forms below are chosen for their
// instruction count.
//
// u = clamp((r2 - r2On)/(r2Off - r2On)) is one multiply-add with the clamp
// modifier: 0 in the plain region, in (0, 1] in the switched one.
//   * Coulomb force: the reference's factor a + r2 (b + r2 (3c + 5d r2)) is the
//     smoothstep 1 + u^2 (2u - 3), exactly 1 in the plain region.
//   * Coulomb energy: s + sc (P - 1) + qShift2 with sc = min(s, 1/inner) and
//     P - 1 = (a - 1) - r2 (b + r2 (c + d r2)) as a cubic in u.  In the plain
//     region sc (P - 1) + qShift2 is the constant qShift1 (the reference's
//     energies meet at the inner cutoff), so no region is selected.  The cubic's
//     leading coefficient is divided out of all of it (eel is E / eScale, scaled
//     back with the item's total), so every step has at most one constant, which
//     is all an instruction can take from scalar registers.
//   * Lennard-Jones in both undamped regions is one polynomial in s = 1/r,
//       E = C12 s^12 + C6 s^6 + C3 s^3 + C0,
//     whose coefficients per type pair and region come from a row table (plain:
//     A, -B, 0, B*bShift6 - A*aShift12; switched: the expanded squares
//     A*aK12*(s^6-aF6)^2 - B*bK6*(s^3-bF3)^2); the region's row offset comes from
//     the high word of u (0 for u = 0) without a compare.
// The damped region (r < dampingCutoff) is a wave-uniform rare path on the raw
// A, B.  The rows hold three times the coefficients, so that the factor 3 of the
// Lennard-Jones force costs nothing: elj is 3 E, divided by 3 with the item's
// total, and fs is minus twice dE/d(r^2).
template <class Factors>
__device__ __forceinline__ double switch_coordinate(const Factors &F, double uShift, double r2)
{
    return fmin(fmax(fma(r2, F.uScale, uShift), 0.0), 1.0);
}

// min(x, s) with s in scalar registers.  fmin of a kernel argument would first
// canonicalise it, one more instruction per use; neither operand is a signalling NaN.
__device__ __forceinline__ double min_uniform(double x, double s)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "s"(s));
    return r;
}

// The damped region's terms (pair_rows and pair_full), a branch of the whole wave (its lanes select), so the usual path
// has no execution-mask bookkeeping.  Its factors and tables are read through the descriptor here: as kernel arguments
// they would hold (and spill) scalar registers over the whole entry loop.  ljScale: the rows' factor.
__device__ __forceinline__ void pair_damped(double r2Damp, double r2, double qq, unsigned long long mact, const SysDesc *D,
                                            int off, double ljScale, double &f, double &e1, double &e2)
{
    if (__builtin_expect((__builtin_amdgcn_ballot_w64(r2 < r2Damp) & mact) != 0ull, 0)) {
        const GAS double *k = as_global(D->damp);
        const bool damped = r2 < r2Damp;
        const double A = as_global(D->ljA)[off >> 6], B = as_global(D->ljB)[off >> 6];
        e1 = damped ? qq * fma(k[1], r2, k[0]) : e1;
        e2 = damped ? ljScale * (A * fma(-k[3], r2, k[2]) - B * fma(-k[5], r2, k[4])) : e2;
        f = damped ? 2.0 * (qq * k[6] + (A * k[3] - B * k[5])) : f;
    }
}

__device__ __forceinline__ void pair_rows(const TiledFactors &F, double r2, double u, double qq, double4 C,
                                          unsigned long long mact, const SysDesc *D, int off, double &fs, double &eel,
                                          double &elj)
{
    const double y = (double)__builtin_amdgcn_rsqf((float)r2);
    const double h = fma(-(r2 * y), y, 1.0);
    const double s = fma(0.5 * y, h, y);
    const double s2 = s * s;
    const double s3 = s2 * s;
    const double s6 = s3 * s3;
    const double Q = fma(u * u, fma(2.0, u, F.minus3), 1.0);
    const double sc = min_uniform(s, F.sOn);
    const double pm1 = fma(fma(u + F.p2, u, F.p1), u, F.p0);
    double e1 = qq * fma(s, F.eInv, fma(sc, pm1, F.qShift2e));
    // inner = s^3 (4 C12 s^6 + 2 C6) + C3 = 2 s^3 (C12 s^6 + t1) + C3, t1 = C12 s^6 + C6.
    const double t1 = fma(C.x, s6, C.y);
    double e2 = fma(t1, s6, fma(C.z, s3, C.w));
    const double inner = fma(s3 + s3, fma(C.x, s6, t1), C.z);
    // Minus twice dE/d(r^2): Coulomb qq s^3 Q, Lennard-Jones 3 s^5 inner (the rows' factor 3).
    double f = s3 * fma(s2, inner, qq * Q);
    pair_damped(F.r2Damp, r2, qq, mact, D, off, 3.0, f, e1, e2);
    fs = f;
    eel = e1;
    elj = e2;
}

// The full-FP64 instance's pair terms: no divide or square root, and every term as close to its exact value as the
// reference's expressions (pair_fp64) come.  Measured on pairs at 200 distances each, default cutoffs, in units of 2^-53 of
// the term's undamped magnitude and as root mean squares (here / pair_fp64 / the mixed kernel's rows with 1/r to 2 ulp):
// at 2-2.8 A Coulomb energy 0.6 / 1.6 / 2.4 and force 0.9 / 0.8 / 1.4, Lennard-Jones energy 1.8 / 2.1 / 3.7 and force
// 2.3 / 2.4 / 4.8; at 8-10 A 3.1 / 7.3 / 7.8, 0.9 / 4.0 / 1.4, 1.0 / 1.1 / 2.9 and 1.5 / 1.6 / 4.4.
//   * s = 1/r: one third-order step from the FP32 seed y, whose square t is exact in FP64, and so is the residual 1 - r2 t
//     to its last bits: only the step's rounding is left.  t + td is 1/r^2 beyond FP64: s2 and s3 each take one rounding
//     of it.
//   * Coulomb energy: s + qShift1 + P0 min(s - 1/inner, 0) + s u (P1 + u (P2 + u P3)), P - 1 about the inner cutoff
//     less its value there, so that nothing large cancels; the plain region's added terms are exactly zero.
//   * Lennard-Jones as the reference squares it: C12 (s^6 - w^2)^2 - C6 (s^3 - w)^2 + C0 (rows 2 C12, 2 C6, 2 C0, w: plain
//     A, B, C0, 0; switched A aK12, B bK6, 0, bF3 = 1/outer^3; elj is 2 E).  Expanded squares cancel towards the outer cutoff.  In the
//     plain region both terms take the rounded s^6 (n: that s^6 less s^3 s^3), whose error then cancels at the minimum.
__device__ __forceinline__ void pair_full(const FullFactors &F, double r2, bool sw, double u, double qq, double4 C,
                                          unsigned long long mact, const SysDesc *D, int off, double &fs, double &eel,
                                          double &elj)
{
    const double y = (double)__builtin_amdgcn_rsqf((float)r2);
    const double t = y * y;
    const double h = fma(-r2, t, 1.0);
    const double s = fma(y * h, fma(0.375, h, 0.5), y);
    const double td = t * fma(h, h, h);
    const double s2 = t + td;
    const double s3 = fma(s, t, s * td);
    const double s6 = s3 * s3;
    const double Q = fma(u * u, fma(2.0, u, F.minus3), 1.0);
    const double R = fma(fma(F.P3, u, F.P2), u, F.P1);
    const double K = fma(F.P0, fmin((s - F.sOn) - F.sOnLow, 0.0), F.q1);
    double e1 = qq * (s + fma(s * u, R, K));
    const double l1 = fma(-C.w, C.w, s6), l2 = s3 - C.w;
    const double nr = fma(-s3, s3, s6);
    const double n = __hiloint2double(sw ? 0 : __double2hiint(nr), __double2loint(nr));    // below 2^-1042 when switched
    const double a = C.x * l1;
    double e2 = fma(a, l1, fma(-C.y, fma(l2, l2, n), C.z));
    const double inner = fma(a + a, s6, -(C.y * fma(l2, s3, n)));
    const double x = s2 * inner;
    double f = fma(2.0, x, fma(s3, qq * Q, x));
    pair_damped(F.r2Damp, r2, qq, mact, D, off, 2.0, f, e1, e2);
    fs = f;
    eel = e1;
    elj = e2;
}

// ------------------------------------------------------------------------------------------------
// Prepare: slot records (origin-relative FP64 position, scaled charge), slot
// types; zero the fixed-point accumulators; reset the work queues.  With
// chk.ref set it also applies CheckForUpdate as NBModelABFS_Update calls it
// (pMolecule-1.9.0/extensions/csource/NBModelABFS.c:538-545, 691-746: some
// free atom moved more than half the buffer since the list was built) and
// tells the guarded launch and the host (PrepareCheck).
// ------------------------------------------------------------------------------------------------
// A guarded launch does nothing when its update test asked for a rebuild.
__device__ __forceinline__ bool guard_skip(const ForceGuard &g)
{
    if (!g.flag) return false;
    // Two relaxed loads that may be in flight together (volatile loads would be issued one after the other).
    const int epoch = g.epoch_ptr ? __hip_atomic_load(g.epoch_ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                  : g.epoch;
    return __hip_atomic_load(g.flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch;
}

__global__ __launch_bounds__(256) void k_prepare(const SysDesc *__restrict__ descs, int tiled, int *__restrict__ heads,
                                                 PrepareCheck chk)
{
    const SysDesc &D = descs[blockIdx.y];
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (heads && blockIdx.y == 0 && blockIdx.x == 0 && threadIdx.x < 8) heads[32 * threadIdx.x] = 0;
    if (blockIdx.x == 0 && D.eacc)
        for (int k = threadIdx.x; k < NB_EACC_WORDS; k += 256) D.eacc[k] = 0;
    if (D.gacc)
        for (int k = blockIdx.x * 256 + threadIdx.x; k < NB_GACC_WORDS_PER_IMAGE * D.nimg; k += gridDim.x * 256)
            D.gacc[k] = 0;
    bool up = false, nonfinite = false;
    if (s < D.n_pad) {
        for (int k = 0; k < 6; k++) D.facc[(size_t)k * D.n_pad + s] = 0;
        const double *xyz = chk.xyz ? chk.xyz : D.xyz;
        const int a = D.slot_atom[s];
        double x = 0.0, y = 0.0, z = 0.0;
        if (a >= 0) {
            x = xyz[3 * (size_t)a];
            y = xyz[3 * (size_t)a + 1];
            z = xyz[3 * (size_t)a + 2];
            nonfinite = !(isfinite(x) && isfinite(y) && isfinite(z));
            if (chk.ref && (!chk.free_flags || (chk.free_flags[a] & 1))) {
#pragma clang fp contract(off)
                const double dx = x - chk.ref[3 * (size_t)a];
                const double dy = y - chk.ref[3 * (size_t)a + 1];
                const double dz = z - chk.ref[3 * (size_t)a + 2];
                up = dx * dx + dy * dy + dz * dz > chk.bufsq;
            }
        }
        if (tiled) {
            double4 v = make_double4(0.0, 0.0, 0.0, 0.0);
            int t = 0;
            if (a >= 0) {
                v = make_double4(x - D.origin[0], y - D.origin[1], z - D.origin[2], D.charge[a] * D.qscale);
                t = D.atype[a];
            }
            D.xyzq[s] = v;
            D.styp[s] = t;
        }
    }
    // A NaN or infinite coordinate fails no distance test (its pairs drop out
    // silently), so it is reported here, where every atom is read.
    raise_error(D.err, nonfinite, NB_ERR_COORD);
    if (chk.counter) {
        // One 64-bit atomic per block carries both its completion (high word) and whether any of its atoms moved (low
        // word).  The last block knows the answer and tells the host and the guarded launch in one word each.  No
        // system-scope fence: nothing else is published, and the fence would write back the accumulators and records of
        // the whole pass (100,002 atoms: 20 us with it, 10 us without).
        const int moved = __syncthreads_or(up);
        if (threadIdx.x == 0) {
            const unsigned long long inc = (1ull << 32) + (moved ? 1ull : 0ull);
            const unsigned long long old = atomicAdd(chk.counter, inc);
            const unsigned long long total = (unsigned long long)gridDim.x * gridDim.y;
            if ((old >> 32) + 1 == total) {
                const bool any = ((old + inc) & 0xffffffffull) != 0;
                *(volatile unsigned long long *)chk.counter = 0ull;
                if (any) *(volatile int *)chk.dflag = chk.epoch;
                *(volatile int *)chk.done = any ? -chk.epoch : chk.epoch;
            }
        }
    }
}

// One lane's FP64 value in scalar registers.
__device__ __forceinline__ double lane_f64(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Cluster-frame image position x' = R x + T of a slot record (charge kept);
// X = R (9, row-major) then T (3), read from LDS at each use (broadcast reads)
// so that the transformation holds no registers across the entry loop.
__device__ __forceinline__ double4 image_slot(double4 v, const volatile double *X)
{
    return make_double4(fma(X[0], v.x, fma(X[1], v.y, fma(X[2], v.z, X[9]))),
                        fma(X[3], v.x, fma(X[4], v.y, fma(X[5], v.z, X[10]))),
                        fma(X[6], v.x, fma(X[7], v.y, fma(X[8], v.z, X[11]))), v.w);
}

// ------------------------------------------------------------------------------------------------
// The 1-4 list (the second pass of NBModelABFS_MMMMEnergy, pMolecule-1.9.0/
// extensions/csource/NBModelABFS.c:228-301): 64 pairs per block (one wave),
// FP64 in the reference's expression order, forces into the fixed-point
// accumulators, the block's two energies (wave sums) into epart14[blk].  Run
// by k_pairs14, or by extra workgroups of the main pair launch.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void pairs14_block(const SysDesc &D, const AbfsFactors &F, int blk, int lane)
{
#pragma clang fp contract(off)
    const int k = blk * 64 + lane;
    double e1 = 0.0, e2 = 0.0;
    bool bad = false;
    if (k < D.n14) {
        const int i = D.p14[2 * k], j = D.p14[2 * k + 1];
        double xij = D.xyz[3 * (size_t)i] - D.xyz[3 * (size_t)j];
        double yij = D.xyz[3 * (size_t)i + 1] - D.xyz[3 * (size_t)j + 1];
        double zij = D.xyz[3 * (size_t)i + 2] - D.xyz[3 * (size_t)j + 2];
        const double r2 = (xij * xij + yij * yij + zij * zij);
        const double qij = (D.escale14 * D.charge[i]) * D.charge[j];
        const int tij = D.ntypes * D.atype[i] + D.atype[j];
        double x1, x2, dF;
        if (pair_fp64(F, r2, qij, D.ljA14[tij], D.ljB14[tij], x1, x2, dF)) {
            e1 = x1;
            e2 = x2;
            const int si = D.atom_slot[i], sj = D.atom_slot[j];
            const double px = xij * (2.0 * dF), py = yij * (2.0 * dF), pz = zij * (2.0 * dF);
            bad |= fx_atomic_add(D.facc, D.n_pad, si, 0, px);
            bad |= fx_atomic_add(D.facc, D.n_pad, si, 1, py);
            bad |= fx_atomic_add(D.facc, D.n_pad, si, 2, pz);
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 0, -px);
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 1, -py);
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 2, -pz);
        }
    }
    e1 = wave_sum_f64(e1);
    e2 = wave_sum_f64(e2);
    if (lane == 0) {
        D.epart14[2 * blk] = e1;
        D.epart14[2 * blk + 1] = e2;
    }
    raise_error(D.err, bad || !isfinite(e1) || !isfinite(e2), NB_ERR_RANGE);
}

// ------------------------------------------------------------------------------------------------
// Tiled force kernel: one work item per workgroup, or a persistent loop over
// per-XCD queues with stealing.  The LJ row table of the item's system sits
// in LDS when it fits; the next entry's j-cluster record and masks are
// fetched while the current one is evaluated.
// ------------------------------------------------------------------------------------------------

// A value read from LDS at an address the caller has made a 32-bit LDS one.
#define LAS __attribute__((address_space(3)))
typedef double f64x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double4 lds_record(const LAS char *p)
{
    const f64x2 u = *(const LAS f64x2 *)p, v = *(const LAS f64x2 *)(p + 16);
    return make_double4(u.x, u.y, v.x, v.y);
}

__device__ __forceinline__ double4 load_slot(const GAS double *__restrict__ xr, int k)
{
    return make_double4(xr[4 * k], xr[4 * k + 1], xr[4 * k + 2], xr[4 * k + 3]);
}

// The j-cluster's records and types: a wave-uniform base plus a 32-bit lane offset.
__device__ __forceinline__ double4 load_j(const GAS double *__restrict__ xr, int J, unsigned off)
{
    // The uniform part of the address stays in scalar registers and the lane's 32-bit offset in one vector register
    // (a 64-bit lane offset hoisted out of the entry loop would cost a register pair and an addition per load).
    unsigned long long base = (unsigned long long)(xr + (size_t)J * (4 * NB_CL));
    asm volatile("" : "+s"(base), "+v"(off));
    const GAS double *p = (const GAS double *)((const GAS char *)base + off);
    return make_double4(p[0], p[1], p[2], p[3]);
}

__device__ __forceinline__ int load_jtype(const GAS int *__restrict__ ty, int J, unsigned off)
{
    unsigned long long base = (unsigned long long)(ty + (size_t)J * NB_CL);
    asm volatile("" : "+s"(base), "+v"(off));
    return *(const GAS int *)((const GAS char *)base + off);
}

// Entry fields through the vector memory path.  Headers: lane k reads (J, cbits)
// of entry first + k, so one load brings a whole item's headers (64 entries) and
// the entry loop takes them from its lanes; each lane reads its own tile-mask
// byte of an entry (64 consecutive bytes).
__device__ __forceinline__ int2 entry_headers(const GAS unsigned char *__restrict__ eb, int first, int count, int lane)
{
    const GAS int *p = (const GAS int *)(eb + (size_t)(first + min(lane, max(count - 1, 0))) * sizeof(Entry));
    return make_int2(p[0], p[1]);
}

__device__ __forceinline__ int entry_bits(const GAS unsigned char *__restrict__ eb, int e, unsigned lane)
{
    unsigned long long base = (unsigned long long)(eb + (size_t)e * sizeof(Entry));
    asm volatile("" : "+s"(base), "+v"(lane));
    return ((const GAS unsigned char *)base + 16)[lane];
}

// Sums over the eight consecutive lanes 8b..8b+7 with DPP moves: quad
// exchanges (xor 1, xor 2), then the half-row mirror (lane i <-> 7-i).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true));
}

// The j-atom's record of an entry: lane a (of the eight of j-atom b) returns
// component min(a, 7 - a) of (sum gx, sum gy, sum gz, J), so that lanes 0..3
// hold the record.  After the two quad steps every lane of a quad has the
// quad's three sums; it keeps one of them and the mirror adds the other quad's
// sum of the same component: 10 instructions instead of three full sums and
// two selects.
__device__ __forceinline__ float j_bits(float, int J) { return __int_as_float(J); }
__device__ __forceinline__ double j_bits(double, int J) { return (double)J; }
__device__ __forceinline__ int bits_j(float v) { return __float_as_int(v); }
__device__ __forceinline__ int bits_j(double v) { return (int)v; }

template <class T>
__device__ __forceinline__ T j_record(T gx, T gy, T gz, int J, int comp)
{
    gx += dpp_move<0xB1>(gx);    // quad_perm [1,0,3,2]
    gy += dpp_move<0xB1>(gy);
    gz += dpp_move<0xB1>(gz);
    gx += dpp_move<0x4E>(gx);    // quad_perm [2,3,0,1]
    gy += dpp_move<0x4E>(gy);
    gz += dpp_move<0x4E>(gz);
    asm("" : "+v"(gx), "+v"(gy), "+v"(gz));    // every lane needs all three: no branches on comp
    T v = comp == 0 ? gx : (comp == 1 ? gy : gz);
    v += dpp_move<0x141>(v);     // row_half_mirror
    return comp == 3 ? j_bits(v, J) : v;
}

// Totals of x (returned by lanes 0..31) and y (lanes 32..63) over the wave:
// one half swap makes the two sums one, then five steps on it.
__device__ __forceinline__ void swap_halves(double &x, double &y)
{
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(y), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(y), false, false);
    x = __hiloint2double(hi[0], lo[0]);
    y = __hiloint2double(hi[1], lo[1]);
}

__device__ __forceinline__ void swap_halves(float &x, float &y)
{
    const auto v = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(y), false, false);
    x = __int_as_float(v[0]);
    y = __int_as_float(v[1]);
}

__device__ __forceinline__ void swap_rows(double &x, double &y)
{
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(x), __double2loint(y), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(x), __double2hiint(y), false, false);
    x = __hiloint2double(hi[0], lo[0]);
    y = __hiloint2double(hi[1], lo[1]);
}

__device__ __forceinline__ void swap_rows(float &x, float &y)
{
    const auto v = __builtin_amdgcn_permlane16_swap(__float_as_int(x), __float_as_int(y), false, false);
    x = __int_as_float(v[0]);
    y = __int_as_float(v[1]);
}

__device__ __forceinline__ double wave_sum2_f64(double x, double y)
{
    swap_halves(x, y);
    double v = x + y;
    v += dpp_move<0xB1>(v);      // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);      // quad_perm [2,3,0,1]
    v += dpp_move<0x141>(v);     // row_half_mirror
    v += dpp_move<0x128>(v);     // row_ror:8
    double w = v;
    swap_rows(v, w);             // the two rows of each half
    return v + w;
}

// i-forces of one component: f[c] holds, on lane 8b + a, the partial of atom a
// of i-cluster c over the j-atoms b; lane 8b + a ends with the sum over b of
// cluster c = b.  A reduction in which every step halves the values as well as
// the lanes: clusters c and c + 4 trade wave halves, c and c + 2 rows, c and
// c + 1 row halves, so no LDS is involved (through LDS it was 24 writes, 24
// reads and two waits per item).
template <class T>
__device__ __forceinline__ T i_force(T (&f)[NB_SCC], int lane)
{
    T g[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        swap_halves(f[c], f[c + 4]);
        g[c] = f[c] + f[c + 4];
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
        swap_rows(g[c], g[c + 2]);
        g[c] += g[c + 2];
    }
    const bool odd = (lane & 8) != 0;
    const T keep = odd ? g[1] : g[0], send = odd ? g[0] : g[1];
    return keep + dpp_move<0x128>(send);     // row_ror:8
}

// LDS of the tiled kernel (dynamic).  A workgroup holds WPG wavefronts, each
// evaluating one work item.  At offset 0 the LJ row table of the group's
// system when it fits (ROWS_LDS: staged once per group), then one region per
// wave: the item's i-cluster records and slot types, then one record per entry
// and j-atom (the three j-force sums and the j-cluster), flushed to the
// fixed-point accumulators every NB_JCHUNK entries.
#define NB_JCHUNK 16
#define NB_LDS_IREC 48          // x, y, z, q and the type's row offset, padded
#define NB_LDS_I_BYTES (NB_SC * NB_LDS_IREC)
#define NB_LDS_ROW_LIMIT 16384
#define NB_LDS_GROUP_LIMIT (160 * 1024 / 4)

static inline size_t tiled_lds_rows(int ntypes, bool rows_lds) { return rows_lds ? (size_t)2 * ntypes * ntypes * 32 : 0; }

// acc: bytes of a force accumulator (4: FP32, the mixed kernel; 8: FP64, the full-FP64 kernel).
static inline size_t tiled_lds_wave(int acc) { return NB_LDS_I_BYTES + (size_t)NB_JCHUNK * 4 * NB_CL * acc; }

// Wave-scope synchronisation of a wave's own LDS region (workgroups of several
// independent waves); a workgroup barrier when the workgroup is one wave.
template <int WPG>
__device__ __forceinline__ void wave_region_sync()
{
    if (WPG == 1) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// Wave sums of three values into the fixed-point words ga[0..5].
__device__ __forceinline__ bool add_sums3(long long *ga, double x, double y, double z, int lane)
{
    const double sx = wave_sum_f64(x), sy = wave_sum_f64(y), sz = wave_sum_f64(z);
    const double v = lane == 0 ? sx : (lane == 1 ? sy : sz);
    return lane < 3 && fx_add(&ga[2 * lane], &ga[2 * lane + 1], v);
}

// What a wave needs before its first tile: its lane's i-record and type, the
// item's entry headers, the first entry's mask byte and j-record.  All of it is
// asked for at once; a group asks before it stages its row table, so that the
// two latencies overlap.
struct ItemStart {
    double4 rec, xj;
    double xf;            // image items: lane k holds word k of the image transform
    int2 head;
    int typ, tj, bits;
};

template <bool IMG>
__device__ __forceinline__ ItemStart item_start(const SysDesc *D, const WorkItem &w, int lane)
{
    const unsigned a = lane & 7, b = lane >> 3;
    const GAS double *xq = (const GAS double *)D->xyzq;
    const GAS int *ty = as_global(D->styp);
    const GAS unsigned char *eb = (const GAS unsigned char *)D->entries;
    ItemStart t;
    t.head = entry_headers(eb, w.first, w.count, lane);
    t.bits = entry_bits(eb, w.first, 8 * a + b);
    t.xf = IMG ? ((const GAS double *)&D->imgxf[max((w.sys >> 16) - 1, 0)])[min(lane, 13)] : 0.0;
    t.rec = load_slot(xq, w.sc * NB_SC + lane);
    t.typ = ty[w.sc * NB_SC + lane];
    t.xj = load_j(xq, w.J0, 32u * b);
    t.tj = load_jtype(ty, w.J0, 4u * b);
    return t;
}

// An item whose fields are the same on every lane, in scalar registers.
__device__ __forceinline__ WorkItem uniform_item(const WorkItem &w)
{
    WorkItem u = {};
    u.sys = __builtin_amdgcn_readfirstlane(w.sys);
    u.sc = __builtin_amdgcn_readfirstlane(w.sc);
    u.first = __builtin_amdgcn_readfirstlane(w.first);
    u.count = __builtin_amdgcn_readfirstlane(w.count);
    u.J0 = __builtin_amdgcn_readfirstlane(w.J0);
    return u;
}

// The factors that an instance of the kernel takes.
template <bool F64>
struct PairFactors {
    using type = typename std::conditional<F64, FullFactors, TiledFactors>::type;
};

// Waves per SIMD.  A tile is a chain of two LDS reads and about forty dependent FP64 instructions, so the issue slots
// fill only with enough waves: five fit in 96 VGPRs, with no spill inside the entry loop, because the loop holds no
// 64-bit lane offsets, one LDS address for all tiles (records at a 16-byte-aligned stride with the type beside the
// charge), FP32 copies of dx, dy, dz across the pair terms and no polynomial factor in vector registers.  16-image batch:
// 680 us per call with three waves, 620 with four, 603 with five.
// A wave costs about 5 us beside its entries, and an entry's loads are a chain as long as its tiles: what a wave needs
// first is asked for at once (ItemStart), and an item's entry headers come with one load.
// IMG: the launch holds image items too (sys >> 16: the image plus one), beside the main list's or alone.  The j-record
// is transformed once per entry; the image's part of the item's end takes four waves per SIMD (107 VGPRs, none spilled; 49
// to 56 scalar registers are, into lanes of vector registers, and some 150 instructions in the loops read them back).  One
// launch, because a second stream's launch starts 15 us after its fork and joins 11 us after its end, and because the
// image items fill the GPU as the main items drain: 23,559 atoms in a 50 A cell, 139 us per call with two launches,
// 126 us with one.
// F64: the full-FP64 instance (NBABFS_TILED_FP64): the same list, tiles, staging and fixed-point sums with pair_full and
// FP64 force vectors, at three waves per SIMD (134 VGPRs; at four the loop keeps two energy sums in scratch).  Us per call
// of 20,001 atoms and of 16 images of 30,000: 75 and 937; at four waves 83 and 934; with the reference's own expressions
// (seven divides and a square root per tile, both regions for a wave that holds both) 141 and 1918; with the mixed kernel's
// rows and 1/r to 2 ulp 73 and 766, but pair terms off by 1.6 to 4 times as much (pair_full).
// WPG: wavefronts per workgroup.  With 4 (the one-item-per-wave launches),
// the row table is staged once for four items and a group's LDS stays small
// enough for five waves per SIMD; the four items of a group belong to one
// system (batches pad each system's items to a multiple of 4 with empty
// ones).  The persistent queues run one wave per group, at four waves per SIMD: their loop over items takes 111 VGPRs, and
// at five it spilled (30,000 atoms on four waves per CU 135 us per call, 131 without the spills; on twelve no difference).
template <bool ROWS_LDS, bool IMG, bool F64, int WPG>
__global__ __launch_bounds__(64 * WPG) __attribute__((amdgpu_waves_per_eu(tiled_waves(F64, IMG, WPG == 1)))) void k_force_tiled(
    const SysDesc *__restrict__ descs, const WorkItem *__restrict__ items, QueueParams qp,
    typename PairFactors<F64>::type F, int rows_bytes, int wave_bytes, ForceGuard guard, int nitems, int nforce_groups, int sys1)
{
    const int lane = threadIdx.x & 63;
    const int wave = WPG == 1 ? 0 : (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // A group's start is a chain of dependent loads (its work item, the system's descriptor, the records the item
    // names).  The loads that depend on nothing go out together with the guard's flag: the work item of a wave
    // with one item, and (sys1 >= 0: every item belongs to system sys1) the descriptor and its row table.
    constexpr bool QUEUE = WPG == 1 && !IMG;       // a persistent launch: items come from the per-XCD queues
    WorkItem w0 = {};
    if (!QUEUE && (int)blockIdx.x < nforce_groups && nitems > 0)
        w0 = items[min((int)blockIdx.x * WPG + wave, nitems - 1)];
    // guard_skip with both loads issued here unconditionally (a null pointer reads the descriptor instead) and
    // their values compared only where the answer is needed.
    const int *gfp = guard.flag ? guard.flag : (const int *)descs;
    const int *gep = guard.epoch_ptr ? guard.epoch_ptr : gfp;
    const int gflag = __hip_atomic_load(gfp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int gepoch = __hip_atomic_load(gep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // Groups past the pair blocks evaluate the 1-4 list of system 0 (single-state launches), one block per wave.
    if ((int)blockIdx.x >= nforce_groups) {
        const int blk = ((int)blockIdx.x - nforce_groups) * WPG + wave;
        if (!guard_skip(guard) && blk < descs[0].n14_blocks) pairs14_block(descs[0], F, blk, lane);
        return;
    }
    // Lane l = 8b + a: a is the i-atom within an i-cluster, b the j-atom of
    // the entry's j-cluster.  The entry masks are stored per l' = 8a + b.
    const int a = lane & 7, b = lane >> 3;
    const int bl = 8 * a + b;
    extern __shared__ __align__(32) unsigned char lds[];
    __shared__ __align__(16) double sXs[IMG ? WPG : 1][12];     // image items: R then T of the item's image
    double *sX = sXs[IMG ? wave : 0];
    using acc_t = typename std::conditional<F64, double, float>::type;
    double4 *sR = (double4 *)lds;
    unsigned char *region = lds + rows_bytes + (size_t)wave * wave_bytes;
    acc_t *sJ = (acc_t *)(region + NB_LDS_I_BYTES);   // [entry][j-atom] of (x, y, z, J)
    // One item per wave: ask for all it needs, then stage the group's row table (the items of a group belong to one
    // system; in a batch, its first item's).
    ItemStart st = {};
    int rows_sys = -1;
    if (!QUEUE) {
        if (ROWS_LDS && !IMG && sys1 < 0) rows_sys = items[(int)blockIdx.x * WPG].sys;
        w0 = uniform_item(w0);
        const SysDesc *D0 = &descs[sys1 >= 0 ? sys1 : (IMG ? (w0.sys & 0xffff) : w0.sys)];
        st = item_start<IMG>(D0, w0, lane);
        if (ROWS_LDS) {
            const SysDesc *DR = rows_sys >= 0 ? &descs[rows_sys] : D0;
            const GAS double *__restrict__ rows0 = as_global(DR->ljrow);
            const int nr = 2 * DR->ntypes * DR->ntypes;
            for (int k = threadIdx.x; k < nr; k += 64 * WPG) sR[k] = load_slot(rows0, k);
            if (WPG > 1) __syncthreads();
        }
    }
    // The guard's answer is needed only now (the loads above are reads; the flag is uniform over the launch).
    if (guard.flag != nullptr && gflag == (guard.epoch_ptr ? gepoch : guard.epoch)) return;
    // One work item per wave (the hardware dispatcher balances the load), or a persistent loop over per-XCD queues whose
    // counters sit on separate 128-byte lines.
    int q = blockIdx.x & 7;
    int tries = 0;
    for (;;) {
        int it;
        WorkItem w = w0;
        if (QUEUE) {
            if (tries >= 8) break;
            int local = 0;
            if (lane == 0) local = atomicAdd(&qp.heads[32 * q], 1);
            local = __builtin_amdgcn_readfirstlane(local);
            const int qs = qp.starts[q], qe = qp.starts[q + 1];
            if (qs + local >= qe) {
                q = (q + 1) & 7;
                tries++;
                continue;
            }
            it = qs + local;
            w = uniform_item(items[it]);
            if (w.count <= 0) continue;
        } else {
            it = (int)blockIdx.x * WPG + wave;
            // Empty items pad a batch's systems to whole groups.
            if (it >= nitems || w.count <= 0) break;
            // An item of another system than the staged rows would be a layout error (reported, never evaluated with the
            // wrong rows).
            if (rows_sys >= 0 && w.sys != rows_sys) {
                raise_error(descs[rows_sys].err, true, NB_ERR_RANGE);
                break;
            }
        }
        const SysDesc *D = &descs[sys1 >= 0 ? sys1 : (IMG ? (w.sys & 0xffff) : w.sys)];
        const GAS double *__restrict__ xq = (const GAS double *)D->xyzq;
        const GAS int *__restrict__ ty = as_global(D->styp);
        const GAS double *__restrict__ rows = as_global(D->ljrow);
        const GAS unsigned char *__restrict__ eb = (const GAS unsigned char *)D->entries;
        long long *facc = D->facc;
        const int n_pad = D->n_pad;
        const int nt = D->ntypes;
        const int I0 = w.sc * NB_SCC;
        // The item's image (-1: main list); all of its entries share it.
        int img = -1;
        double isc = 1.0;
        bool moments = false;
        if (IMG) img = (w.sys >> 16) - 1;
        if (IMG && img >= 0) {
            isc = lane_f64(st.xf, 12);
            moments = lane_f64(st.xf, 13) == 0.0;
        }

        // Pipeline of the entry loop: while entry e is evaluated, entry e+1's j-cluster record and mask byte are in
        // flight.  The indices are clamped, so every iteration issues the same loads and no atomic is pending inside
        // the loop.
        const int e_last = w.first + w.count - 1;
        if (QUEUE) st = item_start<IMG>(D, w, lane);
        const unsigned jrec = 32u * b, jtyp = 4u * b;      // byte offsets in a j-cluster's records and types

        // A persistent wave's region still holds its previous item's data until every lane is past it.
        if (QUEUE) wave_region_sync<WPG>();
        if (IMG && img >= 0 && lane < 12) sX[lane] = st.xf;
        if (ROWS_LDS && QUEUE)
            for (int k = lane; k < 2 * nt * nt; k += 64) sR[k] = load_slot(rows, k);
        {
            double *r = (double *)(region + NB_LDS_IREC * lane);
            r[0] = st.rec.x;
            r[1] = st.rec.y;
            r[2] = st.rec.z;
            r[3] = st.rec.w;
            *(int *)(r + 4) = 64 * nt * st.typ;   // byte offset of the type's first row pair
        }
        int hbase = w.first;                       // entry whose header lane 0 holds
        int2 head = st.head;
        int J = w.J0;
        int cbn = __builtin_amdgcn_readlane(head.y, 0);
        int lbn = st.bits;
        double4 xj = st.xj;
        int tj = 64 * st.tj;
        const int comp = min(a, NB_CL - 1 - a);
        const double fscale = -1.0;            // i-force = fscale times the sum over j
        wave_region_sync<WPG>();
        if (IMG && img >= 0) xj = image_slot(xj, sX);

        acc_t fx[NB_SCC], fy[NB_SCC], fz[NB_SCC];
#pragma unroll
        for (int c = 0; c < NB_SCC; c++) fx[c] = fy[c] = fz[c] = (acc_t)0;
        // Kept in vector registers: its multiply-add already reads one scalar operand.
        double uShift = F.uShift;
        asm("" : "+v"(uShift));
        double eel = 0.0, elj = 0.0;
        // The i-records are read at constant offsets from one address per lane (the compiler would keep one per tile).
        const LAS char *ip = (const LAS char *)(region + NB_LDS_IREC * a);
        asm("" : "+v"(ip));
        bool bad = false;
        for (int e0 = w.first; e0 <= e_last; e0 += NB_JCHUNK) {
        const int e1 = min(e0 + NB_JCHUNK - 1, e_last);
        for (int e = e0; e <= e1; e++) {
            // The next entry's header is on lane en - hbase; an item of more than 64 entries reads the next 64.
            const int cb = cbn, lb = lbn;
            const int en = min(e + 1, e_last);
            if (en - hbase >= 64) {
                hbase = en;
                head = entry_headers(eb, hbase, e_last - hbase + 1, lane);
            }
            const int Jn = __builtin_amdgcn_readlane(head.x, en - hbase);
            cbn = __builtin_amdgcn_readlane(head.y, en - hbase);
            const double4 xjn = load_j(xq, Jn, jrec);
            const int tjn = 64 * load_jtype(ty, Jn, jtyp);
            lbn = entry_bits(eb, en, bl);
            acc_t gx = (acc_t)0, gy = (acc_t)0, gz = (acc_t)0;
#pragma unroll
            for (int c = 0; c < NB_SCC; c++) {
                if (cb & (1 << c)) {
                    const bool inl = (lb & (1 << c)) != 0;
                    double4 xi = lds_record(ip + c * NB_CL * NB_LDS_IREC);
                    int ti = *(const LAS int *)(ip + c * NB_CL * NB_LDS_IREC + 32);
                    // The charge and type are read with the position, not after the branch below: one LDS wait per tile.
                    asm("" : "+v"(xi.w), "+v"(ti));
                    const double dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
                    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
                    const bool inr = r2 <= F.r2Off;
                    // Ballots of the two compares (lane masks as they stand), combined in scalar registers; the
                    // active lanes are that mask again (an execution mask, no per-lane recomputation).
                    const unsigned long long mact = __builtin_amdgcn_ballot_w64(inl) & __builtin_amdgcn_ballot_w64(inr);
                    const bool act = __builtin_amdgcn_inverse_ballot_w64(mact);
                    if (mact != 0ull) {
                        float px = (float)dx, py = (float)dy, pz = (float)dz;
                        if (!F64) asm("" : "+v"(px), "+v"(py), "+v"(pz));   // three registers across the pair terms, not six
                        {
                            const double u = switch_coordinate(F, uShift, r2);
                            const bool sw = F64 && u > 0.0;
                            const int off = ti + tj + (F64 ? (sw ? 32 : 0) : (int)min((unsigned)__double2hiint(u), 32u));
                            const double4 C = ROWS_LDS ? *(const double4 *)((const unsigned char *)sR + off)
                                                       : load_slot(rows, off >> 5);
                            double fs, x1, x2;
                            if constexpr (F64)
                                pair_full(F, r2, sw, u, xi.w * xj.w, C, mact, D, off, fs, x1, x2);
                            else
                                pair_rows(F, r2, u, xi.w * xj.w, C, mact, D, off, fs, x1, x2);
                            // The sums take the active lanes only (the others may hold any value).
                            if (act) {
                                const acc_t f = (acc_t)fs;
                                const acc_t vx = F64 ? (acc_t)dx : (acc_t)px, vy = F64 ? (acc_t)dy : (acc_t)py,
                                            vz = F64 ? (acc_t)dz : (acc_t)pz;
                                fx[c] = fma(f, vx, fx[c]);
                                fy[c] = fma(f, vy, fy[c]);
                                fz[c] = fma(f, vz, fz[c]);
                                gx = fma(f, vx, gx);
                                gy = fma(f, vy, gy);
                                gz = fma(f, vz, gz);
                                eel += x1;
                                elj += x2;
                            }
                        }
                    }
                }
            }
            const acc_t rec = j_record(gx, gy, gz, J, comp);
            // Lanes a and 7 - a hold the same value.
            sJ[(e - e0) * 4 * NB_CL + 4 * b + comp] = rec;
            J = Jn;
            xj = xjn;
            if (IMG && img >= 0) xj = image_slot(xj, sX);      // the j-atom's image position
            tj = tjn;
        }
        // The chunk's j-force sums (written by other lanes) are complete.
        wave_region_sync<WPG>();
        if (!IMG || img < 0) {
            // One record per lane.
            for (int k = lane; k < NB_CL * (e1 - e0 + 1); k += 64) {
                const acc_t *f = &sJ[4 * k];
                const int sj = bits_j(f[3]) * NB_CL + (k & 7);
                bad |= fx_atomic_add3(facc, n_pad, sj, -fscale * (double)f[0], -fscale * (double)f[1],
                                      -fscale * (double)f[2]);
            }
        } else {
            // Image side: g'_j (scaled) is rotated back, g_j += R^T g'_j, and the
            // sums h = sum g'_j and G_ab = sum g'_j,a (x_j - origin)_b are kept
            // for the lattice derivatives (SymmetryParameterGradients_ImageDerivatives,
            // pMolecule-1.9.0/extensions/csource/SymmetryParameterGradients.c:142-216).
            // A pure translation needs only h (the moments' derivative term vanishes).
            const double jsc = -fscale * isc;
            const int nrec = NB_CL * (e1 - e0 + 1);
            long long *ga = D->gacc + (size_t)img * NB_GACC_WORDS_PER_IMAGE +
                            (size_t)(it & (NB_GSLOTS - 1)) * NB_GACC_WORDS_PER_SLOT;
            double hx = 0.0, hy = 0.0, hz = 0.0;
            for (int k = lane; k < nrec; k += 64) {
                const acc_t *f = &sJ[4 * k];
                const int sj = bits_j(f[3]) * NB_CL + (k & 7);
                const double gx = jsc * (double)f[0], gy = jsc * (double)f[1], gz = jsc * (double)f[2];
                bad |= fx_atomic_add3(facc, n_pad, sj, fma(sX[0], gx, fma(sX[3], gy, sX[6] * gz)),
                                      fma(sX[1], gx, fma(sX[4], gy, sX[7] * gz)),
                                      fma(sX[2], gx, fma(sX[5], gy, sX[8] * gz)));
                hx += gx; hy += gy; hz += gz;
            }
            bad |= add_sums3(ga, hx, hy, hz, lane);
            // Row a of the moments, one after the other (nine sums at once would not leave the entry loop its registers).
            if (moments) {
#pragma nounroll
                for (int r = 0; r < 3; r++) {
                    hx = hy = hz = 0.0;
                    for (int k = lane; k < nrec; k += 64) {
                        const acc_t *f = &sJ[4 * k];
                        const double4 xr = load_slot(xq, bits_j(f[3]) * NB_CL + (k & 7));
                        const double g = jsc * (double)f[r];
                        hx = fma(g, xr.x, hx); hy = fma(g, xr.y, hy); hz = fma(g, xr.z, hz);
                    }
                    bad |= add_sums3(ga + 6 * (r + 1), hx, hy, hz, lane);
                }
            }
        }
        wave_region_sync<WPG>();
        }
        // i-forces: lane 8b + a ends with atom a of i-cluster b.
        const double iscale = IMG ? isc * fscale : fscale;
        const acc_t ix = i_force(fx, lane), iy = i_force(fy, lane), iz = i_force(fz, lane);
        bad |= fx_atomic_add3(facc, n_pad, I0 * NB_CL + lane, iscale * (double)ix, iscale * (double)iy,
                              iscale * (double)iz);
        // Energies: lane 0 holds the Coulomb total, lane 32 the Lennard-Jones one.
        if constexpr (F64) {
            elj *= 0.5;
        } else {
            eel *= F.eScale;
            elj *= 1.0 / 3.0;
        }
        const double etot = wave_sum2_f64(eel, elj);
        if ((lane & 31) == 0) {
            const int slot = it & (NB_ESLOTS - 1);
            const int kind = (lane >> 5) + (img >= 0 ? 2 : 0);
            bad |= fx_add(eacc_word(D->eacc, kind, 0, slot), eacc_word(D->eacc, kind, 1, slot),
                          2.0 * (IMG ? isc * etot : etot), 0x1p67);
        }
        raise_error(D->err, bad, NB_ERR_RANGE);
        if (!QUEUE) break;
    }
}

// ------------------------------------------------------------------------------------------------
// Plain FP64 path: one thread per atom over a full (both-direction) CSR list.
// ------------------------------------------------------------------------------------------------
template <int BS>
__device__ __forceinline__ void block_sum2(double &x, double &y)
{
    __shared__ double sx[BS], sy[BS];
    sx[threadIdx.x] = x;
    sy[threadIdx.x] = y;
    __syncthreads();
    for (int o = BS / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            sx[threadIdx.x] += sx[threadIdx.x + o];
            sy[threadIdx.x] += sy[threadIdx.x + o];
        }
        __syncthreads();
    }
    x = sx[0];
    y = sy[0];
}

__global__ __launch_bounds__(256) void k_force_plain(const SysDesc *__restrict__ descs, AbfsFactors F, ForceGuard guard)
{
#pragma clang fp contract(off)
    if (guard_skip(guard)) return;
    // blockIdx.y = system: one launch covers every system of a batch.
    const SysDesc &D = descs[blockIdx.y];
    if ((int)blockIdx.x >= D.n_plain_blocks) return;
    const int *__restrict__ rowptr = D.rowptr;
    const int *__restrict__ cols = D.cols;
    const int i = blockIdx.x * 256 + threadIdx.x;
    double e1 = 0.0, e2 = 0.0;
    if (i < D.n) {
        double gx = 0.0, gy = 0.0, gz = 0.0;
        const double xi = D.xyz[3 * (size_t)i], yi = D.xyz[3 * (size_t)i + 1], zi = D.xyz[3 * (size_t)i + 2];
        const double qi = D.escale * D.charge[i];
        const int ti = D.ntypes * D.atype[i];
        for (int k = rowptr[i]; k < rowptr[i + 1]; k++) {
            const int j = cols[k];
            double xij = xi - D.xyz[3 * (size_t)j];
            double yij = yi - D.xyz[3 * (size_t)j + 1];
            double zij = zi - D.xyz[3 * (size_t)j + 2];
            const double r2 = (xij * xij + yij * yij + zij * zij);
            const double qij = qi * D.charge[j];
            const int tij = ti + D.atype[j];
            double x1, x2, dF;
            if (!pair_fp64(F, r2, qij, D.ljA[tij], D.ljB[tij], x1, x2, dF)) continue;
            e1 += x1;
            e2 += x2;
            gx += xij * (2.0 * dF);
            gy += yij * (2.0 * dF);
            gz += zij * (2.0 * dF);
        }
        D.gplain[3 * (size_t)i] = gx;
        D.gplain[3 * (size_t)i + 1] = gy;
        D.gplain[3 * (size_t)i + 2] = gz;
    }
    block_sum2<256>(e1, e2);
    if (threadIdx.x == 0) {
        D.eplain[2 * blockIdx.x] = e1;
        D.eplain[2 * blockIdx.x + 1] = e2;
    }
}

// ------------------------------------------------------------------------------------------------
// Plain FP64 image pass (MMMMImageEnergy, pMolecule-1.9.0/extensions/csource/NBModelABFS.c:1161-1290, with
// PairwiseInteractionABFS_MMMMEnergy's expression order, PairwiseInteraction.c:292-429): one wavefront per
// image work item, lane l = 8b + a pairing i-atom a of each i-cluster of the super-cluster with j-atom b of
// the entry's j-cluster.  Each item's energies are stored in FP64 and summed in item order by the finalize.  Absolute coordinates; the image coordinate of j is formed as Coordinates3_Rotate +
// _Translate form it (R' x, then + M (t + n)); qi = escale_image * q_i, qij = qi * q_j, A and B times the
// image scale; dF from pair_fp64; i += 2 dF r_ij, j (image side) -= 2 dF r_ij.  j-gradients are summed over
// the 8 lanes of the j-atom, rotated back (R'^T) and added per entry; i-gradients per item; all into the
// fixed-point accumulators, with the energies and the dE/dM sums as in the tiled image instance.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ double sum_lanes_xor(double v, int m0, int m1, int m2)
{
    v += __shfl_xor(v, m0, 64);
    v += __shfl_xor(v, m1, 64);
    v += __shfl_xor(v, m2, 64);
    return v;
}

__global__ __launch_bounds__(64) void k_force_image_fp64(const SysDesc *__restrict__ descs,
                                                         const WorkItem *__restrict__ items, AbfsFactors F,
                                                         ForceGuard guard)
{
#pragma clang fp contract(off)
    if (guard_skip(guard)) return;
    const int it = blockIdx.x;
    const WorkItem w = items[it];
    const SysDesc &D = descs[w.sys & 0xffff];
    const int img = (w.sys >> 16) - 1;
    const ImageXf &X = D.imgxf[img];
    const int lane = threadIdx.x, a = lane & 7, b = lane >> 3;
    const int bl = 8 * a + b;
    const double isc = X.scale, esc = X.escale;
    const bool moments = X.translation == 0.0;
    const int nt = D.ntypes;
    double gi[NB_SCC][3];
    int ia[NB_SCC];
    double xi[NB_SCC][3], qi[NB_SCC];
    int ti[NB_SCC];
#pragma unroll
    for (int c = 0; c < NB_SCC; c++) {
        gi[c][0] = gi[c][1] = gi[c][2] = 0.0;
        ia[c] = D.slot_atom[(w.sc * NB_SCC + c) * NB_CL + a];
        const int i = ia[c] >= 0 ? ia[c] : 0;
        xi[c][0] = D.xyz[3 * (size_t)i];
        xi[c][1] = D.xyz[3 * (size_t)i + 1];
        xi[c][2] = D.xyz[3 * (size_t)i + 2];
        qi[c] = esc * D.charge[i];
        ti[c] = nt * D.atype[i];
    }
    double e1 = 0.0, e2 = 0.0, G[12];
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 12; k++) G[k] = 0.0;
    for (int e = w.first; e < w.first + w.count; e++) {
        const Entry &en = D.entries[e];
        const int J = en.J, cb = en.cbits, lb = en.bits[bl];
        const int j = D.slot_atom[J * NB_CL + b];
        const int jj = j >= 0 ? j : 0;
        const double x0 = D.xyz[3 * (size_t)jj], y0 = D.xyz[3 * (size_t)jj + 1], z0 = D.xyz[3 * (size_t)jj + 2];
        const double xj = (X.R[0] * x0 + X.R[1] * y0 + X.R[2] * z0) + X.Tabs[0];
        const double yj = (X.R[3] * x0 + X.R[4] * y0 + X.R[5] * z0) + X.Tabs[1];
        const double zj = (X.R[6] * x0 + X.R[7] * y0 + X.R[8] * z0) + X.Tabs[2];
        const double qj = D.charge[jj];
        const int tj = D.atype[jj];
        double gx = 0.0, gy = 0.0, gz = 0.0;
#pragma unroll
        for (int c = 0; c < NB_SCC; c++) {
            if (!((cb >> c) & 1) || !((lb >> c) & 1) || ia[c] < 0 || j < 0) continue;
            double xij = xi[c][0] - xj, yij = xi[c][1] - yj, zij = xi[c][2] - zj;
            const double r2 = (xij * xij + yij * yij + zij * zij);
            const double qij = qi[c] * qj;
            const int tij = ti[c] + tj;
            double x1, x2, dF;
            if (!pair_fp64(F, r2, qij, D.ljA[tij] * isc, D.ljB[tij] * isc, x1, x2, dF)) continue;
            e1 += x1;
            e2 += x2;
            xij *= (2.0 * dF);
            yij *= (2.0 * dF);
            zij *= (2.0 * dF);
            gi[c][0] += xij;
            gi[c][1] += yij;
            gi[c][2] += zij;
            gx -= xij;
            gy -= yij;
            gz -= zij;
        }
        // The j-atom's image-side gradient: lanes 8b .. 8b+7.
        gx = sum_lanes_xor(gx, 1, 2, 4);
        gy = sum_lanes_xor(gy, 1, 2, 4);
        gz = sum_lanes_xor(gz, 1, 2, 4);
        if (a == 0 && j >= 0) {
            const int sj = J * NB_CL + b;
            // Coordinates3_Rotate by R'^T.
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 0, X.R[0] * gx + X.R[3] * gy + X.R[6] * gz);
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 1, X.R[1] * gx + X.R[4] * gy + X.R[7] * gz);
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 2, X.R[2] * gx + X.R[5] * gy + X.R[8] * gz);
            G[0] += gx;
            G[1] += gy;
            G[2] += gz;
            if (moments) {
                const double rx = x0 - D.origin[0], ry = y0 - D.origin[1], rz = z0 - D.origin[2];
                G[3] += gx * rx; G[4] += gx * ry; G[5] += gx * rz;
                G[6] += gy * rx; G[7] += gy * ry; G[8] += gy * rz;
                G[9] += gz * rx; G[10] += gz * ry; G[11] += gz * rz;
            }
        }
    }
    // i-gradients: lanes a, a+8, ..., a+56.
#pragma unroll
    for (int c = 0; c < NB_SCC; c++) {
        const double vx = sum_lanes_xor(gi[c][0], 8, 16, 32);
        const double vy = sum_lanes_xor(gi[c][1], 8, 16, 32);
        const double vz = sum_lanes_xor(gi[c][2], 8, 16, 32);
        if (b == 0 && ia[c] >= 0) {
            const int si = (w.sc * NB_SCC + c) * NB_CL + a;
            bad |= fx_atomic_add(D.facc, D.n_pad, si, 0, vx);
            bad |= fx_atomic_add(D.facc, D.n_pad, si, 1, vy);
            bad |= fx_atomic_add(D.facc, D.n_pad, si, 2, vz);
        }
    }
    long long *ga = D.gacc + (size_t)img * NB_GACC_WORDS_PER_IMAGE +
                    (size_t)(it & (NB_GSLOTS - 1)) * NB_GACC_WORDS_PER_SLOT;
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const double v = wave_sum_f64(G[k]);
        if (lane == k && (moments || k < 3)) bad |= fx_add(&ga[2 * k], &ga[2 * k + 1], v);
    }
    e1 = wave_sum_f64(e1);
    e2 = wave_sum_f64(e2);
    if (lane == 0) {
        D.eimgpart[2 * (size_t)it] = e1;
        D.eimgpart[2 * (size_t)it + 1] = e2;
    }
    raise_error(D.err, bad || !isfinite(e1) || !isfinite(e2), NB_ERR_RANGE);
}

// ------------------------------------------------------------------------------------------------
// 1-4 list (NBModelABFS_MMMMEnergy's second pass, NBModelABFS.c:276-294): FP64
// with scale14 and the 1-4 LJ table; gradients into the fixed-point arrays.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_pairs14(const SysDesc *__restrict__ descs, AbfsFactors F, ForceGuard guard)
{
    const SysDesc &D = descs[blockIdx.y];
    if ((int)blockIdx.x >= D.n14_blocks || guard_skip(guard)) return;
    pairs14_block(D, F, blockIdx.x, threadIdx.x);
}

// ------------------------------------------------------------------------------------------------
// Finalize: gradients (fixed point -> FP64, plus the plain-path rows) added
// into the caller's array (or written over it in assign mode); block 0 of each system also sums the energies in a
// fixed order.
// ------------------------------------------------------------------------------------------------
__device__ void sum_range2(const double *__restrict__ p, int m, double &x, double &y)
{
    double sx = 0.0, sy = 0.0;
    for (int k = threadIdx.x; k < m; k += 256) {
        sx += p[2 * (size_t)k];
        sy += p[2 * (size_t)k + 1];
    }
    block_sum2<256>(sx, sy);
    x = sx;
    y = sy;
    __syncthreads();
}

__global__ __launch_bounds__(256) void k_finalize(const SysDesc *__restrict__ descs, int plain, ForceGuard guard)
{
    if (guard_skip(guard)) return;
    const SysDesc &D = descs[blockIdx.y];
    // The last block of each system sums its energies while the others add
    // the gradients (the two are independent, so neither waits for the other).
    // One thread per slot: the fixed-point words are read in slot order
    // (coalesced) and each atom's row is written through slot_atom.
    if (blockIdx.x + 1 != gridDim.x) {
        const int s = blockIdx.x * 256 + threadIdx.x;
        if (s < D.n_pad && D.grad != nullptr) {
            const int i = D.slot_atom[s];
            if (i >= 0) {
                for (int k = 0; k < 3; k++) {
                    double g = fx_value(D.facc, D.n_pad, s, k);
                    if (plain) g += D.gplain[3 * (size_t)i + k];
                    D.grad[3 * (size_t)i + k] = D.grad_assign ? g : D.grad[3 * (size_t)i + k] + g;
                }
            }
        }
        return;
    }
    double el, lj, el14, lj14, iel = 0.0, ilj = 0.0;
    {
        // Exact: each slot's low word is split at 2^48 (its upper part carried
        // into the high word), the words are summed as integers over the 64
        // slots, the total is brought to its unique form (low word in
        // [0, 2^48)) and converted once, so the result does not depend on which
        // items shared a slot.
        __shared__ double sE[NB_EKINDS];
        if (threadIdx.x < 64 * NB_EKINDS) {
            const int t = threadIdx.x & 63, kind = threadIdx.x >> 6;
            long long h = 0, l = 0;
            if (t < NB_ESLOTS) {
                const long long a0 = *eacc_word(D.eacc, kind, 0, t);
                h = *eacc_word(D.eacc, kind, 1, t) + (a0 >> 48);
                l = a0 & ((1ll << 48) - 1);
            }
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) {
                h += __shfl_xor(h, o, 64);
                l += __shfl_xor(l, o, 64);
            }
            if (t == 0) {
                // Canonical words of the total (0 <= low < 2^48), then one rounding.
                h += l >> 48;
                l &= (1ll << 48) - 1;
                sE[kind] = 0.5 * ((double)h * NB_FX_HI_UNIT + (double)l / NB_FX_LO_SCALE);
            }
        }
        __syncthreads();
        el = sE[0];
        lj = sE[1];
        iel = sE[2];
        ilj = sE[3];
    }
    if (plain) {
        sum_range2(D.eplain, D.n_plain_blocks, el, lj);
        el *= 0.5;
        lj *= 0.5;
        if (D.eimgpart) sum_range2(D.eimgpart, D.n_img_items, iel, ilj);
    }
    sum_range2(D.epart14, D.n14_blocks, el14, lj14);
    double qlj = 0.0, qlj14 = 0.0;
    if (D.qljpart) sum_range2(D.qljpart, D.n_qlj, qlj, qlj14);
    if (threadIdx.x == 0) {
        D.energies[0] = el;
        D.energies[1] = lj;
        D.energies[2] = el14;
        D.energies[3] = lj14;
        D.energies[4] = iel;
        D.energies[5] = ilj;
        D.energies[6] = qlj;
        D.energies[7] = qlj14;
        // The call's error bits travel with its energies; the word starts the next call clear.
        int e = 0;
        if (D.err) {
            e = __hip_atomic_exchange(as_global(D.err), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // The plain path's energies are FP64 sums with no fixed-point stage.
            if (plain && !(isfinite(el) && isfinite(lj) && isfinite(iel) && isfinite(ilj))) e |= NB_ERR_RANGE;
        }
        D.energies[NB_ESTATUS] = (double)e;
    }
}

// ------------------------------------------------------------------------------------------------
// QC/MM LJ (NBModelABFS_QCMMEnergyLJ, pMolecule-1.9.0/extensions/csource/NBModelABFS.c:306-378):
// the analytic pair terms with no electrostatics over the QC/MM LJ list (the main LJ table) and
// its 1-4 list (the 1-4 table), NB_QCMM_CHUNKS workgroups per pure QC atom; gradients into the fixed-point
// accumulators, the two energies of each (row, chunk) into qljpart.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_qclj(const SysDesc *__restrict__ descs, AbfsFactors F)
{
#pragma clang fp contract(off)
    const SysDesc &D = descs[0];
    const int r = blockIdx.x, c = blockIdx.y, stride = gridDim.y * 256;
    const int i = D.qlj_atom[r];
    const double xi = D.xyz[3 * (size_t)i], yi = D.xyz[3 * (size_t)i + 1], zi = D.xyz[3 * (size_t)i + 2];
    const int ti = D.ntypes * D.atype[i];
    const int si = D.atom_slot[i];
    double e[2] = {0.0, 0.0}, g[3] = {0.0, 0.0, 0.0};
    bool bad = false;
    for (int list = 0; list < 2; list++) {
        const int *ptr = list ? D.qlj14_ptr : D.qlj_ptr;
        const int *idx = list ? D.qlj14_idx : D.qlj_idx;
        const double *tA = list ? D.ljA14 : D.ljA;
        const double *tB = list ? D.ljB14 : D.ljB;
        for (int k = ptr[r] + c * 256 + threadIdx.x; k < ptr[r + 1]; k += stride) {
            const int j = idx[k];
            double xij = xi - D.xyz[3 * (size_t)j], yij = yi - D.xyz[3 * (size_t)j + 1],
                   zij = zi - D.xyz[3 * (size_t)j + 2];
            const double r2 = xij * xij + yij * yij + zij * zij;
            const int tij = ti + D.atype[j];
            double x1, x2, dF;
            if (!pair_fp64(F, r2, 0.0, tA[tij], tB[tij], x1, x2, dF)) continue;
            e[list] += x2;
            xij *= (2.0 * dF);
            yij *= (2.0 * dF);
            zij *= (2.0 * dF);
            g[0] += xij;
            g[1] += yij;
            g[2] += zij;
            const int sj = D.atom_slot[j];
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 0, -xij);
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 1, -yij);
            bad |= fx_atomic_add(D.facc, D.n_pad, sj, 2, -zij);
        }
    }
    raise_error(D.err, bad, NB_ERR_RANGE);
    // block_sum2's shared arrays are reused: a barrier after each sum.
    block_sum2<256>(e[0], e[1]);
    __syncthreads();
    double gz = g[2];
    block_sum2<256>(g[0], g[1]);
    __syncthreads();
    double zz = 0.0;
    block_sum2<256>(gz, zz);
    bool bad_i = false;
    if (threadIdx.x == 0) {
        D.qljpart[2 * ((size_t)r * gridDim.y + c)] = e[0];
        D.qljpart[2 * ((size_t)r * gridDim.y + c) + 1] = e[1];
        bad_i |= fx_atomic_add(D.facc, D.n_pad, si, 0, g[0]);
        bad_i |= fx_atomic_add(D.facc, D.n_pad, si, 1, g[1]);
        bad_i |= fx_atomic_add(D.facc, D.n_pad, si, 2, gz);
        bad_i |= !isfinite(e[0]) || !isfinite(e[1]);
    }
    raise_error(D.err, bad_i, NB_ERR_RANGE);
}

void launch_qclj(const SysDesc *d_desc, int nrows, const AbfsFactors &F, hipStream_t s)
{
    if (nrows > 0) hipLaunchKernelGGL(k_qclj, dim3(nrows, NB_QCMM_CHUNKS), dim3(256), 0, s, d_desc, F);
}

// ------------------------------------------------------------------------------------------------
// Launchers.
// ------------------------------------------------------------------------------------------------
void launch_prepare(const SysDesc *d_desc, int nsys, int max_npad, int tiled, int *heads, const PrepareCheck &chk,
                    hipStream_t s)
{
    if (nsys <= 0) return;
    hipLaunchKernelGGL(k_prepare, dim3(std::max(nblk(max_npad, 256), 1), nsys), dim3(256), 0, s, d_desc, tiled, heads,
                       chk);
}

template <bool ROWS_LDS, bool IMG, bool F64, int WPG>
static void launch_tiled_instance(dim3 grid, size_t bytes, hipStream_t s, hipEvent_t ev_start, hipEvent_t ev_stop,
                                  const SysDesc *d_desc, const WorkItem *items, QueueParams q,
                                  const typename PairFactors<F64>::type &F,
                                  int rows_bytes, int wave_bytes, ForceGuard g, int nitems, int nforce_groups,
                                  int sys1)
{
    hipExtLaunchKernelGGL((k_force_tiled<ROWS_LDS, IMG, F64, WPG>), grid, dim3(64 * WPG), bytes, s, ev_start, ev_stop, 0,
                          d_desc, items, q, F, rows_bytes, wave_bytes, g, nitems, nforce_groups, sys1);
}

void launch_force_tiled(const SysDesc *d_desc, const WorkItem *items, QueueParams q, const TiledFactors &F,
                        int nblocks, int max_ntypes, ForceGuard g, hipStream_t s, bool images,
                        hipEvent_t ev_start, hipEvent_t ev_stop, int n14_blocks, const FullFactors *full, int sys1)
{
    if (nblocks + n14_blocks <= 0) return;
    // One item per wave, four waves per group, unless the items come from the persistent queues.
    const int wpg = q.heads != nullptr ? 1 : NB_TILED_WPG;
    const int ngroups = nblk(nblocks, wpg);
    const dim3 grid(ngroups + nblk(n14_blocks, wpg));
    const int acc = full ? 8 : 4;
    const int wave_bytes = (int)tiled_lds_wave(acc);
    // The row table goes to LDS when the group's LDS still lets four groups of four waves (or ten single waves) share a CU
    // (five groups do up to 32 KB: ten types with 16 entries per wave take 27 KB).
    const size_t limit = wpg == 1 ? NB_LDS_ROW_LIMIT : NB_LDS_GROUP_LIMIT;
    const bool rows_lds = tiled_lds_rows(max_ntypes, true) + (size_t)wpg * wave_bytes <= limit;
    const int rows_bytes = (int)tiled_lds_rows(max_ntypes, rows_lds);
    const size_t bytes = rows_bytes + (size_t)wpg * wave_bytes;
#define NB_TILED_ARGS(F) grid, bytes, s, ev_start, ev_stop, d_desc, items, q, F, rows_bytes, wave_bytes, g, nblocks, ngroups, \
                      sys1
    if (full) {
        if (wpg == 1) {
            if (rows_lds)
                launch_tiled_instance<true, false, true, 1>(NB_TILED_ARGS(*full));
            else
                launch_tiled_instance<false, false, true, 1>(NB_TILED_ARGS(*full));
        } else {
            if (rows_lds)
                launch_tiled_instance<true, false, true, NB_TILED_WPG>(NB_TILED_ARGS(*full));
            else
                launch_tiled_instance<false, false, true, NB_TILED_WPG>(NB_TILED_ARGS(*full));
        }
    } else if (images) {
        if (rows_lds)
            launch_tiled_instance<true, true, false, NB_TILED_WPG>(NB_TILED_ARGS(F));
        else
            launch_tiled_instance<false, true, false, NB_TILED_WPG>(NB_TILED_ARGS(F));
    } else if (wpg == 1) {
        if (rows_lds)
            launch_tiled_instance<true, false, false, 1>(NB_TILED_ARGS(F));
        else
            launch_tiled_instance<false, false, false, 1>(NB_TILED_ARGS(F));
    } else {
        if (rows_lds)
            launch_tiled_instance<true, false, false, NB_TILED_WPG>(NB_TILED_ARGS(F));
        else
            launch_tiled_instance<false, false, false, NB_TILED_WPG>(NB_TILED_ARGS(F));
    }
#undef NB_TILED_ARGS
}

void launch_force_plain(const SysDesc *d_desc, int nsys, int max_n, const AbfsFactors &F, ForceGuard g, hipStream_t s,
                        hipEvent_t ev_start, hipEvent_t ev_stop)
{
    if (nsys <= 0) return;
    hipExtLaunchKernelGGL(k_force_plain, dim3(max(nblk(max_n, 256), 1), nsys), dim3(256), 0, s, ev_start, ev_stop, 0,
                          d_desc, F, g);
}

void launch_force_image_fp64(const SysDesc *d_desc, const WorkItem *items, int nitems, const AbfsFactors &F,
                             ForceGuard g, hipStream_t s, hipEvent_t ev_start, hipEvent_t ev_stop)
{
    if (nitems > 0)
        hipExtLaunchKernelGGL(k_force_image_fp64, dim3(nitems), dim3(64), 0, s, ev_start, ev_stop, 0, d_desc, items, F, g);
}

void launch_pairs14(const SysDesc *d_desc, int nsys, int max_n14_blocks, const AbfsFactors &F, hipStream_t s,
                    ForceGuard g)
{
    if (nsys > 0 && max_n14_blocks > 0)
        hipLaunchKernelGGL(k_pairs14, dim3(max_n14_blocks, nsys), dim3(64), 0, s, d_desc, F, g);
}

void launch_finalize(const SysDesc *d_desc, int nsys, int max_npad, int plain, hipStream_t s, ForceGuard g)
{
    if (nsys <= 0) return;
    hipLaunchKernelGGL(k_finalize, dim3(nblk(max_npad, 256) + 1, nsys), dim3(256), 0, s, d_desc, plain, g);
}

// ------------------------------------------------------------------------------------------------
// Virial of the last call's gradient (still in the fixed-point accumulators,
// plus the plain path's rows), W_ab = sum_i (x_i - o)_a g_i,b: wave sums in
// FP64 added into fixed point (slot = wave index modulo 64), so the total
// does not depend on which waves shared a slot.  vacc must be zero.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_virial(const SysDesc *__restrict__ descs, int plain)
{
    const SysDesc &D = descs[0];
    const int i = blockIdx.x * 256 + threadIdx.x;
    double g[3] = {0.0, 0.0, 0.0}, x[3] = {0.0, 0.0, 0.0};
    if (i < D.n) {
        const int s = D.atom_slot[i];
        for (int k = 0; k < 3; k++) {
            g[k] = fx_value(D.facc, D.n_pad, s, k);
            if (plain) g[k] += D.gplain[3 * (size_t)i + k];
            x[k] = D.xyz[3 * (size_t)i + k] - D.origin[k];
        }
    }
    const int slot = ((blockIdx.x * 4 + (threadIdx.x >> 6)) & (NB_ESLOTS - 1));
#pragma unroll
    for (int ab = 0; ab < 9; ab++) {
        const double w = wave_sum_f64(x[ab / 3] * g[ab % 3]);
        if ((threadIdx.x & 63) == ab && w != 0.0)
            fx_add(&D.vacc[(2 * ab) * NB_ESLOTS + slot], &D.vacc[(2 * ab + 1) * NB_ESLOTS + slot], w);
    }
}

void launch_virial(const SysDesc *d_desc, int n, int plain, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_virial, dim3(nblk(n, 256)), dim3(256), 0, s, d_desc, plain);
}
