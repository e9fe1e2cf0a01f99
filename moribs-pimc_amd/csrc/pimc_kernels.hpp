// pimc_kernels.hpp -- gfx950 kernels of the sampling hot path.
//
//   k_bisect     linear family: a group of 32 to 256 lanes per (replica, imaginary-time segment).
//                All atoms' beads on the segment's inner slices, plus the linear rotor's axis
//                there, are staged in LDS once and every atom of the selected types is moved in
//                turn, as MCBisectionMove does (mc_piqmc.cc:194-294).  Segments of one offset
//                share only fixed end points, so they run concurrently.
//   k_bisect_nl  the same for the non-linear family, one workgroup per segment.
//   k_centroid_parts  a replica's slices split over workgroups; atoms in turn, Delta V over the
//                part's slices x partners, partials exchanged as numbered words in memory
//                (MCMolecularMove mc_piqmc.cc:54-102).
//   k_rotor      one workgroup per part of a linear rotor's chain (a range of slices): the part's
//                orientations and its rotor-partner geometry live on chip for all sweeps of a
//                launch; each half of the even/odd checkerboard (mc_piqmc.cc:490-512) is a
//                parallel step over slices (MCRotLinStep :781-936), tests on one or two waves
//                and the partner energies of the next half's proposals on the others; parts
//                trade one boundary slice per half-sweep as a record of numbered words (each
//                64-bit word: the publishing half's number over 32 bits of a double), so a poll
//                of the record returns the data with its check.
//   k_est_tiles  one workgroup per (replica, tile of slices): the tile's part of the pair sum of
//                GetPotEnergy_Densities (mc_estim.cc:500-687, every pair, with the g(r),
//                g(r,theta) and (r,theta,chi) bins) and of GetKinEnergy (mc_estim.cc:876-937),
//                beads read once.
//   k_est_final  one workgroup per replica: tiles summed in order (deterministic), GetRotEnergy
//                (mc_estim.cc:939-987) or GetRotE3D with its relative Euler angle bins
//                (:989-1096), and the Cv terms of MCGetAverage (mc_main.cc:551-616).
//   k_pot_slice  batched PotEnergy(atom, pos, it) (mc_piqmc.cc:1796-1965).
//   k_rotor3d_da the non-linear rotor sweep with a surrogate first stage (delayed acceptance).
#pragma once
#include <type_traits>
#include "pimc_device.hpp"
#include "pimc_nl.hpp"
#include "pimc_mlp.hpp"
#include "pimc_plan.hpp"

// A launch's LDS begins on 16 bytes whatever the kernel's own __shared__ data come to.  Behind an odd
// number of doubles it would begin 8 bytes off, and every vec4 of knots, beads or frames in it would
// be read with two instructions or more: on a stretched 1D table k_centroid_parts took 0.31 ms that
// way on 256 chains of 8 atoms at 128 slices and takes 0.15, 4.34 and 3.09 on 4 chains of 100 at 256.
#define DYNAMIC_LDS __attribute__((aligned(16)))

namespace pimc {

struct Run {
    uint32_t seed;
    int u;           // offset within the segment stride (segment order) or time slice (reference order)
    int ref_order;   // 1: one segment/sweep per replica per launch (mc_main.cc order)
    int type_begin, type_end;
};

__device__ __forceinline__ double4 bead(const double4* beads, const Rep& rp, int a, int it) {
    return beads[rp.bead_off + (long long)a * rp.P + it];
}

__device__ __forceinline__ int type_of(const Rep& rp, int a) {
    int t = 0;
    while (t + 1 < rp.ntypes && a >= rp.tbegin[t + 1]) ++t;
    return t;
}

// sum over the block; `red` holds one value per wave (16 for 1024 lanes)
template <typename T>
__device__ __forceinline__ T block_sum(T v, T* red) {
    v = wave_sum(v);
    const int wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[wid] = v;
    __syncthreads();
    T s = 0;
    for (int i = 0; i < nw; ++i) s += red[i];
    return s;
}

__device__ __forceinline__ void rotor_axis(const RotBead* rotb, const Rep& rp, int it, double& nx, double& ny,
                                           double& nz) {
    if (rp.rotkind == 1 && rp.rot_atom >= 0) {
        int ar = rp.rot_atom - rp.tbegin[rp.imtype];
        RotBead rb = rotb[rp.rot_off + (long long)ar * rp.Prot + it / rp.RotRatio];
        nx = rb.nx; ny = rb.ny; nz = rb.nz;
    } else {
        nx = 0; ny = 0; nz = 1;
    }
}

// PotEnergy's dispatch (mc_piqmc.cc:1847-1958) for the non-linear family: pairs of the atom
// type by SPot1D, atom / non-linear rotor pairs by vcord with the rotor's frame at that slice
// (rcom = the rotor, rpt = the atom), rotor / rotor pairs by caleng.  vcord and caleng take the
// positions themselves, so the minimum image (box) reaches the atom pairs only, as there.
template <typename R>
__device__ __forceinline__ double pair_nl(const Lut1D<R>& l1, const vec4_t<R>* __restrict__ k1, const Lut3D<R>& l3,
                                          bool rot_a, bool rot_j, double xa, double ya, double za, double xj,
                                          double yj, double zj, const Frame& fa, const Frame& fj,
                                          const double* box = nullptr) {
    if (rot_a && rot_j) return caleng_v(xa, ya, za, xj, yj, zj, fa, fj);
    if (rot_a) return (double)vcord_v<R>(l3, fa, xa, ya, za, xj, yj, zj);
    if (rot_j) return (double)vcord_v<R>(l3, fj, xj, yj, zj, xa, ya, za);
    const R dx = (R)nearest_image(xa - xj, box, 0), dy = (R)nearest_image(ya - yj, box, 1),
            dz = (R)nearest_image(za - zj, box, 2);
    return (double)spot1d<R>(l1, k1, sqrt(dx * dx + dy * dy + dz * dz));
}

__device__ __forceinline__ const Frame& frame_at(const Frame* __restrict__ frames, const Rep& rp, int a, int it) {
    return frames[rp.rot_off + (long long)(a - rp.nl_atom) * rp.Prot + it / rp.RotRatio];
}

// ------------------------------------------------------------------------- bisection
// LDS written by some lanes of a wave and read by others: a wave's LDS operations complete in
// order, so only the compiler has to keep theirs
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the same among the GW lanes of a group, which may span waves
template <int GW>
__device__ __forceinline__ void group_sync() {
    if constexpr (GW > 64) lds_barrier();
    else wave_sync();
}

// The proposals of one launch of the bisection, ahead of it.  An atom's new midpoints depend on its
// draws and on its segment's end points alone, which no move of the launch changes, so every move's
// are formed here with all lanes busy; inside the moves' chain of dependent steps the generator, the
// logarithm and the cosine were a fifth of the time.  prop has the layout of beads: the midpoint of
// an inner slot at that bead's place, and in .w of slot l + 1 the acceptance draw of level l.  The
// launch runs beside the rotor sweep of the phase before, which leaves most issue slots idle.
// A wave takes a batch of (atom, segment) pairs, so that all its lanes draw.
struct PathItem {
    int r, ty, first, pad;  // pairs first, first + 1, ... of type ty; pair = atom * segments + segment
};

// doubles of a batch's draws; pairs of a batch whose moves have nm midpoints and L levels
__host__ __device__ constexpr int path_ring(int nm, int L) { return 192 > 3 * nm + L ? 192 : 3 * nm + L; }
__host__ __device__ constexpr int path_batch(int nm, int L) { return 192 > 3 * nm + L ? 192 / (3 * nm + L) : 1; }

__global__ __launch_bounds__(256) void k_bisect_paths(const Rep* __restrict__ reps, const Mut* __restrict__ mut,
                                                      const double4* __restrict__ beads, double4* __restrict__ prop,
                                                      const PathItem* __restrict__ items, int ring, Run run) {
    extern __shared__ DYNAMIC_LDS double smem[];
    const int l = threadIdx.x & 63;
    double* gw = smem + (threadIdx.x >> 6) * ring;  // the batch's draws: per pair 3 per midpoint, then one per level
    const PathItem item = items[blockIdx.x * 4 + (threadIdx.x >> 6)];
    if (item.r < 0) return;  // padding of the list
    const Rep& rp = reps[item.r];
    const int S = rp.S, P = rp.P;
    if (run.u >= (run.ref_order ? P : S)) return;
    const int ty = item.ty, L = rp.tlev[ty], St = 1 << L, nm = St - 1, per = 3 * nm + L;
    const int nseg = run.ref_order ? 1 : P / S;
    const int left = rp.tnumb[ty] * nseg - item.first;
    const int nk = left < path_batch(nm, L) ? left : path_batch(nm, L);
    const int ia0 = item.first / nseg, seg0 = item.first - ia0 * nseg;
    const uint32_t pass = mut[item.r].pass;
    const float inv_per = 1.0f / (float)per, inv_nm3 = 1.0f / (float)(3 * nm);
    const double gscale = sqrt(rp.lambda[ty] * rp.tau);  // Gaussian width at the last level
    auto pair_at = [&](int k, int& a, int& s0) {
        int seg = seg0 + k, ia = ia0;
        while (seg >= nseg) {
            seg -= nseg;
            ++ia;
        }
        a = rp.tbegin[ty] + ia;
        s0 = run.ref_order ? run.u : run.u + seg * S;
    };
    // Gaussians of midpoint m (level-major order) and the level acceptance uniforms u, kept as
    // -log(u): the level test exp(-dV) > u (mc_piqmc.cc:265-273) is then dV < -log(u), a comparison.
    // Both kinds take one generator call and one logarithm, on one path
    for (int i = l; i < nk * per; i += 64) {
        const int k = (int)(((float)i + 0.5f) * inv_per), d = i - k * per;
        int a, s0;
        pair_at(k, a, s0);
        const bool gauss = d < 3 * nm;
        const int m = d / 3, id = d - 3 * m;
        const int level = gauss ? 31 - __clz(m + 1) : d - 3 * nm;
        const int q = m + 1 - (1 << level);
        const uint4 w4 = draw(run.seed, rp.key, pass, K_BISECT, 0, (uint32_t)a, (uint32_t)s0,
                              ((uint32_t)level << 24) | (gauss ? ((uint32_t)q << 8) | (uint32_t)id : 0xFFFFu << 8));
        const double u = u53(w4.x, w4.y);
        double v = -log(gauss ? 1.0 - u : u);
        if (gauss) {  // Box-Muller of density exp(-alpha x^2), alpha = 1 / (lambda tau 2^(L - level))
            const int ex = L - level;
            v = sqrt(v) * cospi(2.0 * u53(w4.z, w4.w)) * ((ex & 1 ? 1.4142135623730951 : 1.0) * (double)(1 << (ex >> 1)) * gscale);
            gw[i] = v;
        } else {
            const int it = s0 + 1 + level < P ? s0 + 1 + level : s0 + 1 + level - P;
            prop[rp.bead_off + (long long)a * P + it].w = v;
        }
    }
    wave_sync();
    // coordinate id of slot s: a lane follows its slot down the bisection tree (the midpoints above
    // it are formed again with the same operands)
    for (int i = l; i < nk * 3 * nm; i += 64) {
        const int k = (int)(((float)i + 0.5f) * inv_nm3), c = i - k * 3 * nm;
        const int s = c / 3 + 1, id = c - 3 * (s - 1);
        int a, s0;
        pair_at(k, a, s0);
        const long long b0 = rp.bead_off + (long long)a * P;
        double lo = reinterpret_cast<const double*>(beads + b0 + s0)[id];
        double hi = reinterpret_cast<const double*>(beads + b0 + (s0 + St < P ? s0 + St : s0 + St - P))[id];
        const double* g = gw + k * per;
        double v;
        for (int level = 0;; ++level) {
            const int q = s >> (L - level), mid = (q << (L - level)) + (1 << (L - level - 1));
            v = 0.5 * (lo + hi) + g[3 * ((1 << level) - 1 + q) + id];
            if (s == mid) break;
            if (s < mid) hi = v;
            else lo = v;
        }
        reinterpret_cast<double*>(prop + b0 + (s0 + s < P ? s0 + s : s0 + s - P))[id] = v;
    }
}

// The linear family (atoms and at most one linear rotor): a group of GW lanes per segment.  GW of 32
// or 64 keeps a segment within a wave (two share one), so that nothing waits on a barrier and what
// does not grow with the partners (level sums, tests) costs one wave; GW of 128 or 256 spreads one
// segment over waves, for the few segments of a single chain.  Per segment LDS holds the mover's
// midpoints, the rotor terms and, in the pair precision, the S-1 inner slots of every atom: 12 bytes
// a bead in FP32.  A move sums Delta V of its levels in chunks, each one pass over (midpoint,
// partner) and one reduction: a chunk's midpoints share the group, GW over a power of two lanes each.

// bytes of one segment in LDS (nwf, nhf, part, th, rt, win of k_bisect, in that order)
__host__ __device__ constexpr int bisect_seg_bytes(int N, int S, int rsize) {
    return (8 * rsize * (S - 1) + 8 * (16 + 16) + rsize * (2 * (S - 1) + 3 * N * (S - 1)) + 15) & ~15;
}

// Sum of V(new) - V(old) over U partners of an atom at one slot, from the separations
// d[0 .. U-1] (new position) and d[U .. 2U-1] (old); the first `ok` partners count
template <typename R, bool UT, int U>
__device__ __forceinline__ double atom_terms(const Lut1D<R>& l1, const void* kn, const R (&d)[2 * U][3], int ok) {
    R r[2 * U], v[2 * U];
#pragma unroll
    for (int i = 0; i < 2 * U; ++i) {
        if constexpr (UT) r[i] = fast_sqrt(dot3(d[i][0], d[i][1], d[i][2], d[i][0], d[i][1], d[i][2]));
        else r[i] = fast_sqrt(d[i][0] * d[i][0] + d[i][1] * d[i][1] + d[i][2] * d[i][2]);
    }
    if constexpr (UT) {
        spot1d_u2_many<2 * U>(l1, static_cast<const float2*>(kn), r, v);
    } else {
#pragma unroll
        for (int i = 0; i < 2 * U; ++i) v[i] = spot1d<R>(l1, static_cast<const vec4_t<R>*>(kn), r[i]);
    }
    double acc = 0.0;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const double t = (double)v[i] - (double)v[U + i];
        acc += i < ok ? t : 0.0;
    }
    return acc;
}

// MI: built for contexts that hold a replica under the minimum image (its pairs then take their
// nearest image); without it the kernels carry no trace of it.  UT: FP32 on uniform 1D and 2D
// tables, a launch of its own for the replicas that have them, so that a chain's arithmetic does
// not depend on the replicas beside it.  Uniform FP32 1D knots are staged as (y, y'') pairs.
template <typename R, bool MI, bool UT, int GW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_bisect(
    const Rep* __restrict__ reps, Mut* __restrict__ mut, double4* __restrict__ beads, const RotBead* __restrict__ rotb,
    Tables T, const double4* __restrict__ prop, const int2* __restrict__ work, Run run) {
    extern __shared__ DYNAMIC_LDS double smem[];
    using P4 = vec4_t<R>;
    const int2 wk = work[blockIdx.x];
    const Rep& rp = reps[wk.x];
    const int S = rp.S, P = rp.P, N = rp.natoms, lgS = 31 - __clz(S), S1 = S - 1;
    if (run.u >= (run.ref_order ? P : S)) return;
    const int gl = (int)threadIdx.x & (GW - 1);
    const Lut1D<R> l1 = lut1d<R>(T, rp.pot1d_id);
    const Lut2D<R> l2 = lut2d<R>(T, rp.pot2d_id);
    const double* box = MI && rp.minimage ? rp.box : nullptr;  // MINIMAGE (not with a rotating linear rotor)
    // the 1D knots, shared by the block's segments
    P4* kn = reinterpret_cast<P4*>(smem);
    int kbytes = l1.n * (int)sizeof(P4);
    const bool half = is_fp32<R>() && (UT || l1.uniform);
    if (half) {
        float2* k2 = reinterpret_cast<float2*>(kn);
        for (int i = threadIdx.x; i < l1.n; i += blockDim.x) k2[i] = make_float2((float)l1.k[i].y, (float)l1.k[i].z);
        kbytes = (l1.n * (int)sizeof(float2) + 15) & ~15;
    } else {
        for (int i = threadIdx.x; i < l1.n; i += blockDim.x) kn[i] = l1.k[i];
    }
    __syncthreads();
    const int seg = wk.y + (int)threadIdx.x / GW;
    if (seg >= (run.ref_order ? 1 : P / S)) return;  // no segment for this group: it leaves whole
    const int s0 = run.ref_order ? run.u : run.u + seg * S;
    char* mem = reinterpret_cast<char*>(smem) + kbytes +
                ((int)threadIdx.x / GW) * bisect_seg_bytes(N, S, (int)sizeof(R));
    P4* nwf = reinterpret_cast<P4*>(mem);                // the move's new midpoints, pair precision
    P4* nhf = nwf + S1;                                  // rotor axes
    double* part = reinterpret_cast<double*>(nhf + S1);  // partial sums of a chunk, two buffers of 8
    double* th = part + 16;                              // level tests of this move and the next, 8 each
    R* rt = reinterpret_cast<R*>(th + 16);               // rotor terms (new, old) of every midpoint
    R* win = rt + 2 * S1;                                // [slot - 1][atom][3]
    for (int i = gl; i < N << lgS; i += GW) {
        const int w = i & S1, a = i >> lgS;
        if (w == 0) continue;
        const int it = s0 + w < P ? s0 + w : s0 + w - P;
        const double4 b = bead(beads, rp, a, it);
        R* d = win + ((w - 1) * N + a) * 3;
        d[0] = (R)b.x;
        d[1] = (R)b.y;
        d[2] = (R)b.z;
    }
    for (int w = gl; w < S1; w += GW) {
        double x, y, z;
        rotor_axis(rotb, rp, s0 + 1 + w < P ? s0 + 1 + w : s0 + 1 + w - P, x, y, z);
        P4 q;
        q.x = (R)x;  // the pair functions take the axis in the pair precision
        q.y = (R)y;
        q.z = (R)z;
        q.w = (R)0;
        nhf[w] = q;
    }

    const bool has_rotor = rp.lin_atom >= 0;  // then the last atom
    const int nat = has_rotor ? N - 1 : N;    // atoms
    const double tau = rp.tau;
    // Midpoints whose terms a move's tests needed: of the levels up to its rejection.  A wave of one
    // segment counts them on the scalar unit (on its lanes they were up to 1% of a pass)
    unsigned mids = 0;
    auto any = [](bool b) -> bool {
        if constexpr (GW >= 64) return __builtin_amdgcn_ballot_w64(b) != 0;
        else return b;
    };
    int pb = 0;  // buffer of the next partial sums
    const int tend = run.type_end < rp.ntypes ? run.type_end : rp.ntypes;

    for (int ty = run.type_begin; ty < tend; ++ty) {
        const int L = rp.tlev[ty];
        const int nm = (1 << L) - 1;
        unsigned acc_n = 0;
        // slot gl + 1 of the mover on lane gl: its proposal in registers from one move ahead until
        // it is accepted.  (Moves of more midpoints than lanes read the others where they need them.)
        const int itl = s0 + 1 + gl < P ? s0 + 1 + gl : s0 + 1 + gl - P;
        long long ib = rp.bead_off + (long long)rp.tbegin[ty] * P;
        auto proposal = [&](int i) { return prop[ib + (s0 + 1 + i < P ? s0 + 1 + i : s0 + 1 + i - P)]; };
        auto put = [&](int i, const double4& v, int buf) {
            P4 q;
            q.x = (R)v.x;
            q.y = (R)v.y;
            q.z = (R)v.z;
            q.w = (R)0;
            nwf[i] = q;
            if (i < L) th[8 * buf + i] = v.w;
        };
        // the first three levels one by one (bisect_level_passes).  The bounds that it implies are for
        // the compiler: with the flag alone, or with the rule written out here, the loops are 3% slower
        const bool single = !UT && GW == 256 && !l1.uniform && nat > 64 && rp.level_passes;
        const bool three = L >= 3 && !single;
        const int m3 = gl / (GW / 8), lv3 = m3 < 7 ? 31 - __clz(m3 + 1) : 0;  // the lane's midpoint of the first three levels
        const int slot3 = m3 < 7 && three ? ((m3 + 1 - (1 << lv3)) << (L - lv3)) + (1 << (L - lv3 - 1)) - 1 : 0;
        const double tauh = tau * (double)(1 << (L - 1));
        double4 cur = make_double4(0.0, 0.0, 0.0, 0.0);
        if (gl < nm) cur = prop[ib + itl];
        group_sync<GW>();
        for (int i = gl; i < nm; i += GW) put(i, i == gl ? cur : proposal(i), 0);
        group_sync<GW>();
        for (int ia = 0; ia < rp.tnumb[ty]; ++ia) {
            const int a = rp.tbegin[ty] + ia;
            const double* tst = th + 8 * (ia & 1);  // this move's level tests
            double4 nxt = cur;
            if (gl < nm && ia + 1 < rp.tnumb[ty]) nxt = prop[ib + P + itl];
            auto level_sums = [&](auto mi_c) -> bool {
                // the minimum image as its own instance of the loops, so the plain one is unchanged
                const double* bx = decltype(mi_c)::value ? box : nullptr;
                const bool rot_a = a == rp.lin_atom;
                // the terms with the rotor of every midpoint, new and old on neighbouring lanes: one
                // pass of that code per move.  On uniform FP32 tables the table loads fly while the
                // first chunk's atom terms run
                const bool rterms = has_rotor && !rot_a;
                auto slot_of = [&](int m) {  // of midpoint m, level-major order
                    const int level = 31 - __clz(m + 1), q = m + 1 - (1 << level);
                    return (q << (L - level)) + (1 << (L - level - 1)) - 1;
                };
                // separation from the rotor at midpoint i / 2, of the new (even i) or old position
                auto to_rotor = [&](int i, R (&d)[3], P4& ax) {
                    const int slot = slot_of(i >> 1);
                    const R* pr = win + (slot * N + N - 1) * 3;
                    const R* po = win + (slot * N + a) * 3;
                    const P4 pn = nwf[slot];
                    ax = nhf[slot];
                    d[0] = nearest_image((i & 1 ? po[0] : pn.x) - pr[0], bx, 0);
                    d[1] = nearest_image((i & 1 ? po[1] : pn.y) - pr[1], bx, 1);
                    d[2] = nearest_image((i & 1 ? po[2] : pn.z) - pr[2], bx, 2);
                };
                RotorCell rc{};
                const bool early = UT && 2 * nm <= GW;
                if (rterms)
                    for (int i = gl; i < 2 * nm; i += GW) {
                        R d[3];
                        P4 ax;
                        to_rotor(i, d, ax);
                        if constexpr (UT) {
                            rc = rotor_pair_load(l2, false, d[0], d[1], d[2], ax.x, ax.y, ax.z);
                            if (!early) rt[i] = rotor_pair_value(rc);
                        } else {
                            rt[i] = pair_d<R>(l1, kn, l2, false, true, d[0], d[1], d[2], (double)ax.x, (double)ax.y,
                                              (double)ax.z);
                        }
                    }
                // V(new) - V(old) of the mover at a slot with partners jl, jl + G, ...
                auto pairs = [&](int slot, int jl, int G) -> double {
                    double acc = 0.0;
                    const P4 pn = nwf[slot];
                    const R* po = win + (slot * N + a) * 3;
                    const R xa = po[0], ya = po[1], za = po[2];
                    const R* ws = win + slot * N * 3;
                    if (rot_a) {  // the rotor's partners are the atoms before it
                        const P4 ax = nhf[slot];
                        for (int j = jl; j < nat; j += G) {
                            const R* pj = ws + 3 * j;
                            const R dx = nearest_image(pn.x - pj[0], bx, 0), dy = nearest_image(pn.y - pj[1], bx, 1),
                                    dz = nearest_image(pn.z - pj[2], bx, 2);
                            const R ex = nearest_image(xa - pj[0], bx, 0), ey = nearest_image(ya - pj[1], bx, 1),
                                    ez = nearest_image(za - pj[2], bx, 2);
                            R vn, vo;
                            if constexpr (UT) {
                                const RotorCell kn_ = rotor_pair_load(l2, true, dx, dy, dz, ax.x, ax.y, ax.z);
                                const RotorCell ko_ = rotor_pair_load(l2, true, ex, ey, ez, ax.x, ax.y, ax.z);
                                vn = rotor_pair_value(kn_);
                                vo = rotor_pair_value(ko_);
                            } else {
                                const double nx = ax.x, ny = ax.y, nz = ax.z;
                                vn = pair_d<R>(l1, kn, l2, true, false, dx, dy, dz, nx, ny, nz);
                                vo = pair_d<R>(l1, kn, l2, true, false, ex, ey, ez, nx, ny, nz);
                            }
                            acc += (double)vn - (double)vo;
                        }
                    } else {
                        auto partners = [&](auto u_c) {
                            constexpr int U = decltype(u_c)::value;
                            for (int jp = jl; jp < nat - 1; jp += U * G) {
                                R d[2 * U][3];
#pragma unroll
                                for (int i = 0; i < U; ++i) {
                                    const int jn = i == 0 || jp + i * G < nat - 1 ? jp + i * G : jp;
                                    const R* pj = ws + 3 * (jn + (jn >= a));
                                    const R x = pj[0], y = pj[1], z = pj[2];
                                    d[i][0] = nearest_image(pn.x - x, bx, 0);
                                    d[i][1] = nearest_image(pn.y - y, bx, 1);
                                    d[i][2] = nearest_image(pn.z - z, bx, 2);
                                    d[U + i][0] = nearest_image(xa - x, bx, 0);
                                    d[U + i][1] = nearest_image(ya - y, bx, 1);
                                    d[U + i][2] = nearest_image(za - z, bx, 2);
                                }
                                const int ok = U == 1 || jp + G < nat - 1 ? U : 1;
                                if constexpr (is_fp32<R>() && !UT)
                                    acc += half ? atom_terms<R, true, U>(l1, kn, d, ok) : atom_terms<R, false, U>(l1, kn, d, ok);
                                else
                                    acc += atom_terms<R, UT, U>(l1, kn, d, ok);
                            }
                        };
                        // partners in pairs, so that four look-ups of a lane interleave,
                        // where most lanes have two or more
                        bool two = false;
                        if constexpr (UT) {
                            two = 2 * (nat - 1) > 3 * G;
                            if (two) partners(std::integral_constant<int, 2>{});
                        }
                        if (!two) partners(std::integral_constant<int, 1>{});
                    }
                    return acc;
                };
                double cum = 0.0;
                bool alive = true;
                // The first three levels as one pass: an eighth of the group's lanes per midpoint, the
                // sums of the seven midpoints added in their order.  With the general pass's loops and
                // branches on L for them a move of 64 atoms issued 430 vector and 200 scalar
                // instructions a wave and then read the partial sums one by one: a launch over 16
                // boxes of 64 atoms 153 us, now 108; one chain of 64 145, now 107; the 256-replica
                // scan 410, now 365.
                if (three) {
                    constexpr int G3 = GW / 8;
                    double acc = 0.0;
                    if (m3 < 7) acc = pairs(slot3, gl & (G3 - 1), G3);
                    if (rterms) {
                        if constexpr (UT)
                            if (early && gl < 2 * nm) rt[gl] = rotor_pair_value(rc);
                        group_sync<GW>();
                        if (m3 < 7 && (gl & (G3 - 1)) == 0) acc += (double)rt[2 * m3] - (double)rt[2 * m3 + 1];
                    }
                    acc = group_sum(acc, G3);
                    double* pt = part + 8 * pb;
                    pb ^= 1;
                    if ((gl & (G3 - 1)) == 0) pt[m3] = acc;
                    group_sync<GW>();
                    double p[7], t[3];
#pragma unroll
                    for (int i = 0; i < 7; ++i) p[i] = pt[i];
#pragma unroll
                    for (int i = 0; i < 3; ++i) t[i] = tst[i];
                    // sum over all points up to a level; level acceptance of mc_piqmc.cc:263-273
                    const double c0 = p[0], c1 = (c0 + p[1]) + p[2], c2 = (((c1 + p[3]) + p[4]) + p[5]) + p[6];
                    const double dv0 = c0 * tauh, dv1 = (c1 - 2.0 * c0) * (0.5 * tauh), dv2 = (c2 - 2.0 * c1) * (0.25 * tauh);
                    // without branches: the tests' reads are then under way together
                    const bool b0 = (dv0 < 0.0) | (dv0 < t[0]), b1 = b0 & ((dv1 < 0.0) | (dv1 < t[1]));
                    alive = b1 & ((dv2 < 0.0) | (dv2 < t[2]));
                    mids += 1u + (any(b0) ? 2u : 0u) + (any(b1) ? 4u : 0u);
                    cum = c2;
                }
                for (int l0 = three ? 3 : 0; l0 < L;) {
                    if (GW >= 64 ? !alive : !__any(alive)) break;
                    // levels [l0, l1e) in this pass: the first three together, then one at a time.
                    // Terms of levels behind a rejection are a fifth of all on the 256-replica scan
                    // (half on 8 atoms) and cost less than a pass and a reduction per level: 5.5
                    // against 6.2 ms per pass there, 1.31 against 1.55 on a single 64-atom chain
                    const int l1e = l0 > 0 || single ? l0 + 1 : (L < 3 ? L : 3);
                    const int m0 = (1 << l0) - 1, nmc = (1 << l1e) - 1 - m0;
                    // lanes per midpoint: the chunk's midpoints rounded up to a power of two
                    const int lgn = l0 > 0 ? l0 : (l1e == 1 ? 0 : l1e);
                    const int G = GW >> lgn > 0 ? GW >> lgn : 1;
                    if (alive) {
                        const int lgG = 31 - __clz(G);
                        const int jl = gl & (G - 1);
                        double acc = 0.0;
                        for (int mc = gl >> lgG; mc < nmc; mc += GW >> lgG) {
                            const int slot = slot_of(m0 + mc);
                            acc += pairs(slot, jl, G);
                        }
                        if (rterms) {
                            if constexpr (UT)
                                if (l0 == 0 && early && gl < 2 * nm)
                                    rt[gl] = rotor_pair_value(rc);
                            if (l0 == 0) group_sync<GW>();
                            // a midpoint's rotor terms on one of its lanes
                            if (jl == 0)
                                for (int mc = gl >> lgG; mc < nmc; mc += GW >> lgG)
                                    acc += (double)rt[2 * (m0 + mc)] - (double)rt[2 * (m0 + mc) + 1];
                        }
                        // partial sums of up to 64 lanes of one midpoint (of the whole group when it
                        // has more midpoints than lanes), added in order by every lane
                        const int Gr = lgn > 3 ? (GW < 64 ? GW : 64) : (G < 64 ? G : 64);
                        acc = group_sum(acc, Gr);
                        double* pt = part + 8 * pb;
                        pb ^= 1;
                        if ((gl & (Gr - 1)) == 0) pt[gl / Gr] = acc;
                        group_sync<GW>();
                        // sum over all points up to a level; level acceptance of mc_piqmc.cc:263-273
                        const int per_m = G / Gr > 0 ? G / Gr : 1, np_all = GW / Gr;
                        for (int level = l0, i = 0; level < l1e; ++level) {
                            const double prev = cum;
                            const int i1 = l0 > 0 ? np_all : i + (per_m << level);
                            for (; i < i1; ++i) cum += pt[i];
                            const double deltav = (cum - 2.0 * prev) * (tau * (double)(1 << (L - level - 1)));
                            mids += any(alive) ? 1u << level : 0u;
                            alive = alive && (deltav < 0.0 || deltav < tst[level]);
                        }
                    }
                    l0 = l1e;
                }
                return alive;
            };
            bool accepted;
            if constexpr (MI) accepted = box ? level_sums(std::true_type{}) : level_sums(std::false_type{});
            else accepted = level_sums(std::false_type{});
            // the next move's midpoints and level tests; its loads are waited for here, before an
            // accepted move's stores, which share the wait counter
            if (ia + 1 < rp.tnumb[ty] && gl < nm) put(gl, nxt, (ia + 1) & 1);
            if (accepted) {  // the new midpoints into the window and, in FP64, to HBM
                acc_n += 1;
                for (int i = gl; i < nm; i += GW) {
                    const double4 v = i == gl ? cur : proposal(i);
                    R* d = win + (i * N + a) * 3;
                    d[0] = (R)v.x;
                    d[1] = (R)v.y;
                    d[2] = (R)v.z;
                    beads[ib + (s0 + 1 + i < P ? s0 + 1 + i : s0 + 1 + i - P)] = make_double4(v.x, v.y, v.z, 0.0);
                }
            }
            ib += P;
            if (ia + 1 < rp.tnumb[ty])
                for (int i = gl + GW; i < nm; i += GW) put(i, proposal(i), (ia + 1) & 1);
            cur = nxt;
            group_sync<GW>();
        }
        if (gl == 0) {
            atomicAdd(&mut[wk.x].total[ty][1], (unsigned long long)rp.tnumb[ty]);
            atomicAdd(&mut[wk.x].accep[ty][1], (unsigned long long)acc_n);
        }
    }
    if (gl == 0) atomicAdd(&mut[wk.x].pair_evals[0], 2ull * mids * (unsigned)(N - 1));
}

// Non-linear rotors: one workgroup per segment, its window of all atoms' beads and of the rotors'
// frames in LDS.  A move's first three levels are one pass over (midpoint, partner) with one
// reduction, later levels one each: with few segments the barriers, reductions and idle lanes of a
// pass per level were the time.  Partners that are rotors go to the last lanes, so that one wave and
// not all of them takes the 3D table's path.  33 atoms on 32 segments: 163 us a launch with a pass
// per level, now 128; two rotors on 32768 segments 214 us, now 139.
// The window of all atoms' positions on the segment's S+1 slots is held in the pair precision
// (float4 in FP32 runs, double4 in FP64 runs); new positions come from prop, one atom ahead, and
// accepted ones go to HBM in FP64 at once.  blockDim a multiple of 64.  The rotors' frames at the
// window's slots: fr [nrot*(S+1)].
// MI: built for contexts that hold a replica under the minimum image (its pairs then take their
// nearest image); without it the kernels carry no trace of it
template <typename R, bool MI>
__global__ __launch_bounds__(256) void k_bisect_nl(const Rep* __restrict__ reps, Mut* __restrict__ mut,
                                                   double4* __restrict__ beads, const RotBead* __restrict__ rotb,
                                                   const Frame* __restrict__ frames, Tables T, Tables3 T3,
                                                   const double4* __restrict__ prop, const int2* __restrict__ work, Run run) {
    extern __shared__ DYNAMIC_LDS double smem[];
    __shared__ double red[2][4][3];  // a pass's level sums per wave, two buffers
    const int2 wk = work[blockIdx.x];
    const Rep& rp = reps[wk.x];
    const int tid = threadIdx.x, nth = blockDim.x;
    const int S = rp.S, P = rp.P, N = rp.natoms;
    int s0;
    if (run.ref_order) {
        if (run.u >= P) return;
        s0 = run.u;
    } else {
        if (run.u >= S) return;
        s0 = run.u + wk.y * S;
    }
    const int W = S + 1;
    using P4 = vec4_t<R>;
    // LDS: the level tests of this move and the next, then in the pair precision the window of all
    // atoms' positions (x, y, z, -) and the mover's new midpoints, then the rotor frames and the 1D
    // spline knots
    double* th = smem;
    P4* win = reinterpret_cast<P4*>(smem + 16);
    P4* nwf = win + N * W;
    Frame* fr = reinterpret_cast<Frame*>(nwf + W);
    const int nfr = rp.nrot * W;
    P4* kn = reinterpret_cast<P4*>(fr + nfr);
    const Lut1D<R> l1 = lut1d<R>(T, rp.pot1d_id);
    const Lut3D<R> l3 = lut3d<R>(T3, rp.pot3d_id);
    const double* box = MI && rp.minimage ? rp.box : nullptr;  // MINIMAGE
    for (int i = tid; i < l1.n; i += nth) kn[i] = l1.k[i];
    for (int i = tid; i < nfr; i += nth) {
        const int q = i / W, w = i - q * W;
        fr[i] = frame_at(frames, rp, rp.nl_atom + q, (s0 + w) % P);
    }
    for (int i = tid; i < N * W; i += nth) {
        const int a = i / W, w = i - a * W;
        const double4 b = bead(beads, rp, a, (s0 + w) % P);
        P4 q;
        q.x = (R)b.x;
        q.y = (R)b.y;
        q.z = (R)b.z;
        q.w = (R)0;
        win[i] = q;
    }
    __syncthreads();

    unsigned mids = 0;  // midpoints whose terms a move's tests needed: of the levels up to its rejection
    int pb = 0;  // buffer of the next level sums
    unsigned long long tot[MAXT] = {0, 0, 0, 0}, acc_n[MAXT] = {0, 0, 0, 0};
    const int tend = run.type_end < rp.ntypes ? run.type_end : rp.ntypes;

    for (int ty = run.type_begin; ty < tend; ++ty) {
        const int L = rp.tlev[ty];
        const int St = 1 << L;
        const int nm = St - 1;
        // slot tid + 1 of the mover on lane tid: its proposal in registers from one move ahead until
        // it is accepted
        long long ib = rp.bead_off + (long long)rp.tbegin[ty] * P;
        auto put = [&](int i, const double4& v, int buf) {
            P4 q;
            q.x = (R)v.x;
            q.y = (R)v.y;
            q.z = (R)v.z;
            q.w = (R)0;
            nwf[i + 1] = q;
            if (i < L) th[8 * buf + i] = v.w;
        };
        auto proposal = [&](int i) { return prop[ib + (s0 + 1 + i) % P]; };
        double4 cur = make_double4(0.0, 0.0, 0.0, 0.0);
        if (tid < nm) cur = proposal(tid);
        for (int i = tid; i < nm; i += nth) put(i, i == tid ? cur : proposal(i), 0);
        lds_barrier();
        for (int ia = 0; ia < rp.tnumb[ty]; ++ia) {
            const int a = rp.tbegin[ty] + ia;
            const double* tst = th + 8 * (ia & 1);  // this move's level tests
            double4 nxt = cur;
            if (tid < nm && ia + 1 < rp.tnumb[ty]) nxt = prop[ib + P + (s0 + 1 + tid) % P];
            double cum = 0.0;
            bool accepted = false;
            const bool rot_a = a >= rp.nl_atom;
            const int na = rp.nl_atom - (rot_a ? 0 : 1), nr = rp.nrot - (rot_a ? 1 : 0);  // partners by kind
            for (int level = 0; level < L;) {
                const int end = level == 0 ? min(3, L) : level + 1;  // levels of this pass
                const int m0 = (1 << level) - 1, nmid = (1 << end) - 1 - m0;
                double acc[3] = {0.0, 0.0, 0.0};
                // Delta V at new midpoint m (level-major order) with partner j
                auto item = [&](int m, int j, auto rj_c, const double* bx) {
                    constexpr bool rj = decltype(rj_c)::value;
                    const int lv = 31 - __clz(m + 1), half = 1 << (L - lv - 1);
                    const int slot = half + ((m + 1 - (1 << lv)) << (L - lv));
                    const P4 pj = win[j * W + slot], pa = win[a * W + slot], pn = nwf[slot];
                    const Frame& fa = fr[(rot_a ? a - rp.nl_atom : 0) * W + slot];
                    const Frame& fj = fr[(rj ? j - rp.nl_atom : 0) * W + slot];
                    const double v = pair_nl<R>(l1, kn, l3, rot_a, rj, pn.x, pn.y, pn.z, pj.x, pj.y, pj.z, fa, fj, bx) -
                                     pair_nl<R>(l1, kn, l3, rot_a, rj, pa.x, pa.y, pa.z, pj.x, pj.y, pj.z, fa, fj, bx);
                    acc[0] += lv == level ? v : 0.0;
                    acc[1] += lv == level + 1 ? v : 0.0;
                    acc[2] += lv == level + 2 ? v : 0.0;
                };
                auto items = [&](auto mi_c) {
                    // the minimum image as its own instance of the loop, so the plain one is unchanged
                    const double* bx = decltype(mi_c)::value ? box : nullptr;
                    // item (m, jp) of the atoms: a lane's items advance by nth, so it is carried along
                    // with one division per pass
                    const int dd = na > 0 ? na : 1;
                    const int dq = nth / dd, dj = nth - dq * dd;
                    int q = tid / dd, jp = tid - q * dd;
                    for (int i = tid; i < nmid * na; i += nth) {
                        item(m0 + q, jp + (!rot_a && jp >= a), std::integral_constant<bool, false>{}, bx);
                        jp += dj;
                        q += dq;
                        if (jp >= dd) {
                            jp -= dd;
                            ++q;
                        }
                    }
                    for (int i = nth - 1 - tid; i < nmid * nr; i += nth) {
                        const int m = i / nr, p = i - m * nr;
                        item(m0 + m, rp.nl_atom + p + (rot_a && p >= a - rp.nl_atom), std::integral_constant<bool, true>{}, bx);
                    }
                };
                if constexpr (MI) {
                    if (box) items(std::integral_constant<bool, true>{});
                    else items(std::integral_constant<bool, false>{});
                } else {
                    items(std::integral_constant<bool, false>{});
                }
                const int nlev = end - level, nw = nth >> 6;
                acc[0] = wave_sum(acc[0]);
                if (nlev > 1) {  // together, so that their steps interleave
                    acc[1] = wave_sum(acc[1]);
                    acc[2] = wave_sum(acc[2]);
                }
                if ((tid & 63) == 0)
#pragma unroll
                    for (int k = 0; k < 3; ++k) red[pb][tid >> 6][k] = acc[k];
                lds_barrier();
                double sum[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) {  // at most four waves
                    sum[k] = red[pb][0][k];
#pragma unroll
                    for (int i = 1; i < 4; ++i) sum[k] += i < nw ? red[pb][i][k] : 0.0;
                }
                // sum over all points up to each level; level acceptance of mc_piqmc.cc:263-273
                accepted = true;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    if (k >= nlev) continue;
                    const double prev = cum;
                    cum += sum[k];
                    const double deltav = (cum - 2.0 * prev) * (rp.tau * (double)(1 << (L - (level + k) - 1)));
                    mids += accepted ? 1u << (level + k) : 0u;
                    accepted = accepted && (deltav < 0.0 || deltav < tst[level + k]);
                }
                level = end;
                pb ^= 1;
                if (!accepted) break;
            }
            tot[ty] += 1;
            // the next move's midpoints and level tests; its loads are waited for here, before an
            // accepted move's stores, which share the wait counter
            if (ia + 1 < rp.tnumb[ty] && tid < nm) put(tid, nxt, (ia + 1) & 1);
            if (accepted) {  // the new midpoints into the window and, in FP64, to HBM
                acc_n[ty] += 1;
                for (int i = tid; i < nm; i += nth) {
                    const int slot = 1 + i;
                    const double4 v = i == tid ? cur : proposal(i);
                    P4 q;
                    q.x = (R)v.x;
                    q.y = (R)v.y;
                    q.z = (R)v.z;
                    q.w = (R)0;
                    win[a * W + slot] = q;
                    beads[ib + (s0 + slot) % P] = make_double4(v.x, v.y, v.z, 0.0);
                }
            }
            ib += P;
            if (ia + 1 < rp.tnumb[ty])
                for (int i = tid + nth; i < nm; i += nth) put(i, proposal(i), (ia + 1) & 1);
            cur = nxt;
            lds_barrier();
        }
    }
    if (tid == 0) {
        for (int ty = run.type_begin; ty < tend; ++ty) {
            atomicAdd(&mut[wk.x].total[ty][1], tot[ty]);
            atomicAdd(&mut[wk.x].accep[ty][1], acc_n[ty]);
        }
        atomicAdd(&mut[wk.x].pair_evals[0], 2ull * mids * (unsigned)(N - 1));
    }
}

// ------------------------------------------------------------------------- linear rotor
// The rotor chain of a replica is split into parts of contiguous slices [k0, k1) (even
// length), one workgroup each.  A part builds the rotor-partner geometry of its translational
// slices in LDS once per launch and keeps it for every sweep of the launch (translations do
// not move during rotor sweeps).  Between half-sweeps a part needs one orientation from each
// neighbour: slice k0-1 (odd, moved by the part before) before its even half and slice k1
// (even, moved by the part after) before its odd half.  Each part publishes the boundary slice
// it just moved to rotb and then raises its flag (count of half-sweeps done); the reader spins
// on the flag with a bounded count, so every wave exits.  Boundary values and flags are
// written and read only with device-coherent atomics, and the writer waits for its value
// stores to complete before it stores the flag: the exchange needs no cache write-back or
// invalidation, which on a multi-XCD part would flush the L2 holding everyone's tables.
// Results do not depend on the split: draws are counter-based per (sweep, slice).
// (RotPart: pimc_plan.hpp)

// Polls of a numbered word before a wait gives up and sets the part's error bit (each poll
// sleeps between loads, so this bounds a wait at seconds, far beyond any normal exchange)
constexpr unsigned ROT_SPIN_LIMIT = 1u << 22;

// ------------------------------------------------------------------------- centroid, split
// MCMolecularMove (mc_piqmc.cc:54-102) with a replica's slices split over W workgroups
// (parts [k0, k1) of 0..P-1, RotPart reused): atoms in turn, each part sums Delta V over its
// slices and all partners and publishes the partial as two 64-bit words that carry the atom's
// number (base + ia + 1) above 32 bits of the double; lanes 0..2W-1 poll every part's words
// (bounded spin), and every part then adds the W partials in part order -- the same sum, so the
// same decision -- and moves its own slices of the atom.  Partner positions at a part's slices
// change only inside that part, so no bead data crosses parts.  Partials are double-buffered by
// atom parity: a part can overwrite a buffer only after every part has published the following
// atom, that is after every part has read it.
// Staged: the part's beads are in LDS, FP64, where all parts are small (single and few chains): the
// atoms' chain of sums, exchange and test is then the time, and neither reads nor the stores of an
// accepted move are waited for in it.  The parts' partials are added across a wave's lanes and the
// next atom's draws are formed while they travel.  With one lane adding them, beads in memory and
// barriers that wait for it, a launch over 64 atoms on 64 parts took 495 us, now 345; over 64 atoms
// of 16 boxes on 8 parts each 269, now 223.
template <typename R, int FAM, bool MI, bool Staged>
__global__ __launch_bounds__(256) void k_centroid_parts(const Rep* __restrict__ reps, Mut* __restrict__ mut,
                                                        double4* __restrict__ beads, const RotBead* __restrict__ rotb,
                                                        const Frame* __restrict__ frames, Tables T, Tables3 T3,
                                                        const RotPart* __restrict__ parts, unsigned* __restrict__ flags,
                                                        unsigned long long* __restrict__ slots, int nslots, Run run) {
    extern __shared__ DYNAMIC_LDS double smem[];  // the 1D spline knots, then the beads [3][slice][atom]
    constexpr int NBUF = Staged ? 2 : 1;  // buffers for alternate atoms; unstaged, every atom ends at a barrier
    __shared__ double red[NBUF][4];
    __shared__ double part_sum[NBUF][64];
    __shared__ double s_dv;
    __shared__ int s_err;
    const RotPart pt = parts[blockIdx.x];
    if (pt.r < 0) return;  // padding of the XCD-ordered grid
    const int r = pt.r;
    const Rep& rp = reps[r];
    const int ty = run.type_begin;
    if (ty >= rp.ntypes) return;
    const uint32_t pass = mut[r].pass;
    const int N = rp.natoms, P = rp.P, np = N - 1;
    const int t0 = pt.k0, nt = pt.k1 - pt.k0, W = pt.W;
    const Lut1D<R> l1 = lut1d<R>(T, rp.pot1d_id);
    const Lut2D<R> l2 = lut2d<R>(T, rp.pot2d_id);
    vec4_t<R>* kn = reinterpret_cast<vec4_t<R>*>(smem);
    for (int i = threadIdx.x; i < l1.n; i += blockDim.x) kn[i] = l1.k[i];
    const int nb = nt * N;
    double* lx = reinterpret_cast<double*>(kn + l1.n);
    double* ly = lx + nb;
    double* lz = ly + nb;
    if constexpr (Staged)
        for (int i = threadIdx.x; i < nb; i += blockDim.x) {
            const int j = i / nt, q = i - j * nt;  // a lane's neighbours read neighbouring slices
            const double4 b = bead(beads, rp, j, t0 + q);
            lx[q * N + j] = b.x;
            ly[q * N + j] = b.y;
            lz[q * N + j] = b.z;
        }
    __syncthreads();
    unsigned* myflag = flags + pt.fbase + pt.w;
    const unsigned base = __hip_atomic_load(myflag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const double* box = MI && rp.minimage ? rp.box : nullptr;  // MINIMAGE (not with a rotating linear rotor)
    if (threadIdx.x == 0) s_err = 0;
    unsigned long long acc_n = 0;
    const int lane = threadIdx.x & 63;
    uint4 w0, w1;
    auto draws = [&](int a) {
        w0 = draw(run.seed, rp.key, pass, K_CENTROID, 0, (uint32_t)a, 0, 0);
        w1 = draw(run.seed, rp.key, pass, K_CENTROID, 0, (uint32_t)a, 0, 1);
    };
    if constexpr (Staged) draws(rp.tbegin[ty]);
    for (int ia = 0; ia < rp.tnumb[ty]; ++ia) {
        const int a = rp.tbegin[ty] + ia, ib = ia & (NBUF - 1);
        if constexpr (!Staged) draws(a);  // ahead they cost registers, and a full device a resident part
        const double dx = rp.mcstep[ty] * (u53(w0.x, w0.y) - 0.5);
        const double dy = rp.mcstep[ty] * (u53(w0.z, w0.w) - 0.5);
        const double dz = rp.mcstep[ty] * (u53(w1.x, w1.y) - 0.5);
        const int items = nt * np;
        const bool rot_a = FAM == 1 ? (rp.nl_atom >= 0 && a >= rp.nl_atom) : (a == rp.lin_atom);
        // an atom with the linear rotor last among its partners: atom-atom and rotor terms in
        // separate loops (no wave runs both tables' code)
        const bool split = FAM == 0 && !rot_a && rp.lin_atom == N - 1;
        // the minimum image as its own instance of the loops, so the plain one is unchanged
        auto items_sum = [&](auto mi_c) -> double {
            const double* bx = decltype(mi_c)::value ? box : nullptr;
            auto at = [&](int j, int it) -> double4 {
                if constexpr (Staged) {
                    const int i = (it - t0) * N + j;
                    return make_double4(lx[i], ly[i], lz[i], 0.0);
                } else {
                    return bead(beads, rp, j, it);
                }
            };
            double acc = 0.0;
            if (split) {  // items: nt*(np-1) atom-atom terms first, then the nt rotor terms
                const int np1 = np - 1, n1 = nt * np1;
                // item i = (slice t0 + q, partner index jp); a lane's items advance by blockDim,
                // so (q, jp) is carried along with one division per atom
                const int dd = np1 > 0 ? np1 : 1, nth = (int)blockDim.x;
                const int dq = nth / dd, dj = nth - dq * dd;
                int qa = (int)threadIdx.x / dd, jpa = (int)threadIdx.x - qa * dd;
                for (int i = threadIdx.x; i < items; i += blockDim.x) {
                    const bool rj = i >= n1;
                    const int it = t0 + (rj ? i - n1 : qa), jp = rj ? 0 : jpa;
                    const int j = rj ? N - 1 : jp + (jp >= a);
                    jpa += dj;
                    qa += dq;
                    if (jpa >= dd) {
                        jpa -= dd;
                        ++qa;
                    }
                    const double4 xa = at(a, it), xj = at(j, it);
                    double nx = 0.0, ny = 0.0, nz = 1.0;
                    if (rj) rotor_axis(rotb, rp, it, nx, ny, nz);
                    R vn, vo;
                    if (rj) {
                        vn = pair_v<R>(l1, kn, l2, false, true, xa.x + dx, xa.y + dy, xa.z + dz, xj.x, xj.y, xj.z, nx, ny, nz,
                                       bx);
                        vo = pair_v<R>(l1, kn, l2, false, true, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, nx, ny, nz, bx);
                    } else {
                        vn = pair_v<R>(l1, kn, l2, false, false, xa.x + dx, xa.y + dy, xa.z + dz, xj.x, xj.y, xj.z, 0.0,
                                       0.0, 1.0, bx);
                        vo = pair_v<R>(l1, kn, l2, false, false, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, 0.0, 0.0, 1.0, bx);
                    }
                    acc += (double)vn - (double)vo;
                }
            }
            for (int i = split ? items : (int)threadIdx.x; i < items; i += blockDim.x) {
                const int it = t0 + i / np, jp = i % np;
                const int j = jp + (jp >= a);
                const bool rot_j = FAM == 1 ? (rp.nl_atom >= 0 && j >= rp.nl_atom) : (j == rp.lin_atom);
                const double4 xa = at(a, it), xj = at(j, it);
                if constexpr (FAM == 1) {
                    const Lut3D<R> l3 = lut3d<R>(T3, rp.pot3d_id);
                    const Frame& fa = frame_at(frames, rp, rot_a ? a : rp.nl_atom, it);
                    const Frame& fj = frame_at(frames, rp, rot_j ? j : rp.nl_atom, it);
                    const double vn = pair_nl<R>(l1, kn, l3, rot_a, rot_j, xa.x + dx, xa.y + dy, xa.z + dz, xj.x, xj.y,
                                                 xj.z, fa, fj, bx);
                    const double vo = pair_nl<R>(l1, kn, l3, rot_a, rot_j, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, fa, fj, bx);
                    acc += vn - vo;
                } else {
                    double nx, ny, nz;
                    rotor_axis(rotb, rp, it, nx, ny, nz);
                    const R vn = pair_v<R>(l1, kn, l2, rot_a, rot_j, xa.x + dx, xa.y + dy, xa.z + dz, xj.x, xj.y, xj.z,
                                           nx, ny, nz, bx);
                    const R vo = pair_v<R>(l1, kn, l2, rot_a, rot_j, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, nx, ny, nz, bx);
                    acc += (double)vn - (double)vo;
                }
            }
            return acc;
        };
        double acc;
        if constexpr (MI)
            acc = box ? items_sum(std::integral_constant<bool, true>{}) : items_sum(std::integral_constant<bool, false>{});
        else
            acc = items_sum(std::integral_constant<bool, false>{});
        double partial;
        if constexpr (Staged) {
            acc = wave_sum(acc);
            if (lane == 0) red[ib][threadIdx.x >> 6] = acc;
            lds_barrier();
            partial = ((red[ib][0] + red[ib][1]) + red[ib][2]) + red[ib][3];
        } else {
            partial = block_sum(acc, red[0]);
        }
        const double u = u53(w1.z, w1.w);
        double deltav = partial;
        unsigned long long* buf = slots + ((size_t)(ia & 1) * nslots + pt.fbase) * 2;
        if (W > 1) {
            const unsigned tag = base + (unsigned)ia + 1u;
            if (threadIdx.x < 2) {
                const unsigned long long bits = (unsigned long long)__double_as_longlong(partial);
                __hip_atomic_store(buf + 2 * pt.w + threadIdx.x,
                                   ((unsigned long long)tag << 32) | (threadIdx.x ? bits >> 32 : bits & 0xffffffffull),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if constexpr (Staged)
                if (ia + 1 < rp.tnumb[ty]) draws(a + 1);
            if (threadIdx.x < 2 * W) {  // word 2q + 1 is the high half of part q's partial
                unsigned long long wv;
                unsigned spins = 0;
                for (;;) {
                    wv = __hip_atomic_load(buf + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if ((unsigned)(wv >> 32) == tag) break;
                    if (++spins > ROT_SPIN_LIMIT) {
                        s_err = 8;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(2);
                }
                reinterpret_cast<unsigned*>(part_sum[ib])[threadIdx.x] = (unsigned)wv;
            }
            if constexpr (Staged) lds_barrier();
            else __syncthreads();
            if (s_err) break;  // a part did not arrive: the later atoms' waits would fail as well
            if constexpr (Staged) {
                deltav = wave_sum(lane < W ? part_sum[ib][lane] : 0.0);
            } else {  // on every wave of a full device it costs more than one lane's turn
                if (threadIdx.x == 0) {
                    double sum = 0.0;
                    for (int q = 0; q < W; ++q) sum += part_sum[ib][q];
                    s_dv = sum;
                }
                __syncthreads();
                deltav = s_dv;
            }
        } else if constexpr (Staged) {
            if (ia + 1 < rp.tnumb[ty]) draws(a + 1);
        }
        bool accepted = false;
        if (deltav < 0.0) accepted = true;
        else if (exp(-deltav * rp.tau) > u) accepted = true;
        if (accepted) {
            acc_n += 1;
            for (int it = t0 + (int)threadIdx.x; it < t0 + nt; it += blockDim.x) {
                const long long idx = rp.bead_off + (long long)a * P + it;
                double4 b;
                if constexpr (Staged) {
                    const int i = (it - t0) * N + a;
                    b = make_double4(lx[i] + dx, ly[i] + dy, lz[i] + dz, 0.0);
                    lx[i] = b.x;
                    ly[i] = b.y;
                    lz[i] = b.z;
                } else {
                    b = beads[idx];
                    b = make_double4(b.x + dx, b.y + dy, b.z + dz, 0.0);
                }
                beads[idx] = b;
            }
        }
        if constexpr (Staged) lds_barrier();
        else __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (W > 1)  // every part of the replica ran the same atoms
            __hip_atomic_store(myflag, base + (unsigned)rp.tnumb[ty], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (s_err) atomicOr(&mut[r].err, s_err);
        if (pt.w == 0) {
            atomicAdd(&mut[r].total[ty][0], (unsigned long long)rp.tnumb[ty]);
            atomicAdd(&mut[r].accep[ty][0], acc_n);
        }
        atomicAdd(&mut[r].pair_evals[1], 2ull * (unsigned long long)rp.tnumb[ty] * nt * np);
    }
}

// Sum over items i0, i0 + step, ... < items of a slice of V(r, cos theta) with the rotor axis n:
// cos = -(n . dr)/r (PotRotEnergy mc_piqmc.cc:1967-2044), from the slice's geometry block g.  UT
// (FP32 on a uniform table): g holds unit vectors and distances; the cells of a batch first, then
// all its loads, then the lerps, so that the table look-ups of a lane fly together.
template <typename R, bool UT, int B>
__device__ __forceinline__ void pair_batch(const Lut2D<R>& l2, const vec4_t<R>* g, int i0, int step, int items, R fx, R fy,
                                           R fz, double& acc) {
    if constexpr (UT) {
        int cell[B];
        float wr[B], wc[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int i = i0 + b * step;
            const float4 d = g[i < items ? i : i0];
            const float c = -__builtin_fmaf(d.z, fz, __builtin_fmaf(d.y, fy, rounded_product(d.x, fx)));
            lpot2d_u_cell(l2, d.w, c, cell[b], wr[b], wc[b]);
        }
        float4 q[B];
#pragma unroll
        for (int b = 0; b < B; ++b) q[b] = l2.vc[cell[b]];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const double v = (double)lpot2d_u_lerp(q[b].x, q[b].y, q[b].z, q[b].w, wr[b], wc[b]);
            acc += i0 + b * step < items ? v : 0.0;
        }
    } else {
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int i = i0 + b * step;
            const vec4_t<R> d = g[i < items ? i : i0];
            R c;
            if constexpr (is_fp32<R>()) c = -(fx * d.x + fy * d.y + fz * d.z);
            else c = -((fx * d.x + fy * d.y + fz * d.z) / d.w);
            const double v = (double)lpot2d<R>(l2, d.w, c);
            acc += i < items ? v : 0.0;
        }
    }
}

template <typename R, bool UT>
__device__ __forceinline__ double pair_terms(const Lut2D<R>& l2, const vec4_t<R>* g, int i0, int step, int items, double nx,
                                             double ny, double nz) {
    double acc = 0.0;
    const R fx = (R)nx, fy = (R)ny, fz = (R)nz;
    constexpr int B = UT ? 8 : 2;
    int i = i0;
    for (; i + (B / 2) * step < items; i += B * step) pair_batch<R, UT, B>(l2, g, i, step, items, fx, fy, fz, acc);
    if (i < items) pair_batch<R, UT, B / 2>(l2, g, i, step, items, fx, fy, fz, acc);
    return acc;
}

// One part of a linear rotor's chain: all sweeps of a launch.  The block's waves split the work: the
// first one or two hold the chain of dependent steps, a lane per pair of slices (kl, kl + 1) -- link
// densities, the test, the next proposal --; the others sum the partner energies of the proposals.
// A proposal and its energy depend on the slice's own orientation alone, not on its neighbours, so
// both are formed half a sweep ahead: while the chain waves test parity p, the energy waves work on
// the proposals of parity 1 - p, which the chain waves made in the half before.  A half costs the
// longer of the two instead of their sum, and what a move needs once runs on one lane instead of on
// every lane of its group.
// With every wave doing all of it in turn a half of a 512-slice chain took 5.0 us, now 1.8: bound by
// the exchange with the neighbouring part (a store and a load at agent scope) on chains in several
// parts, by the chain waves' FP64 steps on one part (8 atoms: 4.3 us, now 1.9), and on a full device
// by how many parts are resident (two per CU for their registers; 168 registers spill and cost more
// than the third part gives).  Sweep per pass, 256 replicas: 9.3 -> 4.8 ms.
// LDS (local index kl = k - k0 + 1; kl = 0 and ns+1 are the neighbours' boundary slices): nv[3], Lk
// and the proposals' axes np[3] over ns+2 entries (double), then the geometry block
// geo[(it - k0*RR) * np + jp] (vec4).  Lk[kl] is the density factor rho(n_kl . n_kl+1) of the link
// kl -> kl+1 and a lane's E its slices' partner energy: the "old" values of a move are the "new"
// values of the last accepted move that changed them (for a link to a neighbour part, the value that
// part published with its slice).
constexpr int ROTOR_PARTIALS = 192;       // partial energies of a half: at most one per energy lane
constexpr int ROTOR_KNOTS = 192;          // density knots staged in LDS
constexpr int ROTOR_SLICES_MAX = 256;     // slices of a part where a chain lane holds two
// Longer parts (chains of tens of thousands of slices with hardly any partners) take MPL pairs of
// slices per chain lane: 2 * 128 * 12 slices are more than LDS holds.
constexpr int ROTOR_MPL_LONG = 12;

// Lean: LDS for the part alone, for long parts and for those that leave no room for the partial sums
// and the staged knots (two slices of 1240 partners and more, FP64, two time slices each).  A move's
// energy lanes are then a power of two within a wave, and its sum takes the place of its proposal's
// axis; the knots are staged behind the part (at double knots_at of smem) where the launch has
// room, else read from L2 (knots_at < 0).
template <typename R, bool UT, int MPL, bool Lean>
__global__ __launch_bounds__(256) void k_rotor(const Rep* __restrict__ reps, Mut* __restrict__ mut,
                                               const double4* __restrict__ beads, RotBead* __restrict__ rotb,
                                               Tables T, const RotPart* __restrict__ parts,
                                               unsigned* __restrict__ flags, unsigned long long* __restrict__ xrec, Run run,
                                               int knots_at) {
    static_assert(Lean || MPL == 1, "long parts are lean");
    extern __shared__ DYNAMIC_LDS double smem[];
    __shared__ double pe[Lean ? 1 : 2][Lean ? 1 : ROTOR_PARTIALS];
    __shared__ double4 knots[Lean ? 1 : ROTOR_KNOTS];
    __shared__ unsigned s_acc[2];
    __shared__ int s_err;
    const RotPart pt = parts[blockIdx.x];
    if (pt.r < 0) return;  // padding of the XCD-ordered grid
    const int r = pt.r;
    const Rep& rp = reps[r];
    if (rp.rotkind != 1 || rp.rot_atom < 0) return;
    const int Prot = rp.Prot, RR = rp.RotRatio, P = rp.P, N = rp.natoms;
    int nsweep, j0, jstride;
    if (run.ref_order) {
        if (run.u >= P) return;
        nsweep = 1; j0 = run.u; jstride = 0;
    } else {
        if (run.u >= rp.S) return;
        nsweep = P / rp.S; j0 = run.u; jstride = rp.S;
    }
    const int k0 = pt.k0, ns = pt.k1 - pt.k0, W = pt.W;
    const int np = N - 1;
    const int items = RR * np;
    double* nv = smem;
    double* Lk = nv + 3 * (ns + 2);
    double* na = Lk + (ns + 2);  // axes of the proposals
    vec4_t<R>* geo = reinterpret_cast<vec4_t<R>*>(smem + ((7 * (ns + 2) + 3) & ~3));
    const int ar = rp.rot_atom;
    const long long rbase = rp.rot_off + (long long)(ar - rp.tbegin[rp.imtype]) * Prot;
    unsigned* myflag = flags + pt.fbase + pt.w;  // half-sweeps done by the launches before this one
    if (threadIdx.x == 0) s_err = 0;
    if (threadIdx.x < 2) s_acc[threadIdx.x] = 0;
    // axes of the own slices and of both neighbours' boundary slices; the first energies are those of
    // the current axes
    for (int kl = threadIdx.x; kl < ns + 2; kl += blockDim.x) {
        int k = k0 + kl - 1;
        if (k < 0) k += Prot;
        if (k >= Prot) k -= Prot;
        const RotBead b = rotb[rbase + k];
        nv[3 * kl] = na[3 * kl] = b.nx;
        nv[3 * kl + 1] = na[3 * kl + 1] = b.ny;
        nv[3 * kl + 2] = na[3 * kl + 2] = b.nz;
    }
    // rotor-partner geometry of the part's translational slices (beads of one atom are
    // contiguous in slices, so consecutive lanes take consecutive slices)
    const int nit = ns * RR, it0 = k0 * RR;
    for (int i = threadIdx.x; i < nit * np; i += blockDim.x) {
        const int jp = i / nit, itl = i - jp * nit;
        const int j = jp + (jp >= ar);
        double4 xa = bead(beads, rp, ar, it0 + itl), xj = bead(beads, rp, j, it0 + itl);
        R dx = (R)(xa.x - xj.x), dy = (R)(xa.y - xj.y), dz = (R)(xa.z - xj.z);
        R rr = sqrt(dx * dx + dy * dy + dz * dz);
        vec4_t<R> v;
        if constexpr (is_fp32<R>()) {  // unit vector: a move's cos(theta) is then one dot product
            R ir = (R)1 / rr;
            v.x = dx * ir; v.y = dy * ir; v.z = dz * ir;
        } else {
            v.x = dx; v.y = dy; v.z = dz;
        }
        v.w = rr;
        geo[itl * np + jp] = v;
    }
    const uint32_t pass = mut[r].pass;
    const Lut2D<R> l2 = lut2d<R>(T, rp.pot2d_id);
    const TabRot trt = T.tr[rp.rotdens];
    const double4* hk = T.rk + trt.off + trt.hot;
    if (!Lean || knots_at >= 0) {
        double4* to = Lean ? reinterpret_cast<double4*>(smem + knots_at) : knots;
        for (int i = threadIdx.x; i < trt.n - trt.hot; i += blockDim.x) to[i] = hk[i];
        hk = to;
    }
    const unsigned base = __hip_atomic_load(myflag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int nmoves = ns >> 1;                    // of either parity: k0 and ns are even
    const int nchain = nmoves <= 64 ? 64 : 128;    // lanes of the chain waves
    const bool chain = __builtin_amdgcn_readfirstlane((int)threadIdx.x) < nchain;  // a wave's role, scalar
    // energy lanes: lpm per move, of which each quad or row of 16 leaves one partial sum in pe
    const int nen = (int)blockDim.x - nchain;
    int lpm = Lean ? 1 : nen / nmoves;
    if constexpr (Lean)
        while (lpm < 64 && 2 * lpm * nmoves <= nen) lpm *= 2;
    const int gr = Lean ? lpm : (lpm >= 16 ? 16 : (lpm >= 4 ? 4 : 1));
    lpm -= lpm % gr;
    const int npart = lpm / gr;
    const int le = (int)threadIdx.x - nchain, emv = le / lpm, eli = le - emv * lpm;
    auto energies = [&](int parity) {  // of the proposals of one parity
        for (int m = emv; m < nmoves; m += Lean ? nen / lpm : nmoves) {
            const int kl = 2 * m + parity + 1;
            // without UT the tables of the launch's chains differ in kind: a chain's own decides
            auto terms = [&](auto u_c) {
                return pair_terms<R, decltype(u_c)::value>(l2, geo + (long long)(kl - 1) * items, eli, lpm, items, na[3 * kl],
                                                           na[3 * kl + 1], na[3 * kl + 2]);
            };
            double e;
            if constexpr (is_fp32<R>() && !UT) e = l2.uniform ? terms(std::true_type{}) : terms(std::false_type{});
            else e = terms(std::integral_constant<bool, UT>{});
            e = group_sum(e, gr);
            if constexpr (Lean) {
                if (eli == 0) na[3 * kl] = e;
            } else {
                if ((eli & (gr - 1)) == 0) pe[parity][m * npart + eli / gr] = e;
            }
        }
    };
    auto energy_of = [&](int parity, int mv) {  // sum of the partials of a move
        if constexpr (Lean) return na[3 * (2 * mv + parity + 1)];
        const double* p = &pe[parity][mv * npart];
        double e = p[0];
        if (npart <= 4) {  // read together: one after another they were 0.15 us of a half with three
            double v[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) v[i] = p[i + 1 < npart ? i + 1 : 0];
#pragma unroll
            for (int i = 0; i < 3; ++i) e += i + 1 < npart ? v[i] : 0.0;
        } else {
            for (int i = 1; i < npart; ++i) e += p[i];
        }
        return e;
    };
    __syncthreads();
    if (!chain) {
        energies(0);
        energies(1);
    }
    for (int kl = threadIdx.x; kl <= ns; kl += blockDim.x) {
        double p = nv[3 * kl] * nv[3 * kl + 3] + nv[3 * kl + 1] * nv[3 * kl + 4] + nv[3 * kl + 2] * nv[3 * kl + 5];
        Lk[kl] = rot_rho(T, trt, p);
    }
    __syncthreads();
    // a chain lane's two slices, kl = 2 mv + 1 (even half) and 2 mv + 2 (odd half): the state, and the
    // proposal in hand (its axis is in na)
    struct Slice {
        double phi, cth, E;      // now
        double ph, cost, u;      // proposed, and the test's uniform
        double nx, ny, nz;
    };
    Slice sl[MPL][2] = {};
    auto move_of = [&](int q) { return q * nchain + (int)threadIdx.x; };
    auto propose = [&](Slice& s, int mv, int parity, int sw) {
        const int kl = 2 * mv + parity + 1;
        const uint32_t jsweep = (uint32_t)(j0 + sw * jstride), k = (uint32_t)(k0 + kl - 1);
        const uint4 w0 = draw(run.seed, rp.key, pass, K_ROTLIN, jsweep, (uint32_t)ar, k, 0);
        const uint4 w1 = draw(run.seed, rp.key, pass, K_ROTLIN, jsweep, (uint32_t)ar, k, 1);
        double cost = s.cth + rp.rtstep * (u53(w0.x, w0.y) - 0.5);
        s.ph = s.phi + rp.rtstep * (u53(w0.z, w0.w) - 0.5);
        if (cost > 1.0) cost = 2.0 - cost;
        if (cost < -1.0) cost = -2.0 - cost;
        s.cost = cost;
        s.u = u53(w1.x, w1.y);
        const double sint = sqrt(1.0 - cost * cost);
        double sn, cs;
        sincos(s.ph, &sn, &cs);
        s.nx = sint * cs;
        s.ny = sint * sn;
        s.nz = cost;
        na[3 * kl] = s.nx;
        na[3 * kl + 1] = s.ny;
        na[3 * kl + 2] = s.nz;
    };
    if (chain)
        for (int q = 0; q < MPL; ++q) {
            const int mv = move_of(q);
            if (mv >= nmoves) break;
#pragma unroll
            for (int parity = 0; parity < 2; ++parity) {
                const RotBead b = rotb[rbase + k0 + 2 * mv + parity];
                sl[q][parity].phi = b.phi;
                sl[q][parity].cth = b.cth;
                sl[q][parity].E = energy_of(parity, mv);
            }
        }
    __syncthreads();  // the current axes' energies are read; na and pe are the proposals' from here on
    if (chain)
        for (int q = 0; q < MPL; ++q) {
            const int mv = move_of(q);
            if (mv >= nmoves) break;
            propose(sl[q][0], mv, 0, 0);
            propose(sl[q][1], mv, 1, 0);
        }
    __syncthreads();
    if (!chain) energies(0);
    __syncthreads();
    unsigned nacc = 0;
    int err = 0;
    // The neighbour's boundary slice that half h of the next parity reads: k0-1 before an even half
    // (published by the previous part after its odd half), k1 before an odd half (by the next part
    // after its even half): the orientation and the density of the shared link (the same product of
    // the same operands this part would form), as eight words that each carry the publishing half's
    // number (base + h) above 32 bits of a value.  Eight lanes poll the words themselves, so the data
    // comes with its check; the neighbour cannot publish that record again before this part's next
    // half.  A single part is its own neighbour: local slices 0 and ns are one slice, as are 1 and
    // ns + 1, and links 0 and ns one link, so the move that changes one copy writes the other.
    auto record = [&](int parity) {
        const int nb = parity == 0 ? (pt.w + W - 1) % W : (pt.w + 1) % W;
        return xrec + ((size_t)(pt.fbase + nb) * 2 + (parity == 0 ? 1 : 0)) * 8;
    };
    auto receive = [&](int parity, unsigned h, unsigned long long wv) {
        const int lane = threadIdx.x & 63;
        const unsigned long long* rec = record(parity);
        const unsigned want = base + h;
        const int klr = parity == 0 ? 0 : ns + 1;
        if (lane < 8) {
            unsigned spins = 0;
            while ((unsigned)(wv >> 32) != want) {
                if (++spins > ROT_SPIN_LIMIT) {
                    s_err = 2;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
                wv = __hip_atomic_load(rec + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            const int i = lane >> 1;  // doubles: the orientation, then the link density
            double* dst = i < 3 ? &nv[3 * klr + i] : &Lk[parity == 0 ? 0 : ns];
            reinterpret_cast<unsigned*>(dst)[lane & 1] = (unsigned)wv;
        }
    };
    // parity p of sweep sw on the chain waves: test, update, publish, the proposal of the next sweep,
    // and what the next half needs of the neighbour, which has published it about when this part did:
    // the record is asked for before the proposal and checked after it, while the energy waves work
    auto move = [&](auto p_c, int sw, int q) {
        constexpr int parity = decltype(p_c)::value;
        Slice& s = sl[q][parity];
        const int mv = move_of(q);
        const bool mine = mv < nmoves;
        const int kl = 2 * mv + parity + 1;
        const unsigned h = 2u * (unsigned)sw + (unsigned)parity;  // half-sweeps done before this one
        const int bnd_mv = parity == 0 ? 0 : nmoves - 1;  // the move at the slice that is published
        const int lane = threadIdx.x & 63;
        if (mine) {
            const double p0 = nv[3 * kl - 3] * s.nx + nv[3 * kl - 2] * s.ny + nv[3 * kl - 1] * s.nz;  // n_k-1 . n'
            const double p1 = s.nx * nv[3 * kl + 3] + s.ny * nv[3 * kl + 4] + s.nz * nv[3 * kl + 5];  // n' . n_k+1
            double rho0, rho1;
            rot_rho_hot(T, trt, hk, p0, p1, rho0, rho1);
            const double enew = energy_of(parity, mv);
            double dold = Lk[kl - 1] * Lk[kl];
            if (fabs(dold) < RZERO) dold = 0.0;
            double dnew = rho0 * rho1;
            if (fabs(dnew) < RZERO) dnew = 0.0;
            if (dold < 0.0 || dnew < 0.0) {
                err = 1;  // "Negative rot density" (mc_piqmc.cc:850,886): the move is not taken
            } else {
                // dnew / dold exp(-tau dV) > u (the reference's ratio counts as 1 where dold is zero)
                const double x = exp(-rp.tau * (enew - s.E));
                const bool accepted = dold > RZERO ? dnew * x > s.u * dold : x > s.u;
                if (accepted) {
                    ++nacc;
                    s.cth = s.cost;
                    s.phi = s.ph;
                    s.E = enew;
                    nv[3 * kl] = s.nx;
                    nv[3 * kl + 1] = s.ny;
                    nv[3 * kl + 2] = s.nz;
                    Lk[kl - 1] = rho0;
                    Lk[kl] = rho1;
                    if (W == 1 && (kl == 1 || kl == ns)) {  // the other copy of the slice and link
                        const int km = kl == 1 ? ns + 1 : 0;
                        nv[3 * km] = s.nx;
                        nv[3 * km + 1] = s.ny;
                        nv[3 * km + 2] = s.nz;
                        Lk[kl == 1 ? ns : 0] = kl == 1 ? rho0 : rho1;
                    }
                }
            }
        }
        // publish the boundary slice this half moved (k0 after the even half, k1-1 after the odd)
        const bool publisher = W > 1 && bnd_mv / nchain == q && (bnd_mv % nchain) >> 6 == (int)threadIdx.x >> 6;
        const bool more = !(parity == 1 && sw + 1 == nsweep);  // a half follows in this launch
        unsigned long long wv = 0;
        if (publisher) {
            wave_sync();
            if (lane < 8) {
                // orientation and the density of the link to the neighbour's adjacent slice (Lk[0]
                // after the even half, for the previous part; Lk[ns] after the odd half, for the
                // next), two words per double; no wait for the stores, the reader checks every
                // word's number
                const int kb = parity == 0 ? 1 : ns;
                const int i = lane >> 1;
                const double v = i < 3 ? nv[3 * kb + i] : Lk[parity == 0 ? 0 : ns];
                const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
                const unsigned word = (lane & 1) ? (unsigned)(bits >> 32) : (unsigned)bits;
                __hip_atomic_store(xrec + ((size_t)(pt.fbase + pt.w) * 2 + parity) * 8 + lane,
                                   ((unsigned long long)(base + h + 1u) << 32) | word, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                if (more) wv = __hip_atomic_load(record(1 - parity) + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (mine && sw + 1 < nsweep) propose(s, mv, parity, sw + 1);
        if (publisher && more) receive(1 - parity, h + 1u, wv);
    };
    auto half = [&](auto p_c, int sw) {
        for (int q = 0; q < MPL; ++q)
            if (MPL == 1 || q * nchain < nmoves) move(p_c, sw, q);
    };
    // the two roles in loops of their own, barrier for barrier, so that neither holds the other's
    // registers.  A wait that gave up: leave at once instead of waiting again at every later half
    // (every lane reads s_err after the barrier; it is written again only in the next half)
    if (chain) {
        for (int sw = 0; sw < nsweep; ++sw) {
            half(std::integral_constant<int, 0>{}, sw);
            lds_barrier();
            if (s_err) break;
            half(std::integral_constant<int, 1>{}, sw);
            lds_barrier();
            if (s_err) break;
        }
    } else {
        for (int sw = 0; sw < nsweep; ++sw) {
            energies(1);
            lds_barrier();
            if (s_err) break;
            if (sw + 1 < nsweep) energies(0);
            lds_barrier();
            if (s_err) break;
        }
    }
    if (W > 1 && threadIdx.x == 0)  // every part of the chain ran the same halves
        __hip_atomic_store(myflag, base + 2u * (unsigned)nsweep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (chain)
        for (int q = 0; q < MPL; ++q) {
            const int mv = move_of(q);
            if (mv >= nmoves) break;
#pragma unroll
            for (int parity = 0; parity < 2; ++parity) {
                const int kl = 2 * mv + parity + 1;
                RotBead& b = rotb[rbase + k0 + kl - 1];
                b.phi = sl[q][parity].phi;
                b.cth = sl[q][parity].cth;
                b.nx = nv[3 * kl];
                b.ny = nv[3 * kl + 1];
                b.nz = nv[3 * kl + 2];
            }
        }
    if (chain) {
        const unsigned s = wave_sum(nacc);
        if ((threadIdx.x & 63) == 0) s_acc[threadIdx.x >> 6] = s;
    }
    __syncthreads();
    if (err) atomicOr(&mut[r].err, 1);
    if (threadIdx.x == 0) {
        if (s_err) atomicOr(&mut[r].err, s_err);
        atomicAdd(&mut[r].total[rp.imtype][2], (unsigned long long)nsweep * ns);
        atomicAdd(&mut[r].accep[rp.imtype][2], (unsigned long long)(s_acc[0] + s_acc[1]));
        // the current axes once per launch, then every proposal
        atomicAdd(&mut[r].pair_evals[2], (unsigned long long)(nsweep + 1) * ns * items);
    }
}

// ------------------------------------------------------------------------- non-linear rotors
// The axis that MCRot3Dstep keeps of an accepted move (mc_piqmc.cc:938-1199): a frame's third column
// but for the last bit.  In fixed operations, so that every form of the sweep stores the same bits.
__device__ __forceinline__ void store_axis(RotBead& b, double phi, double cth) {
    const double sint = sqrt(fma(-cth, cth, 1.0));
    double sn, cs;
    sincos(phi, &sn, &cs);
    b.nx = sint * cs;
    b.ny = sint * sn;
    b.nz = cth;
}

// MCRotations3D (mc_piqmc.cc:692-779) with MCRot3Dstep (:938-1199): even slices, then odd;
// at each slice every rotor in turn.  One workgroup per replica and a group of G lanes per
// slice: the density factors rho(t0,t1), rho(t1,t2) (old) and rho(t0,t1'), rho(t1',t2) (new)
// on four lanes, the old and new sums of PotRotE3D (mc_piqmc.cc:2046-2151) over the slice's
// translational slices and partners across the group.  Old energy sums are recomputed for
// every move as the reference does: with two rotors a partner rotor may have moved since.  The
// old density factors are cached per link (Lk[q][k] = rho(slice k, slice k+1) of rotor q): they
// are the new factors of the last accepted move on that link, from the same frames, so a move
// evaluates only its two new links.  Orientations live in rotb and their frames in `frames`; a
// group keeps the frames of all rotors at its slice (and the proposal's) in LDS, so a rotor sees
// the moves of the rotors before it there.
// LDS: Lk [nrot*Prot] doubles, then the groups' frames [groups*(nrot+1)].
template <typename R, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_rotor3d(const Rep* __restrict__ reps, Mut* __restrict__ mut,
                                                 const double4* __restrict__ beads, RotBead* __restrict__ rotb,
                                                 Frame* __restrict__ frames, Tables T, Tables3 T3, const int* __restrict__ replist,
                                                 Run run) {
    extern __shared__ DYNAMIC_LDS double smem[];
    __shared__ unsigned long long red_acc[BLOCK / 64];  // one partial per wave
    __shared__ int s_err;
    const int r = replist[blockIdx.x];
    const Rep& rp = reps[r];
    if (rp.rotkind != 2 || rp.rot3d_id < 0) return;
    const int Prot = rp.Prot, RR = rp.RotRatio, P = rp.P, N = rp.natoms, nrot = rp.nrot;
    int nsweep, j0, jstride;
    if (run.ref_order) {
        if (run.u >= P) return;
        nsweep = 1; j0 = run.u; jstride = 0;
    } else {
        if (run.u >= rp.S) return;
        nsweep = P / rp.S; j0 = run.u; jstride = rp.S;
    }
    const int np = N - 1;
    const int items = RR * np;
    const long long rb0 = rp.rot_off;  // rotor q, slice k at rb0 + q*Prot + k
    const double4* tab = T3.r3 + (long long)rp.rot3d_id * 3 * ROT3D_SIZE;
    const Lut1D<R> l1 = lut1d<R>(T, rp.pot1d_id);
    const Lut3D<R> l3 = lut3d<R>(T3, rp.pot3d_id);
    const int maxmoves = (Prot + 1) / 2;
    int G = 1;
    while (G < 64 && G * 2 * maxmoves <= (int)blockDim.x) G *= 2;
    const int groups = blockDim.x / G;
    const int g = threadIdx.x / G, gl = threadIdx.x % G;
    double* Lk = smem;
    Frame* gf = reinterpret_cast<Frame*>(smem + ((nrot * Prot + 1) & ~1)) + (long long)g * (nrot + 1);
    const uint32_t pass = mut[r].pass;
    const int rtype = rp.imtype;
    const double twopi = 2.0 * PI_D;
    if (threadIdx.x == 0) s_err = 0;
    unsigned long long nacc = 0;
    int err = 0;
    for (int i = threadIdx.x; i < nrot * Prot; i += blockDim.x) {
        const int q = i / Prot, k = i - q * Prot;
        const long long b = rb0 + (long long)q * Prot;
        if (rotden_rho(frames[b + k], frames[b + (k + 1 == Prot ? 0 : k + 1)], tab, Lk[i])) err = 1;
    }
    __syncthreads();
    for (int sw = 0; sw < nsweep; ++sw) {
        const uint32_t jsweep = (uint32_t)(j0 + sw * jstride);
        for (int parity = 0; parity < 2; ++parity) {
            const int nmoves = (Prot - parity + 1) / 2;
            for (int mv = g; mv < nmoves; mv += groups) {
                const int k = 2 * mv + parity;
                int k0 = k - 1, k2 = k + 1;
                if (k0 < 0) k0 += Prot;
                if (k2 >= Prot) k2 -= Prot;
                for (int q = gl; q < nrot; q += G) gf[q] = frames[rb0 + (long long)q * Prot + k];
                __builtin_amdgcn_wave_barrier();
                for (int q = 0; q < nrot; ++q) {
                    const int gatom = rp.nl_atom + q;
                    const long long ik = rb0 + (long long)q * Prot + k;
                    const RotBead cur = rotb[ik];
                    const uint4 w0 = draw(run.seed, rp.key, pass, K_ROT3D, jsweep, (uint32_t)gatom, (uint32_t)k, 0);
                    const uint4 w1 = draw(run.seed, rp.key, pass, K_ROT3D, jsweep, (uint32_t)gatom, (uint32_t)k, 1);
                    const double rand1 = u53(w0.x, w0.y), rand2 = u53(w0.z, w0.w);
                    const double rand3 = u53(w1.x, w1.y), rand4 = u53(w1.z, w1.w);
                    double cost = cur.cth + rp.rtstep * (rand1 - 0.5);
                    double phi = cur.phi + twopi * (rp.rtstep * (rand2 - 0.5));
                    double chi = cur.chi + twopi * (rp.rtstep * (rand3 - 0.5));
                    if (phi < 0.0) phi = twopi + phi;
                    if (chi < 0.0) chi = twopi + chi;
                    phi = fmod_near(phi, twopi);
                    chi = fmod_near(chi, twopi);
                    if (cost > 1.0) cost = 2.0 - cost;
                    if (cost < -1.0) cost = -2.0 - cost;
                    if (gl == 0) gf[nrot] = make_frame(phi, cost, chi);
                    __builtin_amdgcn_wave_barrier();
                    // density factors: old (t0,t1) and (t1,t2) from the link cache, new (t0,t1')
                    // and (t1',t2) on lanes 0 and 1
                    double d[4] = {Lk[q * Prot + k0], Lk[q * Prot + k], 0.0, 0.0};
                    for (int c = 2 + gl; c < 4; c += G) {
                        const Frame& fa = (c == 3) ? gf[nrot] : frames[rb0 + (long long)q * Prot + k0];
                        const Frame& fb = (c == 2) ? gf[nrot] : frames[rb0 + (long long)q * Prot + k2];
                        if (rotden_rho(fa, fb, tab, d[c])) err = 1;
                    }
                    if (G > 1)
                        for (int c = 2; c < 4; ++c) d[c] = __shfl(d[c], (c - 2) % G, G);
                    // PotRotE3D at the old and the proposed orientation
                    double eo = 0.0, en = 0.0;
                    for (int i = gl; i < items; i += G) {
                        const int it = k * RR + i / np, jp = i % np;
                        const int j = jp + (jp >= gatom);
                        const bool rj = j >= rp.nl_atom;
                        const double4 xa = bead(beads, rp, gatom, it), xj = bead(beads, rp, j, it);
                        const Frame& fj = gf[rj ? j - rp.nl_atom : q];
                        eo += pair_nl<R>(l1, l1.k, l3, true, rj, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, gf[q], fj);
                        en += pair_nl<R>(l1, l1.k, l3, true, rj, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, gf[nrot], fj);
                    }
                    for (int o = G >> 1; o > 0; o >>= 1) {  // the two sums' shuffles interleave
                        eo += __shfl_xor(eo, o, G);
                        en += __shfl_xor(en, o, G);
                    }
                    double dold = d[0] * d[1];
                    if (fabs(dold) < RZERO) dold = 0.0;
                    if (dold < 0.0) dold = fabs(dold);
                    double dnew = d[2] * d[3];
                    if (fabs(dnew) < RZERO) dnew = 0.0;
                    if (dnew < 0.0) dnew = fabs(dnew);
                    double rd = (dold > RZERO) ? dnew / dold : 1.0;
                    rd *= exp(-rp.tau * (en - eo));
                    const bool accepted = rd > 1.0 || rd > rand4;
                    if (accepted && gl == 0) {
                        ++nacc;
                        RotBead b = cur;
                        b.cth = cost;
                        b.phi = phi;
                        b.chi = chi;
                        store_axis(b, phi, cost);
                        rotb[ik] = b;
                        frames[ik] = gf[nrot];
                        gf[q] = gf[nrot];
                        Lk[q * Prot + k0] = d[2];
                        Lk[q * Prot + k] = d[3];
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
            __syncthreads();
        }
    }
    if (err) s_err = 1;
    unsigned long long s = block_sum(nacc, red_acc);
    if (threadIdx.x == 0) {
        if (s_err) atomicOr(&mut[r].err, 4);
        const unsigned long long moves = (unsigned long long)nsweep * Prot * nrot;
        atomicAdd(&mut[r].total[rtype][2], moves);
        atomicAdd(&mut[r].accep[rtype][2], s);
        atomicAdd(&mut[r].pair_evals[2], 2ull * moves * (unsigned long long)items);
    }
}

// MCRotations3D by parts: a chain split over W workgroups by slice range [k0, k1) (even length), or
// a short chain as one part.  A half-sweep is a parallel step over the part's slices.  Before its
// even half a part needs the frames of slice k0-1 (the previous part's last, odd) and before its
// odd half those of slice k1 (the next part's first, even).  After its even half a part publishes
// its first slice's frames, after its odd half its last slice's, each with the density of its link
// to the neighbour, as a record of 64-bit words that each carry the publishing half's number above
// 32 bits of a double; the receiver's lanes poll the words themselves, so the data arrives with its
// check, and write the halves into LDS.  A record is rewritten only after the neighbour has read it
// (its next half needs this part's).  Bounded waits set error bit 2.
// Record (part, parity) at pub + part * pub_stride + parity * pub_stride / 2: 2 words per double
// of the nrot frames, then of the nrot link densities.
// Link kl joins local slices kl and kl+1; local slice 0 is k0-1 and ns+1 is k1.  A link's density,
// a rotor's sum over atoms and the pair energy of two rotors are kept as the last accepted move (or
// the launch's start) left them, so a move evaluates its proposal alone.
//
// Two bodies, by the part's length.  Short parts (nrot ns <= ROT3D_AHEAD: few chains, many parts)
// are bound by the chain of half-sweeps and take a group of lanes per move; what depends on the
// slice alone is formed a sweep ahead (rotor3d_ahead).  Long parts (many chains: the device is full)
// are bound by the FP64 instructions of a move and take a lane per move (rotor3d_long).
constexpr int FRAME_D = (int)(sizeof(Frame) / sizeof(double));

struct Rot3dEnv {
    const Rep& rp;
    const double4* beads;
    RotBead* rotb;
    Frame* frames;
    const double4* tab;
    unsigned seed;
    uint32_t pass;
    int nsweep, j0, jstride;
    unsigned base;                    // half-sweeps done by the launches before this one
    unsigned long long* mypub;        // + parity * half_rec
    const unsigned long long *from_prev, *from_next;  // the records an even and an odd half wait for
    int half_rec;
    __device__ __forceinline__ const unsigned long long* from(int parity) const { return parity == 0 ? from_prev : from_next; }
    __device__ __forceinline__ uint32_t sweep(int sw) const { return (uint32_t)(j0 + sw * jstride); }
    __device__ __forceinline__ long long at(int q, int k) const { return rp.rot_off + (long long)q * rp.Prot + k; }
};

// whether the launch has a sweep for this replica
__device__ __forceinline__ bool rotor3d_turn(const Rep& rp, const Run& run) {
    return rp.rotkind == 2 && rp.rot3d_id >= 0 && run.u < (run.ref_order ? rp.P : rp.S);
}

__device__ __forceinline__ Rot3dEnv rotor3d_env(const Rep& rp, uint32_t pass, const double4* beads, RotBead* rotb, Frame* frames,
                                                const Tables3& T3, const RotPart& pt, const unsigned* flags,
                                                unsigned long long* pub, int pub_stride, const Run& run) {
    const int half_rec = pub_stride / 2, W = pt.W;
    auto record = [&](int w, int parity) { return pub + (long long)(pt.fbase + w) * pub_stride + parity * half_rec; };
    return {rp, beads, rotb, frames, T3.r3 + (long long)rp.rot3d_id * 3 * ROT3D_SIZE, run.seed, pass,
            run.ref_order ? 1 : rp.P / rp.S, run.u, run.ref_order ? 0 : rp.S,
            __hip_atomic_load(flags + pt.fbase + pt.w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
            record(pt.w, 0), record((pt.w + W - 1) % W, 1), record((pt.w + 1) % W, 0), half_rec};
}

struct Prop3 {
    double phi, cth, chi, u;
};

// MCRot3Dstep's proposal for rotor q at slice k (mc_piqmc.cc:966-1010)
__device__ __forceinline__ Prop3 rot3d_propose(const Rot3dEnv& e, int q, int k, uint32_t jsweep, double phi, double cth,
                                               double chi) {
    const double twopi = 2.0 * PI_D;
    const uint32_t atom = (uint32_t)(e.rp.nl_atom + q);
    const uint4 w0 = draw(e.seed, e.rp.key, e.pass, K_ROT3D, jsweep, atom, (uint32_t)k, 0);
    const uint4 w1 = draw(e.seed, e.rp.key, e.pass, K_ROT3D, jsweep, atom, (uint32_t)k, 1);
    const double rand1 = u53(w0.x, w0.y), rand2 = u53(w0.z, w0.w), rand3 = u53(w1.x, w1.y);
    Prop3 p;
    p.u = u53(w1.z, w1.w);
    p.cth = cth + e.rp.rtstep * (rand1 - 0.5);
    p.phi = phi + twopi * (e.rp.rtstep * (rand2 - 0.5));
    p.chi = chi + twopi * (e.rp.rtstep * (rand3 - 0.5));
    if (p.phi < 0.0) p.phi = twopi + p.phi;
    if (p.chi < 0.0) p.chi = twopi + p.chi;
    p.phi = fmod_near(p.phi, twopi);
    p.chi = fmod_near(p.chi, twopi);
    if (p.cth > 1.0) p.cth = 2.0 - p.cth;
    if (p.cth < -1.0) p.cth = -2.0 - p.cth;
    return p;
}

// the test of MCRot3Dstep (mc_piqmc.cc:1134-1178): link densities d0 d1 (now) and d2 d3 (proposed)
__device__ __forceinline__ bool rot3d_accept(double d0, double d1, double d2, double d3, double taudv, double u) {
    double dold = d0 * d1;
    if (fabs(dold) < RZERO) dold = 0.0;
    if (dold < 0.0) dold = fabs(dold);
    double dnew = d2 * d3;
    if (fabs(dnew) < RZERO) dnew = 0.0;
    if (dnew < 0.0) dnew = fabs(dnew);
    double rd = (dold > RZERO) ? dnew / dold : 1.0;
    rd *= exp(-taudv);
    return rd > 1.0 || rd > u;
}

__device__ __forceinline__ void rot3d_store(const Rot3dEnv& e, long long i, double phi, double cth, double chi, const Frame& f) {
    RotBead b;
    b.phi = phi;
    b.cth = cth;
    b.chi = chi;
    b.pad0 = 0.0;
    b.pad1 = 0.0;
    store_axis(b, phi, cth);
    e.rotb[i] = b;
    e.frames[i] = f;
}

// one word of the neighbour's record, polled until it carries the half's number
__device__ __forceinline__ unsigned rot3d_word(const unsigned long long* src, unsigned want, int* s_err) {
    unsigned long long w = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned spins = 0;
    while ((unsigned)(w >> 32) != want) {
        if (++spins > ROT_SPIN_LIMIT) {
            *s_err = 2;
            break;
        }
        __builtin_amdgcn_s_sleep(1);
        w = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return (unsigned)w;
}

__device__ __forceinline__ unsigned long long rot3d_pack(double v, int word, unsigned tag) {
    const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    return (unsigned long long)tag << 32 | (word ? bits >> 32 : bits & 0xffffffffull);
}

// Short parts.  A half-sweep of a part is a chain: the neighbour's record, the link densities (angles
// of two frames, a gather from a table of 750 MB), the test, the record for the neighbour.  All else
// of a move depends on its slice alone: the draws, the proposal's frame, its energies with the atoms
// and (two rotors) with the other rotor, moved or not; these are formed right after the slice's
// previous move, while the records travel.  Frames, proposals and energies live in LDS for the
// launch, a group's lanes read a move's alike, one lane per new link evaluates its density, and only
// the waves with a boundary slice trade records, without a barrier of the block.
// With everything formed inside the half and the state in memory, a half of 16 slices and 32 atoms
// took 9.3 us.
// LDS: Lk[q][ns+1], then frames fr[q][ns+2] and proposals' frames fp[q][ns], then sl[q][ns] and, with
// two rotors, pr[ns].
template <typename R, int NROT>
__device__ __forceinline__ void rotor3d_ahead(const Rot3dEnv& e, const RotPart& pt, const Lut3D<R>& l3, double* smem, int* s_err,
                                              unsigned long long& nacc, int& err) {
    struct Slice {
        double phi, cth, chi, E;  // now; E the sum over atoms
        double Enew;
        Prop3 p;
    };
    struct Pair {
        double E, v[3];  // now; of (q0', q1), (q0, q1') and (q0', q1')
    };
    static_assert(sizeof(Slice) == 9 * sizeof(double) && sizeof(Pair) == 4 * sizeof(double), "rotor3d_part_lds");
    const Rep& rp = e.rp;
    const int k0 = pt.k0, ns = pt.k1 - pt.k0, W = pt.W, L = ns + 1, Prot = rp.Prot, RR = rp.RotRatio, nat = rp.nl_atom;
    double* Lk = smem;
    Frame* fr = reinterpret_cast<Frame*>(smem + ((NROT * L + 1) & ~1));
    Frame* fp = fr + NROT * (ns + 2);
    Slice* sl = reinterpret_cast<Slice*>(fp + NROT * ns);
    Pair* pr = reinterpret_cast<Pair*>(sl + NROT * ns);
    const int nmoves = ns >> 1;  // of either parity: k0 and ns are even
    int G = 1;
    while (G < 64 && G * 2 * nmoves <= (int)blockDim.x) G *= 2;
    const int mv = (int)threadIdx.x / G, gl = (int)threadIdx.x & (G - 1), lane = threadIdx.x & 63, gbase = lane & ~(G - 1);
    const bool mine = mv < nmoves;
    const int items_a = RR * nat;
    for (int i = threadIdx.x; i < NROT * (ns + 2); i += blockDim.x) {
        const int q = i / (ns + 2);
        int k = k0 + i - q * (ns + 2) - 1;
        if (k < 0) k += Prot;
        if (k >= Prot) k -= Prot;
        fr[i] = e.frames[e.at(q, k)];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NROT * L; i += blockDim.x) {
        const int q = i / L, kl = i - q * L;
        if (rotden_rho(fr[q * (ns + 2) + kl], fr[q * (ns + 2) + kl + 1], e.tab, Lk[i])) err = 1;
    }
    // separations of the lane's first atom of the sums at its even and odd slice: atoms stay during the launch
    R sep[2][NROT][3];
    auto atom_sum = [&](int parity, int q, int k, const Frame& f) -> double {
        double v = 0.0;
        if (gl < items_a)
            v = (double)vcord_sep<R>(l3, f, parity ? sep[1][q][0] : sep[0][q][0], parity ? sep[1][q][1] : sep[0][q][1],
                                     parity ? sep[1][q][2] : sep[0][q][2]);
        for (int i = gl + G; i < items_a; i += G) {
            const int it = k * RR + i / nat, a = i % nat;
            const double4 xa = bead(e.beads, rp, nat + q, it), xj = bead(e.beads, rp, a, it);
            v += (double)vcord_v<R>(l3, f, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z);
        }
        return group_sum(v, G);
    };
    auto pair = [&](int k, int s, const Frame& f0, const Frame& f1) -> double {
        const double4 x0 = bead(e.beads, rp, nat, k * RR + s), x1 = bead(e.beads, rp, nat + 1, k * RR + s);
        return caleng_v(x0.x, x0.y, x0.z, x1.x, x1.y, x1.z, f0, f1);
    };
    auto ahead = [&](int parity, int sw) {
        const int kl = 2 * mv + parity + 1, k = k0 + kl - 1;
#pragma unroll
        for (int q = 0; q < NROT; ++q) {
            Slice& s = sl[q * ns + kl - 1];
            const Prop3 p = rot3d_propose(e, q, k, e.sweep(sw), s.phi, s.cth, s.chi);
            const Frame f = make_frame(p.phi, p.cth, p.chi);
            double ea = 0.0;
            if (nat > 0) ea = atom_sum(parity, q, k, f);
            if (gl == 0) {
                fp[q * ns + kl - 1] = f;
                s.p = p;
                s.Enew = ea;
            }
        }
        wave_sync();
        if constexpr (NROT == 2) {
            double v0 = 0.0, v1 = 0.0, v2 = 0.0;
#pragma unroll 1
            for (int i = gl; i < 3 * RR; i += G) {
                const int s = i / 3, c = i - 3 * s;
                const double v = pair(k, s, c == 1 ? fr[kl] : fp[kl - 1], c == 0 ? fr[ns + 2 + kl] : fp[ns + kl - 1]);
                v0 += c == 0 ? v : 0.0;
                v1 += c == 1 ? v : 0.0;
                v2 += c == 2 ? v : 0.0;
            }
            v0 = group_sum(v0, G);
            v1 = group_sum(v1, G);
            v2 = group_sum(v2, G);
            if (gl == 0) {
                pr[kl - 1].v[0] = v0;
                pr[kl - 1].v[1] = v1;
                pr[kl - 1].v[2] = v2;
            }
        }
    };
    unsigned moved = 0;  // bit parity * NROT + q: the slice's rotor q was moved in this launch
    if (mine) {
#pragma unroll
        for (int parity = 0; parity < 2; ++parity)
#pragma unroll
            for (int q = 0; q < NROT; ++q) {
                sep[parity][q][0] = sep[parity][q][1] = sep[parity][q][2] = (R)0;
                if (gl < items_a) {
                    const int it = (k0 + 2 * mv + parity) * RR + gl / nat, a = gl % nat;
                    const double4 xa = bead(e.beads, rp, nat + q, it), xj = bead(e.beads, rp, a, it);
                    sep[parity][q][0] = (R)(xj.x - xa.x);
                    sep[parity][q][1] = (R)(xj.y - xa.y);
                    sep[parity][q][2] = (R)(xj.z - xa.z);
                }
            }
#pragma unroll 1
        for (int parity = 0; parity < 2; ++parity) {
            const int kl = 2 * mv + parity + 1, k = k0 + kl - 1;
#pragma unroll
            for (int q = 0; q < NROT; ++q) {
                const RotBead& b = e.rotb[e.at(q, k)];
                double ea = 0.0;
                if (nat > 0) ea = atom_sum(parity, q, k, fr[q * (ns + 2) + kl]);
                if (gl == 0) {
                    Slice& s = sl[q * ns + kl - 1];
                    s.phi = b.phi;
                    s.cth = b.cth;
                    s.chi = b.chi;
                    s.E = ea;
                }
            }
            if constexpr (NROT == 2) {
                double v = 0.0;
#pragma unroll 1
                for (int s = gl; s < RR; s += G) v += pair(k, s, fr[kl], fr[ns + 2 + kl]);
                v = group_sum(v, G);
                if (gl == 0) pr[kl - 1].E = v;
            }
            wave_sync();
            ahead(parity, 0);
        }
    }
    __syncthreads();  // Lk
    const int nwords = 2 * NROT * (FRAME_D + 1);
#pragma unroll 1
    for (int h = 0; h < 2 * e.nsweep; ++h) {
        const int parity = h & 1, sw = h >> 1;
        const int kl = 2 * mv + parity + 1;
        const int bnd = parity == 0 ? 0 : nmoves - 1;  // the move beside the neighbour this half trades with
        const bool trader = W > 1 && (bnd * G) >> 6 == (int)threadIdx.x >> 6;
        if (trader && h > 0) {
            const int kn = parity == 0 ? 0 : ns + 1, ln = parity == 0 ? 0 : ns;
            for (int w = lane; w < nwords; w += 64) {
                const unsigned v = rot3d_word(e.from(parity) + w, e.base + (unsigned)h, s_err);
                const int i = w >> 1;  // the double: frames first, then link densities
                double* d = i < NROT * FRAME_D ? reinterpret_cast<double*>(fr + (i / FRAME_D) * (ns + 2) + kn) + i % FRAME_D
                                               : Lk + (i - NROT * FRAME_D) * L + ln;
                reinterpret_cast<unsigned*>(d)[w & 1] = v;
            }
            wave_sync();
        }
        if (mine) {
            const int c = gl & (2 * NROT - 1), lq = c >> 1, side = c & 1;
            double rho;
            if (rotden_link(fr[lq * (ns + 2) + kl - 1 + 2 * side], fp[lq * ns + kl - 1], side, e.tab, rho)) err = 1;
            bool acc0 = false;
#pragma unroll
            for (int q = 0; q < NROT; ++q) {
                Slice& s = sl[q * ns + kl - 1];
                const double d2 = __shfl(rho, gbase + 2 * q), d3 = __shfl(rho, gbase + 2 * q + 1);
                double dv = s.Enew - s.E, pe = 0.0;
                if constexpr (NROT == 2) {
                    const Pair& p = pr[kl - 1];
                    pe = q == 0 ? p.v[0] : (acc0 ? p.v[2] : p.v[1]);
                    dv = (s.Enew + pe) - (s.E + p.E);
                }
                const bool accepted = rot3d_accept(Lk[q * L + kl - 1], Lk[q * L + kl], d2, d3, rp.tau * dv, s.p.u);
                wave_sync();  // every lane has read the old state
                if (accepted) {
                    if (q == 0) acc0 = true;
                    moved |= 1u << (parity * NROT + q);
                    const double* src = reinterpret_cast<const double*>(fp + q * ns + kl - 1);
                    double* dst = reinterpret_cast<double*>(fr + q * (ns + 2) + kl);
                    // a chain in one part is its own neighbour: slices 0 and ns are one, ns + 1 and 1,
                    // links 0 and ns; the other copy of a boundary slice
                    const bool twin = W == 1 && (kl == 1 || kl == ns);
                    double* dst2 = reinterpret_cast<double*>(fr + q * (ns + 2) + (kl == 1 ? ns + 1 : 0));
                    for (int i = gl; i < FRAME_D; i += G) {
                        dst[i] = src[i];
                        if (twin) dst2[i] = src[i];
                    }
                    if (gl == 0) {
                        ++nacc;
                        s.phi = s.p.phi;
                        s.cth = s.p.cth;
                        s.chi = s.p.chi;
                        s.E = s.Enew;
                        if constexpr (NROT == 2) pr[kl - 1].E = pe;
                        Lk[q * L + kl - 1] = d2;
                        Lk[q * L + kl] = d3;
                        if (twin) Lk[q * L + (kl == 1 ? ns : 0)] = kl == 1 ? d2 : d3;
                    }
                }
                wave_sync();
            }
        }
        if (trader) {  // publish the boundary slice; no wait for the stores, the reader checks every word
            wave_sync();
            const int kb = parity == 0 ? 1 : ns, lb = parity == 0 ? 0 : ns;
            for (int w = lane; w < nwords; w += 64) {
                const int i = w >> 1;
                const double v = i < NROT * FRAME_D ? reinterpret_cast<const double*>(fr + (i / FRAME_D) * (ns + 2) + kb)[i % FRAME_D]
                                                    : Lk[(i - NROT * FRAME_D) * L + lb];
                __hip_atomic_store(e.mypub + parity * e.half_rec + w, rot3d_pack(v, w & 1, e.base + (unsigned)h + 1u), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (mine && sw + 1 < e.nsweep) ahead(parity, sw + 1);
        lds_barrier();
        // a wait that gave up: no later wait of this launch can succeed either, so the part leaves
        // at once (every lane reads s_err after the barrier; it is written again in the next half)
        if (*s_err) break;
    }
    if (mine && gl == 0)
#pragma unroll
        for (int parity = 0; parity < 2; ++parity) {
            const int kl = 2 * mv + parity + 1;
#pragma unroll
            for (int q = 0; q < NROT; ++q) {
                const Slice& s = sl[q * ns + kl - 1];
                if (moved >> (parity * NROT + q) & 1) rot3d_store(e, e.at(q, k0 + kl - 1), s.phi, s.cth, s.chi, fr[q * (ns + 2) + kl]);
            }
        }
}

// Long parts: a lane per move.  With many chains the device is full and the time is a move's FP64
// instructions (two generator calls, the frame, six arc cosines, an energy) and what it reads: its
// neighbours' and partner's frames, its angles, and two gathers for its links.  InLds keeps the chain's
// state in LDS for the launch, which leaves the gathers and positions to memory: of a frame the x and
// z axes (y is their cross product, which differs from the frame's own in its last bit: a link takes
// from y the signs of two sines and, within 1e-8 of theta = pi, an arc cosine; energies take x and z,
// or the proposal's own frame) and of the angles phi and chi, 72 bytes a rotor and slice with
// the link's density, so that two parts of 512 slices of two rotors share a CU; cos theta is on the
// lane (at most one move a lane of either parity).  Even and odd slices lie apart: the lanes' accesses
// then meet no bank twice.
// Otherwise (rotor3d_in_lds) state is read and written in memory.
// LDS: Lk[q][ns+1], Ea[q][ns] (sum over atoms) with atoms, Er[ns] (pair energy) with two rotors, then
// axes[q][ns+2] and angles[q][ns], or the neighbours' frames fnb[2][nrot] (k0-1, then k1).
template <typename R, int NROT, bool InLds>
__device__ __forceinline__ void rotor3d_long(const Rot3dEnv& e, const RotPart& pt, const Lut3D<R>& l3, double* smem, int* s_err,
                                             unsigned long long& nacc, int& err) {
    struct alignas(16) Axes {
        double x[3], z[3];
    };
    struct alignas(16) Angles {
        double phi, chi;
    };
    const Rep& rp = e.rp;
    const int k0 = pt.k0, ns = pt.k1 - pt.k0, L = ns + 1, Prot = rp.Prot, RR = rp.RotRatio, nat = rp.nl_atom;
    double* Lk = smem;
    double* Ea = Lk + NROT * L;
    double* Er = Ea + (nat > 0 ? NROT * ns : 0);
    double* rest = smem + ((NROT * L + (nat > 0 ? NROT * ns : 0) + (NROT - 1) * ns + 1) & ~1);
    Frame* fnb = reinterpret_cast<Frame*>(rest);
    Axes* ax = reinterpret_cast<Axes*>(rest);
    Angles* ang = reinterpret_cast<Angles*>(ax + NROT * (ns + 2));
    const int half_ns = ns >> 1;
    auto axes = [&](int q, int kl) -> Axes& { return ax[q * (ns + 2) + (kl & 1) * (half_ns + 1) + (kl >> 1)]; };
    auto angles = [&](int q, int kl) -> Angles& { return ang[q * ns + ((kl - 1) & 1) * half_ns + ((kl - 1) >> 1)]; };
    auto slice = [&](int kl) {  // of local slice kl
        const int k = k0 + kl - 1;
        return k < 0 ? k + Prot : (k >= Prot ? k - Prot : k);
    };
    // the frame of rotor q at local slice kl (zn left out: it is asked of proposals only)
    auto frame = [&](int q, int kl) -> Frame {
        if constexpr (InLds) {
            const Axes& a = axes(q, kl);
            Frame f;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                f.m[i] = a.x[i];
                f.m[6 + i] = a.z[i];
            }
            f.m[3] = f.m[7] * f.m[2] - f.m[8] * f.m[1];
            f.m[4] = f.m[8] * f.m[0] - f.m[6] * f.m[2];
            f.m[5] = f.m[6] * f.m[1] - f.m[7] * f.m[0];
            f.zn = 1.0;
            return f;
        } else {
            return kl == 0 ? fnb[q] : (kl == ns + 1 ? fnb[NROT + q] : e.frames[e.at(q, k0 + kl - 1)]);
        }
    };
    auto set_axes = [&](int q, int kl, const Frame& f) {
        Axes& a = axes(q, kl);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            a.x[i] = f.m[i];
            a.z[i] = f.m[6 + i];
        }
    };
    // at launch start no neighbour has moved its boundary slice yet (its first move on it waits
    // for this part), so the boundary frames come straight from memory
    if constexpr (InLds) {
        for (int i = threadIdx.x; i < NROT * (ns + 2); i += blockDim.x) {
            const int q = i / (ns + 2), kl = i - q * (ns + 2);
            set_axes(q, kl, e.frames[e.at(q, slice(kl))]);
            if (kl > 0 && kl <= ns) {
                const RotBead& b = e.rotb[e.at(q, slice(kl))];
                angles(q, kl) = {b.phi, b.chi};
            }
        }
    } else {
        for (int i = threadIdx.x; i < 2 * NROT; i += blockDim.x) {
            const int side = i / NROT, q = i - side * NROT;
            fnb[i] = e.frames[e.at(q, slice(side ? ns + 1 : 0))];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NROT * L; i += blockDim.x) {
        const int q = i / L, kl = i - q * L;
        if (rotden_rho(frame(q, kl), frame(q, kl + 1), e.tab, Lk[i])) err = 1;
    }
    auto atom_sum = [&](int q, int k, const Frame& f) -> double {
        double v = 0.0;
        for (int s = 0; s < RR; ++s) {
            const double4 xa = bead(e.beads, rp, nat + q, k * RR + s);
            for (int a = 0; a < nat; ++a) {
                const double4 xj = bead(e.beads, rp, a, k * RR + s);
                v += (double)vcord_v<R>(l3, f, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z);
            }
        }
        return v;
    };
    auto pair = [&](int k, int q, const Frame& f, const Frame& fo) -> double {  // rotor q at f, the other at fo
        double v = 0.0;
#pragma unroll 1
        for (int s = 0; s < RR; ++s) {
            const double4 x = bead(e.beads, rp, nat + q, k * RR + s), xo = bead(e.beads, rp, nat + 1 - q, k * RR + s);
            v += caleng_v(x.x, x.y, x.z, xo.x, xo.y, xo.z, f, fo);
        }
        return v;
    };
    for (int i = threadIdx.x; i < ns; i += blockDim.x) {
        if (nat > 0)
#pragma unroll
            for (int q = 0; q < NROT; ++q) Ea[q * ns + i] = atom_sum(q, k0 + i, e.frames[e.at(q, k0 + i)]);
        if constexpr (NROT == 2) Er[i] = pair(k0 + i, 0, frame(0, i + 1), frame(1, i + 1));
    }
    __syncthreads();
    const int nwords = 2 * NROT * (FRAME_D + 1);
    // InLds: cos theta of the lane's even and odd slice, and which of them were moved (bit parity NROT + q)
    double cth_now[2][NROT];
    unsigned moved = 0;
    if constexpr (InLds) {
#pragma unroll
        for (int i = 0; i < 2 * NROT; ++i)
            if ((int)threadIdx.x < half_ns)
                cth_now[i / NROT][i % NROT] = e.rotb[e.at(i % NROT, k0 + 2 * (int)threadIdx.x + i / NROT)].cth;
    }
    auto cth_of = [&](int parity, int q) -> double {
        const double c0 = parity ? cth_now[1][0] : cth_now[0][0];
        if constexpr (NROT == 1) return c0;
        const double c1 = parity ? cth_now[1][NROT - 1] : cth_now[0][NROT - 1];
        return q ? c1 : c0;
    };
#pragma unroll 1
    for (int h = 0; h < 2 * e.nsweep; ++h) {
        const int parity = h & 1, sw = h >> 1;
        if (h > 0) {
            const int kn = parity == 0 ? 0 : ns + 1, ln = parity == 0 ? 0 : ns;
            for (int w = threadIdx.x; w < nwords; w += blockDim.x) {
                const unsigned v = rot3d_word(e.from(parity) + w, e.base + (unsigned)h, s_err);
                const int i = w >> 1, q = i / FRAME_D, c = i - q * FRAME_D;  // the double: frames first, then link densities
                if (q >= NROT) {
                    reinterpret_cast<unsigned*>(&Lk[(i - NROT * FRAME_D) * L + ln])[w & 1] = v;
                } else if constexpr (InLds) {
                    if (c < 3) reinterpret_cast<unsigned*>(&axes(q, kn).x[c])[w & 1] = v;
                    else if (c >= 6 && c < 9) reinterpret_cast<unsigned*>(&axes(q, kn).z[c - 6])[w & 1] = v;
                } else {
                    reinterpret_cast<unsigned*>(fnb + (parity == 0 ? 0 : NROT))[w] = v;
                }
            }
            __syncthreads();
            if (*s_err) break;  // as in rotor3d_ahead
        }
#pragma unroll 1
        for (int mv = threadIdx.x; mv < half_ns; mv += blockDim.x) {
            const int kl = 2 * mv + parity + 1, k = k0 + kl - 1;
#pragma unroll 1
            for (int q = 0; q < NROT; ++q) {
                const long long ik = e.at(q, k);
                double phi, cth, chi;
                if constexpr (InLds) {
                    phi = angles(q, kl).phi;
                    chi = angles(q, kl).chi;
                    cth = cth_of(parity, q);
                } else {
                    const RotBead& cur = e.rotb[ik];
                    phi = cur.phi;
                    cth = cur.cth;
                    chi = cur.chi;
                }
                const Prop3 p = rot3d_propose(e, q, k, e.sweep(sw), phi, cth, chi);
                const Frame f = make_frame(p.phi, p.cth, p.chi);
                RhoCell left, right;  // the gathers are asked for before the energy and read after it
                if (rotden_cell(frame(q, kl - 1), f, 0, e.tab, left)) err = 1;
                if (rotden_cell(frame(q, kl + 1), f, 1, e.tab, right)) err = 1;
                double ea = 0.0, pe = 0.0, dv = 0.0;
                if (nat > 0) {
                    ea = atom_sum(q, k, f);
                    dv = ea - Ea[q * ns + kl - 1];
                }
                if constexpr (NROT == 2) {  // rotor 1 sees rotor 0's move
                    pe = pair(k, q, f, frame(1 - q, kl));
                    dv = (ea + pe) - ((nat > 0 ? Ea[q * ns + kl - 1] : 0.0) + Er[kl - 1]);
                }
                const double d2 = rho_value(left), d3 = rho_value(right);
                if (rot3d_accept(Lk[q * L + kl - 1], Lk[q * L + kl], d2, d3, rp.tau * dv, p.u)) {
                    ++nacc;
                    if constexpr (InLds) {
                        set_axes(q, kl, f);
                        angles(q, kl) = {p.phi, p.chi};
#pragma unroll
                        for (int i = 0; i < 2 * NROT; ++i)
                            if (i == parity * NROT + q) cth_now[i / NROT][i % NROT] = p.cth;
                        moved |= 1u << (parity * NROT + q);
                    } else {
                        rot3d_store(e, ik, p.phi, p.cth, p.chi, f);
                    }
                    Lk[q * L + kl - 1] = d2;
                    Lk[q * L + kl] = d3;
                    if (nat > 0) Ea[q * ns + kl - 1] = ea;
                    if constexpr (NROT == 2) Er[kl - 1] = pe;
                }
            }
        }
        __syncthreads();
        // publish the boundary slice this half moved; no wait for the stores, the reader checks every word
        const int kb = parity == 0 ? 1 : ns;
        for (int w = threadIdx.x; w < nwords; w += blockDim.x) {
            const int i = w >> 1, q = i / FRAME_D;
            double v;
            if (q >= NROT) {
                v = Lk[(i - NROT * FRAME_D) * L + (parity == 0 ? 0 : ns)];
            } else {
                const Frame f = frame(q, kb);
                v = f.zn;
#pragma unroll
                for (int c = 0; c < 9; ++c)
                    if (c == i - q * FRAME_D) v = f.m[c];
            }
            __hip_atomic_store(e.mypub + parity * e.half_rec + w, rot3d_pack(v, w & 1, e.base + (unsigned)h + 1u), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if constexpr (InLds) {
#pragma unroll 1
        for (int i = 0; i < 2 * NROT; ++i) {
            if (!(moved >> i & 1)) continue;
            const int parity = i / NROT, q = i - parity * NROT, kl = 2 * (int)threadIdx.x + parity + 1;
            const double phi = angles(q, kl).phi, chi = angles(q, kl).chi, cth = cth_of(parity, q);
            rot3d_store(e, e.at(q, k0 + kl - 1), phi, cth, chi, make_frame(phi, cth, chi));
        }
    }
}

template <typename R>
__global__ __launch_bounds__(256, 2) void k_rotor3d_parts(const Rep* __restrict__ reps, Mut* __restrict__ mut,
                                                          const double4* __restrict__ beads, RotBead* __restrict__ rotb,
                                                          Frame* __restrict__ frames, Tables T, Tables3 T3,
                                                          const RotPart* __restrict__ parts, unsigned* __restrict__ flags,
                                                          unsigned long long* __restrict__ pub, int pub_stride, Run run) {
    extern __shared__ DYNAMIC_LDS double smem[];
    __shared__ unsigned long long red_acc[4];
    __shared__ int s_err;
    const RotPart pt = parts[blockIdx.x];
    if (pt.r < 0) return;  // padding of the XCD-ordered grid
    const int r = pt.r;
    const Rep& rp = reps[r];
    if (!rotor3d_turn(rp, run)) return;
    const int ns = pt.k1 - pt.k0, W = pt.W, nrot = rp.nrot;
    const Rot3dEnv e = rotor3d_env(rp, mut[r].pass, beads, rotb, frames, T3, pt, flags, pub, pub_stride, run);
    const Lut3D<R> l3 = lut3d<R>(T3, rp.pot3d_id);
    if (threadIdx.x == 0) s_err = 0;
    unsigned long long nacc = 0;
    int err = 0;
    const bool ahead = nrot * ns <= ROT3D_AHEAD;  // a longer part is one of several (W > 1)
    const bool in_lds = rotor3d_in_lds(ns, nrot, rp.nl_atom > 0);
    auto sweep = [&](auto n_c) {
        constexpr int NROT = decltype(n_c)::value;
        if (ahead) rotor3d_ahead<R, NROT>(e, pt, l3, smem, &s_err, nacc, err);
        else if (in_lds) rotor3d_long<R, NROT, true>(e, pt, l3, smem, &s_err, nacc, err);
        else rotor3d_long<R, NROT, false>(e, pt, l3, smem, &s_err, nacc, err);
    };
    if (nrot == 1) sweep(std::integral_constant<int, 1>{});
    else sweep(std::integral_constant<int, 2>{});
    if (W > 1 && threadIdx.x == 0)  // every part of the chain ran the same halves
        __hip_atomic_store(flags + pt.fbase + pt.w, e.base + 2u * (unsigned)e.nsweep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (err) atomicOr(&mut[r].err, 4);
    unsigned long long sacc = block_sum(nacc, red_acc);
    if (threadIdx.x == 0) {
        if (s_err) atomicOr(&mut[r].err, s_err);
        const unsigned long long slices = (unsigned long long)e.nsweep * ns, items_a = (unsigned long long)(rp.RotRatio * rp.nl_atom);
        atomicAdd(&mut[r].total[rp.imtype][2], slices * nrot);
        atomicAdd(&mut[r].accep[rp.imtype][2], sacc);
        // the atoms' terms of every proposal, the pair terms (two rotors: one per move, though with the
        // energies ahead a third was formed), and the current orientations' once per launch
        const unsigned long long pairs = nrot < 2 ? 0 : (unsigned long long)rp.RotRatio;
        atomicAdd(&mut[r].pair_evals[2], (slices + ns) * nrot * items_a + (slices * 2 + ns) * pairs);
    }
}

// ------------------------------------------------------------------------- restart
// Rotation matrices of every non-linear rotor slice of replica r from its stored angles, with
// the code the moves use when they accept (make_frame), so a resumed chain sees the same bits.
__global__ void k_frames_from_angles(const Rep* __restrict__ reps, const RotBead* __restrict__ rotb,
                                     Frame* __restrict__ frames, int r, int n) {
    const Rep& rp = reps[r];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const RotBead& b = rotb[rp.rot_off + i];
    frames[rp.rot_off + i] = make_frame(b.phi, b.cth, b.chi);
}

// ------------------------------------------------------------------------- rotational correlation
// GetRCF (mc_estim.cc:1098-1139), one sample: for every time origin it0 and offset itc of the
// first rotor of the rotating type, p = n(it0).n(it0+itc) with the unit axes of MCCosine;
// rcf[0][itc] += p and rcf[l][itc] += P_l(p) for l = 1..9.  (The reference adds 1.0 for l >= 1:
// its Legendre call is commented out; here P_l comes from the three-term recurrence.)
// The sum over origins is the same for an offset and its complement to Prot, so offsets up to Prot / 2
// are summed.  Grid (replica, block of RCF_OFFSETS offsets): a block's lanes share the offsets by
// ranges of origins, in FP64, the ranges' sums added in order.  A lane per offset over all origins,
// dividing in the recurrence, took 1.91 ms for 128 chains of 2048 slices, now 0.76.
constexpr int RCF_OFFSETS = 16, RCF_RANGES = 256 / RCF_OFFSETS;
__global__ __launch_bounds__(256) void k_rcf(const Rep* __restrict__ reps, const RotBead* __restrict__ rotb,
                                             const int* __restrict__ list, double* __restrict__ rcf) {
    __shared__ double part[RCF_RANGES][RCF_OFFSETS];
    const Rep& rp = reps[list[blockIdx.x]];
    const int Prot = rp.Prot, last = Prot / 2;  // offsets 0 .. last
    const RotBead* b = rotb + rp.rot_off;
    double* out = rcf + rp.rcf_off;
    const int o = threadIdx.x % RCF_OFFSETS, g = threadIdx.x / RCF_OFFSETS;
    const int from = (int)((long long)Prot * g / RCF_RANGES), end = (int)((long long)Prot * (g + 1) / RCF_RANGES);
    for (int first = blockIdx.y * RCF_OFFSETS; first <= last; first += gridDim.y * RCF_OFFSETS) {
        const int itc = first + o, to = itc <= last ? end : from;
        double acc[RCF_L];
#pragma unroll
        for (int l = 0; l < RCF_L; ++l) acc[l] = 0.0;
        int t1 = from + itc < Prot ? from + itc : from + itc - Prot;
#pragma unroll 2
        for (int it0 = from; it0 < to; ++it0) {
            const double p = b[it0].nx * b[t1].nx + b[it0].ny * b[t1].ny + b[it0].nz * b[t1].nz;
            acc[0] += p;
            double pm = 1.0, pc = p;  // P_0, P_1
            acc[1] += pc;
#pragma unroll
            for (int l = 1; l + 1 < RCF_L; ++l) {
                const double pn = ((2 * l + 1) / (double)(l + 1)) * (p * pc) - (l / (double)(l + 1)) * pm;
                pm = pc;
                pc = pn;
                acc[l + 1] += pc;
            }
            if (++t1 == Prot) t1 = 0;
        }
#pragma unroll
        for (int l = 0; l < RCF_L; ++l) {
            part[g][o] = acc[l];
            __syncthreads();
            if (g == l % RCF_RANGES && itc <= last) {
                double v = 0.0;
                for (int k = 0; k < RCF_RANGES; ++k) v += part[k][o];
                out[(long long)l * Prot + itc] += v;
                if (itc > 0 && 2 * itc != Prot) out[(long long)l * Prot + Prot - itc] += v;
            }
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------------------- delayed acceptance
// MCRotations3D (mc_piqmc.cc:692-779) with the one-stage test of MCRot3Dstep (:1166-1178),
// min(1, rho_new/rho_old * exp(-tau dV)), split into three factors (multi-stage delayed
// acceptance, Christen & Fox 2005), each a Metropolis test of its own:
//   stage 0  min(1, rho_new/rho_old), the density factor, which the move has in hand anyway;
//   stage 1  min(1, exp(-tau (dVs + dVx))), Vs the surrogate network summed over the slice's
//            network pairs and Vx the exact energy of the other pairs;
//   stage 2  min(1, exp(-tau (dV_net - dVs))), the exact network-pair sums.
// Each factor is in detailed balance with its own part of the target, so their product is in
// detailed balance with rho * exp(-tau V) for any surrogate: the stationary distribution is the
// one-stage move's.  A proposal is charged the network only when it passes stage 0, and the exact
// network-pair sums only when it passes stage 1.  Stage 0 takes its uniform from counter word 3
// = 2 (second half), stage 1 the one-stage test's (rand4), stage 2 counter word 3 = 2 (first).
// Network pairs: rotor-atom pairs when the replica has atoms (rotor-rotor pairs of two rotors are
// then exact in stage 1), rotor-rotor pairs when it has none.
//
// Chains are split into parts as k_rotor3d_parts splits them, with the same boundary records
// between half-sweeps (a part of W = 1 is a whole chain and trades with itself).  Within a half,
// rotor q in turn (a move of rotor q at slice k sees the moves of the rotors before it at k, as
// in the one-stage kernel); each wave takes its moves in chunks of DA_MV, lane j the chunk's move
// j: (1) proposal, new link densities and the exact stage-1 terms; (2) stage 0, then the network
// rows of the moves that passed it, listed first, 32 per pass through the matrix cores, summed
// per move in row order; (3) stage 1; (4) stage 2 for the moves that passed -- the whole wave
// sums one move's rotor-atom pairs, or each lane its move's rotor-rotor pairs; (5) updates.  The
// surrogate and exact rotor-atom sums of every own slice at its current orientation are cached
// (atoms do not move during the sweep): a move evaluates only its proposal, and an accepted move
// leaves its new sums as the cached ones.
// LDS: the packed network; Lk [nrot][ns+1], Vs and Ex [nrot][ns] (doubles); the neighbours'
// boundary frames [2 nrot]; per wave DA_MV proposal frames and 32 row outputs (DA_MV and the
// LDS size: pimc_plan.hpp).

// Body-frame features of a rotor-rotor pair for the network: the distance of the centres, the
// cosines of both body z axes (the dipole axis of the TIP4P geometry) with the unit separation
// from rotor q to rotor p, and the cosine between the two z axes.
__device__ __forceinline__ void mlp_rotor_pair_features(const Frame& fq, const Frame& fp, double qx, double qy,
                                                        double qz, double px, double py, double pz, float out[MLP_IN]) {
    const double rx = px - qx, ry = py - qy, rz = pz - qz;
    const double rn = sqrt(rx * rx + ry * ry + rz * rz);
    const double inv = rn > 0.0 ? 1.0 / rn : 0.0;
    out[0] = (float)rn;
    out[1] = (float)((fq.m[6] * rx + fq.m[7] * ry + fq.m[8] * rz) * inv);
    out[2] = (float)((fp.m[6] * rx + fp.m[7] * ry + fp.m[8] * rz) * inv);
    out[3] = (float)(fq.m[6] * fp.m[6] + fq.m[7] * fp.m[7] + fq.m[8] * fp.m[8]);
}

// Short parts of the delayed-acceptance sweep (nrot ns <= ROT3D_AHEAD), where a half-sweep is a chain
// of dependent steps: the neighbour's record, the links' densities, the network's layers, the exact
// sums, the record for the neighbour.  As in rotor3d_ahead the state lives in LDS, proposals are
// formed right after the slice's last move while the records travel, and only the waves with a
// boundary slice trade records.  A wave takes its moves DA_SHORT at a time, lanes j and j + 32 of
// move j one new link each; with at most 32 exact terms a half wave sums a move's.
// With state in memory, both links on one lane and 16 slices a part, a half of 256 slices and 32 atoms
// took 29 us, now 17, of which the network's three layers on a wave are about 5.
// LDS: the network, Lk[q][ns+1], frames fr[q][ns+2] and proposals' frames fp[q][ns], sl[q][ns], then
// 32 row outputs per wave.
constexpr int DA_SHORT = 32;

template <typename R>
__device__ __forceinline__ void rotor3d_da_short(const Rot3dEnv& e, const RotPart& pt, const Lut3D<R>& l3, MlpPacked* W, int* s_err,
                                                 unsigned long long& nacc, unsigned long long& npass, unsigned long long& nnet,
                                                 int& err) {
    struct Slice {
        double phi, cth, chi, V, E;  // now; the network's and the exact sums over atoms
        Prop3 p;
        double u0, u2;               // uniforms of stages 0 and 2 (p.u: stage 1)
    };
    static_assert(sizeof(Slice) == 11 * sizeof(double), "rotor3d_da_part_lds");
    const Rep& rp = e.rp;
    const int k0 = pt.k0, ns = pt.k1 - pt.k0, NP = pt.W, L = ns + 1, Prot = rp.Prot, RR = rp.RotRatio, nrot = rp.nrot, nat = rp.nl_atom;
    const bool net_atoms = nat > 0;  // network pairs: rotor-atom, else rotor-rotor
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, nw = blockDim.x >> 6, j = l & 31, side = l >> 5;
    double* Lk = reinterpret_cast<double*>(W + 1);
    Frame* fr = reinterpret_cast<Frame*>(Lk + ((nrot * L + 1) & ~1));
    Frame* fp = fr + nrot * (ns + 2);
    Slice* sl = reinterpret_cast<Slice*>(fp + nrot * ns);
    float* rowo = reinterpret_cast<float*>(sl + nrot * ns) + wv * 32;
    const double ys = (double)W->ys;
    const int rpm = net_atoms ? RR * nat : RR * (nrot - 1) * 2;  // network rows per move
    const int items_x = RR * nat;                                // exact rotor-atom pairs of a slice
    for (int i = threadIdx.x; i < nrot * (ns + 2); i += blockDim.x) {
        const int q = i / (ns + 2), kl = i - q * (ns + 2);
        int k = k0 + kl - 1;
        if (k < 0) k += Prot;
        if (k >= Prot) k -= Prot;
        fr[i] = e.frames[e.at(q, k)];
        if (kl > 0 && kl <= ns) {
            const RotBead& b = e.rotb[e.at(q, k)];
            Slice& s = sl[q * ns + kl - 1];
            s.phi = b.phi;
            s.cth = b.cth;
            s.chi = b.chi;
            s.V = s.E = 0.0;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nrot * L; i += blockDim.x) {
        const int q = i / L, kl = i - q * L;
        if (rotden_rho(fr[q * (ns + 2) + kl], fr[q * (ns + 2) + kl + 1], e.tab, Lk[i])) err = 1;
    }
    // the network's rows for slices of rotor q, summed per slice: entry i < nm of the list
    // is the slice kl_j of lane src (src_j on lane i); sums of (old, new) rows return in so/sn on lane i
    auto net_rows = [&](int q, int nm, int kl_j, int src_j, bool proposal, double& so, double& sn) {
        so = 0.0;
        sn = 0.0;
        const int total = nm * rpm;
        for (int b = 0; b < total; b += 32) {
            const int row = b + j;
            const int jj = min(row, total - 1) / rpm, jb = __shfl(jj, 0);
            const int klr = __shfl(kl_j, __shfl(src_j, jj));
            float f[MLP_IN] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (row < total) {
                const int idx = row - jj * rpm, k = k0 + klr - 1, gq = nat + q;
                const Frame& now = fr[q * (ns + 2) + klr];
                const Frame& moved = fp[q * ns + klr - 1];
                if (net_atoms) {
                    const int s = idx / nat, a = idx - s * nat, it = k * RR + s;
                    const double4 xa = bead(e.beads, rp, gq, it), xj = bead(e.beads, rp, a, it);
                    const Frame& fq = proposal ? moved : now;
                    mlp_pair_features(fq.m, fq.zn, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, f);
                } else {
                    const int s = (idx >> 1) / (nrot - 1), pp = (idx >> 1) - s * (nrot - 1), p = pp + (pp >= q), it = k * RR + s;
                    const double4 xq = bead(e.beads, rp, gq, it), xp = bead(e.beads, rp, nat + p, it);
                    mlp_rotor_pair_features(proposal && (idx & 1) ? moved : now, fr[p * (ns + 2) + klr], xq.x, xq.y, xq.z, xp.x,
                                            xp.y, xp.z, f);
                }
#pragma unroll
                for (int c = 0; c < MLP_IN; ++c) f[c] = (f[c] - W->xm[c]) * W->xinv[c];
            }
            // an opaque zero offset keeps the weight reads inside the loop (hoisted out they
            // would hold ~130 registers of weights per lane)
            int z = 0;
            __asm__ volatile("" : "+s"(z));
            const float o = mlp_rows32(reinterpret_cast<const MlpPacked*>(reinterpret_cast<const char*>(W) + z), f);
            if (rpm >= 8) {  // entry by entry over the lanes that hold its rows
                for (int i = jb; i * rpm < min(b + 32, total); ++i) {
                    const bool in = l < 32 && row >= i * rpm && row < min((i + 1) * rpm, total);
                    const bool moved = net_atoms || ((row - i * rpm) & 1);
                    const double vn = wave_sum(in && moved ? (double)o : 0.0);
                    if (l == i) sn += vn;
                    if (!net_atoms) {
                        const double vo = wave_sum(in && !moved ? (double)o : 0.0);
                        if (l == i) so += vo;
                    }
                }
                continue;
            }
            if (l < 32) rowo[l] = o;
            wave_sync();
            if (l < nm) {  // the rows of entry l that fall in this batch
                const int r0 = max(l * rpm, b), r1 = min((l + 1) * rpm, b + 32);
                for (int rr = r0; rr < r1; ++rr) {
                    const double v = (double)rowo[rr - b];
                    const bool moved = net_atoms || ((rr - l * rpm) & 1);
                    sn += moved ? v : 0.0;
                    so += moved ? 0.0 : v;
                }
            }
            wave_sync();
        }
    };
    // exact rotor-atom sums of rotor q with frame f at local slice kl, over GL lanes from this one's group
    auto exact_atoms = [&](int q, int kl, const Frame& f, int GL) -> double {
        const int k = k0 + kl - 1, gq = nat + q;
        double v = 0.0;
        for (int i = l & (GL - 1); i < items_x; i += GL) {
            const int s = i / nat, a = i - s * nat, it = k * RR + s;
            const double4 xa = bead(e.beads, rp, gq, it), xj = bead(e.beads, rp, a, it);
            v += (double)vcord_v<R>(l3, f, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z);
        }
        return group_sum(v, GL);
    };
    // exact rotor-rotor terms of rotor q moved, less those of it as it is: the half waves take one each
    auto pair_change = [&](int q, int kl) -> double {
        const int k = k0 + kl - 1;
        const Frame& f = side == 0 ? fp[q * ns + kl - 1] : fr[q * (ns + 2) + kl];
        double v = 0.0;
        for (int p = 0; p < nrot; ++p) {
            if (p == q) continue;
            for (int s = 0; s < RR; ++s) {
                const double4 xa = bead(e.beads, rp, nat + q, k * RR + s), xp = bead(e.beads, rp, nat + p, k * RR + s);
                v += caleng_v(xa.x, xa.y, xa.z, xp.x, xp.y, xp.z, f, fr[p * (ns + 2) + kl]);
            }
        }
        return v;
    };
    auto moves_of_wave = [&](int nmoves) { return nmoves > wv ? (nmoves - wv + nw - 1) / nw : 0; };  // wv, wv + nw, ...
    auto ahead = [&](int parity, int sw) {  // the half waves take a rotor each
        const int mine = moves_of_wave(ns >> 1);
        for (int c0 = 0; c0 < mine; c0 += DA_SHORT) {
            if (c0 + j >= mine || side >= nrot) continue;
            const int kl = 2 * (wv + (c0 + j) * nw) + parity + 1, k = k0 + kl - 1, q = side;
            Slice& s = sl[q * ns + kl - 1];
            s.p = rot3d_propose(e, q, k, e.sweep(sw), s.phi, s.cth, s.chi);
            const uint4 w2 = draw(e.seed, rp.key, e.pass, K_ROT3D, e.sweep(sw), (uint32_t)(nat + q), (uint32_t)k, 2);
            s.u2 = u53(w2.x, w2.y);
            s.u0 = u53(w2.z, w2.w);
            fp[q * ns + kl - 1] = make_frame(s.p.phi, s.p.cth, s.p.chi);
        }
    };
    if (net_atoms) {  // the sums of every own slice at its current orientation
        for (int q = 0; q < nrot; ++q)
            for (int c0 = wv * DA_SHORT; c0 < ns; c0 += nw * DA_SHORT) {
                const int nm = min(DA_SHORT, ns - c0);
                double so, sn;
                net_rows(q, nm, c0 + l + 1, l, false, so, sn);
                if (l < nm) sl[q * ns + c0 + l].V = sn;
                for (int i = 0; i < nm; ++i) {
                    const double v = exact_atoms(q, c0 + i + 1, fr[q * (ns + 2) + c0 + i + 1], 64);
                    if (l == 0) sl[q * ns + c0 + i].E = v;
                }
            }
    }
    __syncthreads();
    ahead(0, 0);
    ahead(1, 0);
    __syncthreads();
    const int nwords = 2 * nrot * (FRAME_D + 1);
    unsigned moved = 0;  // bit 2 parity + q: rotor q of the lane's slice (at most one of either parity: c0 is 0) was moved
#pragma unroll 1
    for (int h = 0; h < 2 * e.nsweep; ++h) {
        const int parity = h & 1, sw = h >> 1;
        const int nmoves = ns >> 1, mine = moves_of_wave(nmoves);  // of either parity: k0 and ns are even
        const bool trader = NP > 1 && (parity == 0 ? 0 : (nmoves - 1) % nw) == wv;  // has the move beside the neighbour
        if (trader && h > 0) {
            const int kn = parity == 0 ? 0 : ns + 1, ln = parity == 0 ? 0 : ns;
            for (int w = l; w < nwords; w += 64) {
                const unsigned v = rot3d_word(e.from(parity) + w, e.base + (unsigned)h, s_err);
                const int i = w >> 1;  // the double: frames first, then link densities
                double* d = i < nrot * FRAME_D ? reinterpret_cast<double*>(fr + (i / FRAME_D) * (ns + 2) + kn) + i % FRAME_D
                                               : Lk + (i - nrot * FRAME_D) * L + ln;
                reinterpret_cast<unsigned*>(d)[w & 1] = v;
            }
            wave_sync();
        }
#pragma unroll 1
        for (int q = 0; q < nrot; ++q) {  // rotor 1 sees rotor 0's move at its slice: the same wave's
#pragma unroll 1
            for (int c0 = 0; c0 < mine; c0 += DA_SHORT) {
                const int nm = min(DA_SHORT, mine - c0);
                const int kl = 2 * (wv + (c0 + min(j, nm - 1)) * nw) + parity + 1;
                Slice& s = sl[q * ns + kl - 1];
                // (1) the new links, and the exact stage-1 terms
                double rho;
                if (rotden_link(fr[q * (ns + 2) + kl - 1 + 2 * side], fp[q * ns + kl - 1], side, e.tab, rho)) err = 1;
                const double d2 = __shfl(rho, j), d3 = __shfl(rho, j + 32);
                double dvx = 0.0;
                if (net_atoms && nrot > 1) {
                    const double v = pair_change(q, kl);
                    dvx = __shfl(v, j) - __shfl(v, j + 32);
                }
                double dold = Lk[q * L + kl - 1] * Lk[q * L + kl];
                if (fabs(dold) < RZERO) dold = 0.0;
                if (dold < 0.0) dold = fabs(dold);
                double dnew = d2 * d3;
                if (fabs(dnew) < RZERO) dnew = 0.0;
                if (dnew < 0.0) dnew = fabs(dnew);
                const double ratio = (dold > RZERO) ? dnew / dold : 1.0;
                // (2) stage 0, then the network rows of the moves that passed it, listed first in lane
                // order (slot: a lane's place in that order, src: the lane whose move fills this place)
                const bool pass0 = l < nm && (ratio > 1.0 || ratio > s.u0);
                const unsigned long long m0 = __ballot(pass0);
                const int n0 = __popcll(m0), below = __popcll(m0 & ((1ull << l) - 1ull));
                const int slot = pass0 ? below : n0 + (l - below);
                const int src = __builtin_amdgcn_ds_permute(slot << 2, l);
                double so = 0.0, sn = 0.0;
                if (n0) {
                    net_rows(q, n0, kl, src, true, so, sn);
                    so = __shfl(so, slot);
                    sn = __shfl(sn, slot);
                }
                // (3) stage 1, the surrogate factor
                bool pass1 = false;
                double dvs = 0.0;
                if (pass0) {
                    if (net_atoms) so = s.V;
                    dvs = ys * (sn - so);
                    const double rd1 = exp(-rp.tau * (dvs + dvx));
                    pass1 = rd1 > 1.0 || rd1 > s.p.u;
                }
                // (4) stage 2: exact network-pair sums of the moves that passed
                double dve = 0.0, ex_new = 0.0;
                unsigned long long todo = __ballot(pass1);
                if (net_atoms) {
                    const int GL = items_x <= 32 ? 32 : 64;
                    while (todo) {
                        const int ja = __ffsll((long long)todo) - 1;
                        todo &= todo - 1;
                        const bool two = GL == 32 && todo;
                        const int jb = two ? __ffsll((long long)todo) - 1 : ja;
                        if (two) todo &= todo - 1;
                        const int klj = __shfl(kl, GL == 32 && side ? jb : ja);
                        const double v = exact_atoms(q, klj, fp[q * ns + klj - 1], GL);
                        const double va = __shfl(v, 0), vb = __shfl(v, 32);
                        if (l == ja || l == jb) {
                            ex_new = l == ja ? va : vb;
                            dve = ex_new - s.E;
                        }
                    }
                } else if (todo) {
                    const double v = pair_change(q, kl);
                    dve = __shfl(v, j) - __shfl(v, j + 32);
                }
                // (5) stage 2 and the update
                if (pass0) {
                    nnet += (unsigned long long)rpm;
                    if (pass1) {
                        ++npass;
                        const double rd2 = exp(-rp.tau * (dve - dvs));
                        if (rd2 > 1.0 || rd2 > s.u2) {
                            ++nacc;
                            const Frame& f = fp[q * ns + kl - 1];
                            fr[q * (ns + 2) + kl] = f;
                            s.phi = s.p.phi;
                            s.cth = s.p.cth;
                            s.chi = s.p.chi;
                            s.V = sn;
                            s.E = ex_new;
                            Lk[q * L + kl - 1] = d2;
                            Lk[q * L + kl] = d3;
                            if (NP == 1 && (kl == 1 || kl == ns)) {  // its own neighbour, as in rotor3d_ahead
                                fr[q * (ns + 2) + (kl == 1 ? ns + 1 : 0)] = f;
                                Lk[q * L + (kl == 1 ? ns : 0)] = kl == 1 ? d2 : d3;
                            }
                            moved |= 1u << (2 * parity + q);
                        }
                    }
                }
                wave_sync();
            }
        }
        if (trader) {  // publish the boundary slice; no wait for the stores, the reader checks every word
            const int kb = parity == 0 ? 1 : ns, lb = parity == 0 ? 0 : ns;
            for (int w = l; w < nwords; w += 64) {
                const int i = w >> 1;
                const double v = i < nrot * FRAME_D ? reinterpret_cast<const double*>(fr + (i / FRAME_D) * (ns + 2) + kb)[i % FRAME_D]
                                                    : Lk[(i - nrot * FRAME_D) * L + lb];
                __hip_atomic_store(e.mypub + parity * e.half_rec + w, rot3d_pack(v, w & 1, e.base + (unsigned)h + 1u), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (sw + 1 < e.nsweep) ahead(parity, sw + 1);
        lds_barrier();
        if (*s_err) break;  // as in rotor3d_ahead
    }
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
        if (!(moved >> i & 1)) continue;
        const int kl = 2 * (wv + l * nw) + (i >> 1) + 1, q = i & 1;
        const Slice& s = sl[q * ns + kl - 1];
        rot3d_store(e, e.at(q, k0 + kl - 1), s.phi, s.cth, s.chi, fr[q * (ns + 2) + kl]);
    }
}

// Longer parts: state in memory, everything of a move inside its half-sweep.
template <typename R>
__device__ __forceinline__ void rotor3d_da_long(const Rot3dEnv& e, const RotPart& pt, const Lut3D<R>& l3, MlpPacked* W, int* s_err,
                                                unsigned long long& nacc, unsigned long long& npass, unsigned long long& nnet,
                                                int& err) {
    const Rep& rp = e.rp;
    const int Prot = rp.Prot, RR = rp.RotRatio, nrot = rp.nrot;
    const int nat = rp.nl_atom;              // atoms come first: 0 .. nat-1
    const bool net_atoms = nat > 0;          // network pairs: rotor-atom, else rotor-rotor
    const int k0 = pt.k0, ns = pt.k1 - pt.k0, NP = pt.W;
    const int L = ns + 1;
    const long long rb0 = rp.rot_off;
    const double4* tab = e.tab;
    const double4* beads = e.beads;
    RotBead* rotb = e.rotb;
    Frame* frames = e.frames;
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, nw = blockDim.x >> 6;
    double* Lk = reinterpret_cast<double*>(W + 1);
    double* Vs = Lk + nrot * L;   // cached surrogate sums (rotor-atom network)
    double* Ex = Vs + nrot * ns;  // cached exact rotor-atom sums
    Frame* fnb = reinterpret_cast<Frame*>(Lk + ((nrot * L + 2 * nrot * ns + 1) & ~1));
    Frame* prop = fnb + 2 * nrot + wv * DA_MV;
    float* rowo = reinterpret_cast<float*>(fnb + 2 * nrot + nw * DA_MV) + wv * 32;
    constexpr int FD = FRAME_D;
    const int nwords = 2 * nrot * (FD + 1);
    const unsigned base = e.base;
    const uint32_t pass = e.pass;
    const double twopi = 2.0 * PI_D;
    const double ys = (double)W->ys;
    // network rows per move: RR x atoms (proposal only; the old sum is cached), or RR x other
    // rotors x (old, new)
    const int rpm = net_atoms ? RR * nat : RR * (nrot - 1) * 2;
    const int items_x = RR * nat;  // exact rotor-atom pairs of a slice
    auto own = [&](int q, int k) -> const Frame& { return frames[rb0 + (long long)q * Prot + k]; };
    for (int i = threadIdx.x; i < 2 * nrot; i += blockDim.x) {
        const int side = i / nrot, q = i - side * nrot;
        int k = side ? k0 + ns : k0 - 1;
        if (k < 0) k += Prot;
        if (k >= Prot) k -= Prot;
        fnb[i] = own(q, k);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nrot * L; i += blockDim.x) {
        const int q = i / L, kl = i - q * L;
        const Frame& fa = kl == 0 ? fnb[q] : own(q, k0 + kl - 1);
        const Frame& fb = kl == ns ? fnb[nrot + q] : own(q, k0 + kl);
        if (rotden_rho(fa, fb, tab, Lk[i])) err = 1;
    }
    // The network's rows for slices of rotor q, summed per slice in row order.  Entry j < nm of
    // the list is the move of lane src (src_j on lane j): its slice is that lane's kl_j and, for
    // the proposal rows, its frame prop[src]; sums of (old, new) rows return in so/sn on lane j.
    auto net_rows = [&](int q, int nm, int kl_j, int src_j, bool proposal, double& so, double& sn) {
        so = 0.0;
        sn = 0.0;
        const int total = nm * rpm;
        for (int b = 0; b < total; b += 32) {
            const int row = b + (l & 31);
            // the row's move and its slice, read from the move's lane with every lane active
            const int jj = min(row, total - 1) / rpm;
            const int sl = __shfl(src_j, jj);
            const int klr = __shfl(kl_j, sl);
            float f[MLP_IN] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (row < total) {
                const int idx = row - jj * rpm;
                const int k = k0 + klr - 1;
                const int gq = rp.nl_atom + q;
                if (net_atoms) {
                    const int s = idx / nat, a = idx - s * nat;
                    const int it = k * RR + s;
                    const double4 xa = bead(beads, rp, gq, it), xj = bead(beads, rp, a, it);
                    const Frame& fq = proposal ? prop[sl] : own(q, k);
                    mlp_pair_features(fq.m, fq.zn, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, f);
                } else {
                    const int which = idx & 1, rest = idx >> 1;
                    const int s = rest / (nrot - 1), pp = rest - s * (nrot - 1);
                    const int p = pp + (pp >= q);
                    const int it = k * RR + s;
                    const double4 xq = bead(beads, rp, gq, it), xp = bead(beads, rp, rp.nl_atom + p, it);
                    const Frame& fq = (proposal && which) ? prop[sl] : own(q, k);
                    mlp_rotor_pair_features(fq, own(p, k), xq.x, xq.y, xq.z, xp.x, xp.y, xp.z, f);
                }
#pragma unroll
                for (int c = 0; c < MLP_IN; ++c) f[c] = (f[c] - W->xm[c]) * W->xinv[c];
            }
            // an opaque zero offset keeps the weight reads inside the loop (hoisted out they
            // would hold ~130 registers of weights per lane)
            int z = 0;
            __asm__ volatile("" : "+s"(z));
            const float o = mlp_rows32(reinterpret_cast<const MlpPacked*>(reinterpret_cast<const char*>(W) + z), f);
            if (l < 32) rowo[l] = o;
            __builtin_amdgcn_wave_barrier();
            if (l < nm) {  // the rows of move l that fall in this batch, in row order
                const int r0 = max(l * rpm, b), r1 = min((l + 1) * rpm, b + 32);
                for (int rr = r0; rr < r1; ++rr) {
                    const int idx = rr - l * rpm;
                    const double v = (double)rowo[rr - b];
                    const bool moved = net_atoms || (idx & 1);
                    sn += moved ? v : 0.0;
                    so += moved ? 0.0 : v;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    };
    // exact rotor-atom sum of rotor q at local slice kl with frame f, over the whole wave
    auto exact_atoms = [&](int q, int kl, const Frame& f) -> double {
        const int k = k0 + kl - 1, gq = rp.nl_atom + q;
        double e = 0.0;
        for (int i = l; i < items_x; i += 64) {
            const int s = i / nat, a = i - s * nat;
            const int it = k * RR + s;
            const double4 xa = bead(beads, rp, gq, it), xj = bead(beads, rp, a, it);
            e += (double)vcord_v<R>(l3, f, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z);
        }
        return wave_sum(e);
    };
    // cached sums of every own slice at its current orientation (rotor-atom network only)
    if (net_atoms) {
        for (int q = 0; q < nrot; ++q) {
            for (int c0 = wv * DA_MV; c0 < ns; c0 += nw * DA_MV) {
                const int nm = min(DA_MV, ns - c0);
                double so, sn;
                net_rows(q, nm, c0 + l + 1, l, false, so, sn);
                if (l < nm) Vs[q * ns + c0 + l] = sn;
                for (int j = 0; j < nm; ++j) {
                    const double e = exact_atoms(q, c0 + j + 1, own(q, k0 + c0 + j));
                    if (l == 0) Ex[q * ns + c0 + j] = e;
                }
            }
        }
    }
    __syncthreads();
    for (int sw = 0; sw < e.nsweep; ++sw) {
        const uint32_t jsweep = e.sweep(sw);
        for (int parity = 0; parity < 2; ++parity) {
            const unsigned h = 2u * (unsigned)sw + (unsigned)parity;
            if (!(sw == 0 && parity == 0)) {
                if (NP == 1) {
                    // one part: the boundary slices are its own, moved in the last half
                    if (threadIdx.x < nrot) {
                        const int q = threadIdx.x;
                        if (parity == 0) {
                            fnb[q] = own(q, Prot - 1);
                            Lk[q * L] = Lk[q * L + ns];
                        } else {
                            fnb[nrot + q] = own(q, 0);
                            Lk[q * L + ns] = Lk[q * L];
                        }
                    }
                } else {
                    unsigned* dstf = reinterpret_cast<unsigned*>(fnb + (parity == 0 ? 0 : nrot));
                    for (int w = threadIdx.x; w < nwords; w += blockDim.x) {
                        const unsigned v = rot3d_word(e.from(parity) + w, base + h, s_err);
                        const int i = w >> 1;
                        if (i < nrot * FD) dstf[w] = v;
                        else reinterpret_cast<unsigned*>(&Lk[(i - nrot * FD) * L + (parity == 0 ? 0 : ns)])[w & 1] = v;
                    }
                }
                __syncthreads();
                if (*s_err) {  // a wait gave up: leave at once (see rotor3d_ahead)
                    sw = e.nsweep;
                    break;
                }
            }
            const int nmoves = (ns - parity + 1) / 2;  // k0 is even: local slice kl has parity (kl - 1) & 1
            const int mine = nmoves > wv ? (nmoves - wv + nw - 1) / nw : 0;  // moves wv, wv + nw, ...
            for (int q = 0; q < nrot; ++q) {
                const int gq = rp.nl_atom + q;
                for (int c0 = 0; c0 < mine; c0 += DA_MV) {
                    const int nm = min(DA_MV, mine - c0);
                    // (1) proposal of move l
                    const int mv = wv + (c0 + l) * nw;
                    const int kl = 2 * mv + parity + 1, k = k0 + kl - 1;
                    const long long ik = rb0 + (long long)q * Prot + k;
                    double cost = 0.0, phi = 0.0, chi = 0.0, ratio = 1.0, d2 = 0.0, d3 = 0.0, dvx = 0.0;
                    double rand4 = 0.0, rand5 = 0.0, rand6 = 0.0;
                    RotBead cur{};
                    if (l < nm) {
                        cur = rotb[ik];
                        const uint4 w0 = draw(e.seed, rp.key, pass, K_ROT3D, jsweep, (uint32_t)gq, (uint32_t)k, 0);
                        const uint4 w1 = draw(e.seed, rp.key, pass, K_ROT3D, jsweep, (uint32_t)gq, (uint32_t)k, 1);
                        const uint4 w2 = draw(e.seed, rp.key, pass, K_ROT3D, jsweep, (uint32_t)gq, (uint32_t)k, 2);
                        const double rand1 = u53(w0.x, w0.y), rand2 = u53(w0.z, w0.w), rand3 = u53(w1.x, w1.y);
                        rand4 = u53(w1.z, w1.w);
                        rand5 = u53(w2.x, w2.y);
                        rand6 = u53(w2.z, w2.w);
                        cost = cur.cth + rp.rtstep * (rand1 - 0.5);
                        phi = cur.phi + twopi * (rp.rtstep * (rand2 - 0.5));
                        chi = cur.chi + twopi * (rp.rtstep * (rand3 - 0.5));
                        if (phi < 0.0) phi = twopi + phi;
                        if (chi < 0.0) chi = twopi + chi;
                        phi = fmod_near(phi, twopi);
                        chi = fmod_near(chi, twopi);
                        if (cost > 1.0) cost = 2.0 - cost;
                        if (cost < -1.0) cost = -2.0 - cost;
                        const Frame fn = make_frame(phi, cost, chi);
                        prop[l] = fn;
                        const Frame& fa = kl == 1 ? fnb[q] : own(q, k - 1);
                        const Frame& fb = kl == ns ? fnb[nrot + q] : own(q, k + 1);
                        if (rotden_rho(fa, fn, tab, d2)) err = 1;
                        if (rotden_rho(fn, fb, tab, d3)) err = 1;
                        double dold = Lk[q * L + kl - 1] * Lk[q * L + kl];
                        if (fabs(dold) < RZERO) dold = 0.0;
                        if (dold < 0.0) dold = fabs(dold);
                        double dnew = d2 * d3;
                        if (fabs(dnew) < RZERO) dnew = 0.0;
                        if (dnew < 0.0) dnew = fabs(dnew);
                        ratio = (dold > RZERO) ? dnew / dold : 1.0;
                        if (net_atoms) {  // rotor-rotor pairs exact in stage 1
                            const Frame& fo = own(q, k);
                            for (int p = 0; p < nrot; ++p) {
                                if (p == q) continue;
                                for (int s = 0; s < RR; ++s) {
                                    const int it = k * RR + s;
                                    const double4 xa = bead(beads, rp, gq, it), xp = bead(beads, rp, rp.nl_atom + p, it);
                                    const Frame& fp = own(p, k);
                                    dvx += caleng_v(xa.x, xa.y, xa.z, xp.x, xp.y, xp.z, fn, fp) -
                                           caleng_v(xa.x, xa.y, xa.z, xp.x, xp.y, xp.z, fo, fp);
                                }
                            }
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                    // (2) stage 0, the density factor alone; the network rows of the moves that
                    // pass it, listed first in lane order (slot: a lane's place in that order,
                    // src: the lane whose move fills this lane's place)
                    const bool pass0 = l < nm && (ratio > 1.0 || ratio > rand6);
                    const unsigned long long m0 = __ballot(pass0);
                    const int n0 = __popcll(m0);
                    const int below = __popcll(m0 & ((1ull << l) - 1ull));
                    const int slot = pass0 ? below : n0 + (l - below);
                    const int src = __builtin_amdgcn_ds_permute(slot << 2, l);
                    double so = 0.0, sn = 0.0;
                    if (n0) {
                        net_rows(q, n0, kl, src, true, so, sn);
                        so = __shfl(so, slot);
                        sn = __shfl(sn, slot);
                    }
                    // (3) stage 1, the surrogate factor
                    bool pass1 = false;
                    double dvs = 0.0;
                    if (pass0) {
                        if (net_atoms) so = Vs[q * ns + kl - 1];
                        dvs = ys * (sn - so);
                        const double rd1 = exp(-rp.tau * (dvs + dvx));
                        pass1 = rd1 > 1.0 || rd1 > rand4;
                    }
                    // (4) stage 2: exact network-pair sums of the moves that passed
                    double dve = 0.0, ex_new = 0.0;
                    if (net_atoms) {
                        unsigned long long todo = __ballot(pass1);
                        while (todo) {
                            const int jj = __ffsll((long long)todo) - 1;
                            todo &= todo - 1;
                            const int klj = __shfl(kl, jj);
                            const double e = exact_atoms(q, klj, prop[jj]);
                            if (l == jj) {
                                ex_new = e;
                                dve = e - Ex[q * ns + klj - 1];
                            }
                        }
                    } else if (pass1) {
                        const Frame& fo = own(q, k);
                        for (int p = 0; p < nrot; ++p) {
                            if (p == q) continue;
                            for (int s = 0; s < RR; ++s) {
                                const int it = k * RR + s;
                                const double4 xa = bead(beads, rp, gq, it), xp = bead(beads, rp, rp.nl_atom + p, it);
                                const Frame& fp = own(p, k);
                                dve += caleng_v(xa.x, xa.y, xa.z, xp.x, xp.y, xp.z, prop[l], fp) -
                                       caleng_v(xa.x, xa.y, xa.z, xp.x, xp.y, xp.z, fo, fp);
                            }
                        }
                    }
                    // (5) stage 2 and the update
                    if (pass0) {
                        nnet += (unsigned long long)rpm;
                        if (pass1) {
                            ++npass;
                            const double rd2 = exp(-rp.tau * (dve - dvs));
                            if (rd2 > 1.0 || rd2 > rand5) {
                                ++nacc;
                                RotBead b = cur;
                                b.cth = cost;
                                b.phi = phi;
                                b.chi = chi;
                                store_axis(b, phi, cost);
                                rotb[ik] = b;
                                frames[ik] = prop[l];
                                Lk[q * L + kl - 1] = d2;
                                Lk[q * L + kl] = d3;
                                if (net_atoms) {
                                    Vs[q * ns + kl - 1] = sn;
                                    Ex[q * ns + kl - 1] = ex_new;
                                }
                            }
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                }
                __syncthreads();  // rotor q + 1 sees rotor q's moves at the same slices
            }
            // publish the boundary slice this half moved (k_rotor3d_parts' record)
            if (NP > 1) {
                const int ks = parity == 0 ? k0 : k0 + ns - 1;
                for (int w = threadIdx.x; w < nwords; w += blockDim.x) {
                    const int i = w >> 1;
                    const double v = i < nrot * FD ? reinterpret_cast<const double*>(&own(i / FD, ks))[i % FD]
                                                   : Lk[(i - nrot * FD) * L + (parity == 0 ? 0 : ns)];
                    __hip_atomic_store(e.mypub + parity * e.half_rec + w, rot3d_pack(v, w & 1, base + h + 1u), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
    }
}

template <typename R>
__global__ __launch_bounds__(256) void k_rotor3d_da(const Rep* __restrict__ reps, Mut* __restrict__ mut,
                                                    const double4* __restrict__ beads, RotBead* __restrict__ rotb,
                                                    Frame* __restrict__ frames, Tables T, Tables3 T3,
                                                    const RotPart* __restrict__ parts, unsigned* __restrict__ flags,
                                                    unsigned long long* __restrict__ pub, int pub_stride, Run run,
                                                    const MlpPacked* __restrict__ Wg) {
    extern __shared__ uint4 mlp_lds[];
    MlpPacked* W = reinterpret_cast<MlpPacked*>(mlp_lds);
    __shared__ unsigned long long red_a[4], red_p[4], red_n[4];
    __shared__ int s_err;
    const RotPart pt = parts[blockIdx.x];
    if (pt.r < 0) return;  // padding of the XCD-ordered grid
    const int r = pt.r;
    const Rep& rp = reps[r];
    if (!rotor3d_turn(rp, run)) return;
    const int ns = pt.k1 - pt.k0, NP = pt.W, RR = rp.RotRatio, nrot = rp.nrot;
    const bool net_atoms = rp.nl_atom > 0;
    const Rot3dEnv e = rotor3d_env(rp, mut[r].pass, beads, rotb, frames, T3, pt, flags, pub, pub_stride, run);
    const Lut3D<R> l3 = lut3d<R>(T3, rp.pot3d_id);
    if (threadIdx.x == 0) s_err = 0;
    unsigned long long nacc = 0, npass = 0, nnet = 0;
    int err = 0;
    mlp_stage(Wg, W);
    __syncthreads();
    if (nrot * ns <= ROT3D_AHEAD) rotor3d_da_short<R>(e, pt, l3, W, &s_err, nacc, npass, nnet, err);
    else rotor3d_da_long<R>(e, pt, l3, W, &s_err, nacc, npass, nnet, err);
    if (threadIdx.x == 0 && NP > 1)  // every part of the chain ran the same halves
        __hip_atomic_store(flags + pt.fbase + pt.w, e.base + 2u * (unsigned)e.nsweep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (err) atomicOr(&mut[r].err, 4);
    const unsigned long long sa = block_sum(nacc, red_a);
    const unsigned long long sp = block_sum(npass, red_p);
    const unsigned long long sn_ = block_sum(nnet, red_n);
    if (threadIdx.x == 0) {
        const int rtype = rp.imtype, items_x = RR * rp.nl_atom;
        if (s_err) atomicOr(&mut[r].err, s_err);
        const unsigned long long moves = (unsigned long long)e.nsweep * ns * nrot;
        atomicAdd(&mut[r].total[rtype][2], moves);
        atomicAdd(&mut[r].accep[rtype][2], sa);
        atomicAdd(&mut[r].da[0], moves);
        atomicAdd(&mut[r].da[1], sp);
        atomicAdd(&mut[r].da[2], sa);
        // exact network-pair evaluations of the moves that reached stage 2
        atomicAdd(&mut[r].pair_evals[2], (net_atoms ? 1ull : 2ull) * sp * (unsigned long long)(net_atoms ? items_x : RR * (nrot - 1)));
        atomicAdd(&mut[r].surrogate_evals, sn_);
    }
}

// Training rows of the surrogate from the current configuration of replica r, for the pairs the
// delayed-acceptance move gives the network.  With atoms: each (rotor q, rotor slice k,
// translational slice it of k, atom a) gives the body-frame features of the pair and its exact
// energy (vcord on the 3D table in FP64, PotRotE3D's atom term); row order q, k, it, a.  Without
// atoms: each (rotor q, slice k, translational slice it, other rotor p) gives the rotor-pair
// features and the TIP4P energy of caleng (PotRotE3D's rotor term).
__global__ void k_surrogate_collect(const Rep* __restrict__ reps, const double4* __restrict__ beads,
                                    const Frame* __restrict__ frames, Tables3 T3, int r, float* __restrict__ X,
                                    float* __restrict__ y, int nrows) {
    const Rep& rp = reps[r];
    const int RR = rp.RotRatio, nat = rp.nl_atom, nrot = rp.nrot, Prot = rp.Prot;
    const int npart = nat > 0 ? nat : nrot - 1;  // partners per translational slice
    const Lut3D<double> l3 = lut3d<double>(T3, rp.pot3d_id);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nrows; i += gridDim.x * blockDim.x) {
        const int per_q = Prot * RR * npart;
        const int q = i / per_q, rem0 = i - q * per_q;
        const int k = rem0 / (RR * npart), rem = rem0 - k * (RR * npart);
        const int it = k * RR + rem / npart, jp = rem % npart;
        const int gq = nat + q;
        const double4 xa = bead(beads, rp, gq, it);
        const Frame& f = frames[rp.rot_off + (long long)q * Prot + k];
        float fe[MLP_IN];
        double e;
        if (nat > 0) {
            const double4 xj = bead(beads, rp, jp, it);
            mlp_pair_features(f.m, f.zn, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z, fe);
            e = (double)vcord_v<double>(l3, f, xa.x, xa.y, xa.z, xj.x, xj.y, xj.z);
        } else {
            const int p = jp + (jp >= q);
            const double4 xp = bead(beads, rp, nat + p, it);
            const Frame& fp = frames[rp.rot_off + (long long)p * Prot + k];
            mlp_rotor_pair_features(f, fp, xa.x, xa.y, xa.z, xp.x, xp.y, xp.z, fe);
            e = caleng_v(xa.x, xa.y, xa.z, xp.x, xp.y, xp.z, f, fp);
        }
        for (int c = 0; c < MLP_IN; ++c) X[(long long)i * MLP_IN + c] = fe[c];
        y[i] = (float)e;
    }
}

// ------------------------------------------------------------------------- read-back
// Counters and the first `most` samples of every replica into host memory that the device writes:
// one launch a run, instead of two copies a replica and getter at 10 to 15 us each.
__global__ __launch_bounds__(64) void k_read_back(const Mut* __restrict__ mut, const Rep* __restrict__ reps,
                                                  const double* __restrict__ samples, int most, Mut* __restrict__ hmut,
                                                  double* __restrict__ hsamples) {
    const int r = blockIdx.x;
    static_assert(sizeof(Mut) % 8 == 0, "copied by words");
    const unsigned long long* src = reinterpret_cast<const unsigned long long*>(mut + r);
    unsigned long long* dst = reinterpret_cast<unsigned long long*>(hmut + r);
    for (int i = threadIdx.x; i < (int)(sizeof(Mut) / 8); i += 64) dst[i] = src[i];
    const int n = 8 * (int)min(mut[r].nsamples, (unsigned)most);
    for (int i = threadIdx.x; i < n; i += 64) hsamples[(long long)r * most * 8 + i] = samples[reps[r].sample_off + i];
}

// A replica's n beads as [3][n] and its m rotor slices as [6][m] (phi, cos theta, chi, axis)
__global__ __launch_bounds__(256) void k_pack_state(const double4* __restrict__ beads, int n, const RotBead* __restrict__ rotb,
                                                    int m, double* __restrict__ out) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n + m; i += gridDim.x * 256) {
        if (i < n) {
            const double4 b = beads[i];
            out[i] = b.x;
            out[n + i] = b.y;
            out[2 * n + i] = b.z;
        } else {
            const RotBead b = rotb[i - n];
            double* o = out + 3 * n + (i - n);
            o[0] = b.phi;
            o[m] = b.cth;
            o[2 * m] = b.chi;
            o[3 * m] = b.nx;
            o[4 * m] = b.ny;
            o[5 * m] = b.nz;
        }
    }
}

__global__ void k_clear_samples(Mut* mut, int n) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) mut[r].nsamples = 0;
}

// ------------------------------------------------------------------------- end of pass
__global__ void k_pass_end(Mut* mut, int n) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) mut[r].pass += 1;
}

// ------------------------------------------------------------------------- estimators
// One workgroup per (replica, tile of est_ts slices).  All atoms' beads on the tile's slices and
// one slice past it are staged in LDS once; lanes then take every pair at every slice of the
// tile, the pairs enumerated as (a, a + d mod N) for d = 1 .. N/2 so that a tile has the same
// work at any N.  g(r) is counted in LDS and added to the replica's bins once per tile.
// part[row_off + tile] = (pair potential of the tile, its kinetic links / (4 beta lambda)).
// The potential and the bins follow GetPotEnergy_Densities (mc_estim.cc:500-687), the kinetic
// term GetKinEnergy (mc_estim.cc:876-937).
template <typename R, int FAM, bool MI>
__global__ __launch_bounds__(256) void k_est_tiles(const Rep* __restrict__ reps, const double4* __restrict__ beads,
                                                   const RotBead* __restrict__ rotb, const Frame* __restrict__ frames,
                                                   Tables T, Tables3 T3, const int2* __restrict__ tiles,
                                                   unsigned* __restrict__ hist, double2* __restrict__ part) {
    extern __shared__ DYNAMIC_LDS double smem[];
    __shared__ double red[16];
    __shared__ unsigned g1s[BINSR];
    const int2 tk = tiles[blockIdx.x];
    const Rep& rp = reps[tk.x];
    const int N = rp.natoms, P = rp.P, TS = rp.est_ts, lts = __ffs(TS) - 1;
    const int s0 = tk.y * TS, nts = min(TS, P - s0), W = nts + 1;
    double* lx = smem;
    double* ly = lx + N * W;
    double* lz = ly + N * W;
    double* ax = lz + N * W;  // rotor axis at the tile's slices
    double* ay = ax + TS;
    double* az = ay + TS;
    int* kind = reinterpret_cast<int*>(az + TS);  // type | molecule kind << 8
    for (int i = threadIdx.x; i < N * W; i += blockDim.x) {
        const int a = i / W, w = i - a * W;
        const int it = s0 + w < P ? s0 + w : s0 + w - P;
        const double4 b = bead(beads, rp, a, it);
        lx[i] = b.x;
        ly[i] = b.y;
        lz[i] = b.z;
    }
    for (int w = threadIdx.x; w < nts; w += blockDim.x) rotor_axis(rotb, rp, s0 + w, ax[w], ay[w], az[w]);
    for (int a = threadIdx.x; a < N; a += blockDim.x) {
        const int t = type_of(rp, a);
        kind[a] = t | (rp.tmol[t] << 8);
    }
    unsigned* g1 = hist ? hist + rp.hist_off : nullptr;
    unsigned* g2h = g1 ? g1 + BINSR : nullptr;
    unsigned* g3 = (g1 && rp.h3_off >= 0) ? g1 + rp.h3_off : nullptr;
    for (int i = threadIdx.x; i < BINSR; i += blockDim.x) g1s[i] = 0u;
    __syncthreads();
    const double* box = MI && rp.minimage ? rp.box : nullptr;  // MINIMAGE (not with a rotating linear rotor)
    double kin = 0.0;
    const Lut1D<R> l1 = lut1d<R>(T, rp.pot1d_id);
    const Lut2D<R> l2 = lut2d<R>(T, rp.pot2d_id);
    const double drad = MAX_RADIUS / (double)BINSR;
    const double dth = 3.14159265358979323846 / (double)(BINST - 1);
    const double dch = 2.0 * 3.14159265358979323846 / (double)(BINSC - 1);
    const int npairs = N * (N - 1) / 2;
    const float invN = 1.0f / (float)N;
    double pot = 0.0;
    // kinetic links (a, s) - (a, s + 1), then the pairs; the minimum image as its own instance
    // of the loops, so the plain one is unchanged
    auto tile_sums = [&](auto mi_c) {
        const double* bx = decltype(mi_c)::value ? box : nullptr;
        for (int i = threadIdx.x; i < N * nts; i += blockDim.x) {
            const int a = i / nts, w = i - a * nts;
            const int j = a * W + w;
            const double dx = nearest_image(lx[j] - lx[j + 1], bx, 0), dy = nearest_image(ly[j] - ly[j + 1], bx, 1),
                         dz = nearest_image(lz[j] - lz[j + 1], bx, 2);
            kin += (dx * dx + dy * dy + dz * dz) / (4.0 * rp.beta * rp.lambda[kind[a] & 255]);
        }
        for (int i = threadIdx.x; i < (npairs << lts); i += blockDim.x) {
            const int w = i & (TS - 1);
            if (w >= nts) continue;
            const int p = i >> lts;
            // p = N (d - 1) + a; the float quotient is exact while N^2 < 2^23
            const int d1 = N < 2896 ? (int)(((float)p + 0.5f) * invN) : p / N;
            const int a0 = p - d1 * N;
            int a1 = a0 + d1 + 1;
            if (a1 >= N) a1 -= N;
            const int k0 = kind[a0], k1 = kind[a1];
            const int t0 = k0 & 255, t1 = k1 & 255, m0 = k0 >> 8, m1 = k1 >> 8;
            const int j0 = a0 * W + w, j1 = a1 * W + w;
            const double ex = nearest_image(lx[j0] - lx[j1], bx, 0), ey = nearest_image(ly[j0] - ly[j1], bx, 1),
                         ez = nearest_image(lz[j0] - lz[j1], bx, 2);
            const R dx = (R)ex, dy = (R)ey, dz = (R)ez;
            const R rr = sqrt(dx * dx + dy * dy + dz * dz);
            if constexpr (FAM == 1) {
                if (m0 == 2 || m1 == 2) {  // mc_estim.cc:582-672: vcord or caleng
                    const Lut3D<R> l3 = lut3d<R>(T3, rp.pot3d_id);
                    const int it = s0 + w;
                    const Frame& f0 = frame_at(frames, rp, m0 == 2 ? a0 : rp.nl_atom, it);
                    const Frame& f1 = frame_at(frames, rp, m1 == 2 ? a1 : rp.nl_atom, it);
                    pot += pair_nl<R>(l1, l1.k, l3, m0 == 2, m1 == 2, lx[j0], ly[j0], lz[j0], lx[j1], ly[j1], lz[j1], f0, f1);
                    if (g3 && m0 != m1) {  // bin_3Ddensity of vcord's FP64 geometry (mc_estim.cc:637,1252-1273)
                        double rad, the, chi;
                        if (m0 == 2) vcord_geometry(f0, lx[j0], ly[j0], lz[j0], lx[j1], ly[j1], lz[j1], rad, the, chi);
                        else vcord_geometry(f1, lx[j1], ly[j1], lz[j1], lx[j0], ly[j0], lz[j0], rad, the, chi);
                        const int br = (int)floor(rad / drad);
                        if (br < BINSR && br >= 0) {
                            const int bt = (int)floor(the / dth);
                            if (bt < BINST && bt >= 0) {
                                const int bc = (int)floor(chi / dch);
                                if (bc < BINSC && bc >= 0) atomicAdd(&g3[(br * BINST + bt) * BINSC + bc], 1u);
                            }
                        }
                    }
                    continue;
                }
            }
            if (m0 == 1 || m1 == 1) {  // axis to the partner: from the rotor to the atom
                const double nx = ax[w], ny = ay[w], nz = az[w];
                R cost = ((R)nx * dx + (R)ny * dy + (R)nz * dz) / rr;
                if (m0 == 1) cost = -cost;
                pot += (double)lpot2d<R>(l2, rr, cost);
                if (g2h) {  // bins from FP64 geometry, as bin_2Ddensity gets it (mc_estim.cc:1233-1250)
                    const double rd = sqrt(ex * ex + ey * ey + ez * ez);
                    double cd = (nx * ex + ny * ey + nz * ez) / rd;
                    if (m0 == 1) cd = -cd;
                    const int br = (int)floor(rd / drad);
                    if (br < BINSR && br >= 0) {
                        const int bt = (int)floor(acos(cd) / dth);
                        if (bt < BINST && bt >= 0) atomicAdd(&g2h[br * BINST + bt], 1u);
                    }
                }
            } else if (t0 == t1 && m0 == 0) {
                pot += (double)spot1d<R>(l1, l1.k, rr);
                if (g1) {  // bin_1Ddensity (mc_estim.cc:1275-1286) on the FP64 distance
                    const int br = (int)floor(sqrt(ex * ex + ey * ey + ez * ez) / drad);
                    if (br < BINSR && br >= 0) atomicAdd(&g1s[br], 1u);
                }
            }
        }
    };
    if constexpr (MI) {
        if (box) tile_sums(std::integral_constant<bool, true>{});
        else tile_sums(std::integral_constant<bool, false>{});
    } else {
        tile_sums(std::integral_constant<bool, false>{});
    }
    const double sp = block_sum(pot, red);
    const double sk = block_sum(kin, red);
    if (g1)
        for (int i = threadIdx.x; i < BINSR; i += blockDim.x)
            if (g1s[i]) atomicAdd(&g1[i], g1s[i]);
    if (threadIdx.x == 0) part[rp.row_off + tk.y] = make_double2(sp, sk);
}

// out (if not null) receives 8 doubles per replica; otherwise the sample ring.
__global__ __launch_bounds__(256) void k_est_final(const Rep* __restrict__ reps, Mut* __restrict__ mut,
                                                   const RotBead* __restrict__ rotb, const Frame* __restrict__ frames,
                                                   Tables T, Tables3 T3,
                                                   const int* __restrict__ replist, const double2* __restrict__ rows,
                                                   double* __restrict__ samples, int sample_cap, double* __restrict__ out,
                                                   unsigned* __restrict__ hist) {
    __shared__ double red[16];
    const int r = replist[blockIdx.x];
    const Rep& rp = reps[r];
    const int N = rp.natoms, P = rp.P;
    // rotational energy, GetRotEnergy mc_estim.cc:939-987
    double srot = 0.0, esq = 0.0, term = 0.0;
    if (rp.rotkind == 1 && rp.rot_atom >= 0 && rp.rotdens >= 0) {
        const long long rbase = rp.rot_off + (long long)(rp.rot_atom - rp.tbegin[rp.imtype]) * rp.Prot;
        double a1 = 0, a2 = 0, a3 = 0;
        for (int k = threadIdx.x; k < rp.Prot; k += blockDim.x) {
            RotBead b0 = rotb[rbase + k], b1 = rotb[rbase + (k + 1) % rp.Prot];
            double p0 = b0.nx * b1.nx + b0.ny * b1.ny + b0.nz * b1.nz;
            double rd = rot_spline(T, rp.rotdens, p0, 0);
            double de = rot_spline(T, rp.rotdens, p0, 1);
            if (fabs(rd) > RZERO) a1 += de / rd;
            a2 += (de / rd) * (de / rd);
            a3 += rot_spline(T, rp.rotdens, p0, 2) / rd;
        }
        srot = block_sum(a1, red);
        term = block_sum(a2, red);
        esq = block_sum(a3, red);
    }
    if (rp.rotkind == 2 && rp.rot3d_id >= 0) {  // GetRotE3D mc_estim.cc:989-1096, per rotor
        const double4* tab = T3.r3 + (long long)rp.rot3d_id * 3 * ROT3D_SIZE;
        // relative Euler angle bins (mc_estim.cc:1046-1058): theta by pi/49, phi and chi by 2 pi/99
        unsigned* hr = (hist && rp.hrel_off >= 0) ? hist + rp.hist_off + rp.hrel_off : nullptr;
        const double dth = PI_D / (double)(BINST - 1), dch = 2.0 * PI_D / (double)(BINSC - 1);
        for (int q = 0; q < rp.nrot; ++q) {
            const long long fb = rp.rot_off + (long long)q * rp.Prot;
            double a1 = 0, a2 = 0, a3 = 0;
            for (int k = threadIdx.x; k < rp.Prot; k += blockDim.x) {
                double rho, er, es, rel[3];
                rotden_frames(frames[fb + k], frames[fb + (k + 1) % rp.Prot], tab, rho, er, es, hr ? rel : nullptr);
                if (hr) {
                    const int bt = (int)floor(rel[1] / dth);
                    if (bt < BINST && bt >= 0) atomicAdd(&hr[bt], 1u);
                    const int bp = (int)floor(rel[0] / dch);
                    if (bp < BINSC && bp >= 0) atomicAdd(&hr[BINST + bp], 1u);
                    const int bc = (int)floor(rel[2] / dch);
                    if (bc < BINSC && bc >= 0) atomicAdd(&hr[BINST + BINSC + bc], 1u);
                }
                a1 += er;
                a2 += es;
                a3 += er * er;
            }
            const double n = (double)rp.Prot;
            srot += block_sum(a1, red) / n;
            esq += block_sum(a2, red) / (n * n);
            term += block_sum(a3, red) / (n * n);
        }
    }
    if (threadIdx.x == 0) {
        double r2avr = 0.0, spot = 0.0;
        const int ntiles = (P + rp.est_ts - 1) / rp.est_ts;
        for (int a = 0; a < ntiles; ++a) {
            double2 v = rows[rp.row_off + a];
            spot += v.x;
            r2avr += v.y;
        }
        spot /= (double)P;
        double skin = (double)P * rp.T * (0.5 * (double)(3 * N) - r2avr);
        double n3 = (double)(3 * N);
        double a = n3 * 0.5 / rp.tau - skin - spot - srot;
        double sCv = -0.5 * n3 / (rp.beta * rp.tau) - a * a + (2.0 / rp.beta) * (0.5 * n3 / rp.tau - skin) + term - esq;
        double b = n3 * 0.5 / rp.tau - skin;
        double sCvt = -0.5 * n3 / (rp.beta * rp.tau) - b * b + (2.0 / rp.beta) * (0.5 * n3 / rp.tau - skin);
        double sCvr = -srot * srot + term - esq;
        double rec[8] = {skin, spot, srot, esq, sCv, sCvt, sCvr, term};
        double* dst = nullptr;
        if (out) dst = out + 8 * r;
        else if (samples) {
            unsigned ns = mut[r].nsamples;
            if ((int)ns < sample_cap) dst = samples + rp.sample_off + 8ll * ns;
            mut[r].nsamples = ns + 1;
        }
        if (dst)
            for (int q = 0; q < 8; ++q) dst[q] = rec[q];
        atomicAdd(&mut[r].pair_evals[3], (unsigned long long)N * (N - 1) / 2 * P);
    }
}

// ------------------------------------------------------------------------- PotEnergy(atom,pos,it)
// A group of POT_LANES lanes per query, partners in turn.  Queries name replicas and slices in any
// order, so every partner's bead is a line of its own from L2: what bounds the batch is how many such
// reads are in flight.  With a lane per query 100003 queries of 20 to 60 partners were 1.5 waves per
// SIMD and took 72 us, and a small batch the latency of all partners in turn; the whole call, copies
// and allocations with it, went from 363 to 354 us.
constexpr int POT_LANES = 8;
template <typename R>
__global__ __launch_bounds__(256) void k_pot_slice(const Rep* __restrict__ reps, const double4* __restrict__ beads,
                            const RotBead* __restrict__ rotb, const Frame* __restrict__ frames, Tables T, Tables3 T3, int nq,
                            const int* __restrict__ qrep,
                            const int* __restrict__ qatom, const int* __restrict__ qit, const double* __restrict__ qpos,
                            double* __restrict__ out) {
    const int l = threadIdx.x % POT_LANES;
    for (long long q = blockIdx.x * (256ll / POT_LANES) + threadIdx.x / POT_LANES; q < nq; q += gridDim.x * (256ll / POT_LANES)) {
        const Rep& rp = reps[qrep[q]];
        int a = qatom[q], it = qit[q];
        const Lut1D<R> l1 = lut1d<R>(T, rp.pot1d_id);
        const Lut2D<R> l2 = lut2d<R>(T, rp.pot2d_id);
        double nx, ny, nz;
        rotor_axis(rotb, rp, it, nx, ny, nz);
        const double* box = rp.minimage ? rp.box : nullptr;
        double s = 0.0;
        for (int j = l; j < rp.natoms; j += POT_LANES) {
            if (j == a) continue;
            double4 xj = bead(beads, rp, j, it);
            if (rp.fam == 1) {
                const bool ra = rp.nl_atom >= 0 && a >= rp.nl_atom, rj = rp.nl_atom >= 0 && j >= rp.nl_atom;
                const Lut3D<R> l3 = lut3d<R>(T3, rp.pot3d_id);
                s += pair_nl<R>(l1, l1.k, l3, ra, rj, qpos[3 * q], qpos[3 * q + 1], qpos[3 * q + 2], xj.x, xj.y, xj.z,
                                frame_at(frames, rp, ra ? a : rp.nl_atom, it), frame_at(frames, rp, rj ? j : rp.nl_atom, it),
                                box);
            } else {
                s += (double)pair_v<R>(l1, l1.k, l2, a == rp.lin_atom, j == rp.lin_atom, qpos[3 * q], qpos[3 * q + 1],
                                       qpos[3 * q + 2], xj.x, xj.y, xj.z, nx, ny, nz, box);
            }
        }
        s = group_sum(s, POT_LANES);
        if (l == 0) out[q] = s;
    }
}

}  // namespace pimc
