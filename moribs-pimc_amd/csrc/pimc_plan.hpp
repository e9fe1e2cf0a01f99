// pimc_plan.hpp -- host-side checks and launch plans that need no device: the validation of a
// replica description, and the split of linear-rotor chains into workgroups.  Plain C++ so
// that the library can run them without a GPU (pimc_check_replica, pimc_plan_rotor_parts).
#pragma once
#include "../../include/moribs_pimc.h"
#include <algorithm>
#include <functional>
#include <string>
#include <vector>

namespace pimc {

// A rotor chain's slice range [k0, k1) run by one workgroup: part w of the W parts of replica
// r, whose exchange flags start at fbase.  Also the slice ranges of the split centroid move.
struct RotPart {
    int r, k0, k1, w, W, fbase, pad0, pad1;
};

// The input checks of MCInit and IOReadParams that apply to the sampled path (mc_setup.cc:384-
// 398, mc_input.cc:210-330), with the reference's messages, plus the limits of this library.
// An empty string means the description is accepted.
inline std::string check_replica(const pimc_replica_desc& d) {
    if (d.ntypes < 1 || d.ntypes > PIMC_MAX_TYPES) return "ntypes out of range";
    if (d.P < 2 || d.P > 65535) return "P out of range";
    int natoms = 0, nmolt = 0, natt = 0;
    bool rotating = false;
    for (int t = 0; t < d.ntypes; ++t) {
        if (d.numb[t] < 1) return "every type needs at least one atom";
        if (d.molecule[t] < 0 || d.molecule[t] > 2) return "unknown molecule kind";
        if (d.molecule[t] == 0 && ++natt > 1) return "No more then one atom/molecule type: densities and potential energy";
        if (d.molecule[t] != 0 && t != d.ntypes - 1) return "Molecules should follow atoms in input file";
        if (d.molecule[t] == 2) {
            ++nmolt;
            if (d.numb[t] > 2) return "GetRotE3D supports at most two non-linear rotors";
            if (d.ntypes > 1 && d.pot3d < 0) return "non-linear rotor without a 3D potential table";
            if (d.Prot > 0 && d.rot3d < 0) return "rotating non-linear rotor without rho/E/E^2 tables";
        }
        if (d.molecule[t] == 1) {
            ++nmolt;
            if (d.numb[t] != 1) return "No more than one linear dopant molecule so far";
        }
        if (d.molecule[t] != 0 && d.Prot > 0) rotating = true;
        if (d.levels[t] < 1 || d.levels[t] > 8) return "bisection levels must be 1..8";
        if ((1 << d.levels[t]) >= d.P) return "Segment size is larger then a number of time slices";
        natoms += d.numb[t];
    }
    if (natoms > 4096) return "too many atoms";
    if (nmolt > 1) return "one molecule type per replica";
    if (d.Prot > 0 && d.P % d.Prot) return "NumbTimes is not proportional to NumbRotTimes";
    if (d.Prot == 1) return "rotational sampling needs at least two rotational slices";
    // the checkerboard sweeps (mc_piqmc.cc:490-512, :728-760) move even slices together, then odd
    // ones: with an odd count slices 0 and Prot-1 are both even and neighbours
    if (rotating && d.Prot % 2) return "the checkerboard rotor sweep needs an even number of rotor slices";
    return std::string();
}

// bisection size classes of the linear family by atom count
inline int bisect_class(int natoms) { return natoms <= 24 ? 0 : (natoms <= 64 ? 1 : 2); }

// Lanes of a segment's group in size class k in a launch of segs segments.  With few segments a chain's
// atoms in turn are the time, and four waves shorten a move; with many the device is full and one
// wave a segment wastes least.  Bisection per pass at 256 and 64 lanes: 40 atoms 1.02 and 1.16 ms on
// 512 segments, 1.28 and 1.24 on 1024; 100 atoms 3.38 and 3.96 ms on 1024, 6.44 and 4.70 on 2048.
// Up to 24 atoms a wave holds the partners as it is (8 atoms: 0.30 and 0.32 ms on 512), and two
// segments share one on a full device (0.445 against 0.470 ms on 4096).
inline int bisect_lanes_by_load(int k, long long segs) {
    if (k == 0) return segs >= 4096 ? 32 : 64;
    return segs <= (k == 1 ? 768 : 1280) ? 256 : 64;
}

// Lanes of the largest block of gw-lane segments that shares the knots in 64 KB, a single wave when
// there are few segments for the device's CUs; lds(block, gw) is a block's LDS.
template <typename Lds>
int bisect_block(int gw, long long segs, const Lds& lds) {
    int block = std::max(gw, segs * gw >= 64 * 1024 ? 256 : 64);
    while (block > std::max(gw, 64) && lds(block, gw) > 64 * 1024) block /= 2;
    return block;
}

// How often a device of ncu CUs fills with segs segments of gw lanes: 16 waves (128 registers) and
// 160 KB a CU.
template <typename Lds>
long long bisect_rounds(int gw, long long segs, int ncu, const Lds& lds) {
    const int block = bisect_block(gw, segs, lds);
    const long long blocks = std::min<long long>(16 * 64 / block, 160 * 1024 / std::max<size_t>(lds(block, gw), 1));
    const long long held = std::max(1LL, blocks) * (block / gw) * ncu;
    return (segs + held - 1) / held;
}

// Lanes of a segment's group in a launch of segs segments of size class k and up to `levels` levels:
// those above, but all 256 where the windows' LDS, not the waves, limits the segments that the device
// holds, and 256 lanes fill it no more often.  Bisection per pass so and with the lanes by load alone:
// FP32, 100 atoms on 1536 segments of 32 slices 39.7 and 59.6 ms; FP64, 100 atoms on 2048 of 8 14.8
// and 24.5, of 16 63 and 132, 200 atoms on 1536 of 16 186 and 522.  Beyond three levels and 24 atoms
// also where the device fills once: 64 atoms in a box on 1024 of 32 13.1 and 20.1.
// stretched: a 1D table on a grid of no one spacing.  An item's knot is then searched for, a chain of
// reads that a uniform grid does without.  The time is those chains, so beyond 24 atoms the lanes are
// those for which the fills of the device, each as long as a segment takes (10, 17 and 29 on 256, 128
// and 64 lanes), are soonest over.  FP32 on 256, 128 and 64: 40 atoms 5.6, 7.1 and 11.5 ms on 1024
// segments of 8 slices, 10.0, 7.4 and 11.5 on 1280; 100 atoms 25.9, 38.7 and 71.5 on 1024, 48.1, 39.8
// and 71.4 on 1280, 102, 85.9 and 144 on 4096, of 4 slices 28.5, 25.3 and 21.3 on 4096; FP64, 100 atoms
// on 2048 of 8 82, 105 and 155.  Two groups of 128 lanes share a block's barrier, and beyond three
// levels each waits for the other's passes: 64 atoms on 2048 of 16 61 ms on 256 lanes, 86 on 128.
// Up to 24 atoms 64 lanes (8 atoms on 4096 segments 0.86 ms, and 1.19 on 32).
template <typename Lds>
int bisect_group(int k, int levels, long long segs, bool stretched, int ncu, const Lds& lds) {
    if (stretched && k > 0) {
        int best = 256;
        long long cost = 10 * bisect_rounds(256, segs, ncu, lds);
        for (const auto& [gw, fill] : {std::pair<int, int>{128, 17}, {64, 29}}) {
            const long long t = fill * bisect_rounds(gw, segs, ncu, lds);
            if (t < cost && !(gw == 128 && levels > 3)) {
                cost = t;
                best = gw;
            }
        }
        return best;
    }
    int gw = stretched ? 64 : bisect_lanes_by_load(k, segs);
    if (gw < 64 && lds(64, gw) > 64 * 1024) gw = 64;
    const long long fills = bisect_rounds(gw, segs, ncu, lds);
    return (fills > 1 || (k > 0 && levels > 3)) && bisect_rounds(256, segs, ncu, lds) <= fills ? 256 : gw;
}

// Whether the bisection on 256 lanes tests its first three levels one by one and not in one pass: where
// a look-up is a search (a stretched 1D table) and the seven midpoints are four searches or more a lane,
// or three where the moves are longer and their first tests reject more, the searches behind a rejection
// cost more than the passes saved.  At once and one by one: 90 atoms on 64 segments of 8 slices 15.9 and
// 17.8 ms, 100 22.7 and 19.7, 300 168 and 122; 64 atoms of 16 slices 26.2 and 31.2, 66 33.7 and 30.4, 100
// 63.8 and 45.6, of 32 slices 118 and 67.6.
inline bool bisect_level_passes(int natoms, int slices, bool stretched) {
    return stretched && natoms > (slices > 8 ? 65 : 98);
}

// Lanes of a non-linear bisection's workgroup, one a segment: a wave or more for a pass over three levels
// of the largest window, fewer where the device (eight waves a CU) would fill more often than a
// segment's time is shortened.  FP32, at 256, 128 and 64 lanes: 13 atoms 0.64 and 0.71 ms (128, 64) on
// 1024 segments, 1.15 and 0.80 on 2048; 25 atoms 0.92, 1.02 and 1.28 on 512, 1.57, 1.09 and 1.31 on 1024,
// 2.51, 2.05 and 2.57 on 2048; 61 atoms 2.36, 2.85 and 4.13 on 512, 4.25, 3.24 and 4.61 on 1024; 101 on
// 1024 7.92, 6.36 and 9.73.  FP64 fills by its windows too: 13 atoms 1.76 and 2.02 (128, 64) on 2048; 25
// atoms 2.16, 1.51 and 1.79 on 1024, 33 3.39, 3.94 and 5.15, and 6.54, 6.12 and 8.27 on 2048, 61 6.57,
// 8.77 and 12.9 on 1024.  So do windows of more than three levels.
inline int bisect_nl_lanes(int natoms, int levels, long long segs, bool fp64) {
    if (natoms <= 10) return 64;
    if (natoms <= 19) return segs > 1024 && !fp64 ? 64 : 128;
    if (levels > 3) return 256;
    if (fp64) return natoms <= 48 && segs > (natoms <= 28 ? 512 : 1024) ? 128 : 256;
    return segs > 512 ? 128 : 256;
}

// Lanes that the autotuner times for a launch: those it has, then the other powers of two that an
// option can ask for.  (32 lanes are a plan's alone: they pay only where it takes them.)
inline std::vector<int> bisect_candidates(int now) {
    std::vector<int> v{now};
    for (int L : {64, 128, 256})
        if (L != now) v.push_back(L);
    return v;
}

// A linear-rotor chain to split: replica r, Prot rotor slices, RotRatio translational slices per
// rotor slice, natoms atoms (the rotor's partners are the natoms - 1 others).
struct RotorChain {
    int r, Prot, RotRatio, natoms;
};

// LDS of a part of ns slices in k_rotor's layout: seven doubles per local slice (two
// neighbours' included) padded to four, then the partner geometry, one vec4 per translational
// slice and partner.
inline size_t rotor_part_lds(int ns, long long per_slice) {
    return (size_t)((7 * (ns + 2) + 3) & ~3) * sizeof(double) + (size_t)((long long)ns * per_slice);
}

constexpr size_t ROTOR_LDS_MAX = 160 * 1024;

// Splits each chain into parts of an even number of slices (the last part may be shorter but is
// even too, since Prot is even), sized so a part's LDS stays within lds_kb and, when
// part_slices_max > 0, at most that many slices.  Parts of a chain wait on one another and are
// all placed on one XCD, so a chain may have at most as many parts as one XCD holds resident at
// the launch's LDS size: cus_per_xcd * blocks_per_cu(lds).  A chain above that is planned again
// with fewer, larger parts; when even those do not fit (a part beyond 160 KB, or one that cannot
// be resident with its neighbours) the plan fails with a message.  parts come out grouped by
// chain in the order given, fbase the index of the chain's first part; lds is the launch's LDS.
inline int plan_linear_rotor(const std::vector<RotorChain>& chains, size_t geo_bytes, int lds_kb, int part_slices_max,
                             int cus_per_xcd, const std::function<int(size_t)>& blocks_per_cu,
                             std::vector<RotPart>& parts, size_t& lds, std::string& err) {
    const long long budget = (long long)lds_kb * 1024;
    const size_t n = chains.size();
    std::vector<int> ns(n), W(n);
    std::vector<long long> per_slice(n);
    auto balance = [](int prot, int w, int& s, int& Wout) {  // even slices per part, W parts
        s = ((prot + w - 1) / w + 1) & ~1;
        if (s >= prot) s = prot;
        Wout = (prot + s - 1) / s;
    };
    for (size_t i = 0; i < n; ++i) {
        const RotorChain& c = chains[i];
        per_slice[i] = (long long)c.RotRatio * (c.natoms - 1) * (long long)geo_bytes;
        int s = (int)std::max<long long>(2, (budget - 16 * (long long)sizeof(double)) /
                                                (7 * (long long)sizeof(double) + per_slice[i])) & ~1;
        if (part_slices_max > 0) s = std::max(2, std::min(s, part_slices_max & ~1));
        if (s >= c.Prot) s = c.Prot;
        balance(c.Prot, (c.Prot + s - 1) / s, ns[i], W[i]);
    }
    for (int iter = 0;; ++iter) {
        lds = 0;
        for (size_t i = 0; i < n; ++i) lds = std::max(lds, rotor_part_lds(ns[i], per_slice[i]));
        if (lds > ROTOR_LDS_MAX) {
            err = "rotor chain exceeds LDS: a part of the linear-rotor sweep needs " + std::to_string(lds) + " bytes";
            return -1;
        }
        if (n == 0) break;
        const long long cap = (long long)cus_per_xcd * std::max(0, blocks_per_cu(lds));
        bool changed = false;
        for (size_t i = 0; i < n; ++i) {
            if (W[i] <= cap) continue;
            if (cap < 1) {
                err = "linear-rotor sweep: parts of " + std::to_string(lds) + " bytes of LDS cannot be resident";
                return -1;
            }
            int s, w;
            balance(chains[i].Prot, (int)std::min<long long>(cap, W[i] - 1), s, w);
            ns[i] = s;
            W[i] = w;
            changed = true;
        }
        if (!changed) break;
        if (iter > 64) {
            err = "linear-rotor sweep: no plan of parts fits one XCD";
            return -1;
        }
    }
    parts.clear();
    for (size_t i = 0; i < n; ++i) {
        const int fbase = (int)parts.size();
        for (int w = 0; w < W[i]; ++w) {
            RotPart q{};
            q.r = chains[i].r;
            q.k0 = w * ns[i];
            q.k1 = std::min(chains[i].Prot, (w + 1) * ns[i]);
            q.w = w;
            q.W = W[i];
            q.fbase = fbase;
            parts.push_back(q);
        }
    }
    return 0;
}

// A part of k_rotor3d_parts with nrot ns up to this takes a group of lanes per move and forms
// proposals ahead.  Two per lane of 256: each move then has the lanes for its new links (two per
// rotor) and the frames fit LDS beside those of other parts.
constexpr int ROT3D_AHEAD = 256;

// A longer part keeps its state in LDS where two parts of its size then share a CU and a lane has one
// move of either parity (rotor3d_long): energies and link densities, and 64 bytes a rotor and slice
// of axes and angles.
constexpr int ROT3D_LANES = 512;
constexpr size_t ROT3D_HALF_CU = 80 * 1024 - 256;
constexpr size_t rotor3d_sums_lds(int ns, int nrot, bool atoms) {
    return (size_t)((nrot * (ns + 1) + (atoms ? nrot * ns : 0) + (nrot - 1) * ns + 1) & ~1) * sizeof(double);
}
constexpr size_t rotor3d_state_lds(int ns, int nrot, bool atoms) {
    return rotor3d_sums_lds(ns, nrot, atoms) + (size_t)nrot * (ns + 2) * 48 + (size_t)nrot * ns * 16;
}
constexpr bool rotor3d_in_lds(int ns, int nrot, bool atoms) {
    return ns <= ROT3D_LANES && rotor3d_state_lds(ns, nrot, atoms) <= ROT3D_HALF_CU;
}

// LDS that parts of up to ns slices of k_rotor3d_parts take with up to nrot rotors.  Short ones: the
// link densities, then the frames of all slices (two neighbours' included) and of the proposals, nine
// doubles a slice and rotor and four a slice with two rotors (rotor3d_ahead).
inline size_t rotor3d_part_lds(int ns, int nrot, size_t frame_bytes) {
    size_t lds = 0;
    for (int nr = 1; nr <= nrot; ++nr) {
        const int na = std::min(ns, ROT3D_AHEAD / nr);
        lds = std::max(lds, (size_t)((nr * (na + 1) + 1) & ~1) * sizeof(double) + (size_t)nr * (2 * na + 2) * frame_bytes +
                                (size_t)na * (9 * nr + (nr > 1 ? 4 : 0)) * sizeof(double));
        if (nr * ns > ROT3D_AHEAD) {
            lds = std::max(lds, rotor3d_sums_lds(ns, nr, true) + (size_t)2 * nr * frame_bytes);
            lds = std::max(lds, std::min(rotor3d_state_lds(std::min(ns, ROT3D_LANES), nr, true), ROT3D_HALF_CU));
        }
    }
    return lds;
}

// LDS of parts of up to ns slices of k_rotor3d_da (delayed acceptance, 256 lanes = 4 waves) with up to
// nrot rotors: the packed network (mlp_bytes), then for short parts (nrot ns <= ROT3D_AHEAD) the link
// densities, the frames of all slices and proposals and eleven doubles a slice and rotor; for longer
// ones the link densities and the two cached sums per own slice, the neighbours' boundary frames and
// DA_MV proposal frames per wave; and 32 row outputs per wave.
constexpr int DA_MV = 64;  // moves a wave takes at once in the long parts: one per lane
inline size_t rotor3d_da_part_lds(int ns, int nrot, size_t frame_bytes, size_t mlp_bytes) {
    size_t lds = 0;
    for (int nr = 1; nr <= nrot; ++nr) {
        const int na = std::min(ns, ROT3D_AHEAD / nr);
        lds = std::max(lds, (size_t)((nr * (na + 1) + 1) & ~1) * sizeof(double) + (size_t)nr * (2 * na + 2) * frame_bytes +
                                (size_t)nr * na * 11 * sizeof(double));
        if (nr * ns > ROT3D_AHEAD)
            lds = std::max(lds, (size_t)((nr * (ns + 1) + 2 * nr * ns + 1) & ~1) * sizeof(double) +
                                    (size_t)(2 * nr + 4 * DA_MV) * frame_bytes);
    }
    return mlp_bytes + lds + (size_t)4 * 32 * sizeof(float);
}

// Split of the non-linear rotor chains: one count W for the launch, a power of two up to 64, the
// largest whose parts hold at least min_slices slices of the longest chain and fit LDS (lds_for(slices)),
// such that the parts of all chains are resident at once (ncu * blocks_per_cu) and the W parts
// of one chain, which wait on one another on one XCD, fit that XCD (cus_per_xcd *
// blocks_per_cu).  Returns 1 when whole chains are better left to one workgroup each.
inline int plan_rotor3d_split(int protmax, int nchains, int ncu, int cus_per_xcd,
                              const std::function<size_t(int)>& lds_for,
                              const std::function<int(size_t)>& blocks_per_cu, int min_slices = 16) {
    int W = 1;
    for (int w = 2; w <= 64; w *= 2) {
        const int ns = ((protmax + w - 1) / w + 1) & ~1;
        const size_t lds = lds_for(ns);
        if (ns < min_slices || lds > ROTOR_LDS_MAX) break;
        const long long occ = std::max(0, blocks_per_cu(lds));
        if ((long long)w * nchains > occ * ncu || (long long)w > occ * cus_per_xcd) break;
        W = w;
    }
    return W;
}

}  // namespace pimc
