/*
 * mpcd_zone.h -- one zone of the snapshot zone redistribution
 * (zone_pass.cpp:62-973), shared by the gfx950 kernels in mpcd_engine.hip and
 * the host logic check in tests/ (ZHD code).
 *
 * The reference's zone kernel is sequential: a shuffled list of dense cells,
 * each of which mutates the counts its successors read.  That order is kept;
 * inside each step the wavefront works together wherever the work is
 * independent by construction: all counter-based draws of a step (shuffle
 * partners, tie breaks, score noise), candidate evaluation and ranking,
 * order-preserving compactions and prefix sums.  On the device a dense cell's
 * candidates and movers are held in lanes and its spread is applied by the
 * lanes at once (dense_cell_wave); the one-lane form of the same functions
 * runs on the host (nl = 1), where the wave primitives reduce to scalars and
 * the barrier to nothing.  A move only records, per particle, the dense pass
 * or the sparse phase that moved it last; the momentum correction, which
 * visits every particle in its final cell, writes the new positions from
 * that record.  The fused kernel (zones with 16-bit indices) runs the passes
 * on four wavefronts and the correction behind them, the zone's state staying
 * in LDS; the form with 32-bit indices runs the passes on one wavefront and
 * hands the state over in global memory (ZoneState) to the correction on four.
 *
 * Memory.  Cell arrays are indexed by the zone-local cell
 * lc = (ix-xs)*zh + (iy-ys) (ascending global cell id); particles by the
 * zone-local index k (the zone's cells' runs of the pass-input binning list,
 * in lc order).  Index arrays use the type IT: uint16_t when the zone has
 * fewer than 65535 cells and particles (the cell arrays and most list links
 * then fit in LDS next to three other zones on a CU), int otherwise.  List
 * links of k < nL live in LDS, the rest in the zone's private global region.
 *
 * Snapshot semantics.  The shifted layout's zones overlap
 * (zone_pass.cpp:191-219 starts them at 0 and T/2 with width T), so two zones
 * may hold the same particle.  Every zone reads the pass input; a zone writes
 * only the particles it owns, i.e. whose input cell has this zone as its
 * owner-map entry (the last zone covering the cell, which is the zone whose
 * result the reference's merge keeps, zone_pass_openmp.cpp:145-153).
 * Positions are written in place (nobody reads them during a pass).
 * Velocities are written in place for particles whose input cell only one
 * zone covers; for cells several zones cover they go to vsx/vsy and are
 * copied back after the pass, so every zone reads inputs.
 *
 * Lists.  A cell's list starts as its input run, consecutive local indices
 * k0..run_end.  What is left of the run stays implicit (pops only move the
 * head along it) and arrivals are linked behind it: the run's last entry
 * links to the first arrival, each arrival to the next.  An append thus
 * writes two links, however long the run is.  A list that is reordered (a
 * sparse donor's), or that takes back a particle of its own run, has every
 * link written (ZF_MAT).  ZF_CHG marks every cell whose list changed; the
 * others cost nothing at the correction.
 */
#pragma once

#include <stdint.h>

#include "mpcd_core.h"

/* every zone function is inlined into the kernel, so the per-lane zone
 * context stays in registers */
#if defined(__HIPCC__)
#define ZHD __host__ __device__ inline __attribute__((always_inline))
#else
#define ZHD inline
#endif

namespace mpcdk {

#if defined(__HIP_DEVICE_COMPILE__)
/* The zone code runs on one wavefront: its barrier orders the lanes' memory
 * operations (workgroup-scope fences) without a workgroup barrier, so a
 * larger workgroup can run it on one of its wavefronts. */
#define ZBAR()                                                 \
    do {                                                       \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup"); \
        __builtin_amdgcn_wave_barrier();                       \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup"); \
    } while (0)
/* compiler-level ordering of LDS accesses between lanes of the one
 * wavefront (the LDS executes a wavefront's accesses in issue order) */
#define ZWSYNC()                                               \
    do {                                                       \
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); \
        __builtin_amdgcn_wave_barrier();                       \
    } while (0)
ZHD unsigned long long wave_ballot(bool f) { return __ballot(f); }
ZHD int wave_popc(unsigned long long m) { return __popcll(m); }
ZHD int wave_shfl_up_add(int v, int lane) {
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}
ZHD int wave_bcast(int v, int src) { return __shfl(v, src, 64); }
/* value of lane l (l uniform across the wavefront) */
ZHD int wave_readlane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
/* v with lane l's value replaced by s (s and l uniform): the compiler has the
 * operation as an intrinsic without a builtin of its own */
extern "C" __device__ int mpcd_intrin_writelane(int s, int l, int v) __asm("llvm.amdgcn.writelane.i32");
__device__ inline __attribute__((always_inline)) int wave_writelane(int s, int l, int v) { return mpcd_intrin_writelane(s, l, v); }
ZHD double wave_readlane_d(double v, int l) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
ZHD int wave_sum(int v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
ZHD double wave_max(double v) {
    for (int o = 32; o > 0; o >>= 1) {
        const double t = __shfl_xor(v, o, 64);
        v = (v < t) ? t : v;
    }
    return v;
}
#else
#define ZBAR() ((void)0)
#define ZWSYNC() ((void)0)
ZHD unsigned long long wave_ballot(bool f) { return f ? 1ull : 0ull; }
ZHD int wave_popc(unsigned long long m) { return __builtin_popcountll(m); }
ZHD int wave_shfl_up_add(int v, int) { return v; }
ZHD int wave_bcast(int v, int) { return v; }
ZHD int wave_readlane(int v, int) { return v; }
ZHD double wave_readlane_d(double v, int) { return v; }
ZHD int wave_sum(int v) { return v; }
ZHD double wave_max(double v) { return v; }
#endif
ZHD unsigned long long lanes_below(int lane) { return (lane >= 64) ? ~0ull : ((1ull << lane) - 1ull); }

struct ZoneParams {
    double highThr, lowThrBulk;
    double lowFrac, highFrac; /* 1/(1+coef), 1+coef */
    double gamma, fluidFracGain, lowThrFloor, highThrFloor;
    double lowLoc1, highLoc1; /* empty-cell thresholds for fluid fraction 1 */
    int useLocal, maxPasses, corrEnabled;
    int dedupe; /* a periodic axis narrower than 5 cells: wrapped neighbours can repeat */
    int odd;    /* dedupe, or thresholds below zero or the low one above the high one: k_zone_fused's kOdd form */
    int quadBins; /* at most 3 neighbour offsets per angular bin, no two of a bin equally far (the wavefront form's
                   * lane layout, in which no tie is left to a draw), and no dense cell its own target */
    /* angular bin (3 bits) of (dx,dy) in [-2,2]^2 at index (dy+2)*5+(dx+2):
     * indices 0..20 in binLo, 21..24 in binHi (registers, not an array that
     * a dynamic index would send to private memory) */
    unsigned long long binLo, binHi;
};

ZHD int zone_bin(const ZoneParams& zp, int idx) {
    return idx < 21 ? (int)((zp.binLo >> (3 * idx)) & 7ull) : (int)((zp.binHi >> (3 * (idx - 21))) & 7ull);
}

/* Candidate of a dense cell's target ranking. */
struct Cand {
    int lc, gc;
    double deficitNeg;
    int cnt, cheb, dist2, bin;
    double tie;
};

struct ZoneRect {
    int xs, xe, ys, ye;
};

struct ZoneOut {
    int nHigh, nLow, movedDense, movedSparse;
    double stats4, stats5;
};

/* (overridable so that a host build can exercise the paths past them) */
#ifndef MPCD_ZONE_MAX_MOVE
#define MPCD_ZONE_MAX_MOVE 64
#endif
#ifndef MPCD_ZONE_TMP_L
#define MPCD_ZONE_TMP_L 256
#endif
constexpr int ZONE_MAX_MOVE = MPCD_ZONE_MAX_MOVE; /* dense movers staged per source cell */
static_assert(ZONE_MAX_MOVE <= 64, "a dense cell's movers are the lanes of one wavefront");
constexpr int ZONE_TMP_L = MPCD_ZONE_TMP_L;       /* donor lists up to this length are shuffled in LDS */

/* per-cell flag bits */
enum : unsigned short {
    ZF_BULK0 = 1,   /* occupied when this pass's maps were built */
    ZF_RECV = 2,    /* received particles */
    ZF_BB = 4,      /* bulk-to-bulk transfer */
    ZF_SKIP = 8,    /* transfer touching a non-bulk cell */
    ZF_MAT = 16,    /* every list link written (else: what is left of the input run, then linked arrivals) */
    ZF_CORR = 32,   /* momentum correction applies */
    ZF_CHG = 64,    /* list changed */
    ZF_OWN = 128,   /* this zone owns the cell's input particles */
    ZF_COVER = 256, /* several zones cover the cell */
    ZF_OUT = 4096   /* in the zone's rectangle but not in its mask */
};

/* Inputs of a zone pass common to all its zones. */
struct ZoneIn {
    Geom g;
    ZoneParams zp;
    const int* gcnt;    /* pass-input binning: counts, run starts, slots */
    const int* gstart;
    const int* glist;
    const unsigned long long* gkey; /* (pid << 32 | slot) of each binning position */
    const int* owner;   /* owner map of the layout, or nullptr: each zone owns its cells */
    const unsigned char* gcover; /* per cell: several zones cover it, or nullptr */
    double *x, *y, *vx, *vy;
    double *vsx, *vsy;  /* side buffer for covered cells */
    /* per cell several zones cover: its owner changed it, so the side buffer
     * holds its particles' velocities (nullptr with gcover) */
    unsigned char* gchg = nullptr;
    /* per-cell velocity sums of the pass input (each cell's run summed in
     * order from zero), or nullptr: the correction sums the runs itself */
    const double *inPx = nullptr, *inPy = nullptr;
    /* non-null: each moved particle's cell change is recorded for the
     * binning update (cell of each slot, departures and arrivals per cell,
     * the list of arrivals: slot and rank among the new cell's, and its
     * length) */
    int *dcid = nullptr, *dout = nullptr, *dinc = nullptr, *darr = nullptr, *darrN = nullptr;
    /* non-null (a single-zone call that reports ZoneKernelStats.diag): per
     * zone cell, the momentum defect and the final list's momentum before
     * the correction (4 doubles), and the count the sparse phase starts
     * from */
    double* dgCell = nullptr;
    int* dgCnt = nullptr;
    /* added to the recorded new cells (an ensemble replica's first cell in
     * the concatenated grid; 0 for a single simulation) */
    int cellOff = 0;
    /* per grid cell, nonzero in the zone (Zone.maskVec, zone_pass.cpp:20-24),
     * or nullptr: the zone is its whole rectangle.  A cell of the rectangle
     * outside the mask keeps its particles and counts but is never in the
     * dense or low lists, a target, a neighbour or a donor. */
    const unsigned char* zmask = nullptr;
};

/* Scalars the lanes share (LDS on the device). */
struct ZoneShared {
    int nOrd, startBin, nr, stage, P, allOwned;
    int mwCount;           /* the multi-wavefront phases' list length */
    int mwNext;            /* and the next list position a wavefront takes */
    int schedWait;         /* nonzero: a wait of the dependency-driven dense phase hit its bound */
    int nHigh, nLow, movedDense, movedSparse;
    int mixed;             /* zone_setup_cells: a cell is not plainly owned */
    unsigned long long off; /* the zone's offset into the particle regions */
    double stats4, stats5;
};

/* A cell's live state: one 8-byte LDS access with 16-bit indices. */
template <class IT>
struct alignas(4 * sizeof(IT)) ZCell {
    IT cnt, head, tail, fl;
};

/* The small scratch of the one-lane forms (and, idle, of the scheduled
 * phases' list building). */
template <class IT>
struct ZScratch {
    Cand cand[24];
    double ordThr[24], nbTie[24], dsc[8], nsm4[4];
    int ord[24], nbGc[24], rnk[24], recvT[48], dord[8], dord2[16];
    IT tmpL[ZONE_TMP_L]; /* a donor list being shuffled */
};

template <class IT>
struct ZoneCtxT {
    typedef IT idx_t;
    Geom g;
    ZoneParams zp;
    int xs, xe, ys, ye, zw, zh, C;
    unsigned zhM; /* lc_col's factor, 0 for zh = 1 */
    int zid, P, nL;
    int allOwned; /* copied from the shared set-up result */
    uint64_t seed;
    const int *gcnt, *gstart, *glist;
    const unsigned long long* gkey;
    double *x, *y, *vx, *vy, *vsx, *vsy;
    unsigned char* gchg; /* changed covered cells, or nullptr */
    const double *inPx, *inPy; /* input run sums per global cell, or nullptr */
    int *dcid, *dout, *dinc, *darr, *darrN; /* cell-change record, or nullptr */
    int cellOff;    /* added to the recorded new cells */
    double* dgCell; /* diagnostics' per-cell record, or nullptr */
    int* dgCnt;     /* diagnostics' sparse-phase start counts, or nullptr */
    IT* nxL;     /* links of k < nL */
    IT* nxG;     /* links of k >= nL (zone's global region, indexed by k) */
    IT* tmpG;    /* donor lists longer than ZONE_TMP_L (zone's global region) */
    double* duG; /* velocity change per cell (zone's global region, 2 per cell) */
    unsigned char* rec; /* last move of each particle by local index (zone's global region, 1 per particle) */
    /* cell arrays */
    ZCell<IT>* cell;
    IT *dl, *k0;
    IT* ext; /* sparse phase: the counts it starts from, zone and ring, (zw+4) x (zh+4) column-major */
    int *colL, *colG; /* per column: first local index, start in the binning list */
    double *lowA, *highA; /* local fluid-fraction thresholds (only with useLocal) */
    IT* halo;             /* pass-input counts of the ring of width 2 around the zone */
    ZScratch<IT>* scr;
    IT* lix; /* per cell: its index in the sparse phase's list (the type's maximum: none, or done); in the dense
              * passes a dense cell's surplus and start bins */
    ZoneShared* sh;
};

/* ---- index and flag access ---- */

template <class IT>
ZHD int iget(IT v) {
    return v == (IT)-1 ? -1 : (int)v;
}
template <class Z>
ZHD bool fget(const Z& z, int lc, unsigned short b) {
    return ((unsigned)z.cell[lc].fl & b) != 0;
}
template <class Z>
ZHD void fset(Z& z, int lc, unsigned short b) {
    z.cell[lc].fl = (typename Z::idx_t)((unsigned)z.cell[lc].fl | b);
}
template <class Z>
ZHD void fclr(Z& z, int lc, unsigned short b) {
    z.cell[lc].fl = (typename Z::idx_t)((unsigned)z.cell[lc].fl & ~(unsigned)b);
}
template <class Z>
ZHD int cnt_of(const Z& z, int lc) {
    return (int)z.cell[lc].cnt;
}
template <class Z>
ZHD void cnt_set(Z& z, int lc, int v) {
    z.cell[lc].cnt = (typename Z::idx_t)v;
}
template <class Z>
ZHD int head_of(const Z& z, int lc) {
    return iget(z.cell[lc].head);
}
template <class Z>
ZHD int tail_of(const Z& z, int lc) {
    return iget(z.cell[lc].tail);
}
template <class Z>
ZHD void head_set(Z& z, int lc, int k) {
    z.cell[lc].head = (typename Z::idx_t)k;
}
template <class Z>
ZHD void tail_set(Z& z, int lc, int k) {
    z.cell[lc].tail = (typename Z::idx_t)k;
}
/* Accesses to the zone's global regions.  On the device they are
 * non-temporal operations: distinct from the working-set accesses, so the
 * compiler never merges the two into one generic (flat) access whose wait
 * would also stall on every outstanding global load. */
#if defined(__HIP_DEVICE_COMPILE__)
#define ZG_LOAD(p) __builtin_nontemporal_load(p)
#define ZG_STORE(p, v) __builtin_nontemporal_store((v), (p))
#else
#define ZG_LOAD(p) (*(p))
#define ZG_STORE(p, v) (*(p) = (v))
#endif

/* The link accessors read both base pointers before choosing: a choice
 * between two fields of the context (rather than two loaded values) would
 * keep the context out of registers. */
template <class Z>
ZHD int nx_get(const Z& z, int k) {
    const typename Z::idx_t* const L = z.nxL;
    const typename Z::idx_t* const G = z.nxG;
    if (k < z.nL) return iget(L[k]);
    return iget(ZG_LOAD(G + k));
}
template <class Z>
ZHD void nx_set(Z& z, int k, int v) {
    typename Z::idx_t* const L = z.nxL;
    typename Z::idx_t* const G = z.nxG;
    if (k < z.nL) L[k] = (typename Z::idx_t)v;
    else ZG_STORE(G + k, (typename Z::idx_t)v);
}

/* ---- geometry ---- */

template <class Z>
ZHD int zone_lc(const Z& z, int gx, int gy) {
    if (gx >= z.xs && gx < z.xe && gy >= z.ys && gy < z.ye) return (gx - z.xs) * z.zh + (gy - z.ys);
    return -1;
}
/* lc / zh.  With 16-bit indices by a multiplication: zhM = floor((2^32-1)/zh) + 1
 * exceeds 2^32/zh by e/zh with e <= zh, and lc e < 2^32, so the high word of
 * lc zhM is the quotient (zh = 1 has no such factor in 32 bits). */
template <class Z>
ZHD int lc_col(const Z& z, int lc) {
    if (sizeof(typename Z::idx_t) == 2)
        return z.zhM ? (int)(((unsigned long long)(unsigned)lc * (unsigned long long)z.zhM) >> 32) : lc;
    return lc / z.zh;
}
template <class Z>
ZHD int lc_gx(const Z& z, int lc) {
    return z.xs + lc_col(z, lc);
}
template <class Z>
ZHD int lc_gy(const Z& z, int lc) {
    return z.ys + lc - z.zh * lc_col(z, lc);
}
template <class Z>
ZHD int lc_gc(const Z& z, int lc) {
    return lc_gy(z, lc) + z.g.Ny * lc_gx(z, lc);
}

/* Slot in z.halo of the cell at zone-relative offset (dx, dy) of the ring of
 * width 2 around the zone: two rows below and above (all zw+4 columns), then
 * two columns left and right (the zh rows between); -1 inside the zone or
 * beyond the ring. */
template <class Z>
ZHD int halo_slot(const Z& z, int dx, int dy) {
    if (dx < -2 || dx >= z.zw + 2 || dy < -2 || dy >= z.zh + 2) return -1;
    const int hx = dx + 2, hy = dy + 2, W4 = z.zw + 4;
    if (hy < 2) return hx * 2 + hy;
    if (hy >= z.zh + 2) return 2 * W4 + hx * 2 + (hy - z.zh - 2);
    if (hx < 2) return 4 * W4 + hx * z.zh + (hy - 2);
    if (hx >= z.zw + 2) return 4 * W4 + 2 * z.zh + (hx - z.zw - 2) * z.zh + (hy - 2);
    return -1;
}
/* extended coordinates (0 .. zw+3, 0 .. zh+3) of ring slot h */
template <class Z>
ZHD void halo_xy(const Z& z, int h, int& hx, int& hy) {
    const int W4 = z.zw + 4;
    if (h < 2 * W4) {
        hx = h / 2;
        hy = h % 2;
    } else if (h < 4 * W4) {
        hx = (h - 2 * W4) / 2;
        hy = z.zh + 2 + (h - 2 * W4) % 2;
    } else if (h < 4 * W4 + 2 * z.zh) {
        hx = lc_col(z, h - 4 * W4);
        hy = 2 + (h - 4 * W4) - hx * z.zh;
    } else {
        const int q = lc_col(z, h - 4 * W4 - 2 * z.zh);
        hx = z.zw + 2 + q;
        hy = 2 + (h - 4 * W4 - 2 * z.zh) - q * z.zh;
    }
}
template <class Z>
ZHD int halo_size(const Z& z) {
    return 4 * (z.zw + 4) + 4 * z.zh;
}
/* the ring slot of global cell (gx, gy) outside the zone, periodic axes
 * taken to the image next to the zone */
template <class Z>
ZHD int halo_of(const Z& z, int gx, int gy) {
    int dx = gx - z.xs, dy = gy - z.ys;
    if (z.g.perx) {
        if (dx < -2) dx += z.g.Nx;
        else if (dx >= z.zw + 2) dx -= z.g.Nx;
    }
    if (z.g.pery) {
        if (dy < -2) dy += z.g.Ny;
        else if (dy >= z.zh + 2) dy -= z.g.Ny;
    }
    return halo_slot(z, dx, dy);
}

/* count at a global cell: live zone count (or the sparse-phase copy), else
 * the pass-input snapshot, from the ring in LDS (a count the index type
 * cannot hold is read from global memory). */
template <class Z>
ZHD int count_at(const Z& z, int gx, int gy, int use_copy) {
    const int lc = zone_lc(z, gx, gy);
    if (lc >= 0) {
        if (!use_copy) return (int)z.cell[lc].cnt;
        const int ix = lc / z.zh;
        return (int)z.ext[(ix + 2) * (z.zh + 4) + (lc - ix * z.zh) + 2];
    }
    const int h = halo_of(z, gx, gy);
    if (h >= 0) {
        const int v = iget(z.halo[h]);
        if (v >= 0) return v;
    }
    return z.gcnt[gy + z.g.Ny * gx];
}

/* 3x3 binomial smoothing without wrap (zone_pass.cpp:296-319).  The
 * weights are multiples of 1/16 and the counts integers, so the weighted
 * sums are exact: they are taken in integers (scaled by 16) and divided once,
 * which is the same correctly rounded quotient. */
template <class Z>
ZHD double nsm_at(const Z& z, int gx, int gy, int use_copy) {
    long long num = 0;
    int den = 0;
    for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
            const int jy = gy + dy, jx = gx + dx;
            if (jy < 0 || jy >= z.g.Ny || jx < 0 || jx >= z.g.Nx) continue;
            const int w = (dx == 0 ? 2 : 1) * (dy == 0 ? 2 : 1); /* 1 2 1 / 2 4 2 / 1 2 1 */
            num += (long long)w * count_at(z, jx, jy, use_copy);
            den += w;
        }
    return (double)num / (double)den;
}

/* nsm_at(.., use_copy = 1) for a point within one cell of the zone: the
 * nine counts are direct reads of the extended array (no branch per
 * neighbour); the same integer sums and quotient. */
template <class Z>
ZHD double nsm_ext(const Z& z, int gx, int gy) {
    int rx = gx - z.xs, ry = gy - z.ys;
    if (z.g.perx) {
        if (rx < -2) rx += z.g.Nx;
        else if (rx >= z.zw + 2) rx -= z.g.Nx;
    }
    if (z.g.pery) {
        if (ry < -2) ry += z.g.Ny;
        else if (ry >= z.zh + 2) ry -= z.g.Ny;
    }
    if (rx < -1 || rx > z.zw || ry < -1 || ry > z.zh) return nsm_at(z, gx, gy, 1);
    const int H = z.zh + 4;
    const int base = (rx + 2) * H + (ry + 2);
    int v[9];
    bool ok[9];
    for (int dx = -1; dx <= 1; ++dx)
        for (int dy = -1; dy <= 1; ++dy) {
            const int t = (dx + 1) * 3 + (dy + 1);
            const int jx = gx + dx, jy = gy + dy;
            ok[t] = jx >= 0 && jx < z.g.Nx && jy >= 0 && jy < z.g.Ny;
            v[t] = ok[t] ? iget(z.ext[base + dx * H + dy]) : 0;
        }
    long long num = 0;
    int den = 0;
    bool far = false;
    for (int t = 0; t < 9; ++t) {
        const int w = (t / 3 == 1 ? 2 : 1) * (t % 3 == 1 ? 2 : 1);
        if (!ok[t]) continue;
        if (v[t] < 0) far = true;
        num += (long long)w * v[t];
        den += w;
    }
    if (far) return nsm_at(z, gx, gy, 1); /* a ring count the index type could not hold */
    return (double)num / (double)den;
}

/* Active thresholds of a zone cell (zone_pass.cpp:321-345, :715-725): the
 * bulk flag is taken when the maps are built; with fluid fraction 1 the
 * empty-cell values are constants, otherwise they are stored per cell. */
template <class Z>
ZHD void zone_maps(Z& z, int lc, int use_copy) {
    const int bulk = z.cell[lc].cnt > 0;
    if (bulk) fset(z, lc, ZF_BULK0);
    else fclr(z, lc, ZF_BULK0);
    if (!z.zp.useLocal) return;
    const double fRaw = nsm_at(z, lc_gx(z, lc), lc_gy(z, lc), use_copy) / dmax(z.zp.gamma, 1e-12);
    const double t = z.zp.fluidFracGain * fRaw;
    const double f = (t < 0.0) ? 0.0 : ((1.0 < t) ? 1.0 : t); /* std::clamp(t, 0, 1) */
    const double gl = z.zp.gamma * f;
    z.lowA[lc] = bulk ? z.zp.lowThrBulk : dmax(z.zp.lowFrac * gl, z.zp.lowThrFloor);
    z.highA[lc] = bulk ? z.zp.highThr : dmax(z.zp.highFrac * gl, z.zp.highThrFloor);
}
template <class Z>
ZHD double low_thr(const Z& z, int lc) {
    if (z.zp.useLocal) return z.lowA[lc];
    const double b = z.zp.lowThrBulk, e = z.zp.lowLoc1;
    return fget(z, lc, ZF_BULK0) ? b : e;
}
template <class Z>
ZHD double high_thr(const Z& z, int lc) {
    if (z.zp.useLocal) return z.highA[lc];
    const double b = z.zp.highThr, e = z.zp.highLoc1;
    return fget(z, lc, ZF_BULK0) ? b : e;
}
template <class Z>
ZHD double thr(const Z& z, int lc, int high) {
    return high ? high_thr(z, lc) : low_thr(z, lc);
}

/* zone_pass.cpp:229-244 */
template <class Z>
ZHD void min_step(const Z& z, int sx, int sy, int tx, int ty, int& ddx, int& ddy) {
    ddx = tx - sx;
    ddy = ty - sy;
    if (z.g.perx) {
        if (ddx > z.g.Nx / 2) ddx -= z.g.Nx;
        if (ddx < -z.g.Nx / 2) ddx += z.g.Nx;
    }
    if (z.g.pery) {
        if (ddy > z.g.Ny / 2) ddy -= z.g.Ny;
        if (ddy < -z.g.Ny / 2) ddy += z.g.Ny;
    }
}

/* zone_pass.cpp:246-261 */
template <class Z>
ZHD int shift_idx(const Z& z, int gx, int gy, int dx, int dy, int& jx, int& jy) {
    jy = gy + dy;
    if (z.g.pery) jy = wrapi(jy, z.g.Ny);
    else if (jy < 0 || jy >= z.g.Ny) return 0;
    jx = gx + dx;
    if (z.g.perx) jx = wrapi(jx, z.g.Nx);
    else if (jx < 0 || jx >= z.g.Nx) return 0;
    return 1;
}

/* ---- particles ---- */

/* column of the zone's k-th particle (the zone's particles are its columns'
 * runs of the binning list, in column order) */
template <class Z>
ZHD int col_of(const Z& z, int k) {
    int lo = 0, hi = z.zw - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (z.colL[mid] <= k) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
template <class Z>
ZHD int slot_in(const Z& z, int k, int col) {
    return z.glist[z.colG[col] + (k - z.colL[col])];
}
/* slot and particle id of the zone's k-th particle in one load */
template <class Z>
ZHD int slot_pid_in(const Z& z, int k, int col, uint32_t& pid) {
    const unsigned long long key = z.gkey[z.colG[col] + (k - z.colL[col])];
    pid = (uint32_t)(key >> 32);
    return (int)(uint32_t)key;
}
template <class Z>
ZHD int slot_of(const Z& z, int k) {
    return slot_in(z, k, col_of(z, k));
}
/* ZF_OWN / ZF_COVER of the input cell of k: the last cell of k's column
 * whose input run starts at or before k */
template <class Z>
ZHD unsigned short own_bits(const Z& z, int k, int col) {
    if (z.allOwned) return ZF_OWN;
    int lo = col * z.zh, hi = lo + z.zh - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if ((int)z.k0[mid] <= k) lo = mid;
        else hi = mid - 1;
    }
    return (unsigned short)((unsigned)z.cell[lo].fl & (ZF_OWN | ZF_COVER));
}

/* last local index of cell lc's input run (k0[lc] - 1 when it is empty): the
 * runs follow each other in lc order */
template <class Z>
ZHD int run_end(const Z& z, int lc) {
    return (lc + 1 < z.C ? (int)z.k0[lc + 1] : z.P) - 1;
}
/* k belongs to cell lc's input run */
template <class Z>
ZHD bool in_run(const Z& z, int lc, int k) {
    return k >= (int)z.k0[lc] && k <= run_end(z, lc);
}
/* entries of a list with head h that are still implicit: what is left of the
 * input run (none once its links are written or the run is used up) */
template <class Z>
ZHD int run_left(const Z& z, int lc, int h) {
    return (h >= 0 && !fget(z, lc, ZF_MAT) && in_run(z, lc, h)) ? run_end(z, lc) - h + 1 : 0;
}

/* successor of k in cell lc's list (implicit run or links) */
template <class Z>
ZHD int next_k(const Z& z, int lc, int k) {
    if (!fget(z, lc, ZF_MAT)) {
        if (k == tail_of(z, lc)) return -1;
        if (k >= (int)z.k0[lc] && k < run_end(z, lc)) return k + 1;
    }
    return nx_get(z, k);
}

/* write the links of what is still implicit in cell lc's list */
template <class Z>
ZHD void ensure_mat(Z& z, int lc) {
    if (fget(z, lc, ZF_MAT)) return;
    const int h = head_of(z, lc), left = run_left(z, lc, h);
    for (int q = 0; q + 1 < left; ++q) nx_set(z, h + q, h + q + 1);
    if (left > 0 && tail_of(z, lc) == h + left - 1) nx_set(z, h + left - 1, -1);
    fset(z, lc, ZF_MAT);
}

/* A list that takes back a particle of its own input run cannot keep the run
 * implicit: its links are written first (one lane). */
template <class Z>
ZHD void ensure_append(Z& z, int lc, int k) {
    if (in_run(z, lc, k)) ensure_mat(z, lc);
}

template <class Z>
ZHD void list_append(Z& z, int lc, int k) {
    ensure_append(z, lc, k);
    fset(z, lc, ZF_CHG);
    nx_set(z, k, -1);
    const int t = tail_of(z, lc);
    if (t < 0) head_set(z, lc, k);
    else nx_set(z, t, k);
    tail_set(z, lc, k);
}

/* A moved particle's new position (zone_pass.cpp:280-294: uniform in its
 * target cell, drawn per dense pass or for the sparse phase) depends only on
 * its last move, so a move records what it was -- ZM_NONE, the dense pass
 * (1..254) or ZM_SPARSE -- and the correction sweep, which visits every
 * particle in its final cell, writes the positions (owned particles only).
 * The serial phases then touch no global memory for moves. */
enum { ZM_NONE = 0, ZM_SPARSE = 255 };
template <class Z>
ZHD void mark_moved(Z& z, int k, int tag) {
    z.rec[k] = (unsigned char)tag;
}
template <class Z>
ZHD void place_moved(Z& z, int lc, int slot, uint32_t pid, int tag) {
    double ux, uy;
    if (tag == ZM_SPARSE) mpcd_draw_sparse_pos(z.seed, pid, &ux, &uy);
    else mpcd_draw_dense_pos(z.seed, tag, pid, &ux, &uy);
    const int ix = lc / z.zh;
    const double nx = (double)(z.xs + ix) * z.g.dxc + z.g.dxc * ux;
    const double ny = (double)(z.ys + (lc - ix * z.zh)) * z.g.dyc + z.g.dyc * uy;
    z.x[slot] = nx;
    z.y[slot] = ny;
    if (z.dcid) {
        /* the cell the binning update will see (a particle is placed once
         * per pass); the pass's own counts stay untouched */
        const int cn = cell_of(z.g, nx, ny) + z.cellOff, co = z.dcid[slot];
        if (cn != co) {
            z.dcid[slot] = cn;
#if defined(__HIP_DEVICE_COMPILE__)
            atomicAdd(&z.dout[co], 1);
            const int r = atomicAdd(&z.dinc[cn], 1);
            /* one place in the list for all lanes here at once */
            const unsigned long long act = wave_ballot(true);
            const int ln = (int)__lane_id();
            int base = 0;
            if (ln == (int)__builtin_ctzll(act)) base = atomicAdd(z.darrN, wave_popc(act));
            base = __builtin_amdgcn_readfirstlane(base) + wave_popc(act & lanes_below(ln));
            reinterpret_cast<int2*>(z.darr)[base] = make_int2(slot, r);
#else
            ++z.dout[co];
            const int j = (*z.darrN)++;
            z.darr[2 * (size_t)j] = slot;
            z.darr[2 * (size_t)j + 1] = z.dinc[cn]++;
#endif
        }
    }
}

/* the bulk/skip masks of a transfer (zone_pass.cpp:492-525) */
template <class Z>
ZHD void transfer_masks(Z& z, int src, const int* rv, int nr) {
    bool allBulk = fget(z, src, ZF_BULK0);
    for (int k = 0; k < nr && allBulk; ++k)
        if (!fget(z, rv[k], ZF_BULK0)) allBulk = false;
    if (allBulk) {
        fset(z, src, ZF_BB);
        for (int k = 0; k < nr; ++k) fset(z, rv[k], ZF_BB);
    } else {
        fset(z, src, ZF_SKIP);
        fclr(z, src, ZF_BB);
        for (int k = 0; k < nr; ++k) {
            fset(z, rv[k], ZF_SKIP);
            fclr(z, rv[k], ZF_BB);
        }
    }
}

ZHD bool cand_less(const Cand& a, const Cand& b) {
    /* (-deficit, -inward (all equal: weight 0), cnt, cheb, dist2, tie) */
    if (a.deficitNeg != b.deficitNeg) return a.deficitNeg < b.deficitNeg;
    if (a.cnt != b.cnt) return a.cnt < b.cnt;
    if (a.cheb != b.cheb) return a.cheb < b.cheb;
    if (a.dist2 != b.dist2) return a.dist2 < b.dist2;
    return a.tie < b.tie;
}

enum { ZC_DENSE = 0, ZC_LOW = 1 };

/* Order-preserving compaction into z.dl of the zone cells above their high
 * threshold (ZC_DENSE) or occupied and below their low threshold (ZC_LOW);
 * all lanes; returns the count (same on every lane). */
template <class Z>
ZHD int zone_compact(Z& z, int lane, int nl, int mode) {
    int base = 0;
    for (int b0 = 0; b0 < z.C; b0 += nl) {
        const int lc = b0 + lane;
        bool f = false;
        if (lc < z.C) {
            const double c = (double)z.cell[lc].cnt;
            f = (mode == ZC_DENSE) ? c > high_thr(z, lc) : (z.cell[lc].cnt > 0 && c < low_thr(z, lc));
            f = f && !fget(z, lc, ZF_OUT);
        }
        const unsigned long long msk = wave_ballot(f);
        if (f) z.dl[base + wave_popc(msk & lanes_below(lane))] = (typename Z::idx_t)lc;
        base += wave_popc(msk);
    }
    return base;
}

/* The shuffles' partner draws, j in [0, i]. */
enum { ZS_DENSE = 0, ZS_LOW = 1, ZS_DONOR = 2, ZS_PARTICLE = 3 };
struct ShufDraw {
    uint64_t seed;
    int kind;
    uint32_t a, b;
    ZHD uint32_t operator()(uint32_t i) const {
        switch (kind) {
            case ZS_DENSE: return mpcd_draw_dense_shuffle(seed, (int)a, i);
            case ZS_LOW: return mpcd_draw_low_shuffle(seed, i);
            case ZS_DONOR: return mpcd_draw_donor_shuffle(seed, a, i);
            default: return mpcd_draw_particle_shuffle(seed, a, b, i);
        }
    }
};

#if defined(__HIP_DEVICE_COMPILE__)
/* Fisher-Yates of the values v of lanes 0..m-1 (m <= 64) with lane i's
 * partner j (in [0, i]) */
__device__ inline __attribute__((always_inline)) int shuffle64(int v, int j, int m) {
    int ii = m - 1;
    for (; ii >= 8; ii -= 8) {
        /* the partners of eight swaps first: off the swaps' own chain */
        int jj[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) jj[t] = wave_readlane(j, ii - t);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int vi = wave_readlane(v, ii - t), vj = wave_readlane(v, jj[t]);
            v = wave_writelane(vj, ii - t, v);
            v = wave_writelane(vi, jj[t], v);
        }
    }
    for (; ii >= 1; --ii) {
        const int jj = wave_readlane(j, ii);
        const int vi = wave_readlane(v, ii), vj = wave_readlane(v, jj);
        v = wave_writelane(vj, ii, v);
        v = wave_writelane(vi, jj, v);
    }
    return v;
}
#endif

/* Fisher-Yates of a[0..m), i = m-1 down to 1, swapping a[i] with a[j(i)],
 * `draw(i)` giving j in [0, i].  The partner draws of a chunk of nl indices
 * are computed by the lanes at once and kept in registers; lane 0 applies
 * the chunk's swaps in order, reading each partner from its lane. */
template <class T>
ZHD void zone_shuffle(T* a, int m, int lane, int nl, ShufDraw draw) {
#if defined(__HIP_DEVICE_COMPILE__)
    if (m <= 128) {
        /* elements q and 64 + q in lane q's registers: a swap is two reads
         * and two writes of single lanes.  (A list in LDS instead makes each
         * swap two dependent accesses of one lane, 259 cycles against 31;
         * a zone of 25 x 25 cells has 50 to 80 dense cells.) */
        int v0 = lane < m ? (int)a[lane] : 0, v1 = 0, j1 = 0;
        const int j0 = (lane >= 1 && lane < m) ? (int)draw((uint32_t)lane) : 0;
        if (m > 64) {
            if (64 + lane < m) {
                v1 = (int)a[64 + lane];
                j1 = (int)draw((uint32_t)(64 + lane));
            }
            for (int ii = m - 65; ii >= 0; --ii) {
                const int jj = wave_readlane(j1, ii), vi = wave_readlane(v1, ii);
                if (jj >= 64) {
                    const int vj = wave_readlane(v1, jj - 64);
                    v1 = wave_writelane(vj, ii, v1);
                    v1 = wave_writelane(vi, jj - 64, v1);
                } else {
                    const int vj = wave_readlane(v0, jj);
                    v1 = wave_writelane(vj, ii, v1);
                    v0 = wave_writelane(vi, jj, v0);
                }
            }
            if (64 + lane < m) a[64 + lane] = (T)v1;
        }
        v0 = shuffle64(v0, j0, imin(m, 64));
        if (lane < m) a[lane] = (T)v0;
        ZBAR();
        return;
    }
#endif
    for (int c0 = ((m - 1) / nl) * nl; c0 >= 0 && m > 1; c0 -= nl) {
        const int i = c0 + lane;
        const int j = (i >= 1 && i < m) ? (int)draw((uint32_t)i) : 0;
        const int hi = imin(m - 1, c0 + nl - 1);
        for (int ii = hi; ii >= imax(1, c0); --ii) {
            const int jj = wave_readlane(j, ii - c0);
            if (lane == 0) {
                const T t = a[ii];
                a[ii] = a[jj];
                a[jj] = t;
            }
        }
    }
    ZBAR();
}

/* ---- dense phase ---- */

/* Admissible targets of dense cell src within Chebyshev range 2 inside the
 * zone, ranked into the round-robin order of rank_dense_targets_unified
 * (zone_pass.cpp:413-490): 8 angular bins from a random start bin, each bin
 * sorted by the candidate key, then one per bin per round.  All lanes; the
 * order lands in z.scr->ord[0..nOrd) with each target's threshold in z.scr->ordThr.
 * Every draw is taken in one round: the tie breaks (t = 0..23, one per
 * neighbour offset) and the start bin (t = 24). */
template <class Z>
ZHD void dense_targets(Z& z, int src, int high, int pass, int phase, int lane, int nl) {
    const int sgx = lc_gx(z, src), sgy = lc_gy(z, src), sgc = lc_gc(z, src);
    for (int t = lane; t < 25; t += nl) {
        if (t < 24) {
            /* neighbour offsets in (dy outer, dx inner) order, centre skipped */
            const int f = t < 12 ? t : t + 1;
            const int dy = f / 5 - 2, dx = f % 5 - 2;
            int jx, jy, gc = -1;
            if (shift_idx(z, sgx, sgy, dx, dy, jx, jy)) {
                const int lc = zone_lc(z, jx, jy);
                if (lc >= 0 && !fget(z, lc, ZF_OUT) && (double)z.cell[lc].cnt < thr(z, lc, high)) gc = jy + z.g.Ny * jx;
            }
            z.scr->nbGc[t] = gc;
            if (gc >= 0) z.scr->nbTie[t] = mpcd_draw_tie(z.seed, pass, phase, (uint32_t)sgc, (uint32_t)gc);
        } else {
            z.sh->startBin = mpcd_draw_start_bin(z.seed, pass, phase, (uint32_t)sgc);
        }
    }
    ZBAR();
#if defined(__HIP_DEVICE_COMPILE__)
    {
        /* one wavefront: neighbour offset o = lane; each candidate stays in
         * its lane's registers and the ranking reads the others by readlane */
        bool keep = false;
        int gc = -1;
        if (lane < 24) {
            gc = z.scr->nbGc[lane];
            keep = gc >= 0;
            if (z.zp.dedupe)
                for (int q = 0; q < lane && keep; ++q)
                    if (z.scr->nbGc[q] == gc) keep = false;
        }
        const unsigned long long msk = wave_ballot(keep);
        const int m = wave_popc(msk);
        int lc = -1, bin = 0, cnt = 0, cheb = 0, dist2 = 0;
        double defn = 0.0, tie = 0.0, th = 0.0;
        if (keep) {
            const int jx = gc / z.g.Ny, jy = gc - jx * z.g.Ny;
            lc = zone_lc(z, jx, jy);
            int ddx, ddy;
            min_step(z, sgx, sgy, jx, jy, ddx, ddy);
            bin = zone_bin(z.zp, (ddy + 2) * 5 + (ddx + 2));
            th = thr(z, lc, high);
            cnt = z.cell[lc].cnt;
            defn = -dmax(0.0, th - (double)cnt);
            cheb = imax(ddx < 0 ? -ddx : ddx, ddy < 0 ? -ddy : ddy);
            dist2 = ddx * ddx + ddy * ddy;
            tie = z.scr->nbTie[lane];
        }
        if (lane == 0) z.sh->nOrd = m;
        if (m == 0) {
            ZBAR();
            return;
        }
        Cand me;
        me.deficitNeg = defn;
        me.cnt = cnt;
        me.cheb = cheb;
        me.dist2 = dist2;
        me.tie = tie;
        /* rank inside the bin: stable order of the candidate key */
        int r = 0;
        for (unsigned long long mm = msk; mm; mm &= mm - 1ull) {
            const int j = __builtin_ctzll(mm);
            Cand o;
            o.deficitNeg = wave_readlane_d(defn, j);
            o.cnt = wave_readlane(cnt, j);
            o.cheb = wave_readlane(cheb, j);
            o.dist2 = wave_readlane(dist2, j);
            o.tie = wave_readlane_d(tie, j);
            const int bj = wave_readlane(bin, j);
            if (keep && j != lane && bj == bin && (cand_less(o, me) || (j < lane && !cand_less(me, o)))) ++r;
        }
        /* round robin position: earlier rounds, then earlier bins from startBin */
        const int sb = z.sh->startBin;
        const int si = (bin - sb + 8) & 7;
        int pos = 0;
        for (unsigned long long mm = msk; mm; mm &= mm - 1ull) {
            const int j = __builtin_ctzll(mm);
            const int rj = wave_readlane(r, j);
            const int sj = (wave_readlane(bin, j) - sb + 8) & 7;
            if (rj < r || (rj == r && sj < si)) ++pos;
        }
        if (keep) {
            z.scr->ord[pos] = lc;
            z.scr->ordThr[pos] = th;
        }
        ZBAR();
    }
#else
    int base = 0;
    for (int b0 = 0; b0 < 24; b0 += nl) {
        const int o = b0 + lane;
        bool keep = false;
        int gc = -1;
        if (o < 24) {
            gc = z.scr->nbGc[o];
            keep = gc >= 0;
            if (z.zp.dedupe)
                for (int q = 0; q < o && keep; ++q)
                    if (z.scr->nbGc[q] == gc) keep = false;
        }
        const unsigned long long msk = wave_ballot(keep);
        if (keep) {
            Cand& c = z.scr->cand[base + wave_popc(msk & lanes_below(lane))];
            const int jx = gc / z.g.Ny, jy = gc - jx * z.g.Ny;
            const int lc = zone_lc(z, jx, jy);
            int ddx, ddy;
            min_step(z, sgx, sgy, jx, jy, ddx, ddy);
            c.lc = lc;
            c.gc = gc;
            c.bin = zone_bin(z.zp, (ddy + 2) * 5 + (ddx + 2));
            c.deficitNeg = -dmax(0.0, thr(z, lc, high) - (double)z.cell[lc].cnt);
            c.cnt = z.cell[lc].cnt;
            c.cheb = imax(ddx < 0 ? -ddx : ddx, ddy < 0 ? -ddy : ddy);
            c.dist2 = ddx * ddx + ddy * ddy;
            c.tie = z.scr->nbTie[o];
        }
        base += wave_popc(msk);
    }
    const int m = base;
    if (lane == 0) z.sh->nOrd = m;
    ZBAR();
    if (m == 0) return;
    /* rank inside the bin: stable order of the candidate key */
    for (int i = lane; i < m; i += nl) {
        const Cand ci = z.scr->cand[i];
        int r = 0;
        for (int j = 0; j < m; ++j) {
            if (j == i || z.scr->cand[j].bin != ci.bin) continue;
            if (cand_less(z.scr->cand[j], ci) || (j < i && !cand_less(ci, z.scr->cand[j]))) ++r;
        }
        z.scr->rnk[i] = r;
    }
    ZBAR();
    /* round robin position: earlier rounds, then earlier bins from startBin */
    const int sb = z.sh->startBin;
    for (int i = lane; i < m; i += nl) {
        const int ri = z.scr->rnk[i];
        const int si = (z.scr->cand[i].bin - sb + 8) & 7;
        int pos = 0;
        for (int j = 0; j < m; ++j) {
            const int rj = z.scr->rnk[j];
            if (rj < ri || (rj == ri && ((z.scr->cand[j].bin - sb + 8) & 7) < si)) ++pos;
        }
        const int lc = z.scr->cand[i].lc;
        z.scr->ord[pos] = lc;
        z.scr->ordThr[pos] = thr(z, lc, high);
    }
    ZBAR();
#endif
}

/* spread_particles_from_dense_source_round_robin (zone_pass.cpp:527-589),
 * lane 0.  The number of candidates at or after position kk
 * that still have a deficit is kept incrementally: within a sweep only the
 * candidate being served changes, and each target appears once. */
template <class Z>
ZHD int spread(Z& z, int src, int needOut, int pass, int* rv, int& nr) {
    int moved = 0;
    const int nOrd = z.sh->nOrd;
    if (needOut <= 0 || nOrd == 0) return 0;
    int avail = cnt_of(z, src);
    if (avail <= 0) return 0;
    while (needOut > 0 && avail > 0) {
        bool progressed = false;
        int R = 0;
        for (int jj = 0; jj < nOrd; ++jj)
            if (imax(0, (int)MPCD_FLOOR(z.scr->ordThr[jj] - (double)cnt_of(z, z.scr->ord[jj]))) > 0) ++R;
        for (int kk = 0; kk < nOrd; ++kk) {
            const int nb = z.scr->ord[kk];
            const int deficit = imax(0, (int)MPCD_FLOOR(z.scr->ordThr[kk] - (double)cnt_of(z, nb)));
            if (deficit <= 0) continue;
            const int remaining = R;
            --R;
            const int quota = imax(1, (int)MPCD_CEIL((double)needOut / (double)imax(1, remaining)));
            const int nt = imax(1, imin(imin(quota, deficit), imin(needOut, avail)));
            fset(z, src, ZF_CHG);
            for (int q = 0; q < nt; ++q) {
                const int k = head_of(z, src);
                const int nk = next_k(z, src, k);
                head_set(z, src, nk);
                if (nk < 0) tail_set(z, src, -1);
                mark_moved(z, k, pass);
                list_append(z, nb, k);
            }
            avail -= nt;
            cnt_set(z, nb, cnt_of(z, nb) + nt);
            bool seen = false;
            for (int k = 0; k < nr; ++k)
                if (rv[k] == nb) seen = true;
            if (!seen) rv[nr++] = nb;
            moved += nt;
            needOut -= nt;
            progressed = true;
            if (needOut <= 0 || avail <= 0) break;
        }
        if (!progressed) break;
    }
    if (moved > 0) cnt_set(z, src, avail);
    return moved;
}

#if defined(__HIP_DEVICE_COMPILE__)
/* ---- dense cells on the device: candidates and movers held in lanes ----
 *
 * Lane p holds candidate p of a ranking and lane q the q-th particle of the
 * source's list (a mover); everything the spread decides is computed by all
 * lanes from readlane values, so the wavefront follows one uniform control
 * path, and the moves and list links are written by the lanes at once.  The
 * results are those of dense_targets + spread + transfer_masks. */


/* value held by lane src (per-lane src) */
ZHD int lane_get(int v, int src) { return __shfl(v, src, 64); }
/* every lane's v to lane dst (dst a permutation of the lanes) */
ZHD int lane_put(int v, int dst) { return __builtin_amdgcn_ds_permute(dst << 2, v); }
ZHD double lane_put_d(double v, int dst) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)lane_put((int)(unsigned)b, dst);
    const unsigned hi = (unsigned)lane_put((int)(unsigned)(b >> 32), dst);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

/* values of the lanes of one's quad, rotated: rotation s hands lane m of a
 * quad the value of lane (m + s) & 3 */
template <int S>
ZHD int quad_rot(int v) {
    constexpr int ctrl = ((0 + S) & 3) | (((1 + S) & 3) << 2) | (((2 + S) & 3) << 4) | (((3 + S) & 3) << 6);
    return __builtin_amdgcn_mov_dpp(v, ctrl, 0xf, 0xf, true);
}
template <int S>
ZHD unsigned long long quad_rot64(unsigned long long v) {
    const unsigned lo = (unsigned)quad_rot<S>((int)(unsigned)v), hi = (unsigned)quad_rot<S>((int)(unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
ZHD int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

/* a periodic axis whose wrapped range-2 neighbours can lie in the zone */
template <class Z>
ZHD bool zone_wrap_x(const Z& z) {
    return z.g.perx && z.zw >= z.g.Nx - 1;
}
template <class Z>
ZHD bool zone_wrap_y(const Z& z) {
    return z.g.pery && z.zh >= z.g.Ny - 1;
}
/* zone-relative coordinate t taken once around an axis of n cells */
ZHD int wrap_near(int t, int n) { return t < 0 ? t + n : (t >= n ? t - n : t); }
/* Below five cells several offsets lead to one cell of a periodic axis, and
 * min_step's alone stands for it: the candidates come out as the general
 * form's dedupe leaves them, whose keys are those of the shortest step.  An
 * offset past half the axis never is; one that wraps is if it is under half
 * (at half of it the one that stays on the axis).  (On one wavefront in the
 * general form a launch of 4 x 1024 x 20 took 216 us, on the four 56; one of
 * 5 x 1024 x 20 takes 60.) */
template <class Z>
ZHD bool past_half(const Z& z, int dx, int dy) {
    return z.zp.odd && ((z.g.perx && 2 * (dx < 0 ? -dx : dx) > z.g.Nx) || (z.g.pery && 2 * (dy < 0 ? -dy : dy) > z.g.Ny));
}
template <class Z>
ZHD bool wrap_step(const Z& z, int d, int& t, int n) {
    const int t0 = t;
    t = wrap_near(t, n);
    return !z.zp.odd || t == t0 || 2 * (d < 0 ? -d : d) < n;
}

/* A dense cell's ranking lives in lanes by angular bin: lanes 4 b + m and
 * 32 + 4 b + m (m < 3) hold the m-th neighbour offset of bin b, the first for
 * the low thresholds (phase 0), the second for the high ones (phase 1).  A
 * candidate is compared with its bin's other members by quad rotations.  The
 * offsets of a bin differ in distance, which the key compares before the tie
 * draw, so no tie draw is ever looked at. */
struct DenseLane {
    int dx, dy, bin, code; /* code: Chebyshev << 4 | squared distance, -1 without an offset */
    double thB, thE;       /* threshold of an occupied and of an empty cell in this lane's phase */
};
template <class Z>
ZHD DenseLane dense_lane(const Z& z, int lane) {
    DenseLane d{0, 0, (lane >> 2) & 7, -1, 0.0, 0.0};
    int seen = 0;
    for (int idx = 0; idx < 25; ++idx) {
        if (idx == 12 || zone_bin(z.zp, idx) != d.bin) continue;
        if (seen == (lane & 3)) {
            d.dx = idx % 5 - 2;
            d.dy = idx / 5 - 2;
            const int ax = d.dx < 0 ? -d.dx : d.dx, ay = d.dy < 0 ? -d.dy : d.dy;
            d.code = (imax(ax, ay) << 4) | (ax * ax + ay * ay);
            if (past_half(z, d.dx, d.dy)) d.code = -1;
        }
        ++seen;
    }
    d.thB = lane < 32 ? z.zp.lowThrBulk : z.zp.highThr;
    d.thE = lane < 32 ? z.zp.lowLoc1 : z.zp.highLoc1;
    return d;
}

/* A dense cell's surplus over its high threshold (an occupied cell's is the
 * bulk one), and its start bins of both phases. */
template <class Z>
ZHD int dense_need(const Z& z, int nc) {
    return imax(0, (int)MPCD_CEIL((double)nc - z.zp.highThr));
}
/* The movers of a dense cell of nc particles fit the wavefront form,
 * min(need + 1, nc) <= 64, and so does the need itself (it exceeds the count
 * where the high threshold lies below zero). */
template <class Z>
ZHD bool dense_count_fits(const Z& z, int nc) {
    const int need = dense_need(z, nc);
    return imin(need + 1, nc) <= ZONE_MAX_MOVE && (!z.zp.odd || (need > 0 && need <= ZONE_MAX_MOVE));
}
/* (a cell that was empty when the pass took its thresholds has another than
 * dense_need's) */
template <class Z>
ZHD bool dense_fits(const Z& z, int c, int nc) {
    return dense_count_fits(z, nc) && (!z.zp.odd || fget(z, c, ZF_BULK0));
}
template <class Z>
ZHD unsigned dense_bins(const Z& z, int c, int pass) {
    const uint32_t gc = (uint32_t)lc_gc(z, c);
    return (unsigned)mpcd_draw_start_bin(z.seed, pass, 0, gc) | ((unsigned)mpcd_draw_start_bin(z.seed, pass, 1, gc) << 3);
}
/* a dense cell can receive: the low threshold lies above the high one */
template <class Z>
ZHD bool dense_receives(const Z& z) {
    return z.zp.odd && z.zp.lowThrBulk > z.zp.highThr;
}
/* both in the cell's lix entry (the surplus of a cell whose movers fit the
 * wavefront is 1 to 64; 0: it can still grow and is taken later) */
template <class Z>
ZHD void dense_word(Z& z, int c, int pass) {
    const int need = dense_receives(z) ? 0 : dense_need(z, cnt_of(z, c));
    z.lix[c] = (typename Z::idx_t)((unsigned)need | (dense_bins(z, c, pass) << 7));
}

/* lanes of `half` set in a ballot, as 32 bits */
ZHD unsigned half_bits(unsigned long long m, int half) { return (unsigned)(m >> (32 * half)); }
/* lanes of m (in half's 32) that the round-robin order puts before this lane
 * within one round: the bins from the start bin sb up to this lane's */
ZHD int round_before(unsigned m, int sb, int bin) {
    const unsigned rot = sb ? (m >> (4 * sb)) | (m << (32 - 4 * sb)) : m;
    return wave_popc((unsigned long long)(rot & ((1u << (4 * ((bin - sb) & 7))) - 1u)));
}

/* One sweep series of spread (zone_pass.cpp:527-589) over the ranking in the
 * lanes: assigns movers used.. to candidates (myT), chains the movers of one
 * candidate in order (nextQ), and keeps each candidate's first and last mover
 * and new count.  All values uniform except the per-lane ones. */
ZHD int spread_plan_wave(int nOrd, double thP, int& cP, int need, int& avail, int& used, int cap, int lane,
                         int& myT, int& nextQ, int& firstQ, int& lastQ) {
    int moved = 0;
    myT = -1;
    firstQ = -1;
    lastQ = -1;
    if (need <= 0 || nOrd == 0 || avail <= 0) return 0;
    while (need > 0 && avail > 0) {
        const int defP = lane < nOrd ? imax(0, (int)MPCD_FLOOR(thP - (double)cP)) : 0;
        unsigned long long mk = wave_ballot(defP > 0);
        if (mk == 0ull) break;
        int R = wave_popc(mk);
        bool stop = false;
        for (; mk; mk &= mk - 1ull) {
            const int kk = (int)__builtin_ctzll(mk);
            const int d = wave_readlane(defP, kk);
            const int remaining = R--;
            /* ceil(need / remaining), both positive and at most 64: need - 1/2
             * over remaining is at least 1/128 from an integer */
            const int quota = 1 + (int)(((float)need - 0.5f) / (float)remaining);
            /* cap (the staged movers) never binds: the callers stage
             * enough for both phases; it only keeps lanes in bounds */
            const int nt = imin(imax(1, imin(imin(quota, d), imin(need, avail))), cap - used);
            if (nt <= 0) {
                stop = true;
                break;
            }
            const int prev = wave_readlane(lastQ, kk);
            if (lane >= used && lane < used + nt) {
                myT = kk;
                nextQ = lane + 1 < used + nt ? lane + 1 : -1;
            }
            if (prev >= 0 && lane == prev) nextQ = used;
            if (lane == kk) {
                cP += nt;
                if (firstQ < 0) firstQ = used;
                lastQ = used + nt - 1;
            }
            used += nt;
            avail -= nt;
            need -= nt;
            moved += nt;
            if (need <= 0 || avail <= 0) {
                stop = true;
                break;
            }
        }
        if (stop) break;
    }
    return moved;
}

/* Applies a plan: records the movers' moves and appends them to their targets
 * in mover order; returns src's next head (src itself is left to the caller,
 * avail: its particles left). */
template <class Z>
ZHD int spread_apply_wave(Z& z, int src, int h, int lane, int moved, int avail, int pass, int myK, int myT, int nextQ,
                          int lcP, int cP, int firstQ, int lastQ) {
    if (moved <= 0) return h;
    /* src first: its next head is read before the movers' links are rewritten */
    const int nh = avail > 0 ? uniform(next_k(z, src, wave_readlane(myK, moved - 1))) : -1;
    const int nk = lane_get(myK, nextQ >= 0 ? nextQ : 0);
    const int fk = lane_get(myK, firstQ >= 0 ? firstQ : 0);
    const int lk = lane_get(myK, lastQ >= 0 ? lastQ : 0);
    /* a target that takes back particles of its own input run (lane q: mover q) */
    const int tl = lane_get(lcP, myT >= 0 ? myT : 0);
    for (unsigned long long bk = wave_ballot(myT >= 0 && in_run(z, tl, myK)); bk; bk &= bk - 1ull) {
        const int lt = wave_readlane(tl, (int)__builtin_ctzll(bk));
        if (lane == 0) ensure_mat(z, lt);
        ZWSYNC();
    }
    ZWSYNC();
    if (myT >= 0) {
        mark_moved(z, myK, pass);
        nx_set(z, myK, nextQ >= 0 ? nk : -1);
    }
    if (firstQ >= 0) {
        const int t = tail_of(z, lcP);
        if (t < 0) head_set(z, lcP, fk);
        else nx_set(z, t, fk);
        tail_set(z, lcP, lk);
        fset(z, lcP, ZF_CHG);
        cnt_set(z, lcP, cP);
    }
    ZWSYNC();
    return nh;
}

/* The first n (<= 64) entries of a list, entry q in lane q: what is left of
 * the run by its indices, the rest along the links (the list holds at least
 * n entries). */
template <class Z>
ZHD int list_entry_wave(const Z& z, int h, int left, int n, int lane) {
    int v = lane < left ? h + lane : -1;
    if (n > left) {
        int k = left > 0 ? nx_get(z, h + left - 1) : h;
        for (int q = left; q < n; ++q) {
            if (lane == q) v = k;
            if (q + 1 < n) k = nx_get(z, k);
        }
    }
    return lane < n ? v : -1;
}

/* One dense cell (zone_pass.cpp:738-779: both target phases, the spreads and
 * the transfer masks) when its movers fit the wavefront:
 * min(need + 1, count) <= 64 (phase 1 moves at most what phase 0 left of
 * need, up to one more by the rounding of its ceil).  bins: dense_bins.
 * Returns the number of particles moved.
 *
 * The ranking (zone_pass.cpp:413-490): rank within the bin by (deficit,
 * count, distances); the round-robin order is by rank, then by bin from the
 * start bin.  When the need is at most the number R of targets with a
 * deficit of one or more, every quota of the spread is ceil(need /
 * remaining) = 1; when no such target has a deficit of two or more, each
 * takes what it can, one.  In both cases the first min(need, R) targets in
 * order take one particle each: no sweep, each receiving lane appends its
 * own particle.  Nine cells of ten of a uniform state go that way.
 *
 * The chain of conflicting cells bounds the passes, so what matters is the
 * instructions between two of its cells: one LDS read per candidate (the
 * cell's state in 8 bytes), three rotations, three ballots, one batch of
 * writes. */
template <class Z>
ZHD int dense_cell_wave(Z& z, const DenseLane& dl, int c, int cx, int cy, int need, unsigned bins, int pass, int lane) {
    typedef typename Z::idx_t IT;
    int tx = cx + dl.dx, ty = cy + dl.dy;
    bool in = dl.code >= 0;
    if (zone_wrap_x(z)) in = in & wrap_step(z, dl.dx, tx, z.g.Nx);
    if (zone_wrap_y(z)) in = in & wrap_step(z, dl.dy, ty, z.g.Ny);
    in = in & ((unsigned)tx < (unsigned)z.zw) & ((unsigned)ty < (unsigned)z.zh);
    const int l = in ? tx * z.zh + ty : c;
    const ZCell<IT> S = z.cell[c];
    const unsigned fS = (unsigned)S.fl;
    int h = uniform(iget(S.head)), avail = uniform((int)S.cnt), moved = 0;
    const int kb = (int)z.k0[c], ke = run_end(z, c);
    int left = uniform((fS & ZF_MAT) || h < kb || h > ke ? 0 : ke - h + 1);
    bool rcvF = false;
    int rg0 = -1, rg1 = -1;
    bool masked = false, allBulk = false;
#pragma nounroll
    for (int half = 0; half < 2; ++half) {
        const ZCell<IT> T = z.cell[l];
        const int cT = (int)T.cnt, tT = iget(T.tail);
        const unsigned fT = (unsigned)T.fl;
        const double th = z.zp.useLocal ? (lane < 32 ? z.lowA[l] : z.highA[l]) : ((fT & ZF_BULK0) ? dl.thB : dl.thE);
        const double def = th - (double)cT;
        const bool keep = in & !(fT & ZF_OUT) & ((lane >> 5) == half) & (def > 0.0);
        /* the key: deficits are positive, so their bits are ordered as their
         * values; a lane without a candidate is never ahead of one */
        const unsigned long long dk = keep ? (unsigned long long)__double_as_longlong(def) : 0ull;
        const unsigned sm = ((unsigned)cT << 8) | (unsigned)(dl.code & 255);
        int r = 0;
        {
            const unsigned long long o1 = quad_rot64<1>(dk), o2 = quad_rot64<2>(dk), o3 = quad_rot64<3>(dk);
            const unsigned s1 = (unsigned)quad_rot<1>((int)sm), s2 = (unsigned)quad_rot<2>((int)sm),
                           s3 = (unsigned)quad_rot<3>((int)sm);
            r += (int)((o1 > dk) | ((o1 == dk) & (s1 < sm)));
            r += (int)((o2 > dk) | ((o2 == dk) & (s2 < sm)));
            r += (int)((o3 > dk) | ((o3 == dk) & (s3 < sm)));
        }
        const int sb = (int)((bins >> (3 * half)) & 7u);
        const bool pd = keep & (def >= 1.0); /* floor(deficit) > 0 */
        const unsigned q0 = half_bits(wave_ballot(pd & (r == 0)), half), q1 = half_bits(wave_ballot(pd & (r == 1)), half),
                       q2 = half_bits(wave_ballot(pd & (r == 2)), half);
        const int n0 = wave_popc(q0), n1 = wave_popc(q1), R = n0 + n1 + wave_popc(q2);
        const bool deep = wave_ballot(pd & (def >= 2.0)) != 0ull;
        if ((need <= R || !deep) && need <= avail) {
            const int mv = imin(need, R);
            if (mv > 0) {
                const int e = (r > 0 ? n0 : 0) + (r > 1 ? n1 : 0) +
                              round_before(r == 0 ? q0 : (r == 1 ? q1 : q2), sb, dl.bin);
                const bool rcv = pd & (e < mv);
                avail -= mv;
                /* the e-th particle of the cell's list, and the list's next head */
                int k, nh = -1;
                bool mat = false;
                if (mv <= left) {
                    k = h + e;
                    if (mv < left) nh = h + mv;
                    else if (avail > 0) nh = uniform(nx_get(z, h + left - 1));
                } else {
                    const int v = list_entry_wave(z, h, left, mv, lane);
                    k = lane_get(v, rcv ? e : 0);
                    if (avail > 0) nh = uniform(next_k(z, c, wave_readlane(v, mv - 1)));
                    /* a particle an earlier pass moved may come home: the target's run gets its links first */
                    for (unsigned long long bk = wave_ballot(rcv & !(fT & ZF_MAT) & (k >= (int)z.k0[l]) & (k <= run_end(z, l)));
                         bk; bk &= bk - 1ull) {
                        if (lane == (int)__builtin_ctzll(bk)) {
                            ensure_mat(z, l);
                            mat = true;
                        }
                        ZWSYNC();
                    }
                }
                /* the cell is done when phase 1 finds nothing above the
                 * threshold; then its masks are known here */
                const int rem = half ? 0 : uniform(dense_need(z, avail));
                unsigned f = fT | ZF_CHG | (mat ? (unsigned)ZF_MAT : 0u);
                if (rem <= 0 && moved == 0) {
                    allBulk = (uniform((int)fS) & ZF_BULK0) && wave_ballot(rcv & !(fT & ZF_BULK0)) == 0ull;
                    f |= ZF_RECV | (allBulk ? ZF_BB : ZF_SKIP);
                    if (!allBulk) f &= ~(unsigned)ZF_BB;
                    masked = true;
                } else {
                    rcvF = rcvF | rcv;
                }
                if (rcv) {
                    nx_set(z, k, -1);
                    if (tT < 0) head_set(z, l, k);
                    else nx_set(z, tT, k);
                    z.cell[l].cnt = (IT)(cT + 1);
                    z.cell[l].tail = (IT)k;
                    z.cell[l].fl = (IT)f;
                    mark_moved(z, k, pass);
                }
                ZWSYNC();
                h = nh;
                left = imax(0, left - mv);
                moved += mv;
            }
        } else {
            /* more need than such targets and a deficit of two or more: the
             * ranking in order into lanes 0..m-1, then the sweeps */
            const unsigned k0 = half_bits(wave_ballot(keep & (r == 0)), half), k1 = half_bits(wave_ballot(keep & (r == 1)), half),
                           k2 = half_bits(wave_ballot(keep & (r == 2)), half);
            const int m0 = wave_popc(k0), m1 = wave_popc(k1), m = m0 + m1 + wave_popc(k2);
            const int pos = (r > 0 ? m0 : 0) + (r > 1 ? m1 : 0) + round_before(r == 0 ? k0 : (r == 1 ? k1 : k2), sb, dl.bin);
            const unsigned long long rest = ~wave_ballot(keep); /* taken by all lanes, outside the choice */
            const int dst = keep ? pos : m + wave_popc(rest & lanes_below(lane));
            const int lcP = lane_put(l, dst);
            int cP = lane_put(cT, dst);
            const double thP = lane_put_d(th, dst);
            const int nStage = imin(need, avail);
            const int myK = list_entry_wave(z, h, left, nStage, lane);
            int used = 0, myT = -1, nextQ = -1, firstQ = -1, lastQ = -1;
            const int mv = spread_plan_wave(m, thP, cP, need, avail, used, nStage, lane, myT, nextQ, firstQ, lastQ);
            h = spread_apply_wave(z, c, h, lane, mv, avail, pass, myK, myT, nextQ, lcP, cP, firstQ, lastQ);
            left = imax(0, left - mv);
            moved += mv;
            const int rc = firstQ >= 0 ? lcP : -1;
            if (half) rg1 = rc;
            else rg0 = rc;
        }
        /* phase 1: high thresholds, for what is left above the high threshold */
        need = uniform(dense_need(z, avail));
        if (need <= 0) break;
    }
    /* transfer masks (zone_pass.cpp:492-525) over both phases' receivers */
    if (!masked) {
        const bool nonBulk = (rcvF && !fget(z, l, ZF_BULK0)) || (rg0 >= 0 && !fget(z, rg0, ZF_BULK0)) ||
                             (rg1 >= 0 && !fget(z, rg1, ZF_BULK0));
        allBulk = (uniform((int)fS) & ZF_BULK0) && wave_ballot(nonBulk) == 0ull;
        const unsigned setb = ZF_RECV | (allBulk ? ZF_BB : ZF_SKIP), keepb = allBulk ? ~0u : ~(unsigned)ZF_BB;
        if (rcvF) z.cell[l].fl = (IT)(((unsigned)z.cell[l].fl | setb) & keepb);
        ZWSYNC();
        if (rg0 >= 0) z.cell[rg0].fl = (IT)(((unsigned)z.cell[rg0].fl | setb) & keepb);
        ZWSYNC();
        if (rg1 >= 0) z.cell[rg1].fl = (IT)(((unsigned)z.cell[rg1].fl | setb) & keepb);
    }
    if (lane == 0) {
        unsigned f = fS | (moved > 0 ? (unsigned)ZF_CHG : 0u) | (allBulk ? ZF_BB : ZF_SKIP);
        if (!allBulk) f &= ~(unsigned)ZF_BB;
        ZCell<IT> w;
        w.cnt = (IT)avail;
        w.head = (IT)h;
        w.tail = avail > 0 ? S.tail : (IT)-1;
        w.fl = (IT)f;
        z.cell[c] = w;
    }
    ZWSYNC();
    return moved;
}
#endif

/* Dense passes (zone_pass.cpp:708-781), all lanes. */
template <class Z>
ZHD void zone_dense_passes(Z& z, int lane, int nl) {
#if defined(__HIP_DEVICE_COMPILE__)
    int nHighW = 0, movedW = 0;
    const DenseLane dlane = dense_lane(z, lane);
#endif
    for (int pass = 1; pass <= z.zp.maxPasses; ++pass) {
        for (int lc = lane; lc < z.C; lc += nl) zone_maps(z, lc, 0);
        ZBAR();
        const int m = zone_compact(z, lane, nl, ZC_DENSE);
        ZBAR();
        zone_shuffle(z.dl, m, lane, nl, ShufDraw{z.seed, ZS_DENSE, (uint32_t)pass, 0u});
        for (int k = 0; k < m; ++k) {
            const int c = (int)z.dl[k];
            const int nc = cnt_of(z, c);
            if (nc <= 0) continue;
            const double hl = high_thr(z, c);
            if ((double)nc <= hl) continue;
            const int needOut = imax(0, (int)MPCD_CEIL((double)nc - hl));
#if defined(__HIP_DEVICE_COMPILE__)
            if (z.zp.quadBins && dense_fits(z, c, nc)) {
                ++nHighW;
                const int cx = lc_col(z, c);
                movedW += dense_cell_wave(z, dlane, c, cx, c - cx * z.zh, needOut, dense_bins(z, c, pass), pass, lane);
                continue;
            }
#endif
            int moved = 0;
            if (lane == 0) {
                ++z.sh->nHigh;
                z.sh->nr = 0;
            }
            if (needOut > 0) {
                dense_targets(z, c, 0, pass, 0, lane, nl);
                if (lane == 0) {
                    int nr = 0;
                    moved += spread(z, c, needOut, pass, z.scr->recvT, nr);
                    z.sh->nr = nr;
                }
                ZBAR();
                const int remaining = imax(0, (int)MPCD_CEIL((double)cnt_of(z, c) - hl));
                if (remaining > 0) {
                    dense_targets(z, c, 1, pass, 1, lane, nl);
                    if (lane == 0) {
                        int nr = z.sh->nr;
                        moved += spread(z, c, remaining, pass, z.scr->recvT, nr);
                        z.sh->nr = nr;
                    }
                }
            }
            if (lane == 0) {
                const int nr = z.sh->nr;
                for (int r = 0; r < nr; ++r) fset(z, z.scr->recvT[r], ZF_RECV);
                transfer_masks(z, c, z.scr->recvT, nr);
                z.sh->movedDense += moved;
            }
            ZBAR();
        }
    }
#if defined(__HIP_DEVICE_COMPILE__)
    if (lane == 0) {
        z.sh->nHigh += nHighW;
        z.sh->movedDense += movedW;
    }
    ZBAR();
#endif
}

#if defined(__HIP_DEVICE_COMPILE__)
/* Order-preserving compaction into z.dl by the four wavefronts from the
 * ballots of each 64-cell chunk (at most 64 chunks); its first ZONE_TMP_L
 * entries also go to scr->tmpL.  Returns the count. */
template <class Z>
__device__ __forceinline__ int zone_compact_mw(Z& z, const unsigned long long* chunkMask, int wave, int lane) {
    const int nch = (z.C + 63) >> 6;
    const int pc = lane < nch ? wave_popc(chunkMask[lane]) : 0;
    const int incl = wave_shfl_up_add(pc, lane);
    for (int ch = wave; ch < nch; ch += 4) {
        const unsigned long long msk = chunkMask[ch];
        const int base = wave_readlane(incl - pc, ch);
        if ((msk >> lane) & 1ull) {
            const int j = base + wave_popc(msk & lanes_below(lane));
            z.dl[j] = (typename Z::idx_t)(ch * 64 + lane);
            if (j < ZONE_TMP_L) z.scr->tmpL[j] = (typename Z::idx_t)(ch * 64 + lane);
        }
    }
    return wave_readlane(incl, 63);
}

/* The dense passes on the four wavefronts of a 256-thread workgroup
 * (device only).  A dense cell's spread reads counts within Chebyshev range 2
 * of it and writes the lists, counts and flags of itself and of targets
 * within range 2; its own count changes only by itself (a dense cell is above
 * its high threshold, a target below it).  Cells of the shuffled list more
 * than 4 cells apart therefore touch disjoint cells and commute.  A cell
 * whose movers exceed a wavefront takes the one-lane form, which uses the
 * zone's shared scratch.
 *
 * The wavefronts take the cells in list order from a counter in LDS; a cell
 * starts once every earlier cell within Chebyshev range 4 is done.  Those are
 * found through pos (the list position of each zone cell), and a finished
 * cell sets its word in done (both in ext, idle in the dense passes).
 * Conflicting cells thus keep the list order and the result is the serial
 * loop's bit for bit, while a wavefront waits only for the cells its own
 * depends on, after everything that does not depend on them.
 * Cells are taken in increasing order and wait only on smaller positions,
 * which are taken already, so the smallest unfinished cell can always run;
 * each wait is bounded all the same (past DS_WAIT_MAX polls it records
 * schedWait, which the kernel reports as an error, and goes on).  A list with
 * a cell that needs the one-lane form (its movers exceed a wavefront, or the
 * grid has no quadBins) or an empty one, or a list that leaves ext no room for
 * pos and done runs on wavefront 0 alone, in list order.  With the low
 * threshold above the high one a dense cell receives too, up to the low
 * threshold: it takes its surplus after its wait, and the list is scheduled
 * if a cell of that many particles fits a wavefront (200 x 100 x 12 with 16
 * above 13.2: 898 us a step, 1328 on one wavefront).
 *
 * What a cell writes lies in LDS, whose accesses the release and acquire
 * order; a zone whose links spill to its global region orders those too. */
constexpr int ZONE_WAVES = 4;
constexpr int DS_WAIT_MAX = 1 << 22;

template <class Z>
__device__ __forceinline__ void sched_release(const Z& z) {
    if (z.P > z.nL) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
}
template <class Z>
__device__ __forceinline__ void sched_acquire(const Z& z) {
    if (z.P > z.nL) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <class Z>
__device__ __forceinline__ void zone_dense_passes_mw(Z& z, int wave, int lane) {
    typedef typename Z::idx_t IT;
    constexpr int NT = 64 * ZONE_WAVES;
    constexpr unsigned NONE = (unsigned)(IT)~(IT)0;
    const int tid = wave * 64 + lane;
    int nHighW = 0, movedW = 0;
    const DenseLane dlane = dense_lane(z, lane);
    if (tid == 0) z.sh->schedWait = 0;
    const int nExt = (z.zw + 4) * (z.zh + 4);
    const bool wrapX = zone_wrap_x(z), wrapY = zone_wrap_y(z);
    /* the 9 x 9 window of a cell: lane t checks offsets t and t + 64 of the 81 */
    const int wx0 = lane / 9 - 4, wy0 = lane % 9 - 4, wx1 = (lane + 64) / 9 - 4, wy1 = (lane + 64) % 9 - 4;
    IT* const pos = z.ext;
    volatile IT* const done = z.ext + z.C;
    unsigned long long* const chunkMask = reinterpret_cast<unsigned long long*>(z.scr->cand); /* idle here */
    for (int pass = 1; pass <= z.zp.maxPasses; ++pass) {
        /* thresholds and the list: chunk ch of 64 cells on wavefront ch % 4 */
        bool one = false;
        for (int ch = wave; ch * 64 < z.C; ch += ZONE_WAVES) {
            const int lc = ch * 64 + lane;
            bool f = false;
            if (lc < z.C) {
                zone_maps(z, lc, 0);
                pos[lc] = (IT)NONE;
                const int nc = cnt_of(z, lc);
                f = (double)nc > high_thr(z, lc) && !fget(z, lc, ZF_OUT);
                one = one || (f && !dense_fits(z, lc, nc));
            }
            const unsigned long long msk = wave_ballot(f);
            if (lane == 0) chunkMask[ch] = msk;
        }
        for (int k = z.C + tid; k < nExt; k += NT) z.ext[k] = (IT)0;
        bool serial = __syncthreads_or(one) || !z.zp.quadBins ||
                      (dense_receives(z) && !dense_count_fits(z, (int)MPCD_CEIL(z.zp.lowThrBulk)));
        const int m = zone_compact_mw(z, chunkMask, wave, lane);
        serial = serial || m + z.C > nExt;
        __syncthreads();
        /* wavefront 0 shuffles; the others meanwhile take each listed cell's
         * surplus and start bins, from the copy of a list that fits it */
        const bool early = m <= ZONE_TMP_L;
        if (wave > 0) {
            if (!serial && early)
                for (int k = tid - 64; k < m; k += NT - 64) dense_word(z, (int)z.scr->tmpL[k], pass);
        } else {
            zone_shuffle(z.dl, m, lane, 64, ShufDraw{z.seed, ZS_DENSE, (uint32_t)pass, 0u});
            if (!serial)
                for (int k = lane; k < m; k += 64) pos[(int)z.dl[k]] = (IT)k;
            if (lane == 0) z.sh->mwNext = 0;
        }
        __syncthreads();
        if (!serial && !early) {
            for (int k = tid; k < m; k += NT) dense_word(z, (int)z.dl[k], pass);
            __syncthreads();
        }
        if (!serial || wave == 0) {
            /* the next position is taken one cell ahead */
            int kv = 0;
            if (lane == 0) kv = atomicAdd(&z.sh->mwNext, 1);
            for (;;) {
                const int k = uniform(kv);
                if (k >= m) break;
                if (lane == 0) kv = atomicAdd(&z.sh->mwNext, 1);
                const int c = uniform((int)z.dl[k]);
                const int cx = lc_col(z, c), cy = c - cx * z.zh;
                if (!serial) {
                    ++nHighW;
                    int x0 = cx + wx0, y0 = cy + wy0, x1 = cx + wx1, y1 = cy + wy1;
                    if (wrapX) {
                        x0 = wrap_near(x0, z.g.Nx);
                        x1 = wrap_near(x1, z.g.Nx);
                    }
                    if (wrapY) {
                        y0 = wrap_near(y0, z.g.Ny);
                        y1 = wrap_near(y1, z.g.Ny);
                    }
                    /* outside the zone: the cell itself, which is not earlier */
                    const bool i0 = ((unsigned)x0 < (unsigned)z.zw) & ((unsigned)y0 < (unsigned)z.zh);
                    const bool i1 = (lane < 17) & ((unsigned)x1 < (unsigned)z.zw) & ((unsigned)y1 < (unsigned)z.zh);
                    const int q0 = (int)pos[i0 ? x0 * z.zh + y0 : c], q1 = (int)pos[i1 ? x1 * z.zh + y1 : c];
                    const unsigned nb = (unsigned)uniform((int)z.lix[c]);
                    const bool w0 = q0 < k, w1 = q1 < k;
                    const int d0 = w0 ? q0 : 0, d1 = w1 ? q1 : 0;
                    for (int polls = 0;; ++polls) {
                        const int v0 = (int)done[d0], v1 = (int)done[d1];
                        if (wave_ballot((w0 & (v0 == 0)) | (w1 & (v1 == 0))) == 0ull) break;
                        if (polls >= DS_WAIT_MAX) {
                            if (lane == 0) z.sh->schedWait = 1;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                    sched_acquire(z);
                    int need = (int)(nb & 127u);
                    if (z.zp.odd && need == 0) need = uniform(dense_need(z, cnt_of(z, c)));
                    movedW += dense_cell_wave(z, dlane, c, cx, cy, need, nb >> 7, pass, lane);
                    sched_release(z);
                    if (lane == 0) done[k] = (IT)1;
                    ZWSYNC();
                    continue;
                }
                const int nc = cnt_of(z, c);
                const double hl = high_thr(z, c);
                if (nc <= 0 || (double)nc <= hl) continue;
                ++nHighW;
                const int needOut = imax(0, (int)MPCD_CEIL((double)nc - hl));
                if (z.zp.quadBins && dense_fits(z, c, nc)) {
                    movedW += dense_cell_wave(z, dlane, c, cx, cy, needOut, dense_bins(z, c, pass), pass, lane);
                } else {
                    /* the one-lane form (serial lists only: wavefront 0, the
                     * zone's shared scratch) */
                    int moved = 0;
                    if (lane == 0) z.sh->nr = 0;
                    dense_targets(z, c, 0, pass, 0, lane, 64);
                    if (lane == 0) {
                        int nr = 0;
                        moved += spread(z, c, needOut, pass, z.scr->recvT, nr);
                        z.sh->nr = nr;
                    }
                    ZBAR();
                    const int remaining = imax(0, (int)MPCD_CEIL((double)cnt_of(z, c) - hl));
                    if (remaining > 0) {
                        dense_targets(z, c, 1, pass, 1, lane, 64);
                        if (lane == 0) {
                            int nr = z.sh->nr;
                            moved += spread(z, c, remaining, pass, z.scr->recvT, nr);
                            z.sh->nr = nr;
                        }
                    }
                    if (lane == 0) {
                        const int nr = z.sh->nr;
                        for (int r = 0; r < nr; ++r) fset(z, z.scr->recvT[r], ZF_RECV);
                        transfer_masks(z, c, z.scr->recvT, nr);
                        z.sh->movedDense += moved;
                    }
                    ZBAR();
                }
            }
        }
        __syncthreads();
    }
    if (lane == 0) {
        atomicAdd(&z.sh->nHigh, nHighW);
        atomicAdd(&z.sh->movedDense, movedW);
    }
    __syncthreads();
}
#else
/* (the host passes of the compilers see a declaration only) */
template <class Z>
ZHD void zone_dense_passes_mw(Z&, int, int) {}
#endif

/* ---- sparse phase ---- */

/* inward_direction_from_local_gradient (zone_pass.cpp:375-411) on the
 * sparse-phase count copy; the four smoothed counts in parallel. */
template <class Z>
ZHD void inward_dir(Z& z, int gx, int gy, int lane, int nl, double& dxo, double& dyo) {
    const int Nx = z.g.Nx, Ny = z.g.Ny;
    /* x pair (xa - xb) * fx, y pair (ya - yb) * fy */
    int xa, xb, ya, yb;
    double fx, fy;
    if (z.g.perx) { xa = wrapi(gx + 1, Nx); xb = wrapi(gx - 1, Nx); fx = 0.5; }
    else if (gx == 0) { xa = gx + 1; xb = gx; fx = 1.0; }
    else if (gx == Nx - 1) { xa = gx; xb = gx - 1; fx = 1.0; }
    else { xa = gx + 1; xb = gx - 1; fx = 0.5; }
    if (z.g.pery) { ya = wrapi(gy + 1, Ny); yb = wrapi(gy - 1, Ny); fy = 0.5; }
    else if (gy == 0) { ya = gy + 1; yb = gy; fy = 1.0; }
    else if (gy == Ny - 1) { ya = gy; yb = gy - 1; fy = 1.0; }
    else { ya = gy + 1; yb = gy - 1; fy = 0.5; }
    for (int t = lane; t < 4; t += nl) {
        const int qx = (t == 0) ? xa : (t == 1) ? xb : gx;
        const int qy = (t == 2) ? ya : (t == 3) ? yb : gy;
        z.scr->nsm4[t] = nsm_ext(z, qx, qy);
    }
    ZBAR();
    dxo = (fx == 0.5) ? 0.5 * (z.scr->nsm4[0] - z.scr->nsm4[1]) : (z.scr->nsm4[0] - z.scr->nsm4[1]);
    dyo = (fy == 0.5) ? 0.5 * (z.scr->nsm4[2] - z.scr->nsm4[3]) : (z.scr->nsm4[2] - z.scr->nsm4[3]);
}

/* One donor transfer of the sparse phase (zone_pass.cpp:818-850): copy
 * donor d's list into tmp (LDS or the zone's global region), Fisher-Yates
 * it, move the first nt to low cell c; all lanes. */
template <class Z, class T>
ZHD void donor_transfer(Z& z, int c, int d, int md, int nt, int cgc, T* tmp, int lane, int nl) {
    typedef typename Z::idx_t IT;
    /* copy the donor list, Fisher-Yates it, move the first nt */
    {
        const int h = head_of(z, d), left = imin(md, run_left(z, d, h));
        for (int q = lane; q < left; q += nl) tmp[q] = (IT)(h + q);
        if (lane == 0) {
            int kk = left > 0 ? (left < md ? nx_get(z, h + left - 1) : -1) : h;
            for (int q = left; q < md; ++q) {
                tmp[q] = (IT)kk;
                kk = nx_get(z, kk);
            }
        }
    }
    ZBAR();
    const int dgc = lc_gc(z, d);
    zone_shuffle(tmp, md, lane, nl,
                 ShufDraw{z.seed, ZS_PARTICLE, (uint32_t)cgc, (uint32_t)dgc});
    /* c's own particles among the movers: its run's links come first */
    bool back = false;
    for (int q = lane; q < nt; q += nl) back = back || in_run(z, c, (int)tmp[q]);
    if (wave_ballot(back) != 0ull) {
        if (lane == 0) ensure_mat(z, c);
        ZBAR();
    }
    /* the movers' records, links of the moved run and of the donor's
     * remaining run, all lanes */
    for (int q = lane; q < md; q += nl) {
        const int kq = (int)tmp[q];
        if (q < nt) {
            mark_moved(z, kq, ZM_SPARSE);
            nx_set(z, kq, q + 1 < nt ? (int)tmp[q + 1] : -1);
        } else {
            nx_set(z, kq, q + 1 < md ? (int)tmp[q + 1] : -1);
        }
    }
    ZBAR();
    if (lane == 0) {
        const int tc = tail_of(z, c);
        if (tc < 0) head_set(z, c, (int)tmp[0]);
        else nx_set(z, tc, (int)tmp[0]);
        tail_set(z, c, (int)tmp[nt - 1]);
        fset(z, c, ZF_CHG);
        fset(z, d, ZF_MAT | ZF_CHG);
        head_set(z, d, md > nt ? (int)tmp[nt] : -1);
        tail_set(z, d, md > nt ? (int)tmp[md - 1] : -1);
        cnt_set(z, d, md - nt);
        cnt_set(z, c, cnt_of(z, c) + nt);
        fset(z, c, ZF_RECV);
        const int rv1[1] = {c};
        transfer_masks(z, d, rv1, 1);
    }
    ZBAR();
}

/* One low cell of the sparse phase (zone_pass.cpp:804-854): its donors among
 * the zone neighbours at range 1, ranked, and the transfers; all lanes of
 * one wavefront.  Returns the particles moved into c. */
template <class Z>
ZHD int sparse_cell(Z& z, int c, int nc, int lowInt, int lane, int nl) {
    const int cgx = lc_gx(z, c), cgy = lc_gy(z, c), cgc = lc_gc(z, c);
    /* zone neighbours at range 1 (local_neighbors_in_zone :263-278) */
    for (int o = lane; o < 8; o += nl) {
        const int f = o < 4 ? o : o + 1;
        const int dy = f / 3 - 1, dx = f % 3 - 1;
        int jx, jy, q = -1;
        if (shift_idx(z, cgx, cgy, dx, dy, jx, jy)) q = zone_lc(z, jx, jy);
        if (q >= 0 && fget(z, q, ZF_OUT)) q = -1;
        z.scr->nbGc[o] = q;
    }
    ZBAR();
    int nn = 0, nd = 0;
    for (int b0 = 0; b0 < 8; b0 += nl) {
        const int o = b0 + lane;
        bool keep = false;
        if (o < 8) {
            const int q = z.scr->nbGc[o];
            keep = q >= 0;
            if (z.zp.dedupe)
                for (int t = 0; t < o && keep; ++t)
                    if (z.scr->nbGc[t] == q) keep = false;
        }
        const unsigned long long mk = wave_ballot(keep);
        nn += wave_popc(mk);
        const bool don = keep && cnt_of(z, z.scr->nbGc[o]) > lowInt;
        const unsigned long long mdn = wave_ballot(don);
        if (don) z.scr->dord[nd + wave_popc(mdn & lanes_below(lane))] = z.scr->nbGc[o];
        nd += wave_popc(mdn);
    }
    ZBAR();
    if (nn == 0) return 0;
    int need = imax(0, lowInt - nc);
    if (need <= 0 || nd == 0) return 0;
    double gxd, gyd;
    inward_dir(z, cgx, cgy, lane, nl, gxd, gyd);
    /* rank_admissible_neighbors_inward (zone_pass.cpp:636-667) */
    zone_shuffle(z.scr->dord, nd, lane, nl, ShufDraw{z.seed, ZS_DONOR, (uint32_t)cgc, 0u});
    const double ndir = mpcd_hypot(gxd, gyd);
    for (int t = lane; t < nd; t += nl) {
        const int q = z.scr->dord[t];
        int ddx, ddy;
        min_step(z, cgx, cgy, lc_gx(z, q), lc_gy(z, q), ddx, ddy);
        const double nstep = mpcd_hypot((double)ddx, (double)ddy);
        double align = 0.0;
        if (ndir >= 1e-14 && nstep >= 1e-14) align = ((double)ddx * gxd + (double)ddy * gyd) / (ndir * nstep);
        const double noise = 1e-9 * mpcd_draw_donor_noise(z.seed, (uint32_t)cgc, (uint32_t)lc_gc(z, q));
        z.scr->dsc[t] = 100.0 * align + nsm_ext(z, lc_gx(z, q), lc_gy(z, q)) + noise;
    }
    ZBAR();
    for (int t = lane; t < nd; t += nl) { /* stable, descending score */
        int r = 0;
        for (int u = 0; u < nd; ++u)
            if (z.scr->dsc[u] > z.scr->dsc[t] || (u < t && !(z.scr->dsc[t] > z.scr->dsc[u]))) ++r;
        z.scr->dord2[r] = z.scr->dord[t];
    }
    ZBAR();
    int moved = 0;
    for (int t = 0; t < nd; ++t) {
        const int d = z.scr->dord2[t];
        const int md = cnt_of(z, d);
        if (md <= 0) continue;
        const int avail = md - lowInt;
        if (avail <= 0) continue;
        const int nt = imin(imin(need, avail), md);
        if (nt <= 0) continue;
        if (md <= ZONE_TMP_L) donor_transfer(z, c, d, md, nt, cgc, z.scr->tmpL, lane, nl);
        else donor_transfer(z, c, d, md, nt, cgc, z.tmpG, lane, nl);
        moved += nt;
        need -= nt;
        if (need <= 0) break;
    }
    return moved;
}

/* the sparse phase's set-up: maps, and the counts it starts from (the zone
 * and its ring) in z.ext; threads tid .. of nt */
template <class Z>
ZHD void sparse_setup(Z& z, int tid, int nt) {
    for (int lc = tid; lc < z.C; lc += nt) zone_maps(z, lc, 0);
    const int H = z.zh + 4, ne = (z.zw + 4) * H;
    for (int e = tid; e < ne; e += nt) {
        const int rx = e / H - 2, ry = e % H - 2;
        const int h = halo_slot(z, rx, ry);
        z.ext[e] = h >= 0 ? z.halo[h] : z.cell[rx * z.zh + ry].cnt;
    }
    if (z.dgCnt)
        for (int lc = tid; lc < z.C; lc += nt) z.dgCnt[lc] = (int)z.cell[lc].cnt;
}

/* Sparse pass (zone_pass.cpp:783-854), all lanes. */
template <class Z>
ZHD void zone_sparse_pass(Z& z, int lane, int nl) {
    sparse_setup(z, lane, nl);
    ZBAR();
    const int m = zone_compact(z, lane, nl, ZC_LOW);
    ZBAR();
    zone_shuffle(z.dl, m, lane, nl, ShufDraw{z.seed, ZS_LOW, 0u, 0u});
    const int lowInt = (int)MPCD_CEIL(z.zp.lowThrBulk);
    for (int k = 0; k < m; ++k) {
        const int c = (int)z.dl[k];
        const int nc = cnt_of(z, c);
        if (nc <= 0) continue;
        if (lane == 0) ++z.sh->nLow;
        const int moved = sparse_cell(z, c, nc, lowInt, lane, nl);
        if (lane == 0) z.sh->movedSparse += moved;
    }
}

#if defined(__HIP_DEVICE_COMPILE__)
/* The sparse phase on the four wavefronts (device only).  A low cell's
 * transfers read and change only itself and its zone neighbours at range 1
 * (its own count changes only by itself: a low cell is never a donor), and
 * the smoothed counts they rank by are the phase's starting counts, so low
 * cells more than 2 apart commute.  The wavefronts take the cells in list
 * order from a counter in LDS, and a cell starts once no earlier unfinished
 * cell lies within range 2 of it (lix, each cell's list index, is cleared
 * when the cell is finished); the waits are bounded as in the dense phase.
 * Conflicting cells keep the list order, so the result is the serial loop's
 * bit for bit.
 *
 * The scores depend on the starting counts and the draws alone, so they are
 * taken for all low cells at once before the loop, eight lanes per cell, into
 * the zone's duG region (free until the correction; longer lists in
 * segments), off the chain of conflicting cells: a cell cost 21,000 cycles
 * with its gradient, noise draws and ranking on that chain.  Two donors of
 * exactly equal score would be ordered by the donor shuffle, and a donor list
 * of more than 64 entries does not fit the wavefront: a segment with either
 * runs on wavefront 0 alone, in list order, in the general form. */
constexpr int SPARSE_REG = 64; /* donor lists up to this length are shuffled in registers */

/* the four smoothed counts of inward_dir by lanes 0..3 of each group of
 * eight, handed to the group */
template <class Z>
__device__ __forceinline__ void inward_dir_group(const Z& z, int gx, int gy, int lane, double& dxo, double& dyo) {
    const int Nx = z.g.Nx, Ny = z.g.Ny, t = lane & 7, g0 = lane & ~7;
    int xa, xb, ya, yb;
    bool hx = true, hy = true;
    if (z.g.perx) { xa = gx + 1 < Nx ? gx + 1 : 0; xb = gx > 0 ? gx - 1 : Nx - 1; }
    else if (gx == 0) { xa = gx + 1; xb = gx; hx = false; }
    else if (gx == Nx - 1) { xa = gx; xb = gx - 1; hx = false; }
    else { xa = gx + 1; xb = gx - 1; }
    if (z.g.pery) { ya = gy + 1 < Ny ? gy + 1 : 0; yb = gy > 0 ? gy - 1 : Ny - 1; }
    else if (gy == 0) { ya = gy + 1; yb = gy; hy = false; }
    else if (gy == Ny - 1) { ya = gy; yb = gy - 1; hy = false; }
    else { ya = gy + 1; yb = gy - 1; }
    const double v = t < 4 ? nsm_ext(z, (t == 0) ? xa : (t == 1) ? xb : gx, (t == 2) ? ya : (t == 3) ? yb : gy) : 0.0;
    const double n0 = __shfl(v, g0, 64), n1 = __shfl(v, g0 + 1, 64), n2 = __shfl(v, g0 + 2, 64), n3 = __shfl(v, g0 + 3, 64);
    dxo = hx ? 0.5 * (n0 - n1) : (n0 - n1);
    dyo = hy ? 0.5 * (n2 - n3) : (n2 - n3);
}

/* zone neighbour o (0..7, the order of local_neighbors_in_zone) of the cell
 * at zone-relative (cx, cy), or -1 */
template <class Z>
__device__ __forceinline__ int sparse_neighbour(const Z& z, int cx, int cy, int o, int& dx, int& dy) {
    const int f = o < 4 ? o : o + 1;
    dy = f / 3 - 1;
    dx = f - 3 * (f / 3) - 1;
    int tx = cx + dx, ty = cy + dy;
    bool in = o < 8;
    if (zone_wrap_x(z)) in = in & wrap_step(z, dx, tx, z.g.Nx);
    if (zone_wrap_y(z)) in = in & wrap_step(z, dy, ty, z.g.Ny);
    in = in & ((unsigned)tx < (unsigned)z.zw) & ((unsigned)ty < (unsigned)z.zh);
    return in ? tx * z.zh + ty : -1;
}

/* One donor transfer with the donor's list (md <= 64) in registers: as
 * donor_transfer.  d, md, nt, dh, left uniform; fd: d's flags. */
template <class Z>
__device__ __forceinline__ void donor_transfer_wave(Z& z, int c, int cgc, int d, int md, int nt, int dh, int left,
                                                    unsigned fd, int lane) {
    typedef typename Z::idx_t IT;
    const int dgc = lc_gc(z, d);
    int j = 0;
    if (lane >= 1 && lane < md)
        j = (int)mpcd_draw_particle_shuffle(z.seed, (uint32_t)cgc, (uint32_t)dgc, (uint32_t)lane);
    int v = list_entry_wave(z, dh, imin(left, md), md, lane);
    v = shuffle64(v, j, md);
    const int vn = __shfl_down(v, 1, 64);
    ZCell<IT> C = z.cell[c];
    unsigned fc = (unsigned)C.fl;
    /* c's own particles among the movers: its run's links come first */
    if (wave_ballot((lane < nt) & !(fc & ZF_MAT) & (v >= (int)z.k0[c]) & (v <= run_end(z, c))) != 0ull) {
        if (lane == 0) ensure_mat(z, c);
        fc |= ZF_MAT;
        ZWSYNC();
    }
    if (lane < md) {
        nx_set(z, v, (lane + 1 == nt || lane + 1 == md) ? -1 : vn);
        if (lane < nt) mark_moved(z, v, ZM_SPARSE);
    }
    const int v0 = wave_readlane(v, 0), vm = wave_readlane(v, nt - 1), vr = wave_readlane(v, nt < md ? nt : 0),
              vl = wave_readlane(v, md - 1);
    ZWSYNC();
    if (lane == 0) {
        const int tc = iget(C.tail);
        if (tc < 0) C.head = (IT)v0;
        else nx_set(z, tc, v0);
        const bool allBulk = (fd & ZF_BULK0) && (fc & ZF_BULK0);
        const unsigned setb = allBulk ? ZF_BB : ZF_SKIP, keepb = allBulk ? ~0u : ~(unsigned)ZF_BB;
        C.cnt = (IT)((int)C.cnt + nt);
        C.tail = (IT)vm;
        C.fl = (IT)((fc | ZF_CHG | ZF_RECV | setb) & keepb);
        z.cell[c] = C;
        ZCell<IT> D;
        D.cnt = (IT)(md - nt);
        D.head = (IT)(md > nt ? vr : -1);
        D.tail = (IT)(md > nt ? vl : -1);
        D.fl = (IT)((fd | ZF_MAT | ZF_CHG | setb) & keepb);
        z.cell[d] = D;
    }
    ZWSYNC();
}

template <class Z>
__device__ __forceinline__ void zone_sparse_pass_mw(Z& z, int wave, int lane) {
    typedef typename Z::idx_t IT;
    static_assert(sizeof(IT) == 2, "the scheduled phases take 16-bit indices");
    constexpr int NT = 64 * ZONE_WAVES;
    const int tid = wave * 64 + lane;
    const IT none = (IT)~(IT)0;
    unsigned long long* const chunkMask = reinterpret_cast<unsigned long long*>(z.scr->cand);
    const int lowInt = (int)MPCD_CEIL(z.zp.lowThrBulk);
    /* maps, the low cells, and the counts the phase starts from (the zone and
     * its ring) in ext */
    for (int ch = wave; ch * 64 < z.C; ch += ZONE_WAVES) {
        const int lc = ch * 64 + lane;
        bool f = false;
        if (lc < z.C) {
            zone_maps(z, lc, 0);
            z.lix[lc] = none;
            const int nc = cnt_of(z, lc);
            f = nc > 0 && (double)nc < low_thr(z, lc) && !fget(z, lc, ZF_OUT);
            const int ix = lc_col(z, lc);
            z.ext[(ix + 2) * (z.zh + 4) + (lc - ix * z.zh) + 2] = (IT)nc;
            if (z.dgCnt) z.dgCnt[lc] = nc;
        }
        const unsigned long long msk = wave_ballot(f);
        if (lane == 0) chunkMask[ch] = msk;
    }
    for (int h = tid; h < halo_size(z); h += NT) {
        int rx, ry;
        halo_xy(z, h, rx, ry);
        z.ext[rx * (z.zh + 4) + ry] = z.halo[h];
    }
    __syncthreads();
    const int m = zone_compact_mw(z, chunkMask, wave, lane);
    __syncthreads();
    if (wave == 0) {
        zone_shuffle(z.dl, m, lane, 64, ShufDraw{z.seed, ZS_LOW, 0u, 0u});
        for (int k = lane; k < m; k += 64) z.lix[(int)z.dl[k]] = (IT)k;
    }
    __syncthreads();
    int nLowW = 0, movedW = 0;
    volatile IT* vlix = z.lix;
    double* const score = z.duG; /* 8 per low cell of the segment */
    const int SEG = imax(1, z.C / 4);
    const bool noSeg = z.C < 4;
    for (int s0 = 0; s0 < m; s0 += SEG) {
        const int s1 = imin(m, s0 + SEG);
        /* scores: eight lanes per low cell */
        bool alone = noSeg;
        if (!noSeg)
            for (int g0 = s0; g0 < s1; g0 += NT / 8) {
                const int k = g0 + (tid >> 3), o = lane & 7;
                const bool act = k < s1;
                const int c = (int)z.dl[act ? k : s0];
                const int cx = lc_col(z, c), cy = c - cx * z.zh;
                int dx, dy;
                int q = sparse_neighbour(z, cx, cy, o, dx, dy);
                const int qs = q >= 0 ? q : c, qx = lc_col(z, qs), qy = qs - qx * z.zh;
                const int n0 = iget(z.ext[(qx + 2) * (z.zh + 4) + qy + 2]);
                const bool don = act && q >= 0 && !fget(z, qs, ZF_OUT) && n0 > lowInt;
                double gxd, gyd;
                inward_dir_group(z, z.xs + cx, z.ys + cy, lane, gxd, gyd);
                double sc = 0.0;
                if (don) {
                    const double ndir = mpcd_hypot(gxd, gyd), nstep = mpcd_hypot((double)dx, (double)dy);
                    double align = 0.0;
                    if (ndir >= 1e-14 && nstep >= 1e-14) align = ((double)dx * gxd + (double)dy * gyd) / (ndir * nstep);
                    const double noise = 1e-9 * mpcd_draw_donor_noise(z.seed, (uint32_t)lc_gc(z, c), (uint32_t)lc_gc(z, qs));
                    sc = 100.0 * align + nsm_ext(z, z.xs + qx, z.ys + qy) + noise;
                }
                if (act) score[8 * (k - s0) + o] = sc;
                alone = alone || (don && n0 > SPARSE_REG);
                const unsigned long long dm = wave_ballot(don) >> (lane & ~7);
                for (int u = 1; u < 8; ++u) {
                    const int p = (o + u) & 7;
                    const double other = __shfl(sc, (lane & ~7) + p, 64);
                    if (don && ((dm >> p) & 1ull) && !(other < sc) && !(other > sc)) alone = true;
                }
            }
        if (tid == 0) z.sh->mwNext = s0;
        __threadfence_block(); /* the scores lie in global memory */
        const bool serial = __syncthreads_or(alone) != 0;
        if (serial) {
            if (wave == 0)
                for (int k = s0; k < s1; ++k) {
                    const int c = (int)z.dl[k];
                    const int nc = cnt_of(z, c);
                    if (nc <= 0) continue;
                    ++nLowW;
                    movedW += sparse_cell(z, c, nc, lowInt, lane, 64);
                }
            /* later segments wait for none of these */
            for (int k = s0 + tid; k < s1; k += NT) z.lix[(int)z.dl[k]] = none;
        } else {
            int kv = 0;
            if (lane == 0) kv = atomicAdd(&z.sh->mwNext, 1);
            for (;;) {
                const int k = uniform(kv);
                if (k >= s1) break;
                if (lane == 0) kv = atomicAdd(&z.sh->mwNext, 1);
                const int c = uniform((int)z.dl[k]);
                const int cx = lc_col(z, c), cy = c - cx * z.zh;
                int dx, dy;
                int q = sparse_neighbour(z, cx, cy, lane, dx, dy);
                const double sc = lane < 8 ? score[8 * (k - s0) + lane] : 0.0;
                const int nc = uniform(cnt_of(z, c)); /* only this treatment changes it */
                /* earlier cells within range 2 (lanes 0..24) */
                int wx = cx + lane / 5 - 2, wy = cy + lane % 5 - 2;
                if (zone_wrap_x(z)) wx = wrap_near(wx, z.g.Nx);
                if (zone_wrap_y(z)) wy = wrap_near(wy, z.g.Ny);
                const bool wi = (lane < 25) & ((unsigned)wx < (unsigned)z.zw) & ((unsigned)wy < (unsigned)z.zh);
                const int wq = wi ? wx * z.zh + wy : c;
                for (int polls = 0;; ++polls) {
                    if (wave_ballot((int)vlix[wq] < k) == 0ull) break;
                    if (polls >= DS_WAIT_MAX) {
                        if (lane == 0) z.sh->schedWait = 1;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                sched_acquire(z);
                ++nLowW;
                int need = imax(0, lowInt - nc);
                const int qs = q >= 0 ? q : c;
                const ZCell<IT> Q = z.cell[qs];
                const int kb = (int)z.k0[qs], ke = run_end(z, qs);
                const int qc = (int)Q.cnt, qh = iget(Q.head);
                const unsigned qf = (unsigned)Q.fl;
                const bool don = (q >= 0) & !(qf & ZF_OUT) & (qc > lowInt);
                const int ql = (qf & ZF_MAT) || qh < kb || qh > ke ? 0 : ke - qh + 1;
                const unsigned long long md0 = wave_ballot(don);
                /* rank by descending score */
                int r = 0;
                for (unsigned long long mm = md0; mm; mm &= mm - 1ull) r += wave_readlane_d(sc, (int)__builtin_ctzll(mm)) > sc ? 1 : 0;
                const int nd = wave_popc(md0);
                for (int t = 0; t < nd && need > 0; ++t) {
                    const int o = (int)__builtin_ctzll(wave_ballot(don & (r == t)));
                    const int md = wave_readlane(qc, o);
                    const int nt = imin(imin(need, md - lowInt), md);
                    if (nt <= 0) continue;
                    donor_transfer_wave(z, c, lc_gc(z, c), wave_readlane(q, o), md, nt, wave_readlane(qh, o),
                                        wave_readlane(ql, o), (unsigned)wave_readlane((int)qf, o), lane);
                    movedW += nt;
                    need -= nt;
                }
                sched_release(z);
                if (lane == 0) vlix[c] = none;
                ZWSYNC();
            }
        }
        __syncthreads();
    }
    if (lane == 0) {
        atomicAdd(&z.sh->nLow, nLowW);
        atomicAdd(&z.sh->movedSparse, movedW);
    }
    __syncthreads();
}
#else
template <class Z>
ZHD void zone_sparse_pass_mw(Z&, int, int) {}
#endif

/* ---- set-up, correction, statistics ---- */

/* zone_setup's flags of the cell with global index gc */
template <class Z>
ZHD unsigned short setup_flags(const Z& z, const ZoneIn& in, int gc) {
    unsigned short f = 0;
    if (!in.owner || in.owner[gc] == z.zid) f |= ZF_OWN;
    if (in.gcover && in.gcover[gc]) f |= ZF_COVER;
    if (in.zmask && !in.zmask[gc]) f |= ZF_OUT;
    return f;
}

/* zone_setup's entry h of the ring of pass-input counts around the zone */
template <class Z>
ZHD void setup_halo(Z& z, int h) {
    int hx, hy;
    halo_xy(z, h, hx, hy);
    int gx = z.xs + hx - 2, gy = z.ys + hy - 2;
    if (z.g.perx) gx = wrapi(gx, z.g.Nx);
    if (z.g.pery) gy = wrapi(gy, z.g.Ny);
    int v = 0;
    if (gx >= 0 && gx < z.g.Nx && gy >= 0 && gy < z.g.Ny) v = z.gcnt[gy + z.g.Ny * gx];
    /* the unsigned 16-bit type keeps its top value for "read the global count" */
    if (sizeof(typename Z::idx_t) == 2 && v >= 0xFFFF) v = -1;
    z.halo[h] = (typename Z::idx_t)v;
}

/* Zone setup (zone_pass.cpp:680-685), all lanes: counts, implicit list of
 * each cell (its run of local indices, from a wave prefix sum over the
 * zone's cells), the column map and the ownership flags. */
template <class Z>
ZHD void zone_setup(Z& z, const ZoneIn& in, int lane, int nl) {
    int base = 0;
    bool mixed = false;
    for (int b0 = 0; b0 < z.C; b0 += nl) {
        const int lc = b0 + lane;
        const int gc = lc < z.C ? lc_gc(z, lc) : 0;
        const int m = lc < z.C ? z.gcnt[gc] : 0;
        const int incl = wave_shfl_up_add(m, lane);
        if (lc < z.C) {
            const int k0 = base + incl - m;
            cnt_set(z, lc, m);
            z.k0[lc] = (typename Z::idx_t)k0;
            head_set(z, lc, m > 0 ? k0 : -1);
            tail_set(z, lc, m > 0 ? k0 + m - 1 : -1);
            const unsigned short f = setup_flags(z, in, gc);
            if ((f & (ZF_OWN | ZF_COVER)) != ZF_OWN) mixed = true;
            z.cell[lc].fl = (typename Z::idx_t)f;
            if (lc % z.zh == 0) {
                z.colL[lc / z.zh] = k0;
                z.colG[lc / z.zh] = z.gstart[gc];
            }
        }
        /* lanes past the zone add 0, so the last lane holds the chunk total */
        base += wave_bcast(incl, nl - 1);
    }
    const bool anyMixed = wave_ballot(mixed) != 0ull;
    /* the ring of pass-input counts around the zone */
    const int nh = halo_size(z);
    for (int h = lane; h < nh; h += nl) setup_halo(z, h);
    if (lane == 0) {
        z.sh->P = base;
        z.sh->allOwned = anyMixed ? 0 : 1;
        z.sh->nHigh = 0;
        z.sh->nLow = 0;
        z.sh->movedDense = 0;
        z.sh->movedSparse = 0;
        z.sh->stats4 = 0.0;
        z.sh->stats5 = 0.0;
    }
}

/* zone_setup on the four wavefronts of a 256-thread workgroup, with two
 * rounds of global loads: a column's cells are one run of the binning, so
 * wavefront 0 takes the columns' starts and lengths (their prefix sum gives
 * the local indices) while the others take the ring; then every cell's run
 * follows from its start and its column's (zone_setup_cells).  The caller
 * takes a workgroup barrier after each; sh->P holds the particle count after
 * the first, zone_setup_all_owned the zone's allOwned after the second. */
template <class Z>
ZHD void zone_setup_columns(Z& z, int wave, int lane) {
    if (wave == 0) {
        int base = 0;
        for (int b0 = 0; b0 < z.zw; b0 += 64) {
            const int col = b0 + lane;
            const int g0 = z.ys + z.g.Ny * (z.xs + (col < z.zw ? col : 0));
            const int s0 = z.gstart[g0], len = col < z.zw ? z.gstart[g0 + z.zh] - s0 : 0;
            const int incl = wave_shfl_up_add(len, lane);
            if (col < z.zw) {
                z.colL[col] = base + incl - len;
                z.colG[col] = s0;
            }
            base += wave_bcast(incl, 63);
        }
        if (lane == 0) {
            z.sh->P = base;
            z.sh->nHigh = 0;
            z.sh->nLow = 0;
            z.sh->movedDense = 0;
            z.sh->movedSparse = 0;
            z.sh->stats4 = 0.0;
            z.sh->stats5 = 0.0;
            z.sh->mixed = 0;
        }
    } else {
        const int nh = halo_size(z);
        for (int h = (wave - 1) * 64 + lane; h < nh; h += 192) setup_halo(z, h);
    }
}
template <class Z>
ZHD void zone_setup_cells(Z& z, const ZoneIn& in, int wave, int lane) {
    typedef typename Z::idx_t IT;
    bool mixed = false;
    for (int lc = wave * 64 + lane; lc < z.C; lc += 256) {
        const int col = lc_col(z, lc), gc = lc_gc(z, lc);
        const int m = z.gcnt[gc], k0 = z.colL[col] + (z.gstart[gc] - z.colG[col]);
        const unsigned short f = setup_flags(z, in, gc);
        mixed = mixed || (f & (ZF_OWN | ZF_COVER)) != ZF_OWN;
        ZCell<IT> c;
        c.cnt = (IT)m;
        c.head = (IT)(m > 0 ? k0 : -1);
        c.tail = (IT)(m > 0 ? k0 + m - 1 : -1);
        c.fl = (IT)f;
        z.cell[lc] = c;
        z.k0[lc] = (IT)k0;
    }
    if (wave_ballot(mixed) != 0ull && lane == 0) z.sh->mixed = 1;
}
template <class Z>
ZHD int zone_setup_all_owned(const Z& z) {
    return z.sh->mixed ? 0 : 1;
}

/* sum over the slots glist[s0 .. s0+n) in order, loads issued 8 at a time */
template <class Z>
ZHD void run_sum(const Z& z, int s0, int n, double& sx, double& sy) {
    for (int j0 = 0; j0 < n; j0 += 8) {
        int sl[8];
        double ax[8], ay[8];
        for (int u = 0; u < 8; ++u) sl[u] = (j0 + u < n) ? z.glist[s0 + j0 + u] : -1;
        for (int u = 0; u < 8; ++u) {
            ax[u] = sl[u] >= 0 ? z.vx[sl[u]] : 0.0;
            ay[u] = sl[u] >= 0 ? z.vy[sl[u]] : 0.0;
        }
        for (int u = 0; u < 8; ++u)
            if (sl[u] >= 0) {
                sx += ax[u];
                sy += ay[u];
            }
    }
}

/* The diagnostics' record of cell lc (zone_pass.cpp:885-897): the momentum
 * defect (input run minus final list) and the final list's momentum, both
 * before the correction. */
template <class Z>
ZHD void diag_cell(Z& z, int lc, double dPx, double dPy, double px, double py) {
    double* d = z.dgCell + 4 * (size_t)lc;
    d[0] = dPx;
    d[1] = dPy;
    d[2] = px;
    d[3] = py;
}

/* the same for an occupied cell nothing changed: its list is its input run */
template <class Z>
ZHD void diag_cell_unchanged(Z& z, int lc) {
    const int gc = lc_gc(z, lc);
    double px = 0.0, py = 0.0;
    run_sum(z, z.gstart[gc], z.gcnt[gc], px, py);
    diag_cell(z, lc, 0.0, 0.0, px, py);
}

/* Momentum correction (zone_pass.cpp:870-909), first half, one lane per
 * cell: the velocity change of a changed cell from the momentum of its
 * input run and of its final list (both in list order).  Reads only; a cell
 * nothing changed has the same list before and after, so its change is
 * exactly zero. */
template <class Z>
ZHD void zone_correct_sums(Z& z, int lc) {
    const int m = cnt_of(z, lc);
    if (!fget(z, lc, ZF_CHG) || m == 0) {
        if (z.dgCell && m > 0 && !fget(z, lc, ZF_OUT)) diag_cell_unchanged(z, lc);
        return;
    }
    const int gc = lc_gc(z, lc);
    double pbx = 0.0, pby = 0.0;
    run_sum(z, z.gstart[gc], z.gcnt[gc], pbx, pby);
    double px = 0.0, py = 0.0;
    int k = head_of(z, lc);
    while (k >= 0) {
        int sl[8];
        double ax[8], ay[8];
        for (int u = 0; u < 8; ++u) {
            sl[u] = -1;
            if (k >= 0) {
                sl[u] = slot_of(z, k);
                k = next_k(z, lc, k);
            }
        }
        for (int u = 0; u < 8; ++u) {
            ax[u] = sl[u] >= 0 ? z.vx[sl[u]] : 0.0;
            ay[u] = sl[u] >= 0 ? z.vy[sl[u]] : 0.0;
        }
        for (int u = 0; u < 8; ++u)
            if (sl[u] >= 0) {
                px += ax[u];
                py += ay[u];
            }
    }
    const double dPx = pbx - px, dPy = pby - py;
    if (z.dgCell) diag_cell(z, lc, dPx, dPy, px, py);
    const double dux = dPx / (double)m, duy = dPy / (double)m;
    z.duG[2 * lc] = dux;
    z.duG[2 * lc + 1] = duy;
    bool corr = z.zp.corrEnabled != 0;
    if (corr && fget(z, lc, ZF_SKIP)) corr = false;
    if (corr && fget(z, lc, ZF_RECV) && !fget(z, lc, ZF_BB)) corr = false;
    if (corr && !(dux != 0.0 || duy != 0.0)) corr = false;
    if (corr) fset(z, lc, ZF_CORR);
}

/* records whether the side buffer holds the velocities of cell lc's input
 * particles (a cell this zone owns and others cover) */
template <class Z>
ZHD void mark_changed(Z& z, int lc, bool chg) {
    if (z.gchg && fget(z, lc, ZF_OWN) && fget(z, lc, ZF_COVER)) z.gchg[lc_gc(z, lc)] = chg ? 1 : 0;
}

/* Second half, one lane per cell: write the velocities of the owned
 * particles of a changed cell; for an unchanged cell that several zones
 * cover, pass its owned particles' input velocities through to the side
 * buffer.  Returns the cell's |du|^2 (0 for an unchanged cell). */
template <class Z>
ZHD double zone_correct_write(Z& z, int lc) {
    mark_changed(z, lc, true);
    if (fget(z, lc, ZF_CHG)) {
        if (cnt_of(z, lc) == 0) return 0.0;
        const bool corr = fget(z, lc, ZF_CORR);
        const double dux = z.duG[2 * lc], duy = z.duG[2 * lc + 1];
        int k = head_of(z, lc);
        while (k >= 0) {
            int sl[8], tg[8];
            uint32_t pd[8];
            unsigned short ow[8];
            double ax[8], ay[8];
            for (int u = 0; u < 8; ++u) {
                sl[u] = -1;
                ow[u] = 0;
                tg[u] = ZM_NONE;
                if (k >= 0) {
                    const int col = col_of(z, k);
                    sl[u] = slot_pid_in(z, k, col, pd[u]);
                    ow[u] = own_bits(z, k, col);
                    tg[u] = z.rec[k];
                    k = next_k(z, lc, k);
                }
            }
            for (int u = 0; u < 8; ++u) {
                const bool w = sl[u] >= 0 && (ow[u] & ZF_OWN);
                ax[u] = w ? z.vx[sl[u]] : 0.0;
                ay[u] = w ? z.vy[sl[u]] : 0.0;
            }
            for (int u = 0; u < 8; ++u) {
                if (sl[u] < 0 || !(ow[u] & ZF_OWN)) continue;
                if (tg[u] != ZM_NONE) place_moved(z, lc, sl[u], pd[u], tg[u]);
                double vx = ax[u], vy = ay[u];
                if (corr) {
                    vx += dux;
                    vy += duy;
                }
                if (ow[u] & ZF_COVER) {
                    z.vsx[sl[u]] = vx;
                    z.vsy[sl[u]] = vy;
                } else {
                    z.vx[sl[u]] = vx;
                    z.vy[sl[u]] = vy;
                }
            }
        }
        return dux * dux + duy * duy;
    }
    if (!fget(z, lc, ZF_COVER) || !fget(z, lc, ZF_OWN)) return 0.0;
    const int gc = lc_gc(z, lc);
    const int s0 = z.gstart[gc], m0 = z.gcnt[gc];
    for (int j0 = 0; j0 < m0; j0 += 8) {
        int sl[8];
        double ax[8], ay[8];
        for (int u = 0; u < 8; ++u) sl[u] = (j0 + u < m0) ? z.glist[s0 + j0 + u] : -1;
        for (int u = 0; u < 8; ++u) {
            ax[u] = sl[u] >= 0 ? z.vx[sl[u]] : 0.0;
            ay[u] = sl[u] >= 0 ? z.vy[sl[u]] : 0.0;
        }
        for (int u = 0; u < 8; ++u)
            if (sl[u] >= 0) {
                z.vsx[sl[u]] = ax[u];
                z.vsy[sl[u]] = ay[u];
            }
    }
    return 0.0;
}

/* Correction of all cells and stats[4], stats[5] of the zone
 * (zone_pass.cpp:870-922), all lanes.  The rms sums |du|^2 over the cells in
 * ascending order: each chunk of nl cells is added lane by lane. */
template <class Z>
ZHD void zone_correct(Z& z, int lane, int nl) {
    for (int lc = lane; lc < z.C; lc += nl) zone_correct_sums(z, lc);
    ZBAR();
    double acc = 0.0, mx = 0.0;
    int nDU = 0;
    for (int b0 = 0; b0 < z.C; b0 += nl) {
        const int lc = b0 + lane;
        const double d = lc < z.C ? zone_correct_write(z, lc) : 0.0;
        mx = dmax(mx, MPCD_SQRT(d));
        unsigned long long pos = wave_ballot(d > 0.0);
        nDU += wave_popc(pos);
        while (pos) {
            const int l = __builtin_ctzll(pos);
            pos &= pos - 1ull;
            acc += wave_readlane_d(d, l);
        }
    }
    mx = wave_max(mx);
    if (lane == 0 && nDU > 0) {
        z.sh->stats4 = MPCD_SQRT(acc / (double)nDU);
        z.sh->stats5 = mx;
    }
}

/* ---- working set ---- */

/* bytes of the per-zone cell arrays and scratch (links excluded) */
template <class IT>
ZHD size_t zone_fixed_bytes(int C, int W, int useLocal) {
    size_t b = 0;
    if (useLocal) b += (size_t)C * 2 * sizeof(double);         /* lowA highA */
    b += sizeof(ZScratch<IT>);                                  /* 8-byte items first */
    b += (size_t)W * 2 * sizeof(int);                           /* colL colG */
    b += (size_t)C * sizeof(ZCell<IT>);                         /* cell */
    b += (size_t)C * 3 * sizeof(IT);                            /* k0 dl lix */
    b += (size_t)(W + 4) * (size_t)(C / (W > 0 ? W : 1) + 4) * sizeof(IT); /* ext */
    b += (size_t)(4 * (W + 4) + 4 * (C / (W > 0 ? W : 1))) * sizeof(IT); /* halo */
    b += 32;                                                    /* alignment after k0 and colG */
    return (b + 15) & ~(size_t)15;
}

/* Carves the working set out of `base` (16-byte aligned); links of k < nL
 * follow the fixed part, nL = what the remaining `bytes` hold. */
template <class IT>
ZHD void zone_carve(ZoneCtxT<IT>& z, unsigned char* base, size_t bytes) {
    const int C = z.C, W = z.zw;
    unsigned char* p = base;
    /* first what the correction keeps (cell arrays, column map), at the
     * offsets of the correction's own LDS layout, so the correction that
     * follows the passes in one kernel finds them in place */
    z.cell = (ZCell<IT>*)p; p += (size_t)C * sizeof(ZCell<IT>);
    z.k0 = (IT*)p; p += (size_t)C * sizeof(IT);
    p = base + (((size_t)(p - base) + 3) & ~(size_t)3);
    z.colL = (int*)p; p += (size_t)W * sizeof(int);
    z.colG = (int*)p; p += (size_t)W * sizeof(int);
    p = base + (((size_t)(p - base) + 15) & ~(size_t)15);
    /* then the passes' scratch */
    if (z.zp.useLocal) {
        z.lowA = (double*)p; p += (size_t)C * sizeof(double);
        z.highA = (double*)p; p += (size_t)C * sizeof(double);
    } else {
        z.lowA = nullptr;
        z.highA = nullptr;
    }
    z.scr = (ZScratch<IT>*)p; p += sizeof(ZScratch<IT>);
    z.dl = (IT*)p; p += (size_t)C * sizeof(IT);
    z.ext = (IT*)p; p += (size_t)(z.zw + 4) * (size_t)(z.zh + 4) * sizeof(IT);
    z.halo = (IT*)p; p += (size_t)halo_size(z) * sizeof(IT);
    z.lix = (IT*)p; p += (size_t)C * sizeof(IT);
    const size_t fixed = zone_fixed_bytes<IT>(C, W, z.zp.useLocal);
    p = base + fixed;
    z.nxL = (IT*)p;
    const size_t rest = bytes > fixed ? bytes - fixed : 0;
    const size_t nl = rest / sizeof(IT);
    z.nL = nl > (size_t)0x7fffffff ? 0x7fffffff : (int)nl;
}

/* Per-lane context of zone zid (1-based) with rectangle r. */
template <class IT>
ZHD void zone_init(ZoneCtxT<IT>& z, const ZoneIn& in, ZoneRect r, int zid, uint64_t seed, ZoneShared* sh) {
    z.g = in.g;
    z.zp = in.zp;
    z.xs = r.xs;
    z.xe = r.xe;
    z.ys = r.ys;
    z.ye = r.ye;
    z.zw = r.xe - r.xs;
    z.zh = r.ye - r.ys;
    z.C = z.zw * z.zh;
    z.zhM = z.zh > 1 ? 0xffffffffu / (unsigned)z.zh + 1u : 0u;
    z.zid = zid;
    z.seed = seed;
    z.gcnt = in.gcnt;
    z.gstart = in.gstart;
    z.glist = in.glist;
    z.gkey = in.gkey;
    z.inPx = in.inPx;
    z.inPy = in.inPy;
    z.dcid = in.dcid;
    z.dout = in.dout;
    z.dinc = in.dinc;
    z.darr = in.darr;
    z.darrN = in.darrN;
    z.cellOff = in.cellOff;
    z.dgCell = in.dgCell;
    z.dgCnt = in.dgCnt;
    z.x = in.x;
    z.y = in.y;
    z.vx = in.vx;
    z.vy = in.vy;
    z.vsx = in.vsx;
    z.vsy = in.vsy;
    z.gchg = in.gchg;
    z.sh = sh;
}

/* The zone after zone_setup and a barrier: both phases. */
template <class Z>
ZHD void zone_passes(Z& z, int lane, int nl) {
    z.P = z.sh->P;
    z.allOwned = z.sh->allOwned;
    for (int k = lane; k < z.P; k += nl) z.rec[k] = (unsigned char)ZM_NONE;
    zone_dense_passes(z, lane, nl);
    zone_sparse_pass(z, lane, nl);
    ZBAR();
}

/* Both phases, the correction and the stats, in one go. */
template <class Z>
ZHD void zone_run(Z& z, int lane, int nl) {
    zone_passes(z, lane, nl);
    zone_correct(z, lane, nl);
}

/* ---- the zone's state between the passes and the correction ----
 *
 * On the device the correction runs in a kernel of its own, with many
 * threads per zone: the pass kernel leaves the cell arrays, the column map
 * and the flags in a per-zone state region of global memory, and the links
 * all in the zone's global link region.  Layout (16-byte aligned):
 * |dsq C doubles|cell C ZCell|hdr 4 ints|colL W ints|colG W ints|k0 C IT| */
template <class IT>
struct ZoneState {
    double* dsq; /* |du|^2 of each cell, for the ordered stats */
    int* hdr;    /* P, allOwned */
    int *colL, *colG;
    ZCell<IT>* cell;
    IT* k0;
};

template <class IT>
ZHD size_t zone_state_bytes(int C, int W) {
    const size_t b = (size_t)C * sizeof(double) + (size_t)C * sizeof(ZCell<IT>) + 4 * sizeof(int) +
                     (size_t)W * 2 * sizeof(int) + (size_t)C * sizeof(IT) + sizeof(ZCell<IT>);
    return (b + 15) & ~(size_t)15;
}

template <class IT>
ZHD ZoneState<IT> zone_state_at(unsigned char* base, int C, int W) {
    ZoneState<IT> st;
    unsigned char* p = base;
    st.dsq = (double*)p; p += (size_t)C * sizeof(double);
    p = base + (((size_t)(p - base) + sizeof(ZCell<IT>) - 1) & ~(sizeof(ZCell<IT>) - 1));
    st.cell = (ZCell<IT>*)p; p += (size_t)C * sizeof(ZCell<IT>);
    st.hdr = (int*)p; p += 4 * sizeof(int);
    st.colL = (int*)p; p += (size_t)W * sizeof(int);
    st.colG = (int*)p; p += (size_t)W * sizeof(int);
    st.k0 = (IT*)p;
    return st;
}

/* all lanes: the state after zone_passes, and the links held in LDS moved
 * to the zone's global link region */
template <class IT>
ZHD void zone_dump(ZoneCtxT<IT>& z, const ZoneState<IT>& st, int lane, int nl) {
    for (int lc = lane; lc < z.C; lc += nl) {
        st.cell[lc] = z.cell[lc];
        st.k0[lc] = z.k0[lc];
    }
    for (int c = lane; c < z.zw; c += nl) {
        st.colL[c] = z.colL[c];
        st.colG[c] = z.colG[c];
    }
    if (lane == 0) {
        st.hdr[0] = z.P;
        st.hdr[1] = z.allOwned;
    }
    const int nk = z.P < z.nL ? z.P : z.nL;
    const IT* const L = z.nxL;
    IT* const G = z.nxG;
    for (int k = lane; k < nk; k += nl) ZG_STORE(G + k, L[k]);
}

/* the correction's view of a dumped zone: cell arrays and column map in the
 * state region, every link in the global link region */
template <class IT>
ZHD void zone_attach_state(ZoneCtxT<IT>& z, const ZoneState<IT>& st) {
    z.cell = st.cell;
    z.k0 = st.k0;
    z.colL = st.colL;
    z.colG = st.colG;
    z.P = st.hdr[0];
    z.allOwned = st.hdr[1];
    z.nxL = nullptr;
    z.nL = 0;
}

/* length of cell lc's input run (its local indices k0[lc] ..) */
template <class Z>
ZHD int in_cnt(const Z& z, int lc) {
    const int col = lc / z.zh;
    const int end = (lc - col * z.zh + 1 < z.zh) ? (int)z.k0[lc + 1] : (col + 1 < z.zw ? (int)z.colL[col + 1] : z.P);
    return end - (int)z.k0[lc];
}

/* ---- the correction kernel's per-cell form (a group of lanes per cell) ----
 * Phase 1 sums every changed cell's input run; after a barrier, phase 2
 * walks each cell's final list once: a list of up to FIN_G x FIN_L entries
 * stays in registers from the sums to the writes (a particle is in exactly
 * one final list, and every input-run read happened in phase 1), a longer
 * one is walked twice.  The moved particles' links are set to their final
 * cell for phase 3, which places them.  Same sums in the same order as
 * zone_correct_sums / zone_correct_write. */
constexpr int FIN_L = 8;
constexpr int FIN_G = 4;

/* column of particle k of cell lc's final list: its own input run lies in
 * lc's column */
template <class Z>
ZHD int fin_col(const Z& z, int lc, int kb, int ke, int k) {
    return (k >= kb && k < ke) ? lc / z.zh : col_of(z, k);
}

template <class Z>
ZHD void fin_write(Z& z, int sl, unsigned short ow, bool corr, double vx, double vy, double dux, double duy) {
    if (!(ow & ZF_OWN)) return;
    if (corr) {
        vx += dux;
        vy += duy;
    }
    if (ow & ZF_COVER) {
        z.vsx[sl] = vx;
        z.vsy[sl] = vy;
    } else {
        z.vx[sl] = vx;
        z.vy[sl] = vy;
    }
}

#if defined(__HIP_DEVICE_COMPILE__)
/* Phase 1 for changed, occupied cell lc on a group of FIN_G lanes: the
 * momentum of its input run (the particles binned into it, before the
 * passes), FIN_G * FIN_L entries at a time, summed in run order as
 * fin_cell_group sums the final list.  Every lane of the group gets the sums. */
template <class Z>
__device__ __forceinline__ void fin_input_sum_group(const Z& z, int lc, int r, int lane, double& pbx, double& pby) {
    constexpr int CH = FIN_G * FIN_L;
    const int gc = lc_gc(z, lc);
    const int s0 = z.gstart[gc], n = z.gcnt[gc];
    const int g0 = lane - r;
    double px = 0.0, py = 0.0;
    for (int c0 = 0; c0 < n; c0 += CH) {
        int sl[FIN_L];
        double ax[FIN_L], ay[FIN_L];
        for (int u = 0; u < FIN_L; ++u) {
            const int e = c0 + FIN_L * r + u;
            sl[u] = e < n ? z.glist[s0 + e] : -1;
        }
        for (int u = 0; u < FIN_L; ++u) {
            ax[u] = sl[u] >= 0 ? z.vx[sl[u]] : 0.0;
            ay[u] = sl[u] >= 0 ? z.vy[sl[u]] : 0.0;
        }
        for (int a = 0; a < FIN_G; ++a) {
            if (r == a)
                for (int u = 0; u < FIN_L; ++u)
                    if (sl[u] >= 0) {
                        px += ax[u];
                        py += ay[u];
                    }
            px = __shfl(px, g0 + a, 64);
            py = __shfl(py, g0 + a, 64);
        }
    }
    pbx = px;
    pby = py;
}

/* A final list as a group walks it: its head, the entries still implicit,
 * and the walk along the links (entry at and local index kw). */
struct FinWalk {
    int h, left, at, kw;
};
template <class Z>
__device__ __forceinline__ FinWalk fin_walk(const Z& z, int lc, int m) {
    FinWalk w;
    w.h = head_of(z, lc);
    w.left = imin(m, run_left(z, lc, w.h));
    w.at = w.left;
    w.kw = w.left > 0 ? (w.left < m ? nx_get(z, w.h + w.left - 1) : -1) : w.h;
    return w;
}
/* entries [c0 + FIN_L r, c0 + FIN_L (r + 1)) of the list of m entries (-1
 * beyond its end): the run's by their indices, the others by the walk, which
 * the whole group takes in step */
template <class Z>
__device__ __forceinline__ void fin_group_entries(const Z& z, FinWalk& w, int m, int c0, int r, int* kk) {
    constexpr int CH = FIN_G * FIN_L;
    const int e0 = c0 + FIN_L * r;
    for (int u = 0; u < FIN_L; ++u) kk[u] = e0 + u < w.left ? w.h + e0 + u : -1;
    const int end = imin(m, c0 + CH);
    while (w.at < end) {
        const int q = w.at - e0;
        for (int u = 0; u < FIN_L; ++u) kk[u] = q == u ? w.kw : kk[u];
        if (++w.at < m) w.kw = nx_get(z, w.kw);
    }
}

/* Phase 2 for changed, occupied cell lc on a group of FIN_G consecutive
 * lanes (r: the lane's rank; every lane of the group passes the same cell).
 * Every entry's link is set to lc, its final cell, once the walk has read
 * it: phase 3 reads the links of the moved particles, and nothing reads the
 * others.
 * The group takes the final list FIN_G * FIN_L entries at a time, lane r
 * entries [FIN_L r, FIN_L (r + 1)) of each chunk, so a list of up to
 * FIN_G * FIN_L entries has each slot and velocity loaded once instead of
 * once per pass.  The momentum sums keep the list order: lane r adds its
 * entries to the running sum lane r - 1 hands on.  A linked list is walked by
 * the whole group in step.  pbx, pby: the cell's input-run momentum.  Returns
 * |du|^2 (the same on every lane of the group). */
template <class Z>
__device__ __forceinline__ double fin_cell_group(Z& z, int lc, int r, int lane, double pbx, double pby) {
    constexpr int CH = FIN_G * FIN_L;
    const int m = cnt_of(z, lc);
    const int kb = (int)z.k0[lc], ke = kb + in_cnt(z, lc);
    FinWalk w = fin_walk(z, lc, m);
    const unsigned short ownLc = (unsigned short)((unsigned)z.cell[lc].fl & (ZF_OWN | ZF_COVER));
    const int g0 = lane - r;
    int kk[FIN_L], sl[FIN_L];
    unsigned short ow[FIN_L];
    double ax[FIN_L], ay[FIN_L];
    double px = 0.0, py = 0.0;
    for (int c0 = 0; c0 < m; c0 += CH) {
        fin_group_entries(z, w, m, c0, r, kk);
        for (int u = 0; u < FIN_L; ++u) {
            sl[u] = -1;
            ow[u] = 0;
            if (kk[u] >= 0) {
                const int col = fin_col(z, lc, kb, ke, kk[u]);
                sl[u] = slot_in(z, kk[u], col);
                ow[u] = (kk[u] >= kb && kk[u] < ke) ? ownLc : own_bits(z, kk[u], col);
            }
        }
        for (int u = 0; u < FIN_L; ++u) {
            ax[u] = sl[u] >= 0 ? z.vx[sl[u]] : 0.0;
            ay[u] = sl[u] >= 0 ? z.vy[sl[u]] : 0.0;
        }
        for (int a = 0; a < FIN_G; ++a) {
            if (r == a)
                for (int u = 0; u < FIN_L; ++u)
                    if (sl[u] >= 0) {
                        px += ax[u];
                        py += ay[u];
                    }
            px = __shfl(px, g0 + a, 64);
            py = __shfl(py, g0 + a, 64);
        }
    }
    if (z.dgCell && r == 0) diag_cell(z, lc, pbx - px, pby - py, px, py);
    const double dux = (pbx - px) / (double)m, duy = (pby - py) / (double)m;
    bool corr = z.zp.corrEnabled != 0;
    if (corr && fget(z, lc, ZF_SKIP)) corr = false;
    if (corr && fget(z, lc, ZF_RECV) && !fget(z, lc, ZF_BB)) corr = false;
    if (corr && !(dux != 0.0 || duy != 0.0)) corr = false;
    if (m > CH) {
        /* a longer list: walk it again for the writes */
        w = fin_walk(z, lc, m);
        for (int c0 = 0; c0 < m; c0 += CH) {
            fin_group_entries(z, w, m, c0, r, kk);
            for (int u = 0; u < FIN_L; ++u) {
                sl[u] = -1;
                ow[u] = 0;
                if (kk[u] >= 0) {
                    const int col = fin_col(z, lc, kb, ke, kk[u]);
                    sl[u] = slot_in(z, kk[u], col);
                    ow[u] = (kk[u] >= kb && kk[u] < ke) ? ownLc : own_bits(z, kk[u], col);
                }
            }
            for (int u = 0; u < FIN_L; ++u) {
                ax[u] = sl[u] >= 0 ? z.vx[sl[u]] : 0.0;
                ay[u] = sl[u] >= 0 ? z.vy[sl[u]] : 0.0;
            }
            for (int u = 0; u < FIN_L; ++u)
                if (sl[u] >= 0) {
                    fin_write(z, sl[u], ow[u], corr, ax[u], ay[u], dux, duy);
                    nx_set(z, kk[u], lc);
                }
        }
    } else {
        for (int u = 0; u < FIN_L; ++u)
            if (sl[u] >= 0) {
                fin_write(z, sl[u], ow[u], corr, ax[u], ay[u], dux, duy);
                nx_set(z, kk[u], lc);
            }
    }
    return dux * dux + duy * duy;
}
/* the value of lane A of one's quad */
template <int A>
__device__ __forceinline__ double quad_bcast_d(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, A * 0x55, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), A * 0x55, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
/* lane A of each quad adds its entries to the running sums, which the quad
 * then holds (absent entries are +0: a running sum from +0 is never -0) */
template <int A>
__device__ __forceinline__ void fin_add(double& px, double& py, const double* ax, const double* ay, int r) {
    if (r == A)
        for (int u = 0; u < FIN_L; ++u) {
            px += ax[u];
            py += ay[u];
        }
    px = quad_bcast_d<A>(px);
    py = quad_bcast_d<A>(py);
}

/* The moved particles a wavefront has met, local index << 16 | final cell,
 * placed 64 at a time. */
struct FinQueue {
    unsigned* q;
    int n;
};
template <class Z>
__device__ __forceinline__ void fin_flush(Z& z, FinQueue& fq, int lane) {
    ZWSYNC();
    if (lane < fq.n) {
        const unsigned e = fq.q[lane];
        const int k = (int)(e >> 16);
        uint32_t pid;
        const int slot = slot_pid_in(z, k, col_of(z, k), pid);
        place_moved(z, (int)(e & 0xffffu), slot, pid, z.rec[k]);
    }
    ZWSYNC();
    fq.n = 0;
}
/* entries u of kk with bit u of mv set, of every lane */
template <class Z>
__device__ __forceinline__ void fin_push(Z& z, FinQueue& fq, unsigned mv, const int* kk, int lc, int lane) {
    int next = 0;
    while (wave_ballot(mv != 0u) != 0ull && next < FIN_L) {
        bool full = false;
#pragma unroll
        for (int u = 0; u < FIN_L; ++u) {
            const bool mine = (mv >> u) & 1u;
            const unsigned long long msk = wave_ballot(mine);
            const int add = wave_popc(msk);
            if (u < next || full || add == 0) continue;
            if (fq.n + add > 64) {
                full = true;
                next = u;
                continue;
            }
            if (mine) fq.q[fq.n + wave_popc(msk & lanes_below(lane))] = ((unsigned)kk[u] << 16) | (unsigned)lc;
            fq.n += add;
        }
        if (!full) break;
        fin_flush(z, fq, lane);
    }
}

/* slots of a group's entries kk: the cell's own run's entries lie in its
 * column, the others' columns by a search all entries take in step.  Returns
 * entry u's ZF_OWN in bit u, its ZF_COVER in bit 8 + u. */
template <class Z>
__device__ __forceinline__ unsigned fin_slots(const Z& z, int lc, int kb, int ke, unsigned ownLc, const int* kk, int* sl) {
    const int own = lc_col(z, lc);
    int lo[FIN_L];
    bool far = false;
    for (int u = 0; u < FIN_L; ++u) {
        lo[u] = own;
        far = far || (kk[u] >= 0 && (kk[u] < kb || kk[u] >= ke));
    }
    if (wave_ballot(far) != 0ull) {
        int hi[FIN_L];
        for (int u = 0; u < FIN_L; ++u) {
            const bool f = kk[u] >= 0 && (kk[u] < kb || kk[u] >= ke);
            lo[u] = f ? 0 : own;
            hi[u] = f ? z.zw - 1 : own;
        }
        for (int s = z.zw - 1; s > 0; s >>= 1)
            for (int u = 0; u < FIN_L; ++u) {
                const int mid = (lo[u] + hi[u] + 1) >> 1;
                const bool up = z.colL[mid] <= kk[u];
                const bool open = lo[u] < hi[u];
                lo[u] = (open & up) ? mid : lo[u];
                hi[u] = (open & !up) ? mid - 1 : hi[u];
            }
    }
    for (int u = 0; u < FIN_L; ++u) sl[u] = kk[u] >= 0 ? z.glist[z.colG[lo[u]] + (kk[u] - z.colL[lo[u]])] : -1;
    unsigned ow = 0u;
    for (int u = 0; u < FIN_L; ++u) {
        unsigned b = ownLc;
        if (!z.allOwned && kk[u] >= 0 && (kk[u] < kb || kk[u] >= ke)) b = own_bits(z, kk[u], lo[u]);
        ow |= ((b & ZF_OWN) ? 1u << u : 0u) | ((b & ZF_COVER) ? 256u << u : 0u);
    }
    return ow;
}

/* a chunk of a group's list: its moved particles to the queue (what the links
 * hold has moved, but for lists whose links were all written), its slots and
 * velocities loaded; returns the ownership bits */
template <class Z>
__device__ __forceinline__ unsigned fin_load(Z& z, FinWalk& w, int lc, int m, int kb, int ke, unsigned f, int left, int c0,
                                             int r, int lane, FinQueue* fq, int* sl, double* ax, double* ay) {
    int kk[FIN_L];
    fin_group_entries(z, w, m, c0, r, kk);
    const unsigned ow = fin_slots(z, lc, kb, ke, f, kk, sl);
    if (fq) {
        unsigned mv = 0u;
        for (int u = 0; u < FIN_L; ++u) {
            bool v = kk[u] >= 0 && c0 + FIN_L * r + u >= left && ((ow >> u) & 1u);
            if (v && (f & ZF_MAT)) v = z.rec[kk[u]] != ZM_NONE;
            mv |= v ? 1u << u : 0u;
        }
        fin_push(z, *fq, mv, kk, lc, lane);
    }
    for (int u = 0; u < FIN_L; ++u) {
        ax[u] = sl[u] >= 0 ? z.vx[sl[u]] : 0.0;
        ay[u] = sl[u] >= 0 ? z.vy[sl[u]] : 0.0;
    }
    return ow;
}
template <class Z>
__device__ __forceinline__ void fin_store(Z& z, const int* sl, unsigned ow, bool corr, const double* ax, const double* ay,
                                          double dux, double duy) {
    for (int u = 0; u < FIN_L; ++u)
        if (sl[u] >= 0 && ((ow >> u) & 1u)) {
            const bool cov = (ow >> (8 + u)) & 1u;
            double* const X = cov ? z.vsx : z.vx;
            double* const Y = cov ? z.vsy : z.vy;
            X[sl[u]] = corr ? ax[u] + dux : ax[u];
            Y[sl[u]] = corr ? ay[u] + duy : ay[u];
        }
}

/* Phase 2 for cell lc of the fused kernel (fin_cell_group's sums and writes);
 * act: the group has a cell (the whole wavefront calls it).  Its moved
 * particles go to the queue.  kLong: lists of more than one chunk, walked
 * twice; the others stay in registers (a form of its own: with both in one,
 * the registers do not hold it, and the spills cost a quarter of the kernel's
 * time at 2048 x 1024 x 20). */
template <bool kLong, class Z>
__device__ __forceinline__ double fin_cell_fused(Z& z, int lc, bool act, int r, int lane, double pbx, double pby,
                                                 FinQueue& fq) {
    constexpr int CH = FIN_G * FIN_L;
    const ZCell<typename Z::idx_t> S = z.cell[lc];
    const unsigned f = (unsigned)S.fl;
    const int m = act ? (int)S.cnt : 0;
    const int kb = (int)z.k0[lc], ke = run_end(z, lc) + 1;
    FinWalk w;
    w.h = iget(S.head);
    w.left = (f & ZF_MAT) || w.h < kb || w.h >= ke ? 0 : imin(m, ke - w.h);
    w.at = w.left;
    w.kw = w.left > 0 ? (w.left < m ? nx_get(z, w.h + w.left - 1) : -1) : w.h;
    const FinWalk w0 = w;
    int sl[FIN_L];
    unsigned ow = 0u;
    double ax[FIN_L], ay[FIN_L];
    double px = 0.0, py = 0.0;
    for (int c0 = 0; c0 == 0 || (kLong && wave_ballot(c0 < m) != 0ull); c0 += CH) {
        ow = fin_load(z, w, lc, m, kb, ke, f, w0.left, c0, r, lane, &fq, sl, ax, ay);
        fin_add<0>(px, py, ax, ay, r);
        fin_add<1>(px, py, ax, ay, r);
        fin_add<2>(px, py, ax, ay, r);
        fin_add<3>(px, py, ax, ay, r);
    }
    if (z.dgCell && r == 0 && act) diag_cell(z, lc, pbx - px, pby - py, px, py);
    const double dux = act ? (pbx - px) / (double)m : 0.0, duy = act ? (pby - py) / (double)m : 0.0;
    const bool corr = z.zp.corrEnabled != 0 && !(f & ZF_SKIP) && !((f & ZF_RECV) && !(f & ZF_BB)) && (dux != 0.0 || duy != 0.0);
    if (!kLong) {
        fin_store(z, sl, ow, corr, ax, ay, dux, duy);
    } else {
        /* loaded again for the writes */
        w = w0;
        for (int c0 = 0; wave_ballot(c0 < m) != 0ull; c0 += CH) {
            ow = fin_load(z, w, lc, m, kb, ke, f, w0.left, c0, r, lane, nullptr, sl, ax, ay);
            fin_store(z, sl, ow, corr, ax, ay, dux, duy);
        }
    }
    return dux * dux + duy * duy;
}

/* The correction of a zone on the 256 threads that ran its passes, its state
 * still in LDS: the changed, occupied cells are listed first, so a group of
 * four lanes always has one (a few hundred of 625 in the base pass, a handful
 * in the shifted one); lists are mostly what is left of an input run, whose
 * entries need no walk; the sums pass between the lanes of a quad in
 * registers; a moved particle is met in its final cell's links and placed
 * from there, with no pass over all particles' records.  dsq: |du|^2 per cell
 * for the ordered stats, or nullptr (no metrics asked). */
template <class Z>
__device__ __forceinline__ void zone_finish_fused(Z& z, int wave, int lane, double* dsq, unsigned* queue) {
    constexpr int NT = 64 * ZONE_WAVES;
    const int tid = wave * 64 + lane;
    unsigned long long* const chunkMask = reinterpret_cast<unsigned long long*>(z.scr->cand);
    for (int ch = wave; ch * 64 < z.C; ch += ZONE_WAVES) {
        const int lc = ch * 64 + lane;
        bool f = false;
        if (lc < z.C) {
            const bool chg = fget(z, lc, ZF_CHG);
            f = chg && cnt_of(z, lc) > 0;
            mark_changed(z, lc, chg);
            if (dsq) dsq[lc] = 0.0;
            if (z.dgCell && !chg && cnt_of(z, lc) > 0 && !fget(z, lc, ZF_OUT)) diag_cell_unchanged(z, lc);
        }
        const unsigned long long msk = wave_ballot(f);
        if (lane == 0) chunkMask[ch] = msk;
    }
    __syncthreads();
    const int m = zone_compact_mw(z, chunkMask, wave, lane);
    __syncthreads();
    const int r = tid % FIN_G, gi = tid / FIN_G;
    /* input-run sums of the changed cells, before any velocity is written
     * (the base pass has them from the reference fields) */
    if (!z.inPx) {
        for (int j = gi; j < m; j += NT / FIN_G) {
            const int lc = (int)z.dl[j];
            double bx, by;
            fin_input_sum_group(z, lc, r, lane, bx, by);
            if (r == 0) {
                z.duG[2 * lc] = bx;
                z.duG[2 * lc + 1] = by;
            }
        }
        __threadfence_block();
        __syncthreads();
    }
    FinQueue fq{queue + 64 * wave, 0};
    bool anyLong = false;
    for (int j0 = 0; j0 < m; j0 += NT / FIN_G) {
        const int lc = (int)z.dl[j0 + gi < m ? j0 + gi : j0];
        const bool act = j0 + gi < m && cnt_of(z, lc) <= FIN_G * FIN_L;
        anyLong = anyLong || cnt_of(z, lc) > FIN_G * FIN_L;
        const int gc = lc_gc(z, lc);
        const double bx = z.inPx ? z.inPx[gc] : z.duG[2 * lc], by = z.inPx ? z.inPy[gc] : z.duG[2 * lc + 1];
        const double d = fin_cell_fused<false>(z, lc, act, r, lane, bx, by, fq);
        if (dsq && act && r == 0) dsq[lc] = d;
    }
    if (wave_ballot(anyLong) != 0ull)
        for (int j0 = 0; j0 < m; j0 += NT / FIN_G) {
            const int lc = (int)z.dl[j0 + gi < m ? j0 + gi : j0];
            const bool act = j0 + gi < m && cnt_of(z, lc) > FIN_G * FIN_L;
            if (wave_ballot(act) == 0ull) continue;
            const int gc = lc_gc(z, lc);
            const double bx = z.inPx ? z.inPx[gc] : z.duG[2 * lc], by = z.inPx ? z.inPy[gc] : z.duG[2 * lc + 1];
            const double d = fin_cell_fused<true>(z, lc, act, r, lane, bx, by, fq);
            if (dsq && act && r == 0) dsq[lc] = d;
        }
    fin_flush(z, fq, lane);
    if (dsq) {
        __threadfence_block();
        __syncthreads();
        if (wave == 0) {
            double rms, mx;
            zone_correct_stats(z, dsq, lane, 64, rms, mx);
            if (lane == 0) {
                z.sh->stats4 = rms;
                z.sh->stats5 = mx;
            }
        }
    }
}
#else
/* (the host passes of the compilers see a declaration only) */
template <class Z>
ZHD void fin_input_sum_group(const Z&, int, int, int, double&, double&) {}
template <class Z>
ZHD double fin_cell_group(Z&, int, int, int, double, double) { return 0.0; }
template <class Z>
ZHD void zone_finish_fused(Z&, int, int, double*, unsigned*) {}
#endif

/* phase 3, all threads of the zone: the new positions of the moved
 * particles (links hold their final cells).  Each wavefront scans its share
 * of the local indices and gathers the moved ones into a queue of one entry
 * per lane, so each batch of draws runs once for up to 64 particles. */
template <class Z>
ZHD void fin_place_batch(Z& z, const int* queue, int n, int lane) {
    if (lane < n) {
        const int kq = queue[lane];
        const int col = col_of(z, kq);
        uint32_t pid;
        const int slot = slot_pid_in(z, kq, col, pid);
        if (own_bits(z, kq, col) & ZF_OWN) place_moved(z, nx_get(z, kq), slot, pid, z.rec[kq]);
    }
}
template <class Z>
ZHD void fin_place(Z& z, int tid, int nthr, int* queue) {
    const int lane = tid & 63;
    int nq = 0;
    for (int b = tid - lane; b < z.P; b += nthr) {
        const int k = b + lane;
        const bool mv = k < z.P && z.rec[k] != ZM_NONE;
        const unsigned long long msk = wave_ballot(mv);
        const int add = wave_popc(msk);
        if (add == 0) continue;
        if (nq + add > 64) {
            ZWSYNC();
            fin_place_batch(z, queue, nq, lane);
            ZWSYNC();
            nq = 0;
        }
        if (mv) queue[nq + wave_popc(msk & lanes_below(lane))] = k;
        nq += add;
    }
    ZWSYNC();
    fin_place_batch(z, queue, nq, lane);
}

/* The stats of zone_correct from the per-cell |du|^2 in cell order (one
 * wavefront: each chunk of nl cells added lane by lane; the loads of four
 * chunks are issued before their adds). */
template <class Z>
ZHD void zone_correct_stats(const Z& z, const double* dsq, int lane, int nl, double& rms, double& mxo) {
    constexpr int NB = 4;
    double acc = 0.0, mx = 0.0;
    int nDU = 0;
    for (int b0 = 0; b0 < z.C; b0 += NB * nl) {
        double dv[NB];
        for (int j = 0; j < NB; ++j) {
            const int lc = b0 + j * nl + lane;
            dv[j] = lc < z.C ? dsq[lc] : 0.0;
        }
        for (int j = 0; j < NB; ++j) {
            const double d = dv[j];
            mx = dmax(mx, MPCD_SQRT(d));
            unsigned long long pos = wave_ballot(d > 0.0);
            nDU += wave_popc(pos);
            while (pos) {
                const int l = __builtin_ctzll(pos);
                pos &= pos - 1ull;
                acc += wave_readlane_d(d, l);
            }
        }
    }
    mxo = wave_max(mx);
    rms = nDU > 0 ? MPCD_SQRT(acc / (double)nDU) : 0.0;
}

}  // namespace mpcdk
