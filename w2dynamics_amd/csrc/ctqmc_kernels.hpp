// Device side of the batched CT-HYB (matrix/"M-V" Z-space) Monte Carlo engine
// for MI355X (gfx950).
//
// One 64-lane wavefront owns one Markov chain and runs NCorr-long sweeps of
// Metropolis steps inside one persistent launch.  Control logic (random draws,
// proposals, window bookkeeping) runs uniformly on all lanes against a chain
// header held in LDS; the heavy parts are lane-parallel:
//   * local trace (Trace.F90:5354-6102): block matrix products
//       K <- Psi_EB(b,s,ca) * diag(exp(-(E-E0) dtau)) * K
//     over the operators of the sliding window, starting from a cached ket at the
//     window's lower edge and contracted with a cached bra at its upper edge; K
//     holds one column per state of the outer superstate, lanes own (row, col)
//     entries, one log scale per matrix, one barrier per operator;
//   * determinant ratio S - R^T M Q and the rank-1 grow/shrink of M = Delta^-1
//     (MatrixUpdate.F90:392-482): lanes own rows of the k x k column-major block;
//   * G(tau)/Legendre accumulation (CTQMC.F90:2252-2440): lanes own (a, c) pairs.
// The random-number stream, proposal and acceptance formulas and the window
// schedule follow the reference exactly, so chain c seeded with seed0 + c makes
// the reference's accept/reject decisions for init_rnd(seed0 + c).
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "../../include/w2dyn_ctqmc.h"
#include "engine.hpp"

namespace w2d {

#define DEV __device__ __forceinline__

// ---------------------------------------------------------------------------
// wave helpers (one wavefront per block)
// ---------------------------------------------------------------------------
DEV int lane_id() { return (int)threadIdx.x; }

typedef __attribute__((address_space(3))) char lds_c;
typedef __attribute__((address_space(3))) unsigned char lds_b;
typedef __attribute__((address_space(3))) double lds_d;
typedef __attribute__((address_space(3))) int lds_i;
typedef __attribute__((address_space(3))) unsigned lds_u;

DEV int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
template <typename T>
DEV T *uni_lds(T *p)
{
    return (T *)(size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(size_t)p);
}

// Cross-lane reductions with DPP row operations (VALU, no LDS traffic): quad
// permutes and row mirrors reduce each 16-lane row, readlane combines the four
// rows; the result is uniform.
template <int CTRL>
DEV int dpp_i(int v)
{
    // permutations within a row: every lane has a source, so no old value
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}

template <int CTRL>
DEV double dpp_d(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(dpp_i<CTRL>(hi), dpp_i<CTRL>(lo));
}

DEV double readlane_d(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

constexpr int DPP_QP_1032 = 0xB1, DPP_QP_2301 = 0x4E, DPP_ROW_HALF_MIRROR = 0x141, DPP_ROW_MIRROR = 0x140;

DEV double wave_max(double v)
{
    v = fmax(v, dpp_d<DPP_QP_1032>(v));
    v = fmax(v, dpp_d<DPP_QP_2301>(v));
    v = fmax(v, dpp_d<DPP_ROW_HALF_MIRROR>(v));
    v = fmax(v, dpp_d<DPP_ROW_MIRROR>(v));
    return fmax(fmax(readlane_d(v, 0), readlane_d(v, 16)), fmax(readlane_d(v, 32), readlane_d(v, 48)));
}

DEV double wave_sum(double v)
{
    v += dpp_d<DPP_QP_1032>(v);
    v += dpp_d<DPP_QP_2301>(v);
    v += dpp_d<DPP_ROW_HALF_MIRROR>(v);
    v += dpp_d<DPP_ROW_MIRROR>(v);
    return (readlane_d(v, 0) + readlane_d(v, 16)) + (readlane_d(v, 32) + readlane_d(v, 48));
}

DEV int wave_isum(int v)
{
    v += dpp_i<DPP_QP_1032>(v);
    v += dpp_i<DPP_QP_2301>(v);
    v += dpp_i<DPP_ROW_HALF_MIRROR>(v);
    v += dpp_i<DPP_ROW_MIRROR>(v);
    return (__builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16)) +
           (__builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48));
}

DEV int wave_imax(int v)
{
    v = max(v, dpp_i<DPP_QP_1032>(v));
    v = max(v, dpp_i<DPP_QP_2301>(v));
    v = max(v, dpp_i<DPP_ROW_HALF_MIRROR>(v));
    v = max(v, dpp_i<DPP_ROW_MIRROR>(v));
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

DEV int wave_imin(int v) { return -wave_imax(-v); }

// Inclusive scans over the lanes: shifts by 1, 2, 4, 8 within the 16-lane
// rows, then the rows' last lanes broadcast to the rows behind (six VALU steps,
// no LDS traffic).
template <int CTRL, int ROWS>
DEV int dpp_mov_i(int old, int v)
{
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
DEV double dpp_mov_d(double old, double v)
{
    return __hiloint2double(dpp_mov_i<CTRL, ROWS>(__double2hiint(old), __double2hiint(v)),
                            dpp_mov_i<CTRL, ROWS>(__double2loint(old), __double2loint(v)));
}
DEV int wave_scan_i(int x)
{
    x += dpp_mov_i<0x111, 0xf>(0, x);
    x += dpp_mov_i<0x112, 0xf>(0, x);
    x += dpp_mov_i<0x114, 0xf>(0, x);
    x += dpp_mov_i<0x118, 0xf>(0, x);
    x += dpp_mov_i<0x142, 0xa>(0, x);
    x += dpp_mov_i<0x143, 0xc>(0, x);
    return x;
}
DEV double wave_scan_d(double x)
{
    x += dpp_mov_d<0x111, 0xf>(0.0, x);
    x += dpp_mov_d<0x112, 0xf>(0.0, x);
    x += dpp_mov_d<0x114, 0xf>(0.0, x);
    x += dpp_mov_d<0x118, 0xf>(0.0, x);
    x += dpp_mov_d<0x142, 0xa>(0.0, x);
    x += dpp_mov_d<0x143, 0xc>(0.0, x);
    return x;
}
DEV double wave_scan_mul(double x)
{
    x *= dpp_mov_d<0x111, 0xf>(1.0, x);
    x *= dpp_mov_d<0x112, 0xf>(1.0, x);
    x *= dpp_mov_d<0x114, 0xf>(1.0, x);
    x *= dpp_mov_d<0x118, 0xf>(1.0, x);
    x *= dpp_mov_d<0x142, 0xa>(1.0, x);
    x *= dpp_mov_d<0x143, 0xc>(1.0, x);
    return x;
}

// hardware FP64 add to device (global) memory, result unused
DEV void global_add(double *p, double v)
{
    typedef __attribute__((address_space(1))) double gdouble;
    (void)__builtin_amdgcn_global_atomic_fadd_f64((gdouble *)p, v);
}

DEV int popc64(unsigned long long m) { return __popcll(m); }

DEV unsigned long long lanemask_le() { return (lane_id() == 63) ? ~0ull : ((2ull << lane_id()) - 1ull); }

DEV void wsync() { __syncthreads(); }

// ---------------------------------------------------------------------------
// random numbers: mt19937 + libstdc++ generate_canonical<double,53> and
// uniform_int_distribution (src/mtrng/random.cc:30-79).  The 624-word state is
// shared in LDS; every lane draws the same numbers, the twist is lane-parallel.
// ---------------------------------------------------------------------------
struct Rng {
    lds_u *mt;      // LDS
    int *idx;       // LDS (uniform): next word, kept there between open and close
    uint32_t w;     // lane l: tempered word base + l
    int pos, base;
};

DEV uint32_t mt_twist_word(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t y = (a & 0x80000000u) | (b & 0x7fffffffu);
    uint32_t v = c ^ (y >> 1);
    if (y & 1u) v ^= 0x9908b0dfu;
    return v;
}

// new mt[i] depends on mt[i+1] (old) and mt[i+397]: old for i < 227, new for
// i >= 227 (from index i-227).  Phases [0,227) [227,454) [454,623) {623}.
__device__ __attribute__((noinline)) void mt_regen(lds_u *mt_)
{
    lds_u *mt = uni_lds(mt_);
    const int l = lane_id();
    uint32_t nv[4];
    int c = 0;
    for (int i = l; i < 227; i += WAVE) nv[c++] = mt_twist_word(mt[i], mt[i + 1], mt[i + 397]);
    wsync();
    c = 0;
    for (int i = l; i < 227; i += WAVE) mt[i] = nv[c++];
    wsync();
    c = 0;
    for (int i = 227 + l; i < 454; i += WAVE) nv[c++] = mt_twist_word(mt[i], mt[i + 1], mt[i - 227]);
    wsync();
    c = 0;
    for (int i = 227 + l; i < 454; i += WAVE) mt[i] = nv[c++];
    wsync();
    c = 0;
    for (int i = 454 + l; i < 623; i += WAVE) nv[c++] = mt_twist_word(mt[i], mt[i + 1], mt[i - 227]);
    wsync();
    c = 0;
    for (int i = 454 + l; i < 623; i += WAVE) mt[i] = nv[c++];
    wsync();
    uint32_t last = mt_twist_word(mt[623], mt[0], mt[396]);
    wsync();
    if (l == 0) mt[623] = last;
    wsync();
}

DEV uint32_t mt_temper(uint32_t y)
{
    y ^= y >> 11;
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= y >> 18;
    return y;
}

DEV void rng_open(Rng &r)
{
    r.pos = uni(*r.idx);
    r.base = -2 * WAVE;
}
DEV void rng_close(Rng &r) { *r.idx = r.pos; }

// The next 64 words, tempered, one per lane: a draw is then a readlane and a
// few scalar instructions instead of LDS round trips for position and word and
// the tempering.  Words beyond the end of the state are those of the next
// block, whose first 227 follow from this block's words alone; the block itself
// is renewed once the position has passed its end.
__device__ __attribute__((noinline)) uint32_t mt_words(lds_u *mt_, int pos_)
{
    lds_u *mt = uni_lds(mt_);
    const int i = uni(pos_) + lane_id();
    uint32_t y = mt[min(i, 623)];
    if (i >= 624) y = mt_twist_word(mt[i - 624], mt[i - 623], mt[i - 624 + 397]);
    return mt_temper(y);
}

// at least n words at hand (n <= 64)
DEV void rng_need(Rng &r, int n)
{
    if (r.pos - r.base > WAVE - n) {
        if (r.pos >= 624) {
            mt_regen(r.mt);
            r.pos -= 624;
        }
        r.base = r.pos;
        r.w = mt_words(r.mt, r.pos);
    }
}

DEV uint32_t mt_next(Rng &r) { return (uint32_t)__builtin_amdgcn_readlane((int)r.w, r.pos++ - r.base); }

// generate_canonical<double,53>: (g1 + g2 2^32) / 2^64, clamped below 1
template <bool CHECK = true>
DEV double grnd(Rng &r)
{
    if (CHECK) rng_need(r, 2);
    const uint32_t g1 = mt_next(r), g2 = mt_next(r);
    const double tmp = 4294967296.0;
    double sum = __dadd_rn((double)g1, __dmul_rn((double)g2, tmp));
    double ret = sum / (tmp * tmp);
    if (ret >= 1.0) ret = 0x1.fffffffffffffp-1;
    return ret;
}

// draws of a function: the position comes from and goes back to LDS
struct RngScope {
    Rng &r;
    DEV explicit RngScope(Rng &x) : r(x) { rng_open(r); }
    DEV ~RngScope() { rng_close(r); }
};

// words a move draws before a look at what is at hand: an insertion takes 14
constexpr int MOVE_WORDS = 24;

template <bool CHECK = true>
DEV int randint(Rng &r, int a, int b)
{
    if (CHECK) rng_need(r, 1);
    uint32_t range = (uint32_t)b - (uint32_t)a + 1u;
    uint64_t prod = (uint64_t)mt_next(r) * (uint64_t)range;
    uint32_t low = (uint32_t)prod;
    if (low < range) {
        uint32_t thr = (uint32_t)(0u - range) % range;
        while (low < thr) {
            rng_need(r, 1);
            prod = (uint64_t)mt_next(r) * (uint64_t)range;
            low = (uint32_t)prod;
        }
    }
    return a + (int)(prod >> 32);
}

// ---------------------------------------------------------------------------
// operator codes: orb | spin << 4 | (ca-1) << 5 ; flavour f = orb + nb*spin
// ---------------------------------------------------------------------------
DEV int op_orb(int c) { return c & 15; }
DEV int op_spin(int c) { return (c >> 4) & 1; }
DEV int op_ca(int c) { return ((c >> 5) & 1) + 1; }
DEV int mk_code(int orb, int spin, int ca) { return orb | (spin << 4) | ((ca - 1) << 5); }

// ---------------------------------------------------------------------------
// chain context: LDS views of the header, model tables and work buffers
// ---------------------------------------------------------------------------
// The kernels' model and layout arguments, read where they lie (constant
// address space: scalar loads), also by functions that are not inlined.
typedef const __attribute__((address_space(4))) DevModel CModel;
typedef const __attribute__((address_space(4))) ChainLayout CLayout;
typedef __attribute__((address_space(1))) char glb_c;
typedef const __attribute__((address_space(4))) char *CArgs;   // a kernel's arguments: model, layout, ...
typedef int iv4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) iv4 lds_i4;
typedef __attribute__((address_space(1))) double glb_d;

// What identifies a chain: the parts of a sweep that are rarely or seldom
// taken (boundary caches, accepted moves, global moves, measurements) are
// functions of their own, so that the loop over proposals stays small and has
// its registers to itself; each rebuilds its view of the chain from this.
struct ChainRef {
    CModel *M;
    CLayout *L;
    char *base;
};

// What the out-of-line functions share of a chain, in LDS, the header among it:
// one variable, since functions find a second one by a look-up in memory at
// their start (1024 chains, 40 sweeps: 1-orbital model 23.3 -> 23.0 ms, 2-orbital
// 40.2 -> 39.9 ms).
struct WalkEnv {
    ChainHdr hdr;
    double egs;
    double flops, bytes;    // algorithmic work of this launch
    const double *opsx;     // operator blocks in the order of the matrix instructions' lanes
    const lds_i4 *tr;       // transition records
    const lds_d *ev;        // energies
    const lds_b *keys;      // key of each superstate, then the superstate of each key (255: none)
    const lds_d *lops;      // operator blocks in LDS (blocks up to 4 states)
    const lds_i4 *sinfo;    // per superstate: lowest energy, size | first energy << 8, width (float)
    lds_d *qa;              // propagators of 16 operators (blocks of 5..16 states); scratch
    int ncol;               // operators per superstate (4 nb)
    int dkey;               // key change by a creator of spin 0 | of spin 1 << 8; 0: no such keys
    int np;                 // removable pairs of the window
    int k0;                 // key of the superstate at the window's lower edge (with the pair counts)
    int ready;              // window list valid and room for any move; cleared by whatever changes that
    int nkmax;              // matrix-instruction steps of the largest block
    int no;                 // states of the outer superstate (valid while ready)
    // LDS addresses: window list and trial list (their buffers swap), pair
    // counts, work vectors, segment caches, tables
    unsigned wtau, wcode, ttau, tcode, pc, q, r, col, row, rk, lb, rkx, lbx, rks, lbs;
    unsigned legc, k, sz, off, trt, evt, opst, mt, dvec, pl, strip;
};
__shared__ WalkEnv s_wenv;

DEV unsigned long long uni64(unsigned long long a)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)a),
                   hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(a >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
DEV const glb_d *uni_glb(const double *p) { return (const glb_d *)uni64((unsigned long long)p); }

// generic pointer to the LDS address a (uniform)
template <typename T>
DEV T *lds_ptr(unsigned a)
{
    typedef __attribute__((address_space(3))) T lds_t;
    return (T *)(lds_t *)(size_t)(unsigned)uni((int)a);
}

struct Ctx {
    CModel &M;
    CLayout &L;
    char *base;          // chain block in global memory
    ChainHdr &h;         // LDS copy
    Rng rng;
    // model tables (LDS)
    const int *sz, *off;
    const int4 *tr;      // per (superstate, operator): target, target size, block offset, target energies offset
    const double *ev, *opsp;   // opsp: operator blocks (LDS or global)
    // chain arrays (global)
    double *tau;
    int *code;
    double *fc, *fa, *minv, *scratch, *kst, *bnd, *bndlog, *part;
    int *fcs, *fas;      // physical row (creator) / column (annihilator) slot of each rank
    int *bndsst;
    // work buffers
    double *wtau;        // window list (LDS): operators [wia, wib) while h.wvalid
    int *wcode;
    int *pc;             // removable-pair count of each window operator (LDS, while h.pc_valid)
    double *ttau;        // trial list / staging buffer (LDS), same capacity
    int *tcode;
    double *K0, *K1;     // trace work matrices (LDS for small blocks)
    double *strip;       // LDS strip of the state for the MFMA walks (blocks above 16 states)
    double *dvec, *Q, *R, *colb, *rowb, *pl;
    // window prefix kets rk[j] (after the first j window operators) and suffix
    // bras lb[m] (after the last m), with their logs and superstates (LDS)
    double *rk, *lb, *rkx, *lbx;
    int *rks, *lbs;
    const double *legc;  // Legendre recursion coefficients (LDS)
    int nm;              // padded block size used for matrix strides
    DEV Ctx(CModel &m, CLayout &l, char *b) : M(m), L(l), base(b), h(s_wenv.hdr) {}
    // algorithmic work, added to the header by save_ctx
    DEV void work(double flops, double bytes)
    {
        s_wenv.flops += flops;
        s_wenv.bytes += bytes;
    }
    DEV ChainRef ref() const { return ChainRef{&M, &L, base}; }
    // window list and trial list of the chain (their buffers swap)
    DEV void lists()
    {
        wtau = lds_ptr<double>(s_wenv.wtau);
        wcode = lds_ptr<int>(s_wenv.wcode);
        ttau = lds_ptr<double>(s_wenv.ttau);
        tcode = lds_ptr<int>(s_wenv.tcode);
    }
    DEV double *mi(int f) { return minv + (long)f * L.kcap * L.kcap; }
    DEV int fl(int c) const { return op_orb(c) + M.nb * op_spin(c); }
    DEV int conn(int s, int c, bool adjoint) const
    {
        int ca = op_ca(c);
        if (adjoint) ca = 3 - ca;
        return tr[((s * M.nb + op_orb(c)) * 2 + op_spin(c)) * 2 + (ca - 1)].x;
    }
};

// The chain's view: chain block in global memory and the dynamic LDS.
template <int NM>
DEV Ctx attach(ChainRef r)
{
    CModel &M = *(CModel *)uni64((unsigned long long)r.M);
    CLayout &L = *(CLayout *)uni64((unsigned long long)r.L);
    char *base = (char *)(glb_c *)uni64((unsigned long long)r.base);
    Ctx c(M, L, base);
    c.nm = NM;
    c.tau = reinterpret_cast<double *>(base + L.tau);
    c.code = reinterpret_cast<int *>(base + L.code);
    c.fc = reinterpret_cast<double *>(base + L.fc);
    c.fa = reinterpret_cast<double *>(base + L.fa);
    c.fcs = reinterpret_cast<int *>(base + L.fcs);
    c.fas = reinterpret_cast<int *>(base + L.fas);
    c.minv = reinterpret_cast<double *>(base + L.minv);
    c.scratch = reinterpret_cast<double *>(base + L.scratch);
    c.kst = reinterpret_cast<double *>(base + L.kst);
    c.bnd = reinterpret_cast<double *>(base + L.bnd);
    c.bndlog = reinterpret_cast<double *>(base + L.bndlog);
    c.bndsst = reinterpret_cast<int *>(base + L.bndsst);
    c.part = reinterpret_cast<double *>(base + L.part);
    c.lists();
    const WalkEnv &e = s_wenv;
    c.pc = lds_ptr<int>(e.pc);
    c.dvec = lds_ptr<double>(e.dvec);
    c.Q = lds_ptr<double>(e.q);
    c.R = lds_ptr<double>(e.r);
    c.colb = lds_ptr<double>(e.col);
    c.rowb = lds_ptr<double>(e.row);
    c.pl = lds_ptr<double>(e.pl);
    if constexpr (NM <= 16) {
        c.rk = NM <= 4 ? lds_ptr<double>(e.rk) : reinterpret_cast<double *>(base + L.grk);
        c.lb = NM <= 4 ? lds_ptr<double>(e.lb) : reinterpret_cast<double *>(base + L.glb);
        c.rkx = lds_ptr<double>(e.rkx);
        c.lbx = lds_ptr<double>(e.lbx);
        c.rks = lds_ptr<int>(e.rks);
        c.lbs = lds_ptr<int>(e.lbs);
    }
    c.legc = lds_ptr<double>(e.legc);
    // work matrices: LDS for blocks up to 4 states (decided at compile time so
    // that their accesses are LDS instructions, not generic ones), HBM above
    if constexpr (NM <= 4) c.K0 = lds_ptr<double>(e.k);
    else c.K0 = reinterpret_cast<double *>(base + L.kwork);
    c.K1 = c.K0 + (long)NM * NM;
    c.strip = NM > 16 ? lds_ptr<double>(e.strip) : nullptr;
    c.sz = lds_ptr<int>(e.sz);
    c.off = lds_ptr<int>(e.off);
    // transition records and energies: LDS for blocks up to 16 states
    if constexpr (NM <= 16) {
        c.tr = (const int4 *)(const void *)lds_ptr<iv4>(e.trt);
        c.ev = lds_ptr<double>(e.evt);
    } else {
        c.tr = M.trans;
        c.ev = M.evals;
    }
    // operator blocks: LDS for blocks up to 4 states
    c.opsp = NM <= 4 ? lds_ptr<double>(e.opst) : M.ops;
    c.rng.mt = (lds_u *)lds_ptr<unsigned>(e.mt);
    c.rng.idx = &s_wenv.hdr.mti;
    return c;
}

// get_HybrF (Trace.F90:1014-1033)
DEV double hybr(CModel &M, double tau, int f)
{
    double sig = 1.0;
    if (tau < 0.0) {
        tau = tau + M.beta;
        sig = -1.0;
    }
    // tau / beta by the reciprocal and one correction step
    double q = tau * M.rbeta;
    q = fma(fma(-q, M.beta, tau), M.rbeta, q);
    const double n = q * (double)(M.nftau - 1);
    const int i = (int)n;
    const double *F = M.ftau + (long)f * M.nftau;
    return sig * (F[i] + (n - (double)i) * (F[i + 1] - F[i]));
}

// ---------------------------------------------------------------------------
// window (Trace.F90:1608-1751)
// ---------------------------------------------------------------------------
DEV void set_window(Ctx &c)
{
    if (c.h.nwin > 1) {
        c.h.tauwin_min = ((double)c.h.wpos / (double)(c.h.nwin + 1)) * c.M.beta;
        c.h.tauwin_max = ((double)(c.h.wpos + 2) / (double)(c.h.nwin + 1)) * c.M.beta;
    }
    c.h.wvalid = 0;
}

DEV double bound_tau(int m, int nwin, double beta)
{
    if (nwin <= 1) return m == 0 ? 0.0 : beta;
    return ((double)m / (double)(nwin + 1)) * beta;
}

// Index of the first operator at or behind x (lower) / behind x (upper): the
// sorted list is counted 256 entries at a time, one memory round trip instead
// of one per bisection step.
template <bool UPPER>
DEV int bound_index(const double *tau, int n, double x)
{
    int cnt = 0;
    for (int b = 0; b < n; b += 4 * WAVE) {
        double t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = b + u * WAVE + lane_id();
            t[u] = tau[min(j, n - 1)];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool in = b + u * WAVE + lane_id() < n;
            cnt += popc64(__ballot(in && (UPPER ? t[u] <= x : t[u] < x)));
        }
    }
    return cnt;
}
DEV int lower_bound_tau(const double *tau, int n, double x) { return bound_index<false>(tau, n, x); }
DEV int upper_bound_tau(const double *tau, int n, double x) { return bound_index<true>(tau, n, x); }

// indices [wia, wib) of the operators inside [tauwin_min, tauwin_max] and
// their copy in the LDS window list; kept across moves until the window
// shifts or a global / tau-shift move rewrites the configuration.  Returns
// false if the window does not fit the LDS list.  Up to 512 operators are read
// in one round trip.
template <int NM>
__device__ __attribute__((noinline)) bool load_window(ChainRef r)
{
    Ctx c = attach<NM>(r);
    constexpr int U = 8;
    const int n = uni(c.h.nop), l = lane_id();
    const double wmin = c.h.tauwin_min, wmax = c.h.tauwin_max;
    int ia = 0, ib = 0;
    double t[U];
    int cd[U];
    for (int b = 0; b < n; b += U * WAVE) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + u * WAVE < n) {
                const int j = min(b + u * WAVE + l, n - 1);
                t[u] = c.tau[j];
                cd[u] = c.code[j];
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + u * WAVE < n) {
                const bool in = b + u * WAVE + l < n;
                ia += popc64(__ballot(in && t[u] < wmin));
                ib += popc64(__ballot(in && t[u] <= wmax));
            }
    }
    if (ib - ia + 2 > c.L.lcap_lds) return false;
    if (n <= U * WAVE) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = u * WAVE + l;
            if (u * WAVE < n && j >= ia && j < ib) {
                c.wtau[j - ia] = t[u];
                c.wcode[j - ia] = cd[u];
            }
        }
    } else {
        for (int j = l; j < ib - ia; j += WAVE) {
            c.wtau[j] = c.tau[ia + j];
            c.wcode[j] = c.code[ia + j];
        }
    }
    c.h.wia = ia;
    c.h.wib = ib;
    c.h.wvalid = 1;
    c.h.pc_valid = 0;
    c.h.rk_n = 0;
    c.h.lb_n = 0;
    wsync();
    return true;
}

// the trial list becomes the window list (after an accepted add / remove)
DEV void swap_lists(Ctx &c)
{
    const unsigned t = s_wenv.wtau, k = s_wenv.wcode;
    s_wenv.wtau = s_wenv.ttau;
    s_wenv.wcode = s_wenv.tcode;
    s_wenv.ttau = t;
    s_wenv.tcode = k;
    c.lists();
}

// ---------------------------------------------------------------------------
// local trace
// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Walks on blocks of at most 16 states (trace engines 1, 4 and 16).
//
// A state matrix (rows: states of the current block, columns: outer states)
// lives in registers in the layout that the FP64 matrix instructions both read
// as operand B and write as D, so an operator K' = A (d o K) never moves data:
//   blocks up to 4:  entry (l/16, l%4) in lane l, the four quads (l/4)%4 of a
//     16-lane row being the four blocks of v_mfma_f64_4x4x4f64;
//   blocks up to 16: entries (4e + l/16, l%16), e = 0..3, i.e. register e is
//     operand B of k-step e of v_mfma_f64_16x16x4f64.
// Rows and columns beyond the block are zero.
// ---------------------------------------------------------------------------
typedef double dbl4 __attribute__((ext_vector_type(4)));
constexpr int DPP_ROW_ROR4 = 0x124, DPP_ROW_ROR8 = 0x128;

template <int NM>
struct State {
    static constexpr int NV = NM <= 4 ? 1 : 4;
    double v[NV];
    DEV static int row(int e) { return NM <= 4 ? lane_id() >> 4 : 4 * e + (lane_id() >> 4); }
    DEV static int col() { return NM <= 4 ? lane_id() & 3 : lane_id() & 15; }
    // row-major (ns x no) matrix
    template <typename P>
    DEV void load(P K, int ns, int no)
    {
#pragma unroll
        for (int e = 0; e < NV; ++e) {
            const bool in = row(e) < ns && col() < no;
            const double x = K[in ? row(e) * no + col() : 0];
            v[e] = in ? x : 0.0;
        }
    }
    template <typename P>
    DEV void store(P K, int ns, int no) const
    {
#pragma unroll
        for (int e = 0; e < NV; ++e)
            if (row(e) < ns && col() < no && (NM > 4 || (lane_id() & 12) == 0)) K[row(e) * no + col()] = v[e];
    }
    DEV void identity(int no)
    {
#pragma unroll
        for (int e = 0; e < NV; ++e) v[e] = row(e) == col() && col() < no ? 1.0 : 0.0;
    }
    // largest modulus of this lane's entries
    DEV double maxabs() const
    {
        double m = fabs(v[0]);
#pragma unroll
        for (int e = 1; e < NV; ++e) m = fmax(m, fabs(v[e]));
        return m;
    }
};

// Thresholds outside which a state matrix is renormalised during a walk; in
// between, the entries are left unscaled (rescaling by powers of two is exact,
// so skipping it changes no rounding).
constexpr double STATE_TINY = 0x1p-64, STATE_HUGE = 0x1p64;
// A walk looks every fourth operator whether its state needs renormalisation,
// unless a propagation of its group spans more than exp(-WALK_DECAY).  A walk
// that starts on a cached state has up to ten propagations between two looks:
// three that the cache holds, three at the end of a group of 63, four more.  They
// keep exp(-500) of the FP64 range, and a product with a cached bra exp(-150) of
// what is left.
constexpr float WALK_DECAY = 50.0f;

// power-of-two renormalisation when the largest entry of the lanes in `mask`
// leaves [2^-64, 2^64]
template <int NM>
DEV void renorm(State<NM> &k, unsigned long long mask, double &lg)
{
    const double m = k.maxabs();
    if ((__ballot(m >= STATE_TINY) & mask) == 0ull || (__ballot(m > STATE_HUGE) & mask) != 0ull) {
        const double mm = wave_max((mask >> lane_id()) & 1ull ? m : 0.0);
        if (mm > 0.0) {
            const int ex = ilogb(mm);
            lg += (double)ex * 0.69314718055994530942;
#pragma unroll
            for (int e = 0; e < State<NM>::NV; ++e) k.v[e] = ldexp(k.v[e], -ex);
        }
    }
}

// Where a walk leaves the state after each operator (at that operator's time):
// state matrices, log scales (lg0 included) and superstates.
template <int NM>
struct Prefix {
    typedef typename std::conditional<(NM <= 4), lds_d *, glb_d *>::type mat;
    mat k;
    lds_d *lg;
    lds_i *sst;
};

template <int NM>
struct WalkOut {
    State<NM> k;
    double lg;
    int s;      // superstate after the walk; -1: an operator without target block
};

// Walk of a state over the n operators of an LDS list: a ket ascending from
// entry 0 (tstart < tau_0 < ... < tend) or, with BRA, a bra descending from
// entry n-1 with the adjoint blocks (tstart > tau_{n-1} > ... > tend):
//   k <- exp(-H (t_end - t_n)) psi_n ... exp(-H (t_2 - t_1)) psi_1 exp(-H (t_1 - t_start)) k.
// Up to 63 operators at a time (lane p holds operator p, the lane behind the
// last one the propagation to tend):
//  (1) the superstate before each operator: superstates carry additive keys
//      (superstate_keys), so it is a scan over the lanes and one table read, and
//      a quantum-number violation ends the walk before any arithmetic; blocks
//      without such keys take one transition record after the other;
//  (2) block offsets, sizes, energies and log factors, all lanes at once;
//  (3) entries (blocks up to 4: block times propagator, four operators per
//      pass, one exp per lane, kept in registers: quad b of pass p holds
//      operator 4p + b) or propagators (blocks up to 16, into LDS);
//  (4) the products.  Blocks up to 4: the state moves one quad on per operator
//      (two DPP moves) to the quad that holds the operator's entries, one
//      matrix instruction each; the other quads carry nothing.  Blocks up to
//      16: ceil(ns/4) chained matrix instructions; the operator blocks lie in
//      global memory in the lanes' own order (512 bytes per k-step, zero beyond
//      the block; 216 KB for the 3-orbital model, shared by all chains), so an
//      operator is three coalesced loads, issued two operators ahead.  Blocks of
//      one state: a product over the lanes.
// The renormalisation check runs per operator only if some propagation of the
// group spans more than exp(-WALK_DECAY), else every fourth operator.
// KEEP: the states after every operator go to px.
template <int NM, bool BRA, bool KEEP>
__device__ __attribute__((noinline)) WalkOut<NM> walk_small(State<NM> k, int s_, double tstart, double tend,
                                                            const lds_d *otau_, const lds_i *ocode_, int n_,
                                                            int no_, double lg0, Prefix<NM> px)
{
    const int l = lane_id();
    const int n = uni(n_), no = uni(no_);
    const lds_d *otau = uni_lds(otau_);
    const lds_i *ocode = uni_lds(ocode_);
    // the environment (uniform)
    const WalkEnv &E = s_wenv;
    const double egs = E.egs;
    const lds_i4 *tr = uni_lds(E.tr), *sinfo = uni_lds(E.sinfo);
    const lds_d *ev = uni_lds(E.ev);
    const lds_b *keys = uni_lds(E.keys);
    const int ncol = uni(E.ncol), dkey = uni(E.dkey);
    int s = uni(s_);
    double lg = lg0;
    WalkOut<NM> out;
    out.s = -1;
    constexpr unsigned long long QUAD0 = 0x000F000F000F000Full;
    int ntns = 0, nss = 0, nts = 0;
    bool last = false;
    for (int c0 = 0; !last; c0 += 63) {
        const int nc = min(63, n - c0);
        last = c0 + nc == n;
        const int m = nc + (last ? 1 : 0);
        // operator of this lane and the time before it
        const int p = c0 + l;
        int cd = 0;
        double t = tend, tp = tstart;
        if (l < nc) {
            cd = ocode[BRA ? n - 1 - p : p];
            t = otau[BRA ? n - 1 - p : p];
        }
        if (l < m && p > 0) tp = otau[BRA ? n - p : p - 1];
        const double dt = l < m ? (BRA ? tp - t : t - tp) : 0.0;
        const int ca = BRA ? 2 - op_ca(cd) : op_ca(cd) - 1;   // 0: creator
        const int col = (op_orb(cd) * 2 + op_spin(cd)) * 2 + ca;
        // (1) superstates before each operator, (2) this lane's blocks
        int sb = s;
        iv4 rec;
        const int sfirst = s;
        if (dkey) {
            int d = (int)(signed char)(op_spin(cd) ? dkey >> 8 : dkey);
            d = l < nc ? (ca ? -d : d) : 0;
            const int key = (int)keys[s] + wave_scan_i(d) - d;
            sb = keys[256 + (key & 255)];
            const bool none = sb == 255;
            sb = none ? 0 : sb;
            rec = tr[sb * ncol + col];
            // the first operator without a target has a valid superstate before it
            if (__ballot(l < nc && (none || rec.x < 0)) != 0ull) return out;
            if (nc > 0) s = __builtin_amdgcn_readlane(rec.x, nc - 1);
            if (l >= nc) sb = s;
        } else {
            for (int kk = 0; kk < nc; ++kk) {
                sb = l == kk ? s : sb;
                s = uni(tr[s * ncol + __builtin_amdgcn_readlane(col, kk)].x);
                if (s < 0) return out;
            }
            if (l >= nc) sb = s;
            rec = tr[sb * ncol + col];
        }
        const iv4 si = sinfo[sb];
        const double e0 = __hiloint2double(si.y, si.x), lc = -(e0 - egs) * dt;
        const int ns = si.z & 255, eo = si.z >> 8;
        if (l >= nc) rec = iv4{s, ns, -1, eo};
        {
            const int nn = l < nc ? rec.y * ns : 0, n1 = l < nc ? ns : 0;
            const int both = wave_isum((nn << 12) | n1);   // at most 63 x 256 and 63 x 16
            ntns += both >> 12;
            nss += both & 0xfff;
            // sum of nt: the sum of ns but for the ends
            nts += (both & 0xfff) + (sinfo[s].z & 255) - (sinfo[sfirst].z & 255);
        }
        if constexpr (KEEP) {
            if (l < nc) px.sst[p] = rec.x;
        }
        if constexpr (NM == 1) {
            // every block is one number, every propagation a log factor only
            const lds_d *lops = uni_lds(E.lops);
            double a = l < nc ? lops[rec.z] : 1.0;
            if constexpr (KEEP) {
                a = wave_scan_mul(a);
                const double sc = wave_scan_d(lc), k0 = readlane_d(k.v[0], 0);
                if (l < nc) {
                    px.k[p] = k0 * a;
                    px.lg[p] = lg + sc;
                }
                k.v[0] *= readlane_d(a, m - 1);
                lg += readlane_d(sc, m - 1);
            } else {
                k.v[0] *= readlane_d(wave_scan_mul(a), 63);
                lg += wave_sum(lc);
            }
        } else if constexpr (NM <= 4) {
            const unsigned chk = __ballot(__int_as_float(si.w) * (float)dt > WALK_DECAY) ? 0u : 3u;
            const lds_d *lops = uni_lds(E.lops);
            const int blk = (l >> 2) & 3, i = l & 3, kr = l >> 4;
            const double sc = KEEP ? wave_scan_d(lc) : wave_sum(lc);   // log factors so far / of the group
            double lr = 0.0;                                           // renormalisations of the group
            const int pack = (rec.z & 0xfffff) | (rec.y << 20) | (ns << 24) | (l >= nc ? 1 << 28 : 0);
            for (int q0 = 0; q0 < m; q0 += 16) {
                // (3) entries A(i, kr) of operators q0 + 4 pass + blk
                double a[4];
#pragma unroll
                for (int ps = 0; ps < 4; ++ps) {
                    a[ps] = 0.0;
                    if (q0 + 4 * ps < m) {
                        const int src = q0 + 4 * ps + blk;
                        const int pk = __shfl(pack, src, WAVE), eq = __shfl(eo, src, WAVE);
                        const double dq = __shfl(dt, src, WAVE);
                        const int nt = (pk >> 20) & 15, nq = (pk >> 24) & 15;
                        const bool in = i < nt && kr < nq, fin = (pk >> 28) != 0;   // fin: the propagation to tend
                        const double pv = lops[in && !fin ? (pk & 0xfffff) + i + kr * nt : 0];
                        const double d = exp(-(ev[eq + (kr < nq ? kr : 0)] - ev[eq]) * dq);
                        a[ps] = in ? (fin ? (i == kr ? d : 0.0) : pv * d) : 0.0;
                    }
                }
                // (4) products
#pragma unroll
                for (int ps = 0; ps < 4; ++ps) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const int t_ = 4 * ps + b;
                        if (q0 + t_ < m) {
                            const double r = dpp_d<DPP_ROW_ROR4>(k.v[0]);
                            k.v[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[ps], r, 0.0, 0, 0, 0);
                            if (b == 3 || chk == 0u) renorm(k, QUAD0 << (4 * b), lr);
                            if constexpr (KEEP) {
                                if (q0 + t_ < nc) {
                                    const int j = c0 + q0 + t_;
                                    if (blk == b) px.k[j * 16 + kr * 4 + i] = k.v[0];
                                    px.lg[j] = lg + lr + readlane_d(sc, q0 + t_);
                                }
                            }
                        }
                    }
                }
            }
            lg += lr + (KEEP ? readlane_d(sc, m - 1) : sc);
            // the state to every quad
            double x = blk == ((m - 1) & 3) ? k.v[0] : 0.0;
            x += dpp_d<DPP_ROW_ROR4>(x);
            k.v[0] = x + dpp_d<DPP_ROW_ROR8>(x);
        } else {
            const unsigned chk = __ballot(__int_as_float(si.w) * (float)dt > WALK_DECAY) ? 0u : 3u;
            const double sc = KEEP ? wave_scan_d(lc) : wave_sum(lc);
            double lren = 0.0;
            auto products = [&](auto nk) {
                constexpr int NK = decltype(nk)::value;
                lds_d *qa = uni_lds(E.qa);
                const glb_d *ops = uni_glb(E.opsx) + l;
                const int lr = l & 15, lk = l >> 4;
                for (int q0 = 0; q0 < m; q0 += 16) {
                    const int mq = min(16, m - q0);
                    // (3) propagators of operators q0 .. q0 + mq - 1, state l % 16
                    wsync();
                    for (int ps = 0; 4 * ps < mq; ++ps) {
                        const int src = min(q0 + 4 * ps + lk, 63);
                        const int nq = __shfl(ns, src, WAVE), eq = __shfl(eo, src, WAVE);
                        const double dq = __shfl(dt, src, WAVE);
                        const double d = exp(-(ev[eq + (lr < nq ? lr : 0)] - ev[eq]) * dq);
                        qa[(4 * ps + lk) * 16 + lr] = lr < nq ? d : 0.0;
                    }
                    wsync();
                    // (4) products
                    const int mp = min(16, nc - q0);   // operators (the propagation to tend comes last)
                    auto load = [&](int t_, double (&a)[NK]) {
                        const int b = __builtin_amdgcn_readlane(rec.w, q0 + min(t_, mp - 1));
                        const glb_d *P = ops + (long)b * (NK * 64);
#pragma unroll
                        for (int e = 0; e < NK; ++e) a[e] = P[e * 64];
                    };
                    auto props = [&](int t_, double (&d)[NK]) {
#pragma unroll
                        for (int e = 0; e < NK; ++e) d[e] = qa[min(t_, 15) * 16 + 4 * e + lk];
                    };
                    auto step = [&](int t_, const double (&a)[NK], const double (&d)[NK]) {
                        const int nq = __builtin_amdgcn_readlane(ns, q0 + t_);
                        dbl4 r = __builtin_amdgcn_mfma_f64_16x16x4f64(a[0], k.v[0] * d[0], dbl4{0.0, 0.0, 0.0, 0.0}, 0, 0, 0);
#pragma unroll
                        for (int e = 1; e < NK; ++e)
                            if (4 * e < nq) r = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], k.v[e] * d[e], r, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; ++e) k.v[e] = r[e];
                    };
                    auto after = [&](int t_) {
                        if (((unsigned)t_ & chk) == chk) renorm(k, ~0ull, lren);
                        if constexpr (KEEP) {
                            const int j = c0 + q0 + t_;
#pragma unroll
                            for (int e = 0; e < 4; ++e) px.k[j * 256 + e * 64 + l] = k.v[e];
                            px.lg[j] = lg + lren + readlane_d(sc, q0 + t_);
                        }
                    };
                    if (mp > 0) {
                        // an odd operator first, then pairs: every load has its
                        // fixed place in the queue
                        double a0[NK], a1[NK], d0[NK], d1[NK];
                        load(0, a0);
                        load(1, a1);
                        int t_ = 0;
                        if (mp & 1) {
                            props(0, d0);
                            step(0, a0, d0);
                            load(1, a0);
                            load(2, a1);
                            after(0);
                            t_ = 1;
                        }
                        props(t_, d0);
                        for (; t_ < mp; t_ += 2) {
                            props(t_ + 1, d1);
                            step(t_, a0, d0);
                            load(t_ + 2, a0);
                            after(t_);
                            props(t_ + 2, d0);
                            step(t_ + 1, a1, d1);
                            load(t_ + 3, a1);
                            after(t_ + 1);
                        }
                    }
                    if (last && q0 + mq == m) {
#pragma unroll
                        for (int e = 0; e < NK; ++e) k.v[e] *= qa[(mq - 1) * 16 + 4 * e + lk];
                    }
                }
            };
            if (uni(E.nkmax) <= 3) products(std::integral_constant<int, 3>());
            else products(std::integral_constant<int, 4>());
            lg += lren + (KEEP ? readlane_d(sc, m - 1) : sc);
        }
    }
    if constexpr (NM > 1) renorm(k, ~0ull, lg);
    if (l == 0) {
        __builtin_amdgcn_ds_atomic_fadd_f64((lds_d *)&s_wenv.flops, (double)(no * (2 * ntns + nss)));
        __builtin_amdgcn_ds_atomic_fadd_f64((lds_d *)&s_wenv.bytes, (double)(8 * no * (nss + nts)));
    }
    out.k = k;
    out.lg = lg;
    out.s = s;
    return out;
}

// sums and scans over the 16 lanes of a row
DEV int row_sum_i(int x)
{
    x += dpp_i<DPP_QP_1032>(x);
    x += dpp_i<DPP_QP_2301>(x);
    x += dpp_i<DPP_ROW_HALF_MIRROR>(x);
    return x + dpp_i<DPP_ROW_MIRROR>(x);
}
DEV double row_sum_d(double x)
{
    x += dpp_d<DPP_QP_1032>(x);
    x += dpp_d<DPP_QP_2301>(x);
    x += dpp_d<DPP_ROW_HALF_MIRROR>(x);
    return x + dpp_d<DPP_ROW_MIRROR>(x);
}
DEV int row_scan_i(int x)
{
    x += dpp_mov_i<0x111, 0xf>(0, x);
    x += dpp_mov_i<0x112, 0xf>(0, x);
    x += dpp_mov_i<0x114, 0xf>(0, x);
    return x + dpp_mov_i<0x118, 0xf>(0, x);
}
DEV double row_scan_d(double x)
{
    x += dpp_mov_d<0x111, 0xf>(0.0, x);
    x += dpp_mov_d<0x112, 0xf>(0.0, x);
    x += dpp_mov_d<0x114, 0xf>(0.0, x);
    return x + dpp_mov_d<0x118, 0xf>(0.0, x);
}
DEV double row_scan_mul(double x)
{
    x *= dpp_mov_d<0x111, 0xf>(1.0, x);
    x *= dpp_mov_d<0x112, 0xf>(1.0, x);
    x *= dpp_mov_d<0x114, 0xf>(1.0, x);
    return x * dpp_mov_d<0x118, 0xf>(1.0, x);
}

// walk_small for lists of up to 15 operators on blocks of up to 4 states whose
// superstates have additive keys (most proposals: a 2-orbital window at
// TaudiffMax = beta / 10 holds 22 operators, a proposal walks the 8 or so
// between its changes).  Every row of 16 lanes holds the whole list (lane p of a
// row operator p, the lane behind the last one the propagation to tend), so scans
// and sums stay within a row; one exponential per lane gives the propagators of
// all operators (lane (state r, operator p) = 16 r + p); operators come in
// groups of four, filled up with identities, so that a group is four matrix
// instructions in a row and one renormalisation check, and the state ends in
// the last quad.
// A chain alone on its SIMD issues an instruction about every five cycles, so
// what counts is their number: about 350 here against 900 for the general walk.
constexpr int WALK_LONG = -2;   // superstate of a walk that walk_row leaves to walk_small
template <int NM, bool BRA, bool KEEP>
__device__ __attribute__((noinline)) WalkOut<NM> walk_row(State<NM> k, int s_, double tstart, double tend,
                                                          const lds_d *otau_, const lds_i *ocode_, int n_, int no_,
                                                          double lg0, Prefix<NM> px)
{
    const int l = lane_id(), p = l & 15;
    const int n = uni(n_), no = uni(no_);
    const lds_d *otau = uni_lds(otau_);
    const lds_i *ocode = uni_lds(ocode_);
    const WalkEnv &E = s_wenv;
    const double egs = E.egs;
    const lds_i4 *tr = uni_lds(E.tr), *sinfo = uni_lds(E.sinfo);
    const lds_d *ev = uni_lds(E.ev), *lops = uni_lds(E.lops);
    const lds_b *keys = uni_lds(E.keys);
    const int ncol = uni(E.ncol), dkey = uni(E.dkey);
    const int s0 = uni(s_);
    WalkOut<NM> out;
    out.s = -1;
    // operator of this lane, the time before it, the superstate before it
    const bool op = p < n;
    const int j = op ? (BRA ? n - 1 - p : p) : 0;
    const int cd = ocode[j];
    const double tj = otau[j], tb = otau[p > 0 && p <= n ? (BRA ? n - p : p - 1) : 0];
    const int key0 = (int)keys[s0];
    const double t = op ? tj : tend, tp = p > 0 ? tb : tstart;
    const double dt = p <= n ? (BRA ? tp - t : t - tp) : 0.0;
    const int ca = BRA ? 2 - op_ca(cd) : op_ca(cd) - 1;   // 0: creator
    const int col = (op_orb(cd) * 2 + op_spin(cd)) * 2 + ca;
    int d = (int)(signed char)(op_spin(cd) ? dkey >> 8 : dkey);
    d = op ? (ca ? -d : d) : 0;
    const int key = key0 + row_scan_i(d) - d;
    int sb = keys[256 + (key & 255)];
    const bool none = sb == 255;
    sb = none ? 0 : sb;
    const iv4 rec = tr[sb * ncol + (op ? col : 0)], si = sinfo[sb];
    if (__ballot((op && (none || rec.x < 0)) || (p == n && none)) != 0ull) return out;
    out.s = __builtin_amdgcn_readlane(sb, n);
    const double e0 = __hiloint2double(si.y, si.x), lc = -(e0 - egs) * dt;
    const int ns = si.z & 255, eo = si.z >> 8;
    if constexpr (KEEP) {
        if (l < n) px.sst[p] = rec.x;
    }
    const double sc = KEEP ? row_scan_d(lc) : row_sum_d(lc);
    double lg = lg0;
    if constexpr (NM == 1) {
        // every block is one number, every propagation a log factor only
        const double a = row_scan_mul(op ? lops[rec.z] : 1.0), k0 = readlane_d(k.v[0], 0);
        if constexpr (KEEP) {
            if (l < n) {
                px.k[p] = k0 * a;
                px.lg[p] = lg + sc;
            }
        }
        k.v[0] *= readlane_d(a, 15);   // zero in the lanes outside the block
    } else {
        // long propagations: a check per operator, left to walk_small by the
        // caller (a function that calls none saves no registers to memory; with
        // the segment caches extended in line, 2-orbital, 1024 chains, 40 sweeps
        // 39.8 -> 38.6 ms)
        if (__ballot(__int_as_float(si.w) * (float)dt > WALK_DECAY) != 0ull) {
            out.s = WALK_LONG;
            return out;
        }
        const int blk = (l >> 2) & 3, i = l & 3, r = l >> 4;
        const double dr = exp(-(ev[eo + (r < ns ? r : 0)] - e0) * dt);
        // block offset, sizes; 1 << 28: the propagation to tend, 1 << 29: beyond it
        const int pack = op ? (rec.z & 0xfffff) | (rec.y << 20) | (ns << 24) : (ns << 20) | (ns << 24) | (p == n ? 1 << 28 : 1 << 29);
        double lgb = lg, lgp = lg;   // scales before this group; of this lane's operator
        double a[4];
#pragma unroll
        for (int ps = 0; ps < 4; ++ps) {
            if (4 * ps <= n) {
                const int src = (l & 48) + 4 * ps + blk;
                const int pk = __shfl(pack, src, WAVE);
                const double dq = __shfl(dr, src, WAVE);
                const int nt = (pk >> 20) & 15, nq = (pk >> 24) & 15, oth = pk >> 28;
                const bool in = i < nt && r < nq;
                const double pv = lops[in && !oth ? (pk & 0xfffff) + i + r * nt : 0];
                a[ps] = oth ? (i == r ? (oth == 2 ? 1.0 : dq) : 0.0) : (in ? pv * dq : 0.0);
            }
        }
#pragma unroll
        for (int ps = 0; ps < 4; ++ps) {
            if (4 * ps <= n) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const double x = dpp_d<DPP_ROW_ROR4>(k.v[0]);
                    k.v[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[ps], x, 0.0, 0, 0, 0);
                    if (b == 3) renorm(k, 0xF000F000F000F000ull, lg);
                    if constexpr (KEEP) {
                        // (entries behind the n-th are rewritten before they are read)
                        if (blk == b && 4 * ps + b < n) px.k[(4 * ps + b) * 16 + r * 4 + i] = k.v[0];
                    }
                }
                if constexpr (KEEP) {
                    // lanes 4 ps .. 4 ps + 2 of the list: scales before this group's check
                    if (p >> 2 == ps) lgp = p == 4 * ps + 3 ? lg : lgb;
                    lgb = lg;
                }
            }
        }
        if constexpr (KEEP) {
            if (l < n) px.lg[p] = lgp + sc;
        }
        // the state to every quad
        double x = blk == 3 ? k.v[0] : 0.0;
        x += dpp_d<DPP_ROW_ROR4>(x);
        k.v[0] = x + dpp_d<DPP_ROW_ROR8>(x);
    }
    {
        const int both = __builtin_amdgcn_readlane(row_sum_i(op ? ((rec.y * ns) << 16) | (ns + rec.y) : 0), 0);
        const int in = __builtin_amdgcn_readlane(row_sum_i(op ? ns : 0), 0);
        if (l == 0) {
            __builtin_amdgcn_ds_atomic_fadd_f64((lds_d *)&s_wenv.flops, (double)(no * (2 * (both >> 16) + in)));
            __builtin_amdgcn_ds_atomic_fadd_f64((lds_d *)&s_wenv.bytes, (double)(8 * no * (both & 0xffff)));
        }
    }
    out.lg = lg + readlane_d(sc, KEEP ? n : 0);
    out.k = k;
    return out;
}

template <int NM, bool BRA, bool KEEP>
DEV WalkOut<NM> walk_any(State<NM> k, int s, double tstart, double tend, const lds_d *otau, const lds_i *ocode, int n,
                         int no, double lg0, Prefix<NM> px)
{
    if constexpr (NM <= 4) {
        if (n <= 15 && uni(s_wenv.dkey)) {
            const WalkOut<NM> o = walk_row<NM, BRA, KEEP>(k, s, tstart, tend, otau, ocode, n, no, lg0, px);
            if (NM == 1 || o.s != WALK_LONG) return o;
        }
    }
    return walk_small<NM, BRA, KEEP>(k, s, tstart, tend, otau, ocode, n, no, lg0, px);
}

// What an operator walk over blocks above 16 states needs, by value (the walk
// is out of line; a reference to the chain context would live in scratch).
struct MfmaEnv {
    const int *sz, *off;   // block sizes and first eigenvalue index per superstate
    const int4 *tr;        // transition records (target, its size, block offset, its energies offset)
    const double *ev, *ops;
    const double *ops16;   // zero-padded operator blocks (multiples of 16 x 16)
    const int *off16;      // their offsets, indexed like tr
    double *dvec;          // LDS: propagator factors of the current block
    double *strip;         // LDS: one 16-column strip of the state (128 x 16)
    double egs;
    int nb;
};

struct MfmaOut {
    double lg;             // log scale added by the walk
    double ntns, nss, nts; // algorithmic work: sum of nt*ns, ns, nt over the operators
    int s;                 // superstate after the walk (-1: quantum-number violation)
};

DEV int mfma_tidx(const MfmaEnv &e, int s, int c, bool adjoint)
{
    int ca = op_ca(c);
    if (adjoint) ca = 3 - ca;
    return ((s * e.nb + op_orb(c)) * 2 + op_spin(c)) * 2 + (ca - 1);
}

DEV int4 mfma_trans(const MfmaEnv &e, int s, int c, bool adjoint) { return e.tr[mfma_tidx(e, s, c, adjoint)]; }

// exp(-(E_k - E_0) dt) of superstate s into LDS, zero up to the next multiple
// of 16 (all lanes read it after the barrier)
DEV void mfma_prop(const MfmaEnv &e, int s, double dt)
{
    const int ns = e.sz[s];
    const double *E = e.ev + e.off[s];
    const double e0 = E[0];
    for (int k = lane_id(); k < (ns + 15) / 16 * 16; k += WAVE)
        e.dvec[k] = k < ns ? (ns > 1 ? exp(-(E[k] - e0) * dt) : 1.0) : 0.0;
    wsync();
}

// out[tp] (tp < NTP) += P diag(dvec) S over nkt groups of 16 k-steps: P the
// zero-padded operator block (leading dimension ldp, global), S the LDS strip
// (rows beyond the block zero).  For v_mfma_f64_16x16x4f64 lane l holds
// A(l%16, l/16) = P(16 tp + l%16, k), B(l/16, l%16) = S(k, l%16), k = k0 + l/16.
// The A fragments of group kt + 1 are loaded before the MFMAs of group kt, so
// that their latency overlaps matrix work.
template <int NTP>
DEV void mfma_kloop(dbl4 (&out)[8], const glb_d *P, int ldp, int nkt, const lds_d *sb, const lds_d *dvec, int lr,
                    int lk)
{
    double a0[4][NTP], a1[4][NTP];
    auto load_a = [&](int kt, double (&a)[4][NTP]) {
#pragma unroll
        for (int ee = 0; ee < 4; ++ee) {
            const glb_d *Pk = P + (long)(16 * kt + 4 * ee + lk) * ldp + lr;
#pragma unroll
            for (int tp = 0; tp < NTP; ++tp) a[ee][tp] = Pk[16 * tp];
        }
    };
    auto step = [&](int kt, const double (&a)[4][NTP]) {
#pragma unroll
        for (int ee = 0; ee < 4; ++ee) {
            const int k = 16 * kt + 4 * ee + lk;
            const double b = sb[k * 16 + lr] * dvec[k];
#pragma unroll
            for (int tp = 0; tp < NTP; ++tp)
                out[tp] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ee][tp], b, out[tp], 0, 0, 0);
        }
    };
    load_a(0, a0);
    int kt = 0;
    for (; kt + 1 < nkt; kt += 2) {
        load_a(kt + 1, a1);
        step(kt, a0);
        if (kt + 2 < nkt) load_a(kt + 2, a0);
        step(kt + 1, a1);
    }
    if (kt < nkt) step(kt, a0);
}

// Walk of a state (ns x no, row-major, entry (r, i) at K[r * no + i]) over
// operators otau/ocode (ascending tau; BRA: taken in descending order with the
// adjoint blocks) from tstart to tend, for blocks above 16 states, on the FP64
// matrix cores (v_mfma_f64_16x16x4f64).  The state is processed in strips of
// 16 columns (outer states); a strip stays in LDS (rows x 16) through every
// operator of the walk, so the state never goes back to memory between
// operators.  Per operator and k-step of 4 rows, lane l reads the B entry
// (row k0 + l/16, column l%16) of the strip times the source block's
// propagator exp(-(E_k - E_0) dt), and one entry of the operator block (nt x
// ns column-major) for each 16-row output tile; the output tiles accumulate
// in registers and are written back to the strip.  Each strip is
// renormalised by powers of two (exactly) when its largest entry leaves
// [2^-64, 2^64]; at the end the strips are brought to a common power of two
// (exactly) and written to Kout.  The common factors exp(-(E_0 - Egs) dt) go
// into the returned log scale.
template <bool BRA>
__device__ __attribute__((noinline)) MfmaOut walk_mfma(const MfmaEnv e, const double *Kin, double *Kout, int s0,
                                                      int no, double tstart, const double *otau, const int *ocode,
                                                      int n, double tend)
{
    MfmaOut o{0.0, 0.0, 0.0, 0.0, -1};
    const int l = lane_id(), lr = l & 15, lk = l >> 4;
    // address spaces made explicit (LDS and global instructions instead of
    // flat ones): the strip and the propagator factors live in LDS, the
    // operator blocks and the state matrices in global memory (blocks above
    // 16 states)
    lds_d *sb = (lds_d *)e.strip;   // [128 rows][16 columns]
    lds_d *dvec = (lds_d *)e.dvec;
    const glb_d *Kg = (const glb_d *)Kin;
    glb_d *Kog = (glb_d *)Kout;
    // superstate path, quantum numbers and the common log factor (uniform)
    int s = s0;
    double t = tstart;
    for (int jj = 0; jj < n; ++jj) {
        const int j = BRA ? n - 1 - jj : jj;
        const double tj = otau[j];
        const int4 tr = mfma_trans(e, s, ocode[j], BRA);
        if (tr.x < 0) return o;
        o.lg += -(e.ev[e.off[s]] - e.egs) * (BRA ? t - tj : tj - t);
        const double ns = (double)e.sz[s], nt = (double)tr.y;
        o.ntns += nt * ns;
        o.nss += ns;
        o.nts += nt;
        s = tr.x;
        t = tj;
    }
    o.lg += -(e.ev[e.off[s]] - e.egs) * (BRA ? t - tend : tend - t);
    const int sfin = s, nsfin = e.sz[sfin], ns0 = e.sz[s0];
    int emax = -2147483647, es_of[8];
    for (int q = 0; q < 8; ++q) es_of[q] = 0;
    for (int q = 0; q * 16 < no; ++q) {
        // rows beyond the block stay zero up to the 16-row padding
        for (int idx = l; idx < (ns0 + 15) / 16 * 256; idx += WAVE) {
            const int r = idx >> 4, i = q * 16 + (idx & 15);
            sb[idx] = (r < ns0 && i < no) ? Kg[(long)r * no + i] : 0.0;
        }
        wsync();
        int es = 0, ns = ns0;
        s = s0;
        t = tstart;
        for (int jj = 0; jj < n; ++jj) {
            const int j = BRA ? n - 1 - jj : jj;
            const double tj = otau[j];
            const int ti = mfma_tidx(e, s, ocode[j], BRA);
            const int4 tr = e.tr[ti];
            // uniform bounds (scalar loop control, no exec-mask branches)
            const int nt = __builtin_amdgcn_readfirstlane(tr.y);
            const int nkt = __builtin_amdgcn_readfirstlane((ns + 15) >> 4);
            const int ntp = __builtin_amdgcn_readfirstlane((nt + 15) >> 4);
            const int ldp = 16 * ntp;
            mfma_prop(e, s, BRA ? t - tj : tj - t);
            const glb_d *P = (const glb_d *)(e.ops16 + __builtin_amdgcn_readfirstlane(e.off16[ti]));
            dbl4 out[8];
#pragma unroll
            for (int tp = 0; tp < 8; ++tp) out[tp] = dbl4{0.0, 0.0, 0.0, 0.0};
            switch (ntp) {   // row tiles as a compile-time count: straight-line loads and MFMAs
            case 1: mfma_kloop<1>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            case 2: mfma_kloop<2>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            case 3: mfma_kloop<3>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            case 4: mfma_kloop<4>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            case 5: mfma_kloop<5>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            case 6: mfma_kloop<6>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            case 7: mfma_kloop<7>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            default: mfma_kloop<8>(out, P, ldp, nkt, sb, dvec, lr, lk); break;
            }
            // rows beyond the target block come out exactly zero (padded A)
            double m = 0.0;
#pragma unroll
            for (int tp = 0; tp < 8; ++tp)
                if (tp < ntp)
#pragma unroll
                    for (int ee = 0; ee < 4; ++ee) m = fmax(m, fabs(out[tp][ee]));
            int ex = 0;
            if (__ballot(m >= STATE_TINY) == 0ull || __ballot(m > STATE_HUGE) != 0ull) {
                const double mm = wave_max(m);
                if (mm > 0.0) ex = ilogb(mm);
            }
            es += ex;
            wsync();   // every lane has read the strip and dvec
#pragma unroll
            for (int tp = 0; tp < 8; ++tp)
                if (tp < ntp)
#pragma unroll
                    for (int ee = 0; ee < 4; ++ee) {
                        const int r = 16 * tp + lk + 4 * ee;
                        sb[r * 16 + lr] = ex ? ldexp(out[tp][ee], -ex) : out[tp][ee];
                    }
            wsync();
            s = tr.x;
            ns = nt;
            t = tj;
        }
        // propagation from the last operator to tend, then the strip to Kout
        mfma_prop(e, s, BRA ? t - tend : tend - t);
        for (int idx = l; idx < ns * 16; idx += WAVE) {
            const int r = idx >> 4, i = q * 16 + (idx & 15);
            if (i < no) Kog[(long)r * no + i] = sb[idx] * dvec[r];
        }
        wsync();
        es_of[q] = es;
        emax = max(emax, es);
    }
    // one power of two for the whole state (exact)
    for (int q = 0; q * 16 < no; ++q)
        if (es_of[q] != emax)
            for (int idx = l; idx < nsfin * 16; idx += WAVE) {
                const int r = idx >> 4, i = q * 16 + (idx & 15);
                if (i < no) Kog[(long)r * no + i] = ldexp(Kog[(long)r * no + i], es_of[q] - emax);
            }
    wsync();
    o.lg += (double)emax * 0.69314718055994530942;
    o.s = sfin;
    return o;
}

DEV MfmaEnv mfma_env(const Ctx &c)
{
    MfmaEnv e;
    e.sz = c.sz, e.off = c.off, e.tr = c.tr, e.ev = c.ev, e.ops = c.opsp, e.dvec = c.dvec, e.strip = c.strip;
    e.ops16 = c.M.ops16, e.off16 = c.M.opoff16;
    e.egs = c.M.egs, e.nb = c.M.nb;
    return e;
}

// algorithmic work of an MFMA walk (states in and out, block products)
DEV void mfma_work(Ctx &c, const MfmaOut &r, int no)
{
    c.work((double)no * (2.0 * r.ntns + r.nss), 8.0 * no * (r.nss + r.nts));
}


// walk_small over a list of this chain (generic pointers into LDS)
template <int NM, bool BRA>
DEV bool walk_list(State<NM> &k, int &s, double &lg, int no, double t0, const double *otau, const int *ocode, int n,
                   double t1)
{
    const WalkOut<NM> o =
        walk_any<NM, BRA, false>(k, s, t0, t1, (const lds_d *)otau, (const lds_i *)ocode, n, no, lg, Prefix<NM>{});
    if (o.s < 0) return false;
    k = o.k;
    s = o.s;
    lg = o.lg;
    return true;
}

// the same for blocks above 16 states: state matrices K / Kw in memory
template <bool BRA>
DEV bool walk_big(Ctx &c, double *&K, double *&Kw, int &s, double &lg, int no, double t0, const double *otau,
                  const int *ocode, int n, double t1)
{
    const MfmaOut r = walk_mfma<BRA>(mfma_env(c), K, Kw, s, no, t0, otau, ocode, n, t1);
    mfma_work(c, r, no);
    if (r.s < 0) return false;
    lg += r.lg;
    s = r.s;
    double *x = K;
    K = Kw;
    Kw = x;
    return true;
}

// stage global operators [j0, j1) into the LDS list (chunks of lcap)
DEV int stage_chunk(Ctx &c, int j0, int j1)
{
    const int n = min(j1 - j0, c.L.lcap_lds);
    for (int b = 0; b < n; b += 4 * WAVE) {
        double t[4];
        int cd[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = j0 + min(b + u * WAVE + lane_id(), n - 1);
            t[u] = c.tau[j], cd[u] = c.code[j];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = b + u * WAVE + lane_id();
            if (j < n) c.ttau[j] = t[u], c.tcode[j] = cd[u];
        }
    }
    wsync();
    return n;
}

// Walk over global operators [j0, j1) in LDS-staged chunks, ascending from t0
// to t1 or (BRA) descending; walk(tstart, n, tend) takes the staged chunk.
template <bool BRA, typename F>
DEV bool walk_staged(Ctx &c, double tstart, int j0, int j1, double tend, F &&walk)
{
    // one walk call site: an empty range is one chunk of no operators
    double t = tstart;
    if constexpr (!BRA) {
        int b = j0;
        do {
            const int n = b < j1 ? stage_chunk(c, b, j1) : 0;
            // the final propagation of a non-last chunk is zero
            const double te = (b + n < j1) ? c.ttau[n - 1] : tend;
            if (!walk(t, n, te)) return false;
            t = te;
            b += n;
            wsync();
        } while (b < j1);
    } else {
        int e = j1;
        do {
            const int b = max(j0, e - c.L.lcap_lds);
            const int n = e > j0 ? stage_chunk(c, b, e) : 0;
            const double te = (b > j0) ? c.ttau[0] : tend;
            if (!walk(t, n, te)) return false;
            t = te;
            e = b;
            wsync();
        } while (e > j0);
    }
    return true;
}

template <int NM, bool BRA>
DEV bool walk_global(Ctx &c, State<NM> &k, int &s, double &lg, int no, double t0, int j0, int j1, double t1)
{
    return walk_staged<BRA>(c, t0, j0, j1, t1, [&](double ta, int n, double tb) {
        return walk_list<NM, BRA>(k, s, lg, no, ta, c.ttau, c.tcode, n, tb);
    });
}

template <bool BRA>
DEV bool walk_global_big(Ctx &c, double *&K, double *&Kw, int &s, double &lg, int no, double t0, int j0, int j1,
                         double t1)
{
    return walk_staged<BRA>(c, t0, j0, j1, t1, [&](double ta, int n, double tb) {
        return walk_big<BRA>(c, K, Kw, s, lg, no, ta, c.ttau, c.tcode, n, tb);
    });
}

DEV void set_identity(double *K, int no)
{
    for (int idx = lane_id(); idx < no * no; idx += WAVE) K[idx] = (idx / no == idx % no) ? 1.0 : 0.0;
    wsync();
}

DEV void copy_mat(double *dst, const double *src, int n)
{
    for (int i = lane_id(); i < n; i += WAVE) dst[i] = src[i];
    wsync();
}

// A local trace: S exp(lg).  x: this lane's part of the part traces of the
// outer states (blocks up to 16 states; above, they are in c.pl and S is the
// sign, lg the logarithm).  The logarithms are taken only where they are kept
// (an accepted move): every column carries the same scale exp(lg), so the
// total is the plain sum of the columns (the log-space sum of addLogTr,
// Trace.F90:286-298, of the same numbers).
struct TraceVal {
    double S, lg, x;
    DEV double log_abs() const { return S == 0.0 ? -DBL_MAX : lg + log(fabs(S)); }
    DEV double sign() const { return S == 0.0 ? 0.0 : copysign(1.0, S); }
};

// from the lanes' products x (ket times bra, summed over the lane's own rows)
template <int NM>
DEV TraceVal trace_of(double x, double lg)
{
    return TraceVal{wave_sum(NM > 4 || (lane_id() & 12) == 0 ? x : 0.0), lg, x};
}

template <int NM, typename P>
DEV TraceVal contract_small(const State<NM> &k, P B, int ns, int no, double lg)
{
    State<NM> b;
    b.load(B, ns, no);
    double x = 0.0;
#pragma unroll
    for (int e = 0; e < State<NM>::NV; ++e) x = fma(k.v[e], b.v[e], x);
    return trace_of<NM>(x, lg);
}

// Contract ket K and bra B (same superstate s, both at the same tau) column by
// column; part traces to c.pl (blocks above 16 states).
DEV TraceVal contract(Ctx &c, const double *K, const double *B, int s, int no, double lg)
{
    const int ns = c.sz[s];
    double part = 0.0;
    for (int i = lane_id(); i < no; i += WAVE) {
        double acc = 0.0;
        for (int r = 0; r < ns; ++r) acc = fma(K[r * no + i], B[r * no + i], acc);
        c.pl[2 * i] = lg + log(fabs(acc));
        c.pl[2 * i + 1] = copysign(1.0, acc);
        part += acc;
    }
    const double S = wave_sum(part);
    wsync();
    if (S == 0.0) return TraceVal{0.0, -DBL_MAX, 0.0};
    return TraceVal{copysign(1.0, S), lg + log(fabs(S)), 0.0};
}

// the trace becomes the chain's: its logarithm, sign and part traces
template <int NM>
DEV void keep_trace(Ctx &c, const TraceVal &T)
{
    const int no = c.sz[c.h.outer];
    c.h.trace_log = T.log_abs();
    c.h.trace_sign = T.sign();
    if constexpr (NM <= 16) {
        double x = T.x;   // columns: sum over the rows
        x += __shfl_xor(x, 16, WAVE);
        x += __shfl_xor(x, 32, WAVE);
        if (lane_id() < no) {
            c.part[2 * lane_id()] = T.lg + log(fabs(x));
            c.part[2 * lane_id() + 1] = copysign(1.0, x);
        }
    } else {
        for (int i = lane_id(); i < 2 * no; i += WAVE) c.part[i] = c.pl[i];
    }
    wsync();
}

// Full trace of the current configuration (global moves, tau shifts,
// set_config, initial state): identity ket on the outer superstate at tau = 0
// through every operator, contracted with the identity bra at beta.
// A configuration that breaks the quantum numbers (an operator without a
// target block) has a zero trace.
template <int NM>
DEV TraceVal full_trace(Ctx &c, int outer)
{
    const int no = c.sz[outer];
    int s = outer;
    double lg = 0.0;
    if constexpr (NM <= 16) {
        State<NM> k;
        k.identity(no);
        if (!walk_global<NM, false>(c, k, s, lg, no, 0.0, 0, c.h.nop, c.M.beta) || s != outer)
            return TraceVal{0.0, -DBL_MAX, 0.0};
        double x = 0.0;
#pragma unroll
        for (int e = 0; e < State<NM>::NV; ++e)
            if (State<NM>::row(e) == State<NM>::col()) x = k.v[e];
        return trace_of<NM>(x, lg);
    } else {
        double *K = c.K0, *Kw = c.K1;
        set_identity(K, no);
        if (!walk_global_big<false>(c, K, Kw, s, lg, no, 0.0, 0, c.h.nop, c.M.beta) || s != outer) {
            wsync();
            return TraceVal{0.0, -DBL_MAX, 0.0};
        }
        set_identity(Kw, no);
        return contract(c, K, Kw, s, no, lg);
    }
}

// ---------------------------------------------------------------------------
// boundary cache: ket at the window's lower edge, bras at every upper edge
// ---------------------------------------------------------------------------
template <int NM>
DEV void rebuild_cache(Ctx &c)
{
    const int outer = c.h.outer, no = c.sz[outer];
    const int p = c.h.nwin > 1 ? c.h.wpos : 0;
    const int nw = c.h.nwin;
    const int top = (nw > 1) ? nw + 1 : 2;
    const int stride = c.nm * c.nm;
    State<NM <= 16 ? NM : 1> k;
    double *B = c.K0, *Bw = c.K1;
    if constexpr (NM <= 16) {
        k.identity(no);
        k.store(c.bnd + (long)top * stride, no, no);
    } else {
        set_identity(B, no);
        copy_mat(c.bnd + (long)top * stride, B, no * no);
    }
    int s = outer;
    double lg = 0.0;
    double tb = c.M.beta;
    int hiidx = c.h.nop;
    if (lane_id() == 0) {
        c.bndlog[top] = lg;
        c.bndsst[top] = s;
    }
    // the whole configuration in the trial list where it fits
    const bool staged = NM <= 16 && c.h.nop <= c.L.lcap_lds;
    if (staged) stage_chunk(c, 0, c.h.nop);
    for (int m = top - 1; m >= p + 2; --m) {
        const double tm = bound_tau(m, nw, c.M.beta);
        const int loidx = staged ? upper_bound_tau(c.ttau, hiidx, tm) : upper_bound_tau(c.tau, hiidx, tm);
        if constexpr (NM <= 16) {
            if (staged) walk_list<NM, true>(k, s, lg, no, tb, c.ttau + loidx, c.tcode + loidx, hiidx - loidx, tm);
            else walk_global<NM, true>(c, k, s, lg, no, tb, loidx, hiidx, tm);
            k.store(c.bnd + (long)m * stride, c.sz[s], no);
        } else {
            walk_global_big<true>(c, B, Bw, s, lg, no, tb, loidx, hiidx, tm);
            copy_mat(c.bnd + (long)m * stride, B, c.sz[s] * no);
        }
        if (lane_id() == 0) {
            c.bndlog[m] = lg;
            c.bndsst[m] = s;
        }
        tb = tm;
        hiidx = loidx;
    }
    s = outer;
    lg = 0.0;
    const double tp = bound_tau(p, nw, c.M.beta);
    const int n0 = staged ? lower_bound_tau(c.ttau, hiidx, tp) : lower_bound_tau(c.tau, hiidx, tp);
    if constexpr (NM <= 16) {
        k.identity(no);
        if (staged) walk_list<NM, false>(k, s, lg, no, 0.0, c.ttau, c.tcode, n0, tp);
        else walk_global<NM, false>(c, k, s, lg, no, 0.0, 0, n0, tp);
        k.store(c.kst, c.sz[s], no);
    } else {
        double *K = c.K0, *Kw = c.K1;
        set_identity(K, no);
        walk_global_big<false>(c, K, Kw, s, lg, no, 0.0, 0, n0, tp);
        copy_mat(c.kst, K, c.sz[s] * no);
    }
    c.h.kst_log = lg;
    c.h.kst_sst = s;
    c.h.cache_pos = p;
    wsync();
}

// Bring the caches to the current window position: advance the ket across
// passed half windows, or rebuild after a wrap / invalidation.
template <int NM>
__device__ __attribute__((noinline)) void move_cache(ChainRef r)
{
    Ctx c = attach<NM>(r);
    const int p = c.h.nwin > 1 ? c.h.wpos : 0;
    c.h.rk_n = 0;
    c.h.lb_n = 0;
    if (c.h.cache_pos < 0 || c.h.cache_pos > p) {
        rebuild_cache<NM>(c);
        return;
    }
    const int no = c.sz[c.h.outer];
    int s = c.h.kst_sst;
    double lg = c.h.kst_log;
    const double ta = bound_tau(c.h.cache_pos, c.h.nwin, c.M.beta);
    const double tb = bound_tau(p, c.h.nwin, c.M.beta);
    const int ia = lower_bound_tau(c.tau, c.h.nop, ta);
    const int ib = lower_bound_tau(c.tau, c.h.nop, tb);
    if constexpr (NM <= 16) {
        State<NM> k;
        k.load(c.kst, c.sz[s], no);
        walk_global<NM, false>(c, k, s, lg, no, ta, ia, ib, tb);
        k.store(c.kst, c.sz[s], no);
    } else {
        double *K = c.K0, *Kw = c.K1;
        copy_mat(K, c.kst, c.sz[s] * no);
        walk_global_big<false>(c, K, Kw, s, lg, no, ta, ia, ib, tb);
        copy_mat(c.kst, K, c.sz[s] * no);
    }
    c.h.kst_log = lg;
    c.h.kst_sst = s;
    c.h.cache_pos = p;
    wsync();
}

template <int NM>
DEV void ensure_cache(Ctx &c)
{
    if (c.h.cache_pos != (c.h.nwin > 1 ? c.h.wpos : 0)) move_cache<NM>(c.ref());
}

// Trace of the LDS trial list between the cached ket and bra; returns false
// on a quantum-number violation (check_sst_sequence, Trace.F90:1243-1302, on a
// superset of the changed span).
template <int NM>
DEV bool window_trace(Ctx &c, int nl, TraceVal &T)
{
    const int no = c.sz[c.h.outer];
    const int p = c.h.nwin > 1 ? c.h.wpos : 0;
    const int top = p + 2;
    const double ta = bound_tau(p, c.h.nwin, c.M.beta), tb = bound_tau(top, c.h.nwin, c.M.beta);
    int s = c.h.kst_sst;
    double lg = c.h.kst_log;
    const double *B = c.bnd + (long)top * c.nm * c.nm;
    if constexpr (NM <= 16) {
        State<NM> k;
        k.load(c.kst, c.sz[s], no);
        if (!walk_list<NM, false>(k, s, lg, no, ta, c.ttau, c.tcode, nl, tb) || s != c.bndsst[top]) return false;
        T = contract_small<NM>(k, B, c.sz[s], no, lg + c.bndlog[top]);
    } else {
        double *K = c.K0, *Kw = c.K1;
        copy_mat(K, c.kst, c.sz[s] * no);
        if (!walk_big<false>(c, K, Kw, s, lg, no, ta, c.ttau, c.tcode, nl, tb)) return false;
        if (s != c.bndsst[top]) return false;
        T = contract(c, K, B, s, no, lg + c.bndlog[top]);
    }
    return true;
}

// ---------------------------------------------------------------------------
// Window segment caches (blocks of up to 16 states).  rk[j] is the ket after the
// window's first j operators, at the time of operator j-1 (rk[0] = the cached
// ket at the window's lower edge); lb[m] is the bra after the window's last m
// operators, at the time of operator nw-m (lb[0] = the cached bra at the upper
// edge).  A proposal then walks only the operators between its changes: an
// insertion at window positions q1 <= q2 walks the two new operators and the
// q2-q1 between them, a removal of w1 < w2 the w2-w1-1 between them.  The
// caches are extended on demand and cut back to their unchanged parts after
// an accepted move; both restart when the window list is reloaded or the
// boundary caches change.  Their log scales and superstates are in LDS; the
// matrices too for blocks up to 4 states (4 x 4, zero beyond the block), above
// they are the lanes' registers as they are (2 KB, coalesced), in the chain
// block.
// ---------------------------------------------------------------------------
template <int NM>
DEV State<NM> seg_load(const double *buf, int j, int ns, int no)
{
    State<NM> k;
    if constexpr (NM == 1) {
        k.load(buf + j, ns, no);
    } else if constexpr (NM <= 4) {
        k.v[0] = buf[j * 16 + 4 * State<NM>::row(0) + State<NM>::col()];
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) k.v[e] = buf[j * 256 + e * 64 + lane_id()];
    }
    return k;
}
template <int NM>
DEV void seg_store(double *buf, int j, int ns, int no, const State<NM> &k)
{
    if constexpr (NM == 1) {
        k.store(buf + j, ns, no);
    } else if constexpr (NM <= 4) {
        if ((lane_id() & 12) == 0) buf[j * 16 + 4 * State<NM>::row(0) + State<NM>::col()] = k.v[0];
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) buf[j * 256 + e * 64 + lane_id()] = k.v[e];
    }
}

// extend rk to `to` operators (BRA = false) or lb (BRA = true); nw: window operators
template <int NM, bool BRA>
DEV void seg_extend(Ctx &c, int nw, int to)
{
    constexpr int S = NM <= 4 ? NM * NM : 256;
    double *buf = BRA ? c.lb : c.rk, *bx = BRA ? c.lbx : c.rkx;
    int *bs = BRA ? c.lbs : c.rks;
    const int no = uni(s_wenv.no);
    const int w = c.h.nwin > 1 ? c.h.wpos : 0;
    int j = uni(BRA ? c.h.lb_n : c.h.rk_n) - 1;
    State<NM> k;
    int s;
    double lg0;
    if (j < 0) {
        // the edge of the window
        s = uni(BRA ? c.bndsst[w + 2] : c.h.kst_sst);
        lg0 = BRA ? c.bndlog[w + 2] : c.h.kst_log;
        k.load(BRA ? c.bnd + (long)(w + 2) * c.nm * c.nm : c.kst, c.sz[s], no);
        seg_store<NM>(buf, 0, c.sz[s], no, k);
        bx[0] = lg0;
        bs[0] = s;
        j = 0;
    } else {
        s = uni(bs[j]);
        lg0 = bx[j];
        k = seg_load<NM>(buf, j, c.sz[s], no);
        // cached as it was between two looks: a cache that grows by one to three
        // operators at a time would never see one
        if constexpr (NM > 1) renorm(k, ~0ull, lg0);
    }
    if (j < to) {
        typedef typename Prefix<NM>::mat mat;
        const Prefix<NM> px{(mat)(buf + (long)(j + 1) * S), (lds_d *)(bx + j + 1), (lds_i *)(bs + j + 1)};
        // window operators j .. to-1 upward, or nw-1-j .. nw-to downward
        const int a = BRA ? nw - to : j;
        const double t0 = j > 0 ? c.wtau[BRA ? nw - j : j - 1] : bound_tau(BRA ? w + 2 : w, c.h.nwin, c.M.beta);
        const double t1 = c.wtau[BRA ? nw - to : to - 1];
        walk_any<NM, BRA, true>(k, s, t0, t1, (const lds_d *)(c.wtau + a), (const lds_i *)(c.wcode + a), to - j,
                                no, lg0, px);
    }
    (BRA ? c.h.lb_n : c.h.rk_n) = to + 1;
    wsync();
}

// Trace of the window with the trial list's entries [a, a + n) replacing the
// window's operators between rk[j0] and lb[m0]; t0 / t1 are the times of
// those two states.  Returns false on a quantum-number violation.
template <int NM>
DEV bool segment_trace(Ctx &c, int nw, int j0, int m0, int a, int n, double t0, double t1, TraceVal &T)
{
    if constexpr (NM <= 16) {
        const int no = uni(s_wenv.no);
        if (c.h.rk_n <= j0) seg_extend<NM, false>(c, nw, j0);
        if (c.h.lb_n <= m0) seg_extend<NM, true>(c, nw, m0);
        int s = c.rks[j0];
        double lg = c.rkx[j0];
        State<NM> k = seg_load<NM>(c.rk, j0, c.sz[s], no);
        if (!walk_list<NM, false>(k, s, lg, no, t0, c.ttau + a, c.tcode + a, n, t1) || s != c.lbs[m0]) return false;
        const State<NM> b = seg_load<NM>(c.lb, m0, c.sz[s], no);
        double x = 0.0;
#pragma unroll
        for (int e = 0; e < State<NM>::NV; ++e) x = fma(k.v[e], b.v[e], x);
        T = trace_of<NM>(x, lg + c.lbx[m0]);
    }
    return true;
}

// The window moves on by half its width (shift_window, Trace.F90:1652-1668).
// While the list and the caches belong to the window left behind, they move
// with it: the ket at the new lower edge is the prefix ket of the last operator
// passed, propagated to the edge; the prefix kets of the upper half stay (LDS
// caches); the list keeps its upper half and is continued from the
// configuration.  Otherwise the next move reloads them.
template <int NM>
__device__ __attribute__((noinline)) void slide_window(ChainRef ref)
{
    Ctx c = attach<NM>(ref);
    s_wenv.ready = 0;
    const int p = uni(c.h.wpos), nw = uni(c.h.wib - c.h.wia), nwin = uni(c.h.nwin), nop = uni(c.h.nop);
    if (nwin <= 1) {
        c.h.wpos = 0;
        return;
    }
    const bool follow = NM <= 16 && c.h.wvalid && c.h.cache_pos == p && p + 1 < nwin && nw <= c.L.sc;
    c.h.wpos = p + 1 == nwin ? 0 : p + 1;
    const double edge0 = bound_tau(p, nwin, c.M.beta);
    set_window(c);
    if constexpr (NM <= 16) {
        if (!follow) return;
        const double wmin = c.h.tauwin_min, wmax = c.h.tauwin_max, edge = bound_tau(p + 1, nwin, c.M.beta);
        int low = 0;   // operators left behind
        for (int j0 = 0; j0 < nw; j0 += WAVE) {
            const int j = j0 + lane_id();
            low += popc64(__ballot(j < nw && c.wtau[j < nw ? j : 0] < wmin));
        }
        // the operators that follow, one round trip
        const int wib = uni(c.h.wib);
        int more = 0;
        for (int j0 = wib; j0 < nop; j0 += WAVE) {
            const int j = min(j0 + lane_id(), nop - 1);
            const double t = c.tau[j];
            const int cd = c.code[j];
            const bool in = j0 + lane_id() < nop && t <= wmax;
            const int cnt = popc64(__ballot(in));
            if (nw - low + more + cnt + 2 > c.L.lcap_lds) return;   // reported by the next move
            if (in) {
                c.ttau[nw - low + more + lane_id()] = t;
                c.tcode[nw - low + more + lane_id()] = cd;
            }
            more += cnt;
            if (cnt < WAVE) break;
        }
        // ket at the new edge
        if (c.h.rk_n <= low) {
            c.h.wpos = p;   // seg_extend starts from the window left behind
            seg_extend<NM, false>(c, nw, low);
            c.h.wpos = p + 1;
        }
        const int s = uni(c.rks[low]), no = c.sz[c.h.outer], ns = c.sz[s];
        State<NM> k = seg_load<NM>(c.rk, low, ns, no);
        const double *E = c.ev + c.off[s];
        const double dt = edge - (low > 0 ? c.wtau[low - 1] : edge0), e0 = E[0];
        double lg = c.rkx[low] - (e0 - c.M.egs) * dt;
        if constexpr (NM > 1) renorm(k, ~0ull, lg);
#pragma unroll
        for (int e = 0; e < State<NM>::NV; ++e) {
            const int r = State<NM>::row(e);
            k.v[e] *= exp(-(E[r < ns ? r : 0] - e0) * dt);
        }
        if constexpr (NM > 1) renorm(k, ~0ull, lg);
        k.store(c.kst, ns, no);
        c.h.kst_log = lg;
        c.h.kst_sst = s;
        c.h.cache_pos = p + 1;
        // list
        for (int j = low + lane_id(); j < nw; j += WAVE) {
            c.ttau[j - low] = c.wtau[j];
            c.tcode[j - low] = c.wcode[j];
        }
        c.h.wia += low;
        c.h.wib = c.h.wia + nw - low + more;
        c.h.wvalid = 1;
        c.h.pc_valid = 0;
        c.h.lb_n = 0;
        if constexpr (NM <= 4) {
            // prefix kets low + 1 .. rk_n - 1 become 1 .. rk_n - 1 - low
            constexpr int S2 = NM * NM;
            const int rn = uni(c.h.rk_n) - low;
            for (int i = S2 + lane_id(); i - lane_id() < rn * S2; i += WAVE) {
                const double x = i < rn * S2 ? c.rk[low * S2 + i] : 0.0;
                wsync();
                if (i < rn * S2) c.rk[i] = x;
                wsync();
            }
            for (int i = 1 + lane_id(); i - lane_id() < rn; i += WAVE) {
                const double x = i < rn ? c.rkx[low + i] : 0.0;
                const int q = i < rn ? c.rks[low + i] : 0;
                wsync();
                if (i < rn) c.rkx[i] = x, c.rks[i] = q;
                wsync();
            }
            seg_store<NM>(c.rk, 0, ns, no, k);
            c.rkx[0] = lg;
            c.rks[0] = s;
            c.h.rk_n = rn;
        } else {
            c.h.rk_n = 0;
        }
        wsync();
        swap_lists(c);
    }
}

// Trace of a proposal: the window with its operators [j0, nw - m0) replaced by
// the n entries of the trial list from a = j0 on; nl: length of the whole
// trial list.  ok: no quantum-number violation.
struct Proposal {
    TraceVal T;
    int ok;
};
template <int NM>
__device__ __attribute__((noinline)) Proposal trace_proposal(ChainRef r, int nw_, int j0_, int m0_, int n_)
{
    Ctx c = attach<NM>(r);
    const int nw = uni(nw_), j0 = uni(j0_), m0 = uni(m0_), n = uni(n_);
    Proposal p;
    p.T = TraceVal{0.0, 0.0, 0.0};
    if (NM <= 16 && nw <= c.L.sc) {
        const int w = c.h.nwin > 1 ? c.h.wpos : 0;
        const double t0 = j0 > 0 ? c.wtau[j0 - 1] : bound_tau(w, c.h.nwin, c.M.beta);
        const double t1 = m0 > 0 ? c.wtau[nw - m0] : bound_tau(w + 2, c.h.nwin, c.M.beta);
        p.ok = segment_trace<NM>(c, nw, j0, m0, j0, n, t0, t1, p.T);
    } else {
        p.ok = window_trace<NM>(c, j0 + n + m0, p.T);
    }
    return p;
}

// change of a superstate's key by an operator (superstate_keys)
DEV int key_delta(int dkey, int code)
{
    const int d = (int)(signed char)(op_spin(code) ? dkey >> 8 : dkey);
    return op_ca(code) == 1 ? d : -d;
}

// ---------------------------------------------------------------------------
// removable pairs (ensure_valid_NPairs_diag, Trace.F90:1769-1810): for every
// window operator the later operators of its flavour and the other type no
// further than taudiff_max behind it.  pc[j] holds the counts of the first j+1
// window operators together, so that the total is known and the pick of a
// removal is one comparison per lane; kept until the window list changes.
//
// The upper 8 bits of pc[j] are the key of the superstate behind operator j (at
// most 2^19 pairs in a list of 1024): an operator pair put in or taken out
// shifts the keys between its two places by its first operator's change and
// leaves the others, so whether a proposal breaks quantum numbers is a look-up
// per operator between them, before any walk (blocked).  Three to five proposals in
// ten end there; the walk found out only after the segment caches were extended
// for it (2-orbital model 7 K cycles; the look-up is three LDS round trips).
// 1024 chains: 2-orbital, 40 sweeps 42.8 -> 40.2 ms; 1-orbital 24.2 -> 23.3 ms;
// 2-orbital in one window, 256 chains, 10 sweeps 6.8 -> 6.2 ms.
// ---------------------------------------------------------------------------
constexpr int PC_PAIRS = 0xffffff;
struct Keys {
    const lds_b *keys;    // key of each superstate, superstate of each key
    const lds_i4 *tr;
    int ncol, dkey;       // dkey 0: no such keys
    int k0;               // key at the window's lower edge
};
template <int NM>
DEV Keys window_keys()
{
    Keys q{nullptr, nullptr, 0, 0, 0};
    if constexpr (NM <= 16) {
        const WalkEnv &E = s_wenv;
        q.keys = uni_lds(E.keys);
        q.tr = uni_lds(E.tr);
        q.ncol = uni(E.ncol);
        q.dkey = uni(E.dkey);
        q.k0 = uni(E.k0);
    }
    return q;
}
// Whether quantum numbers stop one of n operators: operator i in front of window
// position q + max(i - lead, 0), the keys from i = lead on shifted.
DEV bool blocked(const Keys &ks, const int *pc, const int *code, int q, int n, int lead, int shift)
{
    bool bad = false;
    for (int i0 = 0; i0 < n; i0 += WAVE) {
        const bool in = i0 + lane_id() < n;
        const int i = in ? i0 + lane_id() : 0, a = q + max(i - lead, 0), cd = code[i];
        const int key = (a > 0 ? pc[max(a - 1, 0)] >> 24 : ks.k0) + (i >= lead ? shift : 0);
        const int s = ks.keys[256 + (key & 255)];
        const int col = (op_orb(cd) * 2 + op_spin(cd)) * 2 + op_ca(cd) - 1;
        const iv4 rec = ks.tr[(s == 255 ? 0 : s) * ks.ncol + col];
        bad |= in & ((s == 255) | (rec.x < 0));
    }
    return __ballot(bad) != 0ull;
}
template <int NM>
__device__ __attribute__((noinline)) void count_pairs(ChainRef r)
{
    Ctx c = attach<NM>(r);
    const int nw = uni(c.h.wib - c.h.wia);
    const double tdm = c.h.taudiff_max, wmax = c.h.tauwin_max;
    Keys ks = window_keys<NM>();
    if (ks.dkey) s_wenv.k0 = ks.k0 = ks.keys[uni(c.h.kst_sst)];
    int carry = (int)((unsigned)ks.k0 << 24);
    for (int j0 = 0; j0 < nw; j0 += WAVE) {
        const int j = j0 + lane_id();
        int cnt = 0;
        if (j < nw) {
            const double lim = fmin(wmax, c.wtau[j] + tdm);
            const int want = c.wcode[j] ^ 32;   // same flavour, other type
            // the list is read four entries at a time so that the LDS loads overlap
            for (int k = j + 1; k < nw; k += 4) {
                double tk[4];
                int ck[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    tk[u] = k + u < nw ? c.wtau[k + u] : DBL_MAX;
                    ck[u] = k + u < nw ? c.wcode[k + u] : -1;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) cnt += tk[u] <= lim && ck[u] == want;
                if (tk[3] > lim) break;
            }
        }
        if (ks.dkey && j < nw) cnt += (int)((unsigned)key_delta(ks.dkey, c.wcode[j]) << 24);
        const int inc = wave_scan_i(cnt) + carry;
        if (j < nw) c.pc[j] = inc;
        carry = __builtin_amdgcn_readlane(inc, 63);
    }
    s_wenv.np = carry & PC_PAIRS;
    c.h.pc_valid = 1;
    wsync();
}

// ---------------------------------------------------------------------------
// configuration sign: get_Sign with get_BlockSign and get_permaltca
// (Trace.F90:3479-3615).  Parities of
//   BlockSign: sum over operators j of the counts of later operators of the
//     flavours (b', s') with b' < o_j, plus (o_j, s'=0) when s_j = 1;
//   permaltca: sum over creators of the count of later same-flavour operators,
//     plus 1 for an odd number of pairs;
// computed per flavour g with ballots over chunks of 64 operators.
// ---------------------------------------------------------------------------
DEV double config_sign(Ctx &c)
{
    const int n = c.h.nop, nb = c.M.nb, nf = c.M.nf;
    // stage the operator codes in LDS (the trial buffer is free here)
    const int *codes = c.code;
    if (n <= 2 * c.L.lcap_lds) {
        int *st = reinterpret_cast<int *>(c.ttau);
        for (int j = lane_id(); j < n; j += WAVE) st[j] = c.code[j];
        wsync();
        codes = st;
    }
    int parity = 0, alt = 0;
    for (int g = 0; g < nf; ++g) {
        const int bg = g % nb, sg = g / nb;
        const int mg = 2 * c.h.kf[g];
        int before = 0;   // flavour-g operators before the current chunk
        for (int b0 = 0; b0 < n; b0 += WAVE) {
            const int j = b0 + lane_id();
            int cj = 0;
            bool isg = false;
            if (j < n) {
                cj = codes[j];
                isg = c.fl(cj) == g;
            }
            const unsigned long long mask = __ballot(isg);
            if (j < n) {
                const int upto = before + popc64(mask & lanemask_le());   // flavour g up to j
                const int later = mg - upto;
                const int oj = op_orb(cj), sj = op_spin(cj);
                const bool in_set = (bg < oj) || (sj == 1 && bg == oj && sg == 0);
                if (in_set) parity ^= later & 1;
                if (isg && op_ca(cj) == 1) alt ^= later & 1;
            }
            before += popc64(mask);
        }
    }
    wsync();
    parity = wave_isum(parity) & 1;
    alt = wave_isum(alt) & 1;
    if ((n / 2) % 2 == 1) alt ^= 1;
    const double block = parity ? -1.0 : 1.0, altsign = alt ? -1.0 : 1.0;
    return c.h.trace_sign * c.h.det_sign * block * altsign;
}

// ---------------------------------------------------------------------------
// hybridisation matrix algebra (MatrixUpdate.F90)
// ---------------------------------------------------------------------------
// Lanes over the elements (i, j) of a k x k block without divisions: groups of
// 16, 32 or 64 lanes hold a column each, so lane l keeps row i = l mod G and
// takes the columns g, g + 64/G, ...
struct MatLanes {
    int i, g, step;
    DEV explicit MatLanes(int k)
    {
        const int l = lane_id();
        if (k <= 16) i = l & 15, g = l >> 4, step = 4;
        else if (k <= 32) i = l & 31, g = l >> 5, step = 2;
        else i = l, g = 0, step = 1;
    }
    // sum over the lanes that hold the same row
    DEV double rows(double v) const
    {
        if (step >= 2) v += __shfl_xor(v, 32, WAVE);
        if (step == 4) v += __shfl_xor(v, 16, WAVE);
        return v;
    }
};

// The block loops below are chains of memory round trips (the inverses of a
// batch lie in HBM or the last-level cache): f(c) steps of `step` columns each,
// N at a time with all their loads ahead of their arithmetic, as long as every
// lane group has them; the last ones, at most four, go together, their column
// clamped to the last one and masked.
template <int N, typename Body>
DEV int batches(int u, int full, const Body &body)
{
    for (; u + N <= full; u += N) body(std::integral_constant<int, N>(), u);
    return u;
}

template <typename Body, typename Tail>
DEV void in_batches(int k, const MatLanes &ml, const Body &body, const Tail &tail)
{
    const int full = k / ml.step;   // steps that every lane group has
    int u = 0;
    if (ml.step == 1) u = batches<16>(u, full, body);
    u = batches<8>(u, full, body);
    u = batches<4>(u, full, body);
    if (u * ml.step < k) tail(u);
}

// M(i,j) += (a col(i)) row(j)
DEV void rank1(Ctx &c, double *Mf, int k, double a, const double *col, const double *row)
{
    const int ld = c.L.kcap;
    for (int i0 = 0; i0 < k; i0 += WAVE) {
        const MatLanes ml(k - i0);
        const int i = i0 + ml.i;
        const bool in = i < k;
        const double ci = in ? a * col[i] : 0.0;
        double *p = Mf + (in ? i : 0) + (long)ml.g * ld;
        const double *q = row + ml.g;
        const long ps = (long)ml.step * ld;
        in_batches(
            k, ml,
            [&](auto n, int) {
                constexpr int N = decltype(n)::value;
                double m[N], r[N];
#pragma unroll
                for (int v = 0; v < N; ++v) m[v] = p[v * ps];
#pragma unroll
                for (int v = 0; v < N; ++v) r[v] = q[v * ml.step];
                if (in) {
#pragma unroll
                    for (int v = 0; v < N; ++v) p[v * ps] = fma(ci, r[v], m[v]);
                }
                p += N * ps;
                q += N * ml.step;
            },
            [&](int u) {
                const int left = k - 1 - (u * ml.step + ml.g);   // columns behind this one
                double m[4], r[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int d = min(v * ml.step, left);
                    m[v] = p[(long)d * ld];
                    r[v] = q[d];
                }
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (in && v * ml.step <= left) p[v * ps] = fma(ci, r[v], m[v]);
            });
    }
}

// R^T M Q of an order-k block (get_DetRatAdd); leaves M Q in colb.
DEV double detrat_add(Ctx &c, const double *Mf, int k)
{
    const int ld = c.L.kcap;
    double part = 0.0;
    for (int i0 = 0; i0 < k; i0 += WAVE) {
        const MatLanes ml(k - i0);
        const int i = i0 + ml.i;
        const bool in = i < k;
        const double *p = Mf + (in ? i : 0) + (long)ml.g * ld, *q = c.Q + ml.g;
        const long ps = (long)ml.step * ld;
        double acc = 0.0;
        in_batches(
            k, ml,
            [&](auto n, int) {
                constexpr int N = decltype(n)::value;
                double m[N];
#pragma unroll
                for (int v = 0; v < N; ++v) m[v] = p[v * ps];
#pragma unroll
                for (int v = 0; v < N; ++v) acc = fma(m[v], q[v * ml.step], acc);
                p += N * ps;
                q += N * ml.step;
            },
            [&](int u) {
                const int left = k - 1 - (u * ml.step + ml.g);
                double m[4], r[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int d = min(v * ml.step, left);
                    m[v] = p[(long)d * ld];
                    r[v] = v * ml.step <= left ? q[d] : 0.0;
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) acc = fma(m[v], r[v], acc);
            });
        acc = ml.rows(acc);
        if (in && ml.g == 0) {
            c.colb[i] = acc;
            part = fma(c.R[i], acc, part);
        }
    }
    return wave_sum(part);
}

// Bordering update to order k+1, get_MatAdd (MatrixUpdate.F90:410-442), on
// physical storage: the new creator takes physical row k, the new annihilator
// physical column k, so no entry moves.  c.Q holds Q by physical column, c.R
// holds R by physical row, c.colb M Q (detrat_add).
//   col(i) = -(M Q)_i / dr,  row(j) = -(R M)_j / dr,
//   M(i,j) += dr col(i) row(j),  M(i,k) = col(i),  M(k,j) = row(j),  M(k,k) = 1/dr
DEV void mat_add_phys(Ctx &c, double *Mf, int k, double dr)
{
    const int ld = c.L.kcap;
    const int l = lane_id();
    double *col = c.colb, *row = c.rowb;
    // columns of M against R: the lane's column is contiguous
    for (int j0 = 0; j0 < k; j0 += WAVE) {
        const MatLanes ml(k - j0);
        const int j = j0 + ml.i;
        const double *p = Mf + (long)min(j, k - 1) * ld + ml.g, *r = c.R + ml.g;
        double v = 0.0;
        in_batches(
            k, ml,
            [&](auto n, int) {
                constexpr int N = decltype(n)::value;
                double m[N];
#pragma unroll
                for (int w = 0; w < N; ++w) m[w] = p[w * ml.step];
#pragma unroll
                for (int w = 0; w < N; ++w) v = fma(r[w * ml.step], m[w], v);
                p += N * ml.step;
                r += N * ml.step;
            },
            [&](int u) {
                const int left = k - 1 - (u * ml.step + ml.g);
                double m[4], q[4];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int d = min(w * ml.step, left);
                    m[w] = p[d];
                    q[w] = w * ml.step <= left ? r[d] : 0.0;
                }
#pragma unroll
                for (int w = 0; w < 4; ++w) v = fma(q[w], m[w], v);
            });
        v = ml.rows(v);
        if (j < k && ml.g == 0) row[j] = -v / dr;
    }
    for (int i = l; i < k; i += WAVE) col[i] = -col[i] / dr;
    wsync();
    rank1(c, Mf, k, dr, col, row);
    for (int i = l; i < k; i += WAVE) {
        Mf[i + (long)k * ld] = col[i];
        Mf[k + (long)i * ld] = row[i];
    }
    if (l == 0) Mf[k + (long)k * ld] = 1.0 / dr;
    wsync();
}

// Removal of the creator in physical row sc and the annihilator in physical
// column sa, get_MatRem (MatrixUpdate.F90:455-482):
//   M(i,j) -= M(i,sa) M(sc,j) / M(sc,sa);
// then the last physical row / column move into the freed slots.
DEV void mat_rem_phys(Ctx &c, double *Mf, int k, int sc, int sa)
{
    const int ld = c.L.kcap;
    const int l = lane_id();
    double *colp = c.colb, *rowp = c.rowb;
    for (int i = l; i < k; i += WAVE) {
        colp[i] = Mf[i + (long)sa * ld];
        rowp[i] = Mf[sc + (long)i * ld];
    }
    wsync();
    rank1(c, Mf, k, -(1.0 / rowp[sa]), colp, rowp);
    wsync();
    const int last = k - 1;
    if (sc != last) {
        for (int j = l; j < k; j += WAVE) Mf[sc + (long)j * ld] = Mf[last + (long)j * ld];
        wsync();
    }
    if (sa != last) {
        for (int i = l; i < k; i += WAVE) Mf[i + (long)sa * ld] = Mf[i + (long)last * ld];
        wsync();
    }
}

// log|det| and sign from pivots: the product by mantissa and exponent, one
// logarithm at the end
struct PivotProduct {
    double m = 1.0;
    int e = 0;
    DEV void mul(double d, bool swapped)
    {
        m *= swapped ? -d : d;
        const int x = ilogb(m);
        m = ldexp(m, -x);
        e += x;
    }
    DEV double log_abs() const { return log(fabs(m)) + (double)e * 0.69314718055994530942; }
    DEV double sign() const { return m >= 0.0 ? 1.0 : -1.0; }
};

// Pivot of column col among the rows col .. k-1 (largest modulus, lowest row
// among ties), swapped into row col; false if the column is zero.
template <typename P>
DEV bool pivot_row(P A, int k, int ld, int col, int &bi)
{
    const int l = lane_id();
    double best = -1.0;
    bi = 0x7fffffff;
    for (int r = l; r < k; r += WAVE) {
        const double v = r >= col ? fabs(A[r + (long)col * ld]) : -1.0;
        if (v > best) best = v, bi = r;
    }
    const double wb = wave_max(best);
    bi = wave_imin(best == wb ? bi : 0x7fffffff);
    if (!(wb > 0.0)) return false;
    if (bi != col) {
        for (int j = l; j < k; j += WAVE) {
            const double t = A[col + (long)j * ld], u = A[bi + (long)j * ld];
            A[col + (long)j * ld] = u;
            A[bi + (long)j * ld] = t;
        }
    }
    wsync();
    return true;
}

// LU with partial pivoting of A (k x k, ld) in place; log|det| and sign as
// get_LogDetFull (MatrixUpdate.F90:302-339).  Returns false if singular.
template <typename P>
DEV bool lu_inplace(P A, int k, int ld, double &dl, double &ds)
{
    const MatLanes ml(k);
    PivotProduct det;
    for (int col = 0; col < k; ++col) {
        int bi;
        if (!pivot_row(A, k, ld, col, bi)) {
            dl = 0.0;
            ds = 1.0;
            return false;
        }
        const double d = A[col + (long)col * ld];
        det.mul(d, bi != col);
        const double rd = 1.0 / d;
        for (int i0 = 0; i0 < k; i0 += WAVE) {
            const int i = i0 + ml.i;
            if (i > col && i < k) {
                const double f = A[i + (long)col * ld] * rd;
                for (int j = col + 1 + ml.g; j < k; j += ml.step) A[i + (long)j * ld] -= f * A[col + (long)j * ld];
            }
        }
        wsync();
    }
    dl = det.log_abs();
    ds = det.sign();
    return true;
}

// Inverse of A (k x k, ld) in place by Gauss-Jordan elimination with partial
// pivoting, and the determinant from its pivots; piv: k ints.
template <typename P>
DEV bool gj_inverse(P A, int k, int ld, int *piv, double &dl, double &ds)
{
    const int l = lane_id();
    const MatLanes ml(k);
    PivotProduct det;
    for (int col = 0; col < k; ++col) {
        int bi;
        if (!pivot_row(A, k, ld, col, bi)) {
            dl = 0.0;
            ds = 1.0;
            return false;
        }
        const double d = A[col + (long)col * ld], rd = 1.0 / d;
        det.mul(d, bi != col);
        if (l == 0) piv[col] = bi;
        wsync();
        // the pivot row, with the pivot's place taken by the inverse's column
        for (int j = l; j < k; j += WAVE) A[col + (long)j * ld] = j == col ? rd : A[col + (long)j * ld] * rd;
        wsync();
        for (int i0 = 0; i0 < k; i0 += WAVE) {
            const int i = i0 + ml.i;
            const bool in = i < k && i != col;
            const double f = in ? A[i + (long)col * ld] : 0.0;
            wsync();
            if (in)
                for (int j = ml.g; j < k; j += ml.step)
                    A[i + (long)j * ld] = fma(-f, A[col + (long)j * ld], j == col ? 0.0 : A[i + (long)j * ld]);
        }
        wsync();
    }
    // undo the row swaps as column swaps
    for (int col = k - 1; col >= 0; --col) {
        const int b = uni(piv[col]);
        if (b == col) continue;
        for (int i = l; i < k; i += WAVE) {
            const double t = A[i + (long)col * ld], u = A[i + (long)b * ld];
            A[i + (long)col * ld] = u;
            A[i + (long)b * ld] = t;
        }
        wsync();
    }
    dl = det.log_abs();
    ds = det.sign();
    return true;
}

// Delta_f(row = annihilator rank, col = creator rank) = F(tau_a - tau_c)
// (get_InvFullHybr, Trace.F90:2279-2333) from the per-flavour lists
template <typename P>
DEV void build_delta(Ctx &c, int f, int k, P D, int ld, const double *fcl, const double *fal)
{
    const double *ct = fcl + (long)f * c.L.kcap, *at = fal + (long)f * c.L.kcap;
    const MatLanes ml(k);
    for (int i0 = 0; i0 < k; i0 += WAVE) {
        const int r = i0 + ml.i;
        const double ta = at[min(r, k - 1)];
        for (int j0 = ml.g; j0 < k; j0 += 4 * ml.step) {
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = hybr(c.M, ta - ct[min(j0 + u * ml.step, k - 1)], f);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (r < k && j0 + u * ml.step < k) D[r + (long)(j0 + u * ml.step) * ld] = v[u];
        }
    }
    wsync();
}

// LDS work area for one k x k block: the window segment caches (blocks up to 4
// states) or the trial list (blocks up to 16), both free during the moves that
// need it; its size in doubles
template <int NM>
DEV lds_d *block_area(Ctx &c, long &cap)
{
    if constexpr (NM <= 4) {
        cap = 2L * (c.L.sc + 1) * NM * NM;
        c.h.rk_n = 0;
        c.h.lb_n = 0;
        return (lds_d *)c.rk;
    } else if constexpr (NM <= 16) {
        cap = 3L * (c.L.lcap_lds & ~1) / 2;   // times and codes lie behind each other
        return (lds_d *)c.ttau;
    } else {
        cap = 0;
        return nullptr;
    }
}

// determinant of Delta_f of the given lists
template <int NM>
DEV bool delta_det(Ctx &c, int f, int k, const double *fcl, const double *fal, double &dl, double &ds)
{
    long cap;
    lds_d *A = block_area<NM>(c, cap);
    if ((long)k * k <= cap) {
        build_delta(c, f, k, A, k, fcl, fal);
        return lu_inplace(A, k, k, dl, ds);
    }
    build_delta(c, f, k, c.scratch, c.L.kcap, fcl, fal);
    return lu_inplace(c.scratch, k, c.L.kcap, dl, ds);
}

// M_f = Delta_f^{-1} of the chain's lists (physical order = ranks), and det Delta_f
template <int NM>
DEV bool delta_inverse(Ctx &c, int f, int k, double &dl, double &ds)
{
    long cap;
    lds_d *A = block_area<NM>(c, cap);
    int *piv = reinterpret_cast<int *>(c.R);
    double *Mf = c.mi(f);
    const int ld = c.L.kcap;
    if ((long)k * k <= cap) {
        build_delta(c, f, k, A, k, c.fc, c.fa);
        const bool ok = gj_inverse(A, k, k, piv, dl, ds);
        const MatLanes ml(k);
        for (int i0 = 0; i0 < k; i0 += WAVE) {
            const int i = i0 + ml.i;
            if (i < k)
                for (int j = ml.g; j < k; j += ml.step) Mf[i + (long)j * ld] = A[i + (long)j * k];
        }
        wsync();
        return ok;
    }
    build_delta(c, f, k, Mf, ld, c.fc, c.fa);
    return gj_inverse(Mf, k, ld, piv, dl, ds);
}

// ---------------------------------------------------------------------------
// array edits (lane-parallel shifts; chunks ordered so nothing is overwritten
// before it is read)
// ---------------------------------------------------------------------------
// Move the operators [from, to) by `by` places (either sign).  Rounds of 4
// operators per lane: all loads of a round complete before its stores, and
// rounds run from the end that is written into first, so nothing is
// overwritten unread.
DEV void move_ops(Ctx &c, int from, int to, int by)
{
    constexpr int U = 4, R = U * WAVE;
    const int l = lane_id();
    const int cnt = to - from;
    if (cnt <= 0 || by == 0) return;
    const int nr = (cnt + R - 1) / R;
    for (int q = 0; q < nr; ++q) {
        const int b = from + (by > 0 ? nr - 1 - q : q) * R + l;
        double t[U];
        int cd[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + u * WAVE < to) t[u] = c.tau[b + u * WAVE], cd[u] = c.code[b + u * WAVE];
        wsync();
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b + u * WAVE < to) c.tau[b + u * WAVE + by] = t[u], c.code[b + u * WAVE + by] = cd[u];
        wsync();
    }
}

// A pair joins the flavour lists (sorted times and their physical slots) of
// length k: creator tc at rank pc, annihilator ta at rank pa, both in slot k.
DEV void lists_insert(Ctx &c, long fo, int k, int pc, double tc, int pa, double ta)
{
    double *fc = c.fc + fo, *fa = c.fa + fo;
    int *fcs = c.fcs + fo, *fas = c.fas + fo;
    for (int b = k / WAVE * WAVE; b >= 0; b -= WAVE) {
        const int j = b + lane_id();
        const bool mc = j > pc && j <= k, ma = j > pa && j <= k;
        double vc = tc, va = ta;
        int sc = k, sa = k;
        if (mc) vc = fc[j - 1], sc = fcs[j - 1];
        if (ma) va = fa[j - 1], sa = fas[j - 1];
        wsync();
        if (mc || j == pc) fc[j] = vc, fcs[j] = sc;
        if (ma || j == pa) fa[j] = va, fas[j] = sa;
        wsync();
    }
}

// The creator of rank pc (slot sc) and the annihilator of rank pa (slot sa)
// leave the flavour lists of length k; the operators that owned the last slot
// take the freed ones.
DEV void lists_remove(Ctx &c, long fo, int k, int pc, int sc, int pa, int sa)
{
    double *fc = c.fc + fo, *fa = c.fa + fo;
    int *fcs = c.fcs + fo, *fas = c.fas + fo;
    for (int b = 0; b < k; b += WAVE) {
        const int j = b + lane_id();
        const bool in = j < k - 1;
        double vc = 0.0, va = 0.0;
        int xc = 0, xa = 0;
        if (in) {
            const int jc = j + (j >= pc), ja = j + (j >= pa);
            vc = fc[jc], xc = fcs[jc];
            va = fa[ja], xa = fas[ja];
        }
        wsync();
        if (in) {
            fc[j] = vc, fcs[j] = xc == k - 1 ? sc : xc;
            fa[j] = va, fas[j] = xa == k - 1 ? sa : xa;
        }
        wsync();
    }
}

// parallel count of entries < x in a sorted list of n
DEV int count_below_par(const double *arr, int n, double x)
{
    int cnt = 0;
    for (int j = lane_id(); j < n; j += WAVE) cnt += arr[j] < x;
    return wave_isum(cnt);
}

// ---------------------------------------------------------------------------
// moves
// ---------------------------------------------------------------------------
enum { OUT_REJ = 0, OUT_ACC = 1, OUT_QN = 2 };
enum { ERR_CAP = 3, ERR_SING = 4, ERR_STATE_DEV = 6 };

// write the LDS trial list into the global operator list at wia (its length
// nl replaces the window's nw operators: the tail [wib, nop) moves first); the
// trial list then serves as the window list
DEV void commit_window(Ctx &c, int nl)
{
    const int nw = c.h.wib - c.h.wia;
    move_ops(c, c.h.wib, c.h.nop, nl - nw);
    for (int j = lane_id(); j < nl; j += WAVE) {
        c.tau[c.h.wia + j] = c.ttau[j];
        c.code[c.h.wia + j] = c.tcode[j];
    }
    wsync();
    c.h.nop += nl - nw;
    c.h.wib = c.h.wia + nl;
    swap_lists(c);
}

// An accepted insertion or removal of a pair of flavour f spanning dt
// (CTQMC.F90:3579-3587, 4119-4127): the histogram AccPair over NAccPair bins
// of [0, AccPairMax] and, while the calibration list is open, the distance.
DEV void record_pair(Ctx &c, int f, double dt)
{
    if (lane_id() == 0) {
        double *ap = reinterpret_cast<double *>(c.base + c.L.accpair) + (long)f * c.L.naccpair_cap;
        const int bin = min(c.h.naccpair, (int)floor(dt / c.h.accpair_max * (double)c.h.naccpair) + 1);
        global_add(ap + bin - 1, 1.0);
        if (c.h.apt_index <= c.h.apt_n) reinterpret_cast<double *>(c.base + c.L.aptau)[c.h.apt_index - 1] = dt;
    }
    if (c.h.apt_index <= c.h.apt_n) c.h.apt_index++;
}

// Sign of the whole configuration.  Accepted insertions and removals carry the
// sign on from move to move; behind a zero trace there is none to carry.
template <int NM>
__device__ __attribute__((noinline)) void sign_anew(ChainRef r)
{
    Ctx c = attach<NM>(r);
    c.h.cfgsign = -config_sign(c);
}

// an accepted insertion / removal: what the proposal found
struct AddMove {
    int f, k, nl, q1, q2, fp_c, fp_a;   // flavour, its order, length of the trial list, insertion points, FPos
    double ta, tc, S, dr_sign;          // times, determinant ratio and its sign with the permutation's
    double cfg_ratio;                   // change of the configuration sign but for the trace's
    TraceVal T;
};
struct RemMove {
    int f, k, nl, w1, w2, fp_c, fp_a, sc, sa;   // window indices of the pair, its physical slots
    double dt, S, dr_sign, cfg_ratio;
    TraceVal T;
};

// accept: M, operator list, flavour lists, weights, sign
template <int NM>
__device__ __attribute__((noinline)) void accept_add(ChainRef ref, AddMove m)
{
    Ctx c = attach<NM>(ref);
    const int f = uni(m.f), k = uni(m.k), nl = uni(m.nl), q1 = uni(m.q1), q2 = uni(m.q2), fp_c = uni(m.fp_c),
              fp_a = uni(m.fp_a), nw = nl - 2;
    const double S = m.S, tc = m.tc, ta = m.ta;
    const long fo = (long)f * c.L.kcap;
    const bool seg = NM <= 16 && nw <= c.L.sc;
    mat_add_phys(c, c.mi(f), k, S);
    c.work(6.0 * k * k, 8.0 * k * k + 8.0 * (k + 1) * (k + 1));
    s_wenv.ready = 0;
    commit_window(c, nl);
    c.h.pc_valid = 0;
    // segment caches: the first q1 and the last nw - q2 window operators are unchanged
    c.h.rk_n = seg ? min(c.h.rk_n, q1 + 1) : 0;
    c.h.lb_n = seg ? min(c.h.lb_n, nw - q2 + 1) : 0;
    lists_insert(c, fo, k, fp_c - 1, tc, fp_a - 1, ta);
    c.h.kf[f] = k + 1;
    c.h.kfmax[f] = max(c.h.kfmax[f], k + 1);
    record_pair(c, f, fabs(ta - tc));
    c.h.det_log += log(fabs(S));
    c.h.det_sign *= m.dr_sign;
    c.h.cfgsign *= m.cfg_ratio * c.h.trace_sign;
    keep_trace<NM>(c, m.T);
    c.h.cfgsign *= c.h.trace_sign;
    c.h.acc_add++;
}

// |new weight / old weight| of a trace T and a determinant ratio S: one
// exponential; through the logarithms where that could leave the FP64 range
DEV double weight_ratio(const TraceVal &T, double S, double trace_log)
{
    const double d = T.lg - trace_log;
    if (fabs(d) < 500.0) return fabs(T.S * S) * exp(d);
    return exp((T.log_abs() - trace_log) + log(fabs(S)));
}

// StepAdd (CTQMC.F90:3353-3612), change_outer = false
template <int NM>
DEV int step_add(Ctx &c)
{
    CModel &M = c.M;
    const double wmin = c.h.tauwin_min, wmax = c.h.tauwin_max, tdm = c.h.taudiff_max;
    const int nw = uni(c.h.wib - c.h.wia);
    const double width = wmax - wmin;
    const double tref = wmin + width * grnd<false>(c.rng);
    double tdf = width;
    const int orb = randint<false>(c.rng, 1, M.nb) - 1;
    const int spin = randint<false>(c.rng, 1, 2) - 1;
    const double tmin = fmax(tref - tdm, wmin);
    const double w2 = fmin(tref + tdm, wmax) - tmin;
    const double t2 = tmin + w2 * grnd<false>(c.rng);
    tdf *= w2;
    const int f = orb + M.nb * spin;
    if (t2 == tref) return OUT_QN;
    const int k = uni(c.h.kf[f]);
    ensure_cache<NM>(c);
    if (!c.h.pc_valid) count_pairs<NM>(c.ref());
    // equal times (process_OperAdd, Trace.F90:4287-4380), insertion points, the
    // removable pairs that the two operators form with those of the window, and
    // the trial list: the window with t1 before index q1 and t2o before index q2
    const double ta = tref, tc = t2;
    const double t1 = fmin(ta, tc), t2o = fmax(ta, tc);
    const int code_a = mk_code(orb, spin, 2), code_c = mk_code(orb, spin, 1);
    int q1 = 0, q2 = 0, np = uni(s_wenv.np) + (t2o <= t1 + tdm ? 1 : 0);
    bool eq = false;
    for (int j0 = 0; j0 < nw; j0 += WAVE) {
        const int j = j0 + lane_id();
        const bool in = j < nw;
        const double x = in ? c.wtau[j] : DBL_MAX;
        const int cd = in ? c.wcode[j] : 0;
        const bool b1 = x < t1, b2 = x < t2o;
        eq = eq || __ballot(x == t1 || x == t2o) != 0ull;
        q1 += popc64(__ballot(b1));
        q2 += popc64(__ballot(b2));
        const double mate = cd == code_c ? ta : tc;
        const bool pair = in && (cd == code_c || cd == code_a) && fmax(x, mate) <= fmin(x, mate) + tdm;
        np += popc64(__ballot(pair));
        if (in) {
            const int d = j + !b1 + !b2;
            c.ttau[d] = x;
            c.tcode[d] = cd;
        }
    }
    if (eq) return OUT_QN;
    if (lane_id() < 2) {
        const bool second = lane_id() == 1;
        const int d = second ? q2 + 1 : q1;
        c.ttau[d] = second ? t2o : t1;
        c.tcode[d] = ((ta < tc) != second) ? code_a : code_c;
    }
    wsync();
    const Keys ks = window_keys<NM>();
    if (ks.dkey && blocked(ks, c.pc, c.tcode + q1, q1, q2 - q1 + 2, 1, key_delta(ks.dkey, ta < tc ? code_a : code_c)))
        return OUT_QN;
    const int nl = nw + 2;
    const Proposal pr = trace_proposal<NM>(c.ref(), nw, q1, nw - q2, q2 - q1 + 2);
    if (!pr.ok) return OUT_QN;
    const TraceVal T = pr.T;
    // det ratio, get_LogDetRatPairAdd (Trace.F90:2775-2832): Q (annihilators) and
    // R (creators) placed by physical slot, the lane behind the last rank takes
    // S0 = F(ta - tc); FPos = 1 + earlier operators of the type
    const long fo = (long)f * c.L.kcap;
    const double *ctl = c.fc + fo, *atl = c.fa + fo;
    const int *csl = c.fcs + fo, *asl = c.fas + fo;
    int fp_c = 1, fp_a = 1, sgn = q2 - q1 + (ta > tc) + 1;
    double S0 = 0.0;
    for (int j0 = 0; j0 <= k; j0 += WAVE) {
        const int j = j0 + lane_id();
        const bool in = j < k;
        double xa = ta, xc = tc;
        int sa = 0, sc = 0;
        if (in) xa = atl[j], xc = ctl[j], sa = asl[j], sc = csl[j];
        const double q = hybr(M, xa - tc, f), r = hybr(M, ta - xc, f);
        if (in) {
            c.Q[sa] = q;
            c.R[sc] = r;
        }
        if (k - j0 < WAVE) S0 = readlane_d(q, k - j0);
        const bool a_lt = in && xa < ta, c_lt = in && xc < tc;
        fp_a += popc64(__ballot(a_lt));
        fp_c += popc64(__ballot(c_lt));
        // sign change of the operator order (config_sign): operators of other
        // flavours between the pair, creators of its own between them, and
        // operators of its own behind the new creator
        const bool abet = in && xa > t1 && xa < t2o;
        sgn += popc64(__ballot(abet)) + popc64(__ballot(in && xc > tc)) + popc64(__ballot(in && xa > tc));
    }
    wsync();
    const double S = S0 - detrat_add(c, c.mi(f), k);
    c.work(2.0 * k * k, 8.0 * k * k);
    const double sig = ((fp_c - fp_a) & 1) ? -1.0 : 1.0;
    const double dr_sign = copysign(1.0, S) * sig;
    const double rnd = grnd<false>(c.rng);
    const double wr = weight_ratio(T, S, c.h.trace_log);
    const double prob = fabs(((1.0 * tdf) * (double)(2 * M.nb)) / (double)np * wr);
    if (!(rnd < prob)) return OUT_REJ;
    accept_add<NM>(c.ref(), AddMove{f, k, nl, q1, q2, fp_c, fp_a, ta, tc, S, dr_sign,
                                    (sgn & 1) ? -dr_sign : dr_sign, T});
    c.lists();
    if (c.h.cfgsign == 0.0) sign_anew<NM>(c.ref());
    return OUT_ACC;
}

template <int NM>
__device__ __attribute__((noinline)) void accept_rem(ChainRef ref, RemMove m)
{
    Ctx c = attach<NM>(ref);
    const int f = uni(m.f), k = uni(m.k), nl = uni(m.nl), w1 = uni(m.w1), w2 = uni(m.w2), fp_c = uni(m.fp_c),
              fp_a = uni(m.fp_a), sc = uni(m.sc), sa = uni(m.sa), nw = nl + 2;
    const double S = m.S;
    const long fo = (long)f * c.L.kcap;
    const bool seg = NM <= 16 && nw <= c.L.sc;
    mat_rem_phys(c, c.mi(f), k, sc, sa);
    c.work(3.0 * k * k, 8.0 * k * k + 8.0 * (k - 1) * (k - 1));
    s_wenv.ready = 0;
    commit_window(c, nl);
    c.h.pc_valid = 0;
    // segment caches: the first w1 and the last nw - 1 - w2 window operators are unchanged
    c.h.rk_n = seg ? min(c.h.rk_n, w1 + 1) : 0;
    c.h.lb_n = seg ? min(c.h.lb_n, nw - w2) : 0;
    lists_remove(c, fo, k, fp_c - 1, sc, fp_a - 1, sa);
    c.h.kf[f] = k - 1;
    record_pair(c, f, m.dt);
    c.h.det_log += log(fabs(S));
    c.h.det_sign *= m.dr_sign;
    c.h.cfgsign *= m.cfg_ratio * c.h.trace_sign;
    keep_trace<NM>(c, m.T);
    c.h.cfgsign *= c.h.trace_sign;
    c.h.acc_rem++;
}

// StepRem (CTQMC.F90:3892-4150) with gen_OperRemove (Trace.F90:4851-4977)
template <int NM>
DEV int step_rem(Ctx &c)
{
    CModel &M = c.M;
    const int nw = uni(c.h.wib - c.h.wia);
    ensure_cache<NM>(c);
    if (!c.h.pc_valid) count_pairs<NM>(c.ref());
    const int np = uni(s_wenv.np);
    if (np <= 0) return OUT_QN;
    int pick = randint<false>(c.rng, 1, np);
    // the pick-th pair: the operator w1 whose running count reaches it, and
    // among the later operators of its flavour and the other type the one that
    // the rest of the count names
    int w1 = -1, w2 = -1, want = pick;
    for (int j0 = 0; j0 < nw && w1 < 0; j0 += WAVE) {
        const int j = j0 + lane_id();
        const int pc = j < nw ? c.pc[j] & PC_PAIRS : 0;
        const unsigned long long at = __ballot(j < nw && pc >= pick);
        const int b = at ? __builtin_ctzll(at) : WAVE;
        if (b > 0) want = pick - __builtin_amdgcn_readlane(pc, b - 1);
        if (at) w1 = j0 + b;
    }
    if (w1 < 0) {
        c.h.err = ERR_STATE_DEV, s_wenv.ready = 0;
        return OUT_REJ;
    }
    const int c1 = uni(c.wcode[w1]);
    for (int j0 = w1 / WAVE * WAVE; j0 < nw && w2 < 0; j0 += WAVE) {
        const int j = j0 + lane_id();
        unsigned long long mate = __ballot(j > w1 && j < nw && c.wcode[j < nw ? j : 0] == (c1 ^ 32));
        const int n = popc64(mate);
        if (n < want) {
            want -= n;
            continue;
        }
        for (; want > 1; --want) mate &= mate - 1;
        w2 = j0 + __builtin_ctzll(mate);
    }
    if (w2 < 0) {
        c.h.err = ERR_STATE_DEV, s_wenv.ready = 0;
        return OUT_REJ;
    }
    const Keys ks = window_keys<NM>();
    if (ks.dkey && w2 > w1 + 1 &&
        blocked(ks, c.pc, c.wcode + w1 + 1, w1 + 1, w2 - w1 - 1, 0, -key_delta(ks.dkey, c1)))
        return OUT_QN;
    const double t1 = c.wtau[w1], t2 = c.wtau[w2];
    const double wmin = c.h.tauwin_min, wmax = c.h.tauwin_max, tdm = c.h.taudiff_max;
    const int f = c.fl(c1);
    const int k = uni(c.h.kf[f]);
    const double tc = op_ca(c1) == 1 ? t1 : t2, ta = op_ca(c1) == 1 ? t2 : t1;
    const double hprf = (double)np / ((wmax - wmin) * (fmin(ta + tdm, wmax) - fmax(ta - tdm, wmin)));
    // trial list: the window without entries w1 < w2
    const int nl = nw - 2;
    for (int j = lane_id(); j < nw; j += WAVE) {
        const double x = c.wtau[j];
        const int cd = c.wcode[j];
        if (j != w1 && j != w2) {
            const int d = j - (j > w1) - (j > w2);
            c.ttau[d] = x;
            c.tcode[d] = cd;
        }
    }
    wsync();
    const Proposal pr = trace_proposal<NM>(c.ref(), nw, w1, nw - 1 - w2, w2 - w1 - 1);
    if (!pr.ok) return OUT_QN;
    const TraceVal T = pr.T;
    // ranks and slots of the pair; sign change as in step_add
    const long fo = (long)f * c.L.kcap;
    const double *ctl = c.fc + fo, *atl = c.fa + fo;
    const int *csl = c.fcs + fo, *asl = c.fas + fo;
    int fp_c = 1, fp_a = 1, sc = 0, sa = 0, sgn = w2 - w1 - 1 + 1;
    for (int j0 = 0; j0 < k; j0 += WAVE) {
        const int j = j0 + lane_id();
        const bool in = j < k;
        double xa = 0.0, xc = 0.0;
        int xsa = 0, xsc = 0;
        if (in) xa = atl[j], xc = ctl[j], xsa = asl[j], xsc = csl[j];
        fp_a += popc64(__ballot(in && xa < ta));
        fp_c += popc64(__ballot(in && xc < tc));
        if (fp_a - 1 >= j0 && fp_a - 1 < j0 + WAVE) sa = __builtin_amdgcn_readlane(xsa, fp_a - 1 - j0);
        if (fp_c - 1 >= j0 && fp_c - 1 < j0 + WAVE) sc = __builtin_amdgcn_readlane(xsc, fp_c - 1 - j0);
        const bool abet = in && xa > t1 && xa < t2;
        sgn += popc64(__ballot(abet)) + popc64(__ballot(in && xc > tc)) + popc64(__ballot(in && xa > tc));
    }
    // get_LogDetRatPairRem (Trace.F90:2937-2963): M(FPos(1), FPos(2))
    const double S = c.mi(f)[sc + (long)sa * c.L.kcap];
    const double sig = ((fp_c - fp_a) & 1) ? -1.0 : 1.0;
    const double dr_sign = copysign(1.0, S) * sig;
    const double wr = weight_ratio(T, S, c.h.trace_log);
    const double prob = fabs(((1.0 * hprf) / (double)(2 * M.nb)) * wr);
    const double rnd = grnd<false>(c.rng);
    if (!(rnd < prob)) return OUT_REJ;
    if (fabs(S) < 1e-12) {
        c.h.err = ERR_SING, s_wenv.ready = 0;
        return OUT_REJ;
    }
    accept_rem<NM>(c.ref(), RemMove{f, k, nl, w1, w2, fp_c, fp_a, sc, sa, t2 - t1, S, dr_sign,
                                    (sgn & 1) ? -dr_sign : dr_sign, T});
    c.lists();
    if (c.h.cfgsign == 0.0) sign_anew<NM>(c.ref());
    return OUT_ACC;
}

// relabel flavours / swap c and c+ (globalUpdate, Trace.F90:2126-2188)
DEV void global_update(Ctx &c, const int *gu)
{
    CModel &M = c.M;
    for (int j = lane_id(); j < c.h.nop; j += WAVE) {
        const int cj = c.code[j];
        const int idx = op_orb(cj) + M.nb * op_spin(cj) + 1;
        const int g = gu[idx];
        int ca = op_ca(cj);
        if (gu[0] != 0) ca = 3 - ca;
        c.code[j] = mk_code((g - 1) % M.nb, (g - 1) / M.nb, ca);
    }
    wsync();
}

// per-flavour tau lists and orders from the operator list: ballot-compact the
// creators / annihilators of every flavour in each 64-operator chunk (lane g of
// the counts: creators of flavour g, lane 32 + g its annihilators).  With slot
// lists given, slots are reset to the identity (logical = physical order).
DEV void rebuild_flavour_lists(Ctx &c, double *dfc, double *dfa, int *dkf, int *dfcs, int *dfas)
{
    CModel &M = c.M;
    const long kc = c.L.kcap;
    const int n = uni(c.h.nop), l = lane_id(), nf = M.nf;
    const unsigned long long below = l == 0 ? 0ull : (~0ull >> (64 - l));
    int counts = 0;
    for (int b0 = 0; b0 < n; b0 += WAVE) {
        const int j = b0 + l;
        const int cj = j < n ? c.code[j] : 0;
        const double tj = j < n ? c.tau[j] : 0.0;
        const int fj = j < n ? c.fl(cj) : -1;
        const bool cre = op_ca(cj) == 1;
        for (int g = 0; g < nf; ++g) {
            const bool isc = fj == g && cre, isa = fj == g && !cre;
            const unsigned long long mc = __ballot(isc), ma = __ballot(isa);
            const int nc = __builtin_amdgcn_readlane(counts, g), na = __builtin_amdgcn_readlane(counts, 32 + g);
            if (isc) dfc[g * kc + nc + popc64(mc & below)] = tj;
            if (isa) dfa[g * kc + na + popc64(ma & below)] = tj;
            counts += (l == g ? popc64(mc) : 0) + (l == 32 + g ? popc64(ma) : 0);
        }
    }
    for (int g = 0; g < nf; ++g) {
        const int nc = __builtin_amdgcn_readlane(counts, g);
        if (dfcs)
            for (int r = l; r < nc; r += WAVE) {
                dfcs[g * kc + r] = r;
                dfas[g * kc + r] = r;
            }
        if (l == 0) dkf[g] = nc;
    }
    wsync();
}

DEV void all_outer(Ctx &c, unsigned long long *okmask)
{
    for (int w = 0; w < MAXSST / WAVE; ++w) {
        const int left = c.M.nsst - w * WAVE;
        okmask[w] = left <= 0 ? 0ull : left >= WAVE ? ~0ull : (1ull << left) - 1ull;
    }
}

// Which of the superstates set in okmask (one bit each) give a valid cyclic
// sequence of the configuration; the others' bits are cleared, the number of
// the ones left returned.  With additive keys the lanes take 64 operators at a
// time, else a superstate each.
template <int NM>
DEV int valid_outer(Ctx &c, unsigned long long *okmask)
{
    const int n = uni(c.h.nop), l = lane_id();
    int total = 0;
    if constexpr (NM <= 16) {
        const int dkey = uni(s_wenv.dkey), ncol = uni(s_wenv.ncol);
        if (dkey) {
            const lds_b *keys = uni_lds(s_wenv.keys);
            int carry = 0;
            for (int j0 = 0; j0 < n; j0 += WAVE) {
                const bool in = j0 + l < n;
                const int cd = in ? c.code[j0 + l] : 0;
                const int d = in ? key_delta(dkey, cd) : 0;
                const int sum = wave_scan_i(d), pre = carry + sum - d;
                const int col = (op_orb(cd) * 2 + op_spin(cd)) * 2 + op_ca(cd) - 1;
                carry += __builtin_amdgcn_readlane(sum, 63);
                for (int w = 0; w * WAVE < c.M.nsst; ++w) {
                    unsigned long long left = okmask[w], ok = left;
                    for (; left; left &= left - 1) {
                        const int b = __builtin_ctzll(left);
                        const int sb = keys[256 + (((int)keys[w * WAVE + b] + pre) & 255)];
                        const int t = c.tr[(sb == 255 ? 0 : sb) * ncol + col].x;
                        if (__ballot(in && (sb == 255 || t < 0)) != 0ull) ok &= ~(1ull << b);
                    }
                    okmask[w] = ok;
                }
            }
            for (int w = 0; w * WAVE < c.M.nsst; ++w) {
                if ((carry & 255) != 0) okmask[w] = 0ull;
                total += popc64(okmask[w]);
            }
            return total;
        }
    }
    for (int s0 = 0; s0 < c.M.nsst; s0 += WAVE) {
        const int s = s0 + l;
        bool ok = false;
        if (s < c.M.nsst && ((okmask[s0 / WAVE] >> l) & 1ull)) {
            int cur = s;
            for (int j = 0; j < n && cur >= 0; ++j) cur = c.conn(cur, c.code[j], false);
            ok = (cur == s);
        }
        const unsigned long long m = __ballot(ok);
        okmask[s0 / WAVE] = m;
        total += popc64(m);
    }
    return total;
}

// superstate before operator `first` of the configuration
template <int NM>
DEV int sst_before(Ctx &c, int first)
{
    int s = uni(c.h.outer);
    if constexpr (NM <= 16) {
        const int dkey = uni(s_wenv.dkey);
        if (dkey) {
            int sum = 0;
            for (int j = lane_id(); j < first; j += WAVE) sum += key_delta(dkey, c.code[j]);
            const lds_b *keys = uni_lds(s_wenv.keys);
            return uni((int)keys[256 + (((int)keys[s] + wave_isum(sum)) & 255)]);
        }
    }
    for (int i = 0; i < first; ++i) s = c.conn(s, c.code[i], false);
    return s;
}

// StepGlob (CTQMC.F90:4433-4554)
template <int NM>
__device__ __attribute__((noinline)) int step_glob(ChainRef ref)
{
    Ctx c = attach<NM>(ref);
    s_wenv.ready = 0;
    const RngScope rs(c.rng);
    CModel &M = c.M;
    c.h.try_glob++;
    if (c.h.nop == 0) return OUT_REJ;
    const int nf = M.nf, nb = M.nb;
    int gu[MAXF + 1], igu[MAXF + 1];
    const double r = grnd(c.rng);
    bool spinflip = false;
    if (r < 0.3) {
        spinflip = true;
        gu[0] = 0;
        for (int i = 1; i <= nb; ++i) gu[i] = i + nb;
        for (int i = nb + 1; i <= 2 * nb; ++i) gu[i] = i - nb;
    } else if (r < 0.6) {
        gu[0] = 1;
        for (int i = 1; i <= nf; ++i) gu[i] = i;
    } else if (NM <= 16 && r < 0.8 && M.nsym > 0) {
        // gen_SymUpdate (Trace.F90:1166-1182): a user permutation or its inverse
        // (engines up to 16 states; the MFMA engine refuses NSymMove)
        if constexpr (NM <= 16) {
            const int isym = randint(c.rng, 1, 2 * M.nsym);
            gu[0] = 0;
            for (int i = 1; i <= nf; ++i) gu[i] = M.symmoves[(isym - 1) * nf + (i - 1)];
        }
    } else {
        for (int i = 1; i <= nf; ++i) gu[i] = i;
        for (int j = 1; j <= nf; ++j) {   // rand_perm (Trace.F90:1065-1080)
            const int i = randint(c.rng, j, nf);
            const int t = gu[j];
            gu[j] = gu[i];
            gu[i] = t;
        }
        gu[0] = randint(c.rng, 0, 1);
    }
    for (int i = 1; i <= nf; ++i) igu[gu[i]] = i;
    igu[0] = gu[0];
    const int old_outer = c.h.outer;
    double sst_factor;
    unsigned long long okm[MAXSST / WAVE];   // valid outer superstates, one bit each
    if (spinflip && M.has_szt) {
        // perform_spinflip_check_qn (Trace.F90:1306-1339)
        const int st = M.first_state[c.h.outer];
        const int dn = st & ((1 << nb) - 1), up = (st >> nb) & ((1 << nb) - 1);
        const int nst = up | (dn << nb);
        c.h.outer = M.state_sst[nst];
        global_update(c, gu);
        okm[0] = okm[1] = okm[2] = okm[3] = 0;
        okm[c.h.outer / WAVE] = 1ull << (c.h.outer % WAVE);
        sst_factor = valid_outer<NM>(c, okm) ? 1.0 : 0.0;
    } else {
        // perform_global_check_qn (Trace.F90:1345-1383)
        all_outer(c, okm);
        const int pold = valid_outer<NM>(c, okm);
        global_update(c, gu);
        all_outer(c, okm);
        const int pnew = valid_outer<NM>(c, okm);
        if (pnew <= 0) {
            sst_factor = 0.0;
        } else {
            sst_factor = (double)pnew / (double)pold;
            int kk = randint(c.rng, 1, pnew);
            for (int s = 0; s < M.nsst; ++s)
                if (((okm[s / WAVE] >> (s % WAVE)) & 1ull) && --kk <= 0) {
                    c.h.outer = s;
                    break;
                }
        }
    }
    if (sst_factor == 0.0) {
        c.h.outer = old_outer;
        global_update(c, igu);
        return c.h.qn_rej++, OUT_QN;
    }
    // flavour lists of the relabelled configuration in the operator scratch
    const long kc = c.L.kcap;
    double *tfc = c.scratch + c.L.kmat, *tfa = tfc + nf * kc;
    int *tkf = reinterpret_cast<int *>(tfa + nf * kc);
    rebuild_flavour_lists(c, tfc, tfa, tkf, nullptr, nullptr);
    // det(new Delta) * det(old M) (get_InvFullHybr, get_FullLogDet)
    double dnl = 0.0, dns = 1.0;
    bool sing = false;
    for (int f = 0; f < nf; ++f) {
        const int k = tkf[f];
        if (k > 0) {
            double l, s;
            if (!delta_det<NM>(c, f, k, tfc, tfa, l, s)) sing = true;
            dnl += l;
            dns *= s;
        }
        c.work((2.0 / 3.0) * k * k * k, 8.0 * k * k);
    }
    // det(old M) = 1 / det(old Delta), which the chain carries
    const double dol = -c.h.det_log;
    const TraceVal T = full_trace<NM>(c, c.h.outer);
    const double wr = exp((T.log_abs() - c.h.trace_log) + (dnl + dol));
    const double rr = grnd(c.rng);   // drawn even for a singular Delta (prob = 0)
    if (!sing && rr < fabs(wr * sst_factor)) {
        rebuild_flavour_lists(c, c.fc, c.fa, c.h.kf, c.fcs, c.fas);
        for (int f = 0; f < nf; ++f) {
            const int k = c.h.kf[f];
            if (k == 0) continue;
            double l, s;
            delta_inverse<NM>(c, f, k, l, s);
            c.work(2.0 * k * k * k, 8.0 * k * k);
        }
        c.h.det_log = dnl;
        c.h.det_sign = dns;
        keep_trace<NM>(c, T);
        c.h.cfgsign = -config_sign(c);
        c.h.cache_pos = -1;
        c.h.wvalid = 0;   // relabelled codes: reload the window list
        c.h.acc_glob++;
        return OUT_ACC;
    }
    c.h.outer = old_outer;
    global_update(c, igu);
    return OUT_REJ;
}

// empty-trace weights of every superstate into c.Q (sum returned)
template <int NM>
DEV double empty_weights(Ctx &c)
{
    double sum = 0.0;
    for (int q = 0; q < c.M.nsst; ++q) {
        const TraceVal T = full_trace<NM>(c, q);
        const double v = T.sign() * exp(T.log_abs());
        if (lane_id() == 0) c.Q[q] = v;
        sum += v;
    }
    wsync();
    return sum;
}

// choose the outer superstate proportional to the empty traces (init_Trace,
// Trace.F90:640-670; StepChangeOuter, CTQMC.F90:4569-4637)
template <int NM>
DEV void choose_outer(Ctx &c)
{
    const double sum = empty_weights<NM>(c);
    const double r = grnd(c.rng);
    double acc = 0.0;
    int pick = c.M.nsst - 1;
    for (int q = 0; q < c.M.nsst; ++q) {
        const double v = c.Q[q] / sum;
        acc += v;
        if (acc >= r && v != 0.0) {
            pick = q;
            break;
        }
    }
    c.h.outer = pick;
    keep_trace<NM>(c, full_trace<NM>(c, pick));
    c.h.cache_pos = -1;
    c.h.pc_valid = 0;   // the key at the window's lower edge
}

// StepShiftTau_proper (CTQMC.F90:4641-4835) + update_InvFullHybrShiftTau_diag
// (Trace.F90:2355-2457)
template <int NM>
__device__ __attribute__((noinline)) int step_shift(ChainRef ref)
{
    Ctx c = attach<NM>(ref);
    s_wenv.ready = 0;
    const RngScope rs(c.rng);
    CModel &M = c.M;
    if (c.h.nop == 0) {
        choose_outer<NM>(c);
        c.h.cfgsign = -config_sign(c);
        return OUT_REJ;
    }
    const double dtau = grnd(c.rng) * M.beta;
    if (dtau == 0.0 || dtau == M.beta) return OUT_REJ;
    c.h.try_shift++;
    const int n = c.h.nop, nf = M.nf;
    int first = lower_bound_tau(c.tau, n, dtau);
    if (first == n) first = 0;
    const int s = sst_before<NM>(c, first);
    // rotate through the operator scratch area behind the matrix scratch
    double *opscr = c.scratch + c.L.kmat;
    double *old_tau = opscr;
    int *old_code = reinterpret_cast<int *>(opscr + n);
    for (int i = lane_id(); i < n; i += WAVE) {
        old_tau[i] = c.tau[i];
        old_code[i] = c.code[i];
    }
    wsync();
    for (int i = lane_id(); i < n; i += WAVE) {
        const int src = (first + i) % n;
        const double t = old_tau[src] - dtau;
        c.tau[i] = t - floor(t / M.beta) * M.beta;
        c.code[i] = old_code[src];
    }
    wsync();
    const int old_outer = c.h.outer, old_pos = c.h.wpos;
    const double old_min = c.h.tauwin_min, old_max = c.h.tauwin_max;
    c.h.outer = s;
    if (c.h.nwin > 1) {
        const int nw = c.h.nwin;
        const int a = (int)floor((dtau / M.beta) * (double)(nw + 1));
        const int am = ((a % nw) + nw) % nw;
        const int p = old_pos - am;
        c.h.wpos = ((p % nw) + nw) % nw;
    } else {
        c.h.wpos = 0;
    }
    set_window(c);
    const TraceVal T = full_trace<NM>(c, c.h.outer);
    const double ratio = T.sign() * c.h.trace_sign * exp(T.log_abs() - c.h.trace_log);
    if (grnd(c.rng) < fabs(1.0 * ratio * 1.0)) {
        keep_trace<NM>(c, T);
        double detrat = 1.0;
        const int ld = c.L.kcap;
        const long kc = c.L.kcap;
        for (int f = 0; f < nf; ++f) {
            const int k = c.h.kf[f];
            double *fcf = c.fc + f * kc, *faf = c.fa + f * kc;
            int *fcsf = c.fcs + f * kc, *fasf = c.fas + f * kc;
            const int w1 = count_below_par(fcf, k, dtau);
            const int w2 = count_below_par(faf, k, dtau);
            double *Mf = c.mi(f);
            if (!((w1 == 0 && w2 == 0) || (w1 == k && w2 == k))) {
                // negate the physical rows of wrapped creators and columns of
                // wrapped annihilators (entries wrapped on both sides keep sign)
                double *rneg = c.colb, *cneg = c.rowb;
                for (int r = lane_id(); r < k; r += WAVE) {
                    rneg[fcsf[r]] = r < w1 ? 1.0 : 0.0;
                    cneg[fasf[r]] = r < w2 ? 1.0 : 0.0;
                }
                wsync();
                for (int idx = lane_id(); idx < k * k; idx += WAVE) {
                    const int i = idx % k, j = idx / k;
                    if (rneg[i] != cneg[j]) Mf[i + (long)j * ld] = -Mf[i + (long)j * ld];
                }
                wsync();
            }
            // rotate ranks: the wrapped operators move to the end, taus shifted
            // like the operator list
            int *rs = reinterpret_cast<int *>(c.R);
            for (int r = lane_id(); r < k; r += WAVE) {
                const int src = (r + w1) % k;
                const double t = fcf[src] - dtau;
                c.Q[r] = t - floor(t / M.beta) * M.beta;
                rs[r] = fcsf[src];
            }
            wsync();
            for (int r = lane_id(); r < k; r += WAVE) {
                fcf[r] = c.Q[r];
                fcsf[r] = rs[r];
            }
            wsync();
            for (int r = lane_id(); r < k; r += WAVE) {
                const int src = (r + w2) % k;
                const double t = faf[src] - dtau;
                c.Q[r] = t - floor(t / M.beta) * M.beta;
                rs[r] = fasf[src];
            }
            wsync();
            for (int r = lane_id(); r < k; r += WAVE) {
                faf[r] = c.Q[r];
                fasf[r] = rs[r];
            }
            wsync();
            if (k % 2 != 0 && (w1 + w2) % 2 != 0) detrat = -detrat;
        }
        c.h.det_sign *= detrat;
        c.h.cfgsign = -config_sign(c);
        c.h.cache_pos = -1;
        c.h.acc_shift++;
        return OUT_ACC;
    }
    for (int i = lane_id(); i < n; i += WAVE) {
        c.tau[i] = old_tau[i];
        c.code[i] = old_code[i];
    }
    wsync();
    c.h.outer = old_outer;
    c.h.wpos = old_pos;
    c.h.tauwin_min = old_min;
    c.h.tauwin_max = old_max;
    c.h.wvalid = 0;
    return OUT_REJ;
}

// Whether the next move fits the chain's memory whatever it proposes: every
// flavour can take one more pair and the window plus a pair fits the LDS
// lists.  Checked before the move's first random draw, so a chain that has no
// room stops with its state and random stream intact and continues exactly
// where it stopped once the host has enlarged its memory.  Loads the window
// list (as the next insertion or removal would).  A chain that has stopped on
// an error is not ready either.
template <int NM>
__device__ __attribute__((noinline)) bool make_ready(ChainRef r)
{
    Ctx c = attach<NM>(r);
    if (c.h.err != 0 || c.h.halt != HALT_NONE) return false;
    int km = 0;
    for (int f = lane_id(); f < c.M.nf; f += WAVE) km = c.h.kf[f];
    km = wave_imax(km);
    const bool ok = km + 1 <= c.L.kcap && c.h.nop + 2 <= c.L.cap && (c.h.wvalid || load_window<NM>(r)) &&
                    c.h.wib - c.h.wia + 2 <= c.L.lcap_lds;
    if (!ok) c.h.halt = HALT_CAP;
    s_wenv.ready = ok;
    s_wenv.no = c.sz[c.h.outer];
    wsync();
    return ok;
}

// A count of moves in 32 bits: a launch has at most LAUNCH_MOVES moves, so what
// lies further ahead is as good as never.
DEV int near(long long n) { return (int)min(n, (long long)0x7fffffff); }

// What a sweep counts in registers: insertion and removal attempts, proposals
// rejected by quantum numbers, and the attempts since the last multiple of
// nslide (where nslide exceeds 32 bits: such that the next multiple comes up at
// near(nslide), 0 only at a multiple).
struct Tally {
    int add, rem, qn, slide;
};

// one Metropolis step with the dispatch of ctqmc_warmup / ctqmc_measure
// (CTQMC.F90:8213-8254, 8432-8533) and the window-shift rule
template <int NM>
DEV void one_move(Ctx &c, Tally &ty, int &kind, int &out)
{
    CModel &M = c.M;
    rng_need(c.rng, MOVE_WORDS);
    const double r = grnd<false>(c.rng);
    if (r <= 1.0 - M.p_shift - M.p_glob) {
        c.rng.pos += 4;   // the draws of Percentage4OperatorMove and PercentageOuterMove
        if (r < (1.0 - M.p_shift - M.p_glob) / 2.0) {
            kind = 1;
            ty.add++;
            out = step_add<NM>(c);
        } else {
            kind = 2;
            ty.rem++;
            out = step_rem<NM>(c);
        }
        ty.qn += out == OUT_QN;
        if (++ty.slide == near(M.nslide)) ty.slide = 0;
    } else {
        rng_close(c.rng);
        if (r <= 1.0 - M.p_shift) {
            kind = 3;
            out = step_glob<NM>(c.ref());
        } else {
            kind = 4;
            out = step_shift<NM>(c.ref());
        }
        rng_open(c.rng);
    }
    // every nslide-th attempt; after a global move or shift the count, and with
    // it this condition, stands
    if (ty.slide == 0) {
        slide_window<NM>(c.ref());
        c.lists();
    }
}

// ---------------------------------------------------------------------------
// measurements
// ---------------------------------------------------------------------------
// Reduce-scatter of 16 values over the 16 lanes of a DPP row: afterwards lane
// i of the row holds the sum over the row of v[i & 15].  Pairing steps: row
// mirror (i <-> 15-i), half-row mirror (i <-> 7-i), quad swaps (i <-> i^2,
// i <-> i^1); at each step a lane keeps the half its position selects and
// receives the partner's copy of that half.
DEV double row_reduce_scatter16(double (&v)[16])
{
    const int i = lane_id() & 15;
    {
        const bool hi = i >= 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const double keep = hi ? v[j + 8] : v[j], give = hi ? v[j] : v[j + 8];
            v[j] = keep + dpp_d<DPP_ROW_MIRROR>(give);
        }
    }
    {
        const bool hi = (i & 7) >= 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double keep = hi ? v[j + 4] : v[j], give = hi ? v[j] : v[j + 4];
            v[j] = keep + dpp_d<DPP_ROW_HALF_MIRROR>(give);
        }
    }
    {
        const bool hi = (i & 3) >= 2;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const double keep = hi ? v[j + 2] : v[j], give = hi ? v[j] : v[j + 2];
            v[j] = keep + dpp_d<DPP_QP_2301>(give);
        }
    }
    const bool hi = (i & 1) != 0;
    const double keep = hi ? v[1] : v[0], give = hi ? v[0] : v[1];
    return keep + dpp_d<DPP_QP_1032>(give);
}

// MeasGtauRem (CTQMC.F90:2252-2440): lanes over (annihilator, creator) pairs,
// up to four pairs per lane.  G(tau) bins by atomic adds; the Legendre sums run
// the Bonnet recursion of all pairs side by side, fold 16 orders at a time with
// row_reduce_scatter16 and add them to the chain's sums.  Bound by instruction
// issue of one wave; the orders are a loop of 16 at a time and not unrolled: the
// unrolled form was 24 KB of code per flavour that every measurement fetched
// anew (2-orbital model: 208 K cycles per measurement, 3-orbital 632 K).
struct GtauArgs {
    int nf, ntau, nleg, kcap;
    double beta, rbeta, cfgsign;
    const double *legc;
    const int *kf;
    const double *fc, *fa, *minv;
    const int *fcs, *fas;
    double *gtau, *gleg;
    double *mstep, *dstep;   // this measurement's row of Gtau_mean_step / Gtau_mid_step (or null)
};

// the pairs p0 .. p0 + 64 PPL - 1 of flavour f (k of them each way): lane l
// takes p0 + l + 64 u
template <int PPL>
DEV void gtau_pairs(const GtauArgs &a, int f, int k, int p0)
{
    const int ld = a.kcap, npair = k * k;
    const double *ctl = a.fc + (long)f * a.kcap, *atl = a.fa + (long)f * a.kcap;
    const int *csl = a.fcs + (long)f * a.kcap, *asl = a.fas + (long)f * a.kcap;
    const double *Mf = a.minv + (long)f * a.kcap * a.kcap;
    const float rk = 1.0f / (float)k;
    double Mv[PPL], x[PPL], pl[PPL], plm1[PPL], ta[PPL], tc[PPL], m[PPL];
#pragma unroll
    for (int u = 0; u < PPL; ++u) {
        const int p = min(p0 + lane_id() + WAVE * u, npair - 1);
        int ai = (int)((float)p * rk);   // annihilator rank p / k (k <= 4096: off by one at most)
        ai -= ai * k > p;
        ai += (ai + 1) * k <= p;
        const int ci = p - ai * k;       // creator rank
        ta[u] = atl[ai];
        tc[u] = ctl[ci];
        m[u] = Mf[csl[ci] + (long)asl[ai] * ld];
    }
#pragma unroll
    for (int u = 0; u < PPL; ++u) {
        const bool in = p0 + lane_id() + WAVE * u < npair;
        const double d = ta[u] - tc[u];
        const bool fwd = d > 0.0;
        const double dt = fwd ? d : a.beta + ta[u] - tc[u];
        // dt / beta by the reciprocal and one correction step
        double q = dt * a.rbeta;
        q = fma(fma(-q, a.beta, dt), a.rbeta, q);
        const int idt = min((int)(q * (double)a.ntau) + 1, a.ntau);
        x[u] = in ? 2.0 / a.beta * dt - 1.0 : 0.0;
        Mv[u] = in ? (fwd ? m[u] : -m[u]) * a.cfgsign : 0.0;
        if (in) {
            global_add(&a.gtau[(long)f * a.ntau + idt - 1], Mv[u]);
            // step-resolved sums (CTQMC.F90:2394-2401): M * cfgsign of
            // every pair, and of pairs with |ta - tc| / beta in [0.4, 0.6]
            if (a.mstep) global_add(&a.mstep[f], Mv[u] * a.cfgsign);
            if (a.dstep) {
                const double r = fabs(d) / a.beta;
                if (r >= 0.4 && r <= 0.6) global_add(&a.dstep[f], Mv[u] * a.cfgsign);
            }
        }
        pl[u] = 1.0;
        plm1[u] = 0.0;
    }
    double *gl = a.gleg + (long)f * a.nleg;
#pragma unroll 1
    for (int lb = 0; lb < a.nleg; lb += 16) {
        double v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            // order l = lb + j from pl, then the next: P_{l+1} = c1 x P_l - c2 P_{l-1}
            const int l = min(lb + j, a.nleg - 1);
            const double c1 = a.legc[2 * l], c2 = a.legc[2 * l + 1];
            double sum = 0.0;
#pragma unroll
            for (int u = 0; u < PPL; ++u) {
                sum = fma(Mv[u], pl[u], sum);
                const double nx = c1 * x[u] * pl[u] - c2 * plm1[u];
                plm1[u] = pl[u];
                pl[u] = nx;
            }
            v[j] = sum;
        }
        double r = row_reduce_scatter16(v);
        r += __shfl_xor(r, 16, WAVE);
        r += __shfl_xor(r, 32, WAVE);
        if (lane_id() < 16 && lb + lane_id() < a.nleg) global_add(gl + lb + lane_id(), r);
    }
}

__device__ __attribute__((noinline)) double2 meas_gtau(const GtauArgs a)
{
    double wflops = 0.0, wbytes = 0.0;
#pragma unroll 1
    for (int f = 0; f < a.nf; ++f) {
        const int k = uni(a.kf[f]), npair = k * k;
        wflops += (double)k * k * (5.0 * a.nleg + 4.0);
        wbytes += 8.0 * k * k;
        int p0 = 0;
#pragma unroll 1
        for (; npair - p0 > 2 * WAVE; p0 += 4 * WAVE) gtau_pairs<4>(a, f, k, p0);
        if (npair - p0 > WAVE) gtau_pairs<2>(a, f, k, p0);
        else if (npair - p0 > 0) gtau_pairs<1>(a, f, k, p0);
    }
    wsync();
    return make_double2(wflops, wbytes);
}

// gtau_accum%add() of the binning accumulator (AccumGtau = 2,
// autocorracc_add, Accumulators.F90:298-340): this measurement's G(tau) bins
// (gbuf, filled by atomics) go into the sum and into level 0 by the Welford
// update; when the low bits of the count n are ones the finished bin of each
// level (mean of its halves) rolls over to the next.  Lanes over components;
// the roll-over depth depends on n only, so it is uniform.  Bound by round trips
// to memory: eight components a lane go together, level by level, all their loads
// ahead of their arithmetic (4 flavours of 1000 bins: one by one 176 K cycles a
// measurement; one chain, 16 measurements 13.3 -> 12.5 ms).
DEV void autocorr_add(CModel &M, double *gbuf, double *gacc, double *gtau, long long n0)
{
    constexpr int U = 8;
    const long nc = (long)M.nf * M.ntau;
    double *spill = gacc, *mean = gacc + nc * M.nlev, *sq = gacc + 2 * nc * M.nlev;
    wsync();
    for (long i0 = lane_id(); i0 - lane_id() < nc; i0 += U * WAVE) {
        // v: this level's value; s, m, q: its half-filled bin, mean and squares
        double v[U], g[U], s[U], m[U], q[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long i = min(i0 + u * WAVE, nc - 1);
            // the bins were written by atomics at L2: read past the vector L1
            v[u] = __hip_atomic_load(gbuf + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            g[u] = gtau[i], s[u] = spill[i], m[u] = mean[i], q[u] = sq[i];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long i = i0 + u * WAVE;
            if (i < nc) gbuf[i] = 0.0, gtau[i] = g[u] + v[u];
        }
        long long n = n0;
        for (int lvl = 0;; ++lvl) {
            const bool roll = (n & 1) != 0 && lvl + 1 < M.nlev;
            const long at = (long)lvl * nc;
            const double cnt = (double)(n + 1);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const long i = i0 + u * WAVE;
                s[u] += v[u];
                const double d1 = v[u] - m[u];
                m[u] += d1 / cnt;
                q[u] += d1 * (v[u] - m[u]);
                if (i < nc) spill[at + i] = roll ? 0.0 : s[u], mean[at + i] = m[u], sq[at + i] = q[u];
                v[u] = s[u] / 2.0;
            }
            if (!roll) break;
            n >>= 1;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const long i = at + nc + min(i0 + u * WAVE, nc - 1);
                s[u] = spill[i], m[u] = mean[i], q[u] = sq[i];
            }
        }
    }
    wsync();
}

// MeasDensityMatrix_beta_half (CTQMC.F90:3088-3151) with update_b2_states_eb
// (Trace.F90:6213-6469): ket from 0 to beta/2, bra from beta to beta/2
template <int NM>
DEV void meas_dm(Ctx &c, double *dm)
{
    CModel &M = c.M;
    const int outer = c.h.outer, no = c.sz[outer];
    if (c.h.nop != 0) {
        const double bh = M.beta / 2.0;
        const int nk = upper_bound_tau(c.tau, c.h.nop, bh);   // ops with tau <= beta/2
        int s = outer, sb = outer;
        double kl = 0.0, bl = 0.0;
        double *Ks, *B;
        if constexpr (NM <= 16) {
            // both halves in registers, then to the work matrices
            Ks = c.K0;
            B = c.K1;
            State<NM> k;
            k.identity(no);
            walk_global<NM, false>(c, k, s, kl, no, 0.0, 0, nk, bh);
            k.store(Ks, c.sz[s], no);
            k.identity(no);
            walk_global<NM, true>(c, k, sb, bl, no, M.beta, nk, c.h.nop, bh);
            k.store(B, c.sz[sb], no);
            wsync();
        } else {
            double *K = c.K0, *Kw = c.K1;
            set_identity(K, no);
            walk_global_big<false>(c, K, Kw, s, kl, no, 0.0, 0, nk, bh);
            Ks = c.scratch;
            copy_mat(Ks, K, c.sz[s] * no);
            B = c.K0;
            double *Bw = c.K1;
            set_identity(B, no);
            walk_global_big<true>(c, B, Bw, sb, bl, no, M.beta, nk, c.h.nop, bh);
        }
        const int n = c.sz[s];
        double *blk = dm + M.dmoff[s];
        const double fac = c.h.trace_sign * (-c.h.cfgsign) * exp(kl + bl - c.h.trace_log);
        for (int idx = lane_id(); idx < n * n; idx += WAVE) {
            const int s1 = idx % n, s2 = idx / n;
            double acc = 0.0;
            for (int i = 0; i < no; ++i) acc = fma(B[s1 * no + i], Ks[s2 * no + i], acc);
            blk[s1 + (long)s2 * n] += fac * acc;
        }
        wsync();
    } else {
        double *blk = dm + M.dmoff[outer];
        for (int i = lane_id(); i < no; i += WAVE) {
            const double v = c.part[2 * i + 1] * c.h.trace_sign * exp(c.part[2 * i] - c.h.trace_log);
            blk[i + (long)i * no] -= c.h.cfgsign * v;
        }
        wsync();
    }
}

// ---------------------------------------------------------------------------
// parameter derivatives (no counterpart in the reference)
// ---------------------------------------------------------------------------
// d ln|w| / d theta of a configuration, w = det(Delta) Tr[...]:
//  * d ln|det Delta| = sum_f tr(Delta_f^{-1} dDelta_f): each (creator,
//    annihilator) pair of a flavour times dF/dtheta(tau_a - tau_c), looked up
//    like get_HybrF (Trace.F90:1014-1033) on the derivative table;
//  * d ln|Tr| by forward tangents: each state matrix K carries dK_t beside it.
//    Over dt in block s (levels E_k relative to the block's lowest)
//      K <- P K,   dK_t <- P dK_t - (D_t o Phi) K,
//    P = diag(exp(-dt E_k)), D_t = V^T (dH/dtheta_t) V in the eigenbasis and
//    Phi_kl = (exp(-dt E_k) - exp(-dt E_l)) / (E_l - E_k) (dt exp(-dt E_k) for
//    equal levels); an operator block maps K and every dK_t alike, and one
//    power of two rescales them together.  The ket from 0 and the bra from
//    beta meet at beta/2 (as the density-matrix measurement), where the trace,
//    its tangents, the density-matrix sample and that sample's explicit
//    derivative are contracted.
constexpr int MAXTHETA = 4;

struct TanEnv {
    CModel *M;
    const int *sz, *off;
    const int4 *tr;
    const double *ev, *ops, *tau;
    const int *code;
    double *w;            // derivative work area of the chain
    int nm, nth;
};

DEV TanEnv tan_env(const Ctx &c)
{
    TanEnv e;
    e.M = &c.M, e.sz = c.sz, e.off = c.off, e.tr = c.tr, e.ev = c.ev, e.ops = c.opsp, e.tau = c.tau;
    e.code = c.code, e.w = reinterpret_cast<double *>(c.base + c.L.dwork), e.nm = c.nm, e.nth = c.M.ntheta;
    return e;
}

// divided difference of exp(-dt E) at two levels relative to the block's lowest
DEV double phi_div(double ek, double el, double dt)
{
    const double a = fmin(ek, el), y = fabs(ek - el) * dt;
    const double g = y > 0.0 ? -expm1(-y) / y : 1.0;
    return dt * exp(-a * dt) * g;
}

DEV int4 tan_trans(const TanEnv &e, int s, int code, bool adjoint)
{
    int ca = op_ca(code);
    if (adjoint) ca = 3 - ca;
    return e.tr[((s * e.M->nb + op_orb(code)) * 2 + op_spin(code)) * 2 + (ca - 1)];
}

// segment of length dt in block s: dKw_t = P dK_t - (D_t o Phi) K, then K <- P K
DEV void tan_prop(const TanEnv &e, int s, double dt, double *K, const double *dK, double *dKw, int no)
{
    CModel &M = *e.M;
    const int ns = e.sz[s];
    const long nm2 = (long)e.nm * e.nm;
    const double *E = e.ev + e.off[s];
    double *Phi = e.w, *pv = e.w + (4L + 3L * e.nth) * nm2;
    for (int idx = lane_id(); idx < ns * ns; idx += WAVE)
        Phi[idx] = phi_div(E[idx % ns] - E[0], E[idx / ns] - E[0], dt);
    for (int k = lane_id(); k < ns; k += WAVE) pv[k] = exp(-(E[k] - E[0]) * dt);
    wsync();
    for (int t = 0; t < e.nth; ++t) {
        const double *D = M.dblk + (long)t * M.dmsize + M.dmoff[s];
        const double *dk = dK + t * nm2;
        double *dw = dKw + t * nm2;
        for (int idx = lane_id(); idx < ns * no; idx += WAVE) {
            const int k = idx / no, i = idx - k * no;
            double acc = pv[k] * dk[idx];
            for (int l = 0; l < ns; ++l) acc = fma(-D[k + l * ns] * Phi[k + l * ns], K[l * no + i], acc);
            dw[idx] = acc;
        }
    }
    wsync();
    for (int idx = lane_id(); idx < ns * no; idx += WAVE) K[idx] *= pv[idx / no];
    wsync();
}

// operator block P (nt x ns, column-major): Kw = P K, dKw_t = P dK_t
DEV void tan_apply(const TanEnv &e, const double *P, int nt, int ns, int no, const double *K, double *Kw,
                   const double *dK, double *dKw)
{
    const long nm2 = (long)e.nm * e.nm;
    for (int t = -1; t < e.nth; ++t) {
        const double *src = t < 0 ? K : dK + t * nm2;
        double *dst = t < 0 ? Kw : dKw + t * nm2;
        for (int idx = lane_id(); idx < nt * no; idx += WAVE) {
            const int r = idx / no, i = idx - r * no;
            double acc = 0.0;
            for (int c = 0; c < ns; ++c) acc = fma(P[r + c * nt], src[c * no + i], acc);
            dst[idx] = acc;
        }
    }
    wsync();
}

// one power of two for K and its tangents when their largest entry leaves [2^-64, 2^64]
DEV void tan_renorm(const TanEnv &e, double *K, double *dK, int n, double &lg)
{
    const long nm2 = (long)e.nm * e.nm;
    double m = 0.0;
    for (int idx = lane_id(); idx < n; idx += WAVE) {
        m = fmax(m, fabs(K[idx]));
        for (int t = 0; t < e.nth; ++t) m = fmax(m, fabs(dK[t * nm2 + idx]));
    }
    const double mm = wave_max(m);
    if (mm > 0.0 && (mm < STATE_TINY || mm > STATE_HUGE)) {
        const int ex = ilogb(mm);
        for (int idx = lane_id(); idx < n; idx += WAVE) {
            K[idx] = ldexp(K[idx], -ex);
            for (int t = 0; t < e.nth; ++t) dK[t * nm2 + idx] = ldexp(dK[t * nm2 + idx], -ex);
        }
        lg += (double)ex * 0.69314718055994530942;
    }
    wsync();
}

// Walk over operators [j0, j1) of the configuration (BRA: descending, adjoint
// blocks) from tstart to tend with tangents; false on a quantum-number violation
template <bool BRA>
DEV bool tan_walk(const TanEnv &e, double *&K, double *&Kw, double *&dK, double *&dKw, int &s, double &lg, int no,
                  double tstart, int j0, int j1, double tend)
{
    CModel &M = *e.M;
    double t = tstart;
    for (int jj = 0; jj < j1 - j0; ++jj) {
        const int j = BRA ? j1 - 1 - jj : j0 + jj;
        const double tj = e.tau[j];
        const int4 tr = tan_trans(e, s, e.code[j], BRA);
        if (tr.x < 0) return false;
        const double dt = BRA ? t - tj : tj - t;
        tan_prop(e, s, dt, K, dK, dKw, no);
        lg += -(e.ev[e.off[s]] - M.egs) * dt;
        tan_apply(e, e.ops + tr.z, tr.y, e.sz[s], no, K, Kw, dKw, dK);
        double *x = K;
        K = Kw, Kw = x;
        tan_renorm(e, K, dK, tr.y * no, lg);
        s = tr.x;
        t = tj;
    }
    const double dt = BRA ? t - tend : tend - t;
    tan_prop(e, s, dt, K, dK, dKw, no);
    lg += -(e.ev[e.off[s]] - M.egs) * dt;
    double *x = dK;
    dK = dKw, dKw = x;
    tan_renorm(e, K, dK, e.sz[s] * no, lg);
    return true;
}

struct HalfTangents {
    const double *K, *dK, *B, *dB;   // ket and bra at beta/2 (rows of block smid x outer states) and tangents
    double kl, bl;                    // their log scales
    int smid, no;
    bool ok;
};

// ket from 0 and bra from beta to beta/2 with tangents
DEV HalfTangents half_tangents(const TanEnv &e, int nop, int outer)
{
    CModel &M = *e.M;
    const long nm2 = (long)e.nm * e.nm;
    double *A0 = e.w + nm2, *A1 = A0 + nm2, *A2 = A1 + nm2;
    double *T0 = A2 + nm2, *T1 = T0 + e.nth * nm2, *T2 = T1 + e.nth * nm2;
    HalfTangents r;
    const int no = e.sz[outer];
    r.no = no;
    const double bh = M.beta / 2.0;
    const int nk = upper_bound_tau(e.tau, nop, bh);
    double *K = A0, *Kw = A1, *dK = T0, *dKw = T1;
    for (int idx = lane_id(); idx < no * no; idx += WAVE) {
        K[idx] = (idx / no == idx % no) ? 1.0 : 0.0;
        for (int t = 0; t < e.nth; ++t) dK[t * nm2 + idx] = 0.0;
    }
    wsync();
    int s = outer;
    r.kl = 0.0;
    r.ok = tan_walk<false>(e, K, Kw, dK, dKw, s, r.kl, no, 0.0, 0, nk, bh);
    r.smid = s;
    const int nmid = e.sz[s];
    for (int idx = lane_id(); idx < nmid * no; idx += WAVE) {
        A2[idx] = K[idx];
        for (int t = 0; t < e.nth; ++t) T2[t * nm2 + idx] = dK[t * nm2 + idx];
    }
    wsync();
    double *B = A0, *Bw = A1, *dB = T0, *dBw = T1;
    for (int idx = lane_id(); idx < no * no; idx += WAVE) {
        B[idx] = (idx / no == idx % no) ? 1.0 : 0.0;
        for (int t = 0; t < e.nth; ++t) dB[t * nm2 + idx] = 0.0;
    }
    wsync();
    int sb = outer;
    r.bl = 0.0;
    r.ok = r.ok && tan_walk<true>(e, B, Bw, dB, dBw, sb, r.bl, no, M.beta, nk, nop, bh) && sb == s;
    r.K = A2, r.dK = T2, r.B = B, r.dB = dB;
    return r;
}

// d ln|Tr| / d theta from the beta/2 contraction
DEV void trace_tangent(const TanEnv &e, const HalfTangents &h, double *dlt)
{
    const long nm2 = (long)e.nm * e.nm;
    const int n = e.sz[h.smid] * h.no;
    double tr = 0.0;
    for (int idx = lane_id(); idx < n; idx += WAVE) tr += h.B[idx] * h.K[idx];
    tr = wave_sum(tr);
    for (int t = 0; t < e.nth; ++t) {
        double d = 0.0;
        for (int idx = lane_id(); idx < n; idx += WAVE)
            d += h.dB[t * nm2 + idx] * h.K[idx] + h.B[idx] * h.dK[t * nm2 + idx];
        dlt[t] = wave_sum(d) / tr;
    }
}

// What a derivative pass needs, by value (the pass is out of line so that it
// does not add to the sweep's registers; a reference to the chain context
// would live in scratch).
struct ScoreArgs {
    TanEnv e;
    const double *fc, *fa, *minv;
    const int *fcs, *fas;
    int kf[MAXF];
    int kcap, nop, outer;
    double cfgsign, trace_sign, trace_log;
    double *scsum, *scg, *scdm, *scdmx;   // score sums of the chain
    double *gbuf, *gtau;                  // this measurement's G(tau) bins, the G(tau) sums
};

DEV ScoreArgs score_args(const Ctx &c, double *gbuf, double *gtau)
{
    ScoreArgs a;
    a.e = tan_env(c);
    a.fc = c.fc, a.fa = c.fa, a.minv = c.minv, a.fcs = c.fcs, a.fas = c.fas;
    for (int f = 0; f < MAXF; ++f) a.kf[f] = c.h.kf[f];
    a.kcap = c.L.kcap, a.nop = c.h.nop, a.outer = c.h.outer;
    a.cfgsign = c.h.cfgsign, a.trace_sign = c.h.trace_sign, a.trace_log = c.h.trace_log;
    a.scsum = reinterpret_cast<double *>(c.base + c.L.scsum);
    a.scg = reinterpret_cast<double *>(c.base + c.L.scg);
    a.scdm = reinterpret_cast<double *>(c.base + c.L.scdm);
    a.scdmx = reinterpret_cast<double *>(c.base + c.L.scdmx);
    a.gbuf = gbuf, a.gtau = gtau;
    return a;
}

// d ln|det| / d theta = sum_f tr(Delta_f^{-1} dDelta_f)
DEV void det_tangent(const ScoreArgs &a, double *dld)
{
    CModel &M = *a.e.M;
    const int ld = a.kcap;
    double acc[MAXTHETA] = {0.0, 0.0, 0.0, 0.0};
    for (int f = 0; f < M.nf; ++f) {
        const int k = a.kf[f];
        const double *ctl = a.fc + (long)f * ld, *atl = a.fa + (long)f * ld;
        const int *csl = a.fcs + (long)f * ld, *asl = a.fas + (long)f * ld;
        const double *Mf = a.minv + (long)f * ld * ld;
        for (int p = lane_id(); p < k * k; p += WAVE) {
            const int ai = p / k, ci = p - ai * k;
            const double m = Mf[csl[ci] + (long)asl[ai] * ld];
            double tau = atl[ai] - ctl[ci], sig = 1.0;
            if (tau < 0.0) {
                tau += M.beta;
                sig = -1.0;
            }
            const double x = tau / M.beta * (double)(M.nftau - 1);
            const int i = (int)x;
            for (int t = 0; t < M.ntheta; ++t) {
                const double *F = M.dftau + ((long)t * M.nf + f) * M.nftau;
                acc[t] += m * sig * (F[i] + (x - (double)i) * (F[i + 1] - F[i]));
            }
        }
    }
    for (int t = 0; t < M.ntheta; ++t) dld[t] = wave_sum(acc[t]);
}

// One derivative pass over the configuration.  out != null: d ln|det| /
// d theta_t -> out[2 t], d ln|Tr| / d theta_t -> out[2 t + 1].  accumulate:
// the score-function sums of a measurement (s_t = d ln|w| / d theta_t):
// Sum sign s_t, Sum s_t x this measurement's G(tau) bins (gbuf, which is then
// added to the G(tau) sums unless the binning accumulator does that), Sum
// s_t x density-matrix sample and Sum d(sample)/dtheta_t at fixed
// configuration (the beta/2 sample depends on H explicitly).
__device__ __attribute__((noinline)) void score_pass(const ScoreArgs a, double *out, bool accumulate)
{
    CModel &M = *a.e.M;
    const TanEnv &e = a.e;
    const long nm2 = (long)e.nm * e.nm;
    double dld[MAXTHETA], dlt[MAXTHETA], sc[MAXTHETA];
    det_tangent(a, dld);
    const HalfTangents h = half_tangents(e, a.nop, a.outer);
    trace_tangent(e, h, dlt);
    if (out && lane_id() == 0)
        for (int t = 0; t < M.ntheta; ++t) {
            out[2 * t] = dld[t];
            out[2 * t + 1] = h.ok ? dlt[t] : __builtin_nan("");
        }
    if (!accumulate) return;
    for (int t = 0; t < M.ntheta; ++t) sc[t] = dld[t] + dlt[t];
    if (lane_id() == 0)
        for (int t = 0; t < M.ntheta; ++t) a.scsum[t] += a.cfgsign * sc[t];
    if (M.meas_dm) {
        const int n = e.sz[h.smid], no = h.no;
        const long off = M.dmoff[h.smid];
        const double fac = a.trace_sign * (-a.cfgsign) * exp(h.kl + h.bl - a.trace_log);
        for (int idx = lane_id(); idx < n * n; idx += WAVE) {
            const int s1 = idx % n, s2 = idx / n;
            double smp = 0.0;
            for (int i = 0; i < no; ++i) smp = fma(h.B[s1 * no + i], h.K[s2 * no + i], smp);
            smp *= fac;
            for (int t = 0; t < M.ntheta; ++t) {
                double x = 0.0;
                for (int i = 0; i < no; ++i)
                    x += h.dB[t * nm2 + s1 * no + i] * h.K[s2 * no + i] + h.B[s1 * no + i] * h.dK[t * nm2 + s2 * no + i];
                a.scdm[t * M.dmsize + off + idx] += sc[t] * smp;
                a.scdmx[t * M.dmsize + off + idx] += fac * x - smp * dlt[t];
            }
        }
    }
    // this measurement's G(tau) bins: written by atomics at L2, read past the vector L1
    wsync();
    const long nc = (long)M.nf * M.ntau;
    for (long i = lane_id(); i < nc; i += WAVE) {
        const double v = __hip_atomic_load(a.gbuf + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int t = 0; t < M.ntheta; ++t) a.scg[t * nc + i] += sc[t] * v;
        if (M.accum != 2) {
            a.gtau[i] += v;
            a.gbuf[i] = 0.0;
        }
    }
    wsync();
}

// MeasSign, MeasOuterHistograms, MeasExpOrder (CTQMC.F90:3264-3350): visits
// of the outer superstate and of each of its states, superstate sign, state
// signs (trace sign x part-trace sign x configuration sign), trace
// contributions exp(log part trace) per state and summed per superstate, and
// the order histogram
DEV void meas_misc(Ctx &c, double *histo, double *outer_hist)
{
    CModel &M = c.M;
    const int outer = c.h.outer, no = c.sz[outer], off = c.off[outer];
    double *ohst = reinterpret_cast<double *>(c.base + c.L.ohst);
    double *shss = reinterpret_cast<double *>(c.base + c.L.shss);
    double *shst = reinterpret_cast<double *>(c.base + c.L.shst);
    double *tcss = reinterpret_cast<double *>(c.base + c.L.tcss);
    double *tcst = reinterpret_cast<double *>(c.base + c.L.tcst);
    c.h.meas_sign += c.h.cfgsign;
    double tc = 0.0;
    for (int i = lane_id(); i < no; i += WAVE) {
        const double e = exp(c.part[2 * i]);
        ohst[off + i] += 1.0;
        shst[off + i] += c.h.trace_sign * c.part[2 * i + 1] * c.h.cfgsign;
        tcst[off + i] += e;
        tc += e;
    }
    tc = wave_sum(tc);
    if (lane_id() == 0) {
        outer_hist[outer] += 1.0;
        shss[outer] += c.h.cfgsign;
        tcss[outer] += tc;
        for (int f = 0; f < M.nf; ++f) {
            int k = c.h.kf[f];
            if (k > M.maxhisto) k = M.maxhisto;
            histo[(long)f * (M.maxhisto + 1) + k] += 1.0;
        }
    }
    wsync();
}


// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// the chain a header pointer belongs to, in the header array behind the blocks
DEV ChainHdr *global_hdr(CLayout &L, char *base, int chain)
{
    return reinterpret_cast<ChainHdr *>(base - (long)chain * L.stride + L.hdrs) + chain;
}

// Start of a kernel: header, RNG state and model tables into LDS.
template <int NM>
DEV Ctx make_ctx(char *chains, int chain, CArgs args, char *lds)
{
    CModel &M = *(CModel *)args;
    CLayout &L = *(CLayout *)(args + (sizeof(DevModel) + 7) / 8 * 8);
    {
        WalkEnv &e = s_wenv;
        const unsigned d = (unsigned)(size_t)(lds_c *)lds;
        e.wtau = d + (unsigned)L.l_wtau, e.wcode = d + (unsigned)L.l_wcode;
        e.ttau = d + (unsigned)L.l_ttau, e.tcode = d + (unsigned)L.l_tcode;
        e.pc = d + (unsigned)L.l_pc, e.dvec = d + (unsigned)L.l_dvec, e.pl = d + (unsigned)L.l_pl;
        e.q = d + (unsigned)L.l_q, e.r = d + (unsigned)L.l_r;
        e.col = d + (unsigned)L.l_col, e.row = d + (unsigned)L.l_row;
        e.rk = d + (unsigned)L.l_rk, e.lb = d + (unsigned)L.l_lb;
        e.rkx = d + (unsigned)L.l_rkx, e.lbx = d + (unsigned)L.l_lbx;
        e.rks = d + (unsigned)L.l_rks, e.lbs = d + (unsigned)L.l_lbs;
        e.legc = d + (unsigned)L.l_legc, e.k = d + (unsigned)L.l_k, e.strip = d + (unsigned)L.l_strip;
        e.sz = d + (unsigned)L.l_sz, e.off = d + (unsigned)L.l_off;
        e.trt = d + (unsigned)L.l_tr, e.evt = d + (unsigned)L.l_ev, e.opst = d + (unsigned)L.l_ops;
        e.mt = d + (unsigned)L.l_mt;
        e.ready = 0;
    }
    wsync();
    char *base = chains + (long)chain * L.stride;
    Ctx c = attach<NM>(ChainRef{&M, &L, base});
    const int *gh = reinterpret_cast<const int *>(global_hdr(L, base, chain));
    int *lh = reinterpret_cast<int *>(&s_wenv.hdr);
    for (int i = lane_id(); i < (int)(sizeof(ChainHdr) / 4); i += WAVE) lh[i] = gh[i];
    const uint32_t *gmt = reinterpret_cast<const uint32_t *>(base + L.mt);
    for (int i = lane_id(); i < 624; i += WAVE) c.rng.mt[i] = gmt[i];
    for (int i = lane_id(); i < M.nsst; i += WAVE) {
        const_cast<int *>(c.sz)[i] = M.sizes[i];
        const_cast<int *>(c.off)[i] = M.offsets[i];
    }
    for (int i = lane_id(); i < 2 * M.nleg; i += WAVE) const_cast<double *>(c.legc)[i] = M.legc[i];
    const int ncn = M.nsst * M.nb * 4;
    if constexpr (NM <= 16) {
        for (int i = lane_id(); i < M.nstates; i += WAVE) const_cast<double *>(c.ev)[i] = M.evals[i];
        for (int i = lane_id(); i < ncn; i += WAVE) const_cast<int4 *>(c.tr)[i] = M.trans[i];
        // what the walks read
        int *si = (int *)(lds_i *)(lds_c *)(lds + L.l_sinfo);
        for (int q = lane_id(); q < M.nsst; q += WAVE) {
            const int n = M.sizes[q], o = M.offsets[q];
            const double e0 = M.evals[o];
            si[4 * q] = __double2loint(e0);
            si[4 * q + 1] = __double2hiint(e0);
            si[4 * q + 2] = n | (o << 8);
            si[4 * q + 3] = __float_as_int((float)(M.evals[o + n - 1] - e0));
        }
        unsigned char *kb = (unsigned char *)(lds_b *)(lds_c *)(lds + L.l_keys);
        for (int q = lane_id(); q < 512; q += WAVE) kb[q] = M.dkey ? M.keys[q] : 255;
        WalkEnv &e = s_wenv;
        e.opsx = M.opsx;
        e.tr = (const lds_i4 *)c.tr;
        e.ev = (const lds_d *)c.ev;
        e.keys = (const lds_b *)kb;
        e.sinfo = (const lds_i4 *)(const void *)si;
        e.qa = NM > 4 ? (lds_d *)(lds_c *)(lds + L.l_qa) : nullptr;
        e.lops = (const lds_d *)c.ev;
        if constexpr (NM <= 4) {
            for (long i = lane_id(); i < M.nops; i += WAVE) const_cast<double *>(c.opsp)[i] = M.ops[i];
            e.lops = (const lds_d *)c.opsp;
        }
        e.ncol = 4 * M.nb;
        e.dkey = M.dkey;
        e.nkmax = (M.nmax + 3) / 4;
    }
    s_wenv.egs = M.egs;
    s_wenv.flops = s_wenv.bytes = 0.0;
    wsync();
    s_wenv.hdr.wvalid = 0;   // the LDS window list does not survive a launch
    wsync();
    return c;
}

DEV void save_ctx(Ctx &c, int chain)
{
    c.h.alg_flops += s_wenv.flops;
    c.h.alg_bytes += s_wenv.bytes;
    uint32_t *gmt = reinterpret_cast<uint32_t *>(c.base + c.L.mt);
    for (int i = lane_id(); i < 624; i += WAVE) gmt[i] = c.rng.mt[i];
    int *gh = reinterpret_cast<int *>(global_hdr(c.L, c.base, chain));
    const int *lh = reinterpret_cast<const int *>(&c.h);
    wsync();
    for (int i = lane_id(); i < (int)(sizeof(ChainHdr) / 4); i += WAVE) gh[i] = lh[i];
    wsync();
}

// Calibration: phase 1 ends once the distance list is full, phase 2 once every
// flavour has calib.z accepted pairs (CTQMC.F90:8128-8175)
template <int NM>
__device__ __attribute__((noinline)) bool calib_done(ChainRef r, int3 calib)
{
    Ctx c = attach<NM>(r);
    if (calib.x == 1) return c.h.apt_index > c.h.apt_n;
    const double *ap = reinterpret_cast<const double *>(c.base + c.L.accpair);
    int short_f = 0;
    for (int f = 0; f < c.M.nf; ++f) {
        double n = 0.0;
        // the counts are written by atomics at L2: read past the vector L1
        for (int b = lane_id(); b < c.h.naccpair; b += WAVE)
            n += __hip_atomic_load(ap + (long)f * c.L.naccpair_cap + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        short_f += wave_sum(n) < (double)calib.z;
    }
    return short_f == 0;
}

// all measurements of the current configuration
template <int NM, bool SCORE>
__device__ __attribute__((noinline)) void measure(ChainRef r)
{
    Ctx c = attach<NM>(r);
    CModel &M = c.M;
    CLayout &L = c.L;
    char *base = c.base;
    double *gtau = reinterpret_cast<double *>(base + L.gtau);
    double *gleg = reinterpret_cast<double *>(base + L.gleg);
    double *gbuf = reinterpret_cast<double *>(base + L.gbuf);
    c.h.cnt_meas++;
    meas_misc(c, reinterpret_cast<double *>(base + L.histo), reinterpret_cast<double *>(base + L.outer));
    if (M.meas_dm) meas_dm<NM>(c, reinterpret_cast<double *>(base + L.dm));
    GtauArgs ga;
    ga.nf = M.nf, ga.ntau = M.ntau, ga.nleg = M.nleg, ga.kcap = L.kcap;
    ga.beta = M.beta, ga.rbeta = M.rbeta, ga.cfgsign = c.h.cfgsign, ga.legc = c.legc;
    ga.kf = c.h.kf, ga.fc = c.fc, ga.fa = c.fa, ga.minv = c.minv, ga.fcs = c.fcs, ga.fas = c.fas;
    ga.gtau = (M.accum == 2 || SCORE) ? gbuf : gtau, ga.gleg = gleg;
    const long long mi = c.h.cnt_meas - 1;   // g_inmeas - 1
    const bool st = mi < M.nmstep;
    ga.mstep = (st && M.step_mean) ? reinterpret_cast<double *>(base + L.gmstep) + mi * M.nf : nullptr;
    ga.dstep = (st && M.step_mid) ? reinterpret_cast<double *>(base + L.gdstep) + mi * M.nf : nullptr;
    // sign_step is set when the configuration has a pair (CTQMC.F90:2402)
    if (st && M.step_sign && c.h.nop > 0 && lane_id() == 0)
        reinterpret_cast<double *>(base + L.sstep)[mi] = c.h.cfgsign;
    const double2 wk = meas_gtau(ga);
    c.work(wk.x, wk.y);
    if constexpr (SCORE) score_pass(score_args(c, gbuf, gtau), nullptr, true);
    if (M.accum == 2)
        autocorr_add(M, gbuf, reinterpret_cast<double *>(base + L.gacc), gtau, c.h.cnt_meas - 1);
}

// Sweep kernel: each block advances chain blockIdx.x until it has done
// `target` moves in the current warmup / measure call (header field pos); if
// ncorr > 0 it measures after every ncorr-th move of the call.  A chain stops
// early, state intact, when the next move might not fit its memory
// (HALT_CAP) or when the host has raised the abort word (HALT_ABORT, polled
// at measurement boundaries and every 128 warm-up moves; the reference checks
// its signal flag before every move, CTQMC.F90:8212, 8436).  rec != nullptr
// records every step of chain `only` at rec[pos - rec_base] (parity mode;
// other chains return at once).
// SCORE: the measurements add the score-function sums (a separate
// instantiation, so that the derivative pass costs the plain sweep nothing)
template <int NM, bool SCORE>
__global__ void __launch_bounds__(WAVE) sweep_kernel(DevModel M, ChainLayout L, char *chains, long long target,
                                                     long long ncorr, int only, w2d_move_record *rec,
                                                     long long rec_base, const int *abort_word, int3 calib,
                                                     const int *order)
{
    // order: the chain each workgroup runs (longest first, so that the
    // launch's tail is short), or null for workgroup = chain.  The order is
    // rewritten by order_kernel before every launch: it is read with a
    // device-coherent vector load, never through the scalar cache (which is
    // not coherent with the vector stores of an earlier kernel)
    const int chain = order ? __builtin_amdgcn_readfirstlane(__hip_atomic_load(
                                  order + blockIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                            : (int)blockIdx.x;
    if (only >= 0 && chain != only) return;
    extern __shared__ __align__(16) char lds[];
    Ctx c = make_ctx<NM>(chains, chain, (CArgs)__builtin_amdgcn_kernarg_segment_ptr(), lds);
    rng_open(c.rng);
    wsync();
    const long long pos0 = c.h.pos;
    const int todo = near(target - pos0);   // moves of this launch
    // moves until the next measurement, check of the calibration, look at the
    // abort word (warm-up); counted down instead of divided
    const long long step = ncorr > 0 ? ncorr : 128;
    const int every = near(step);
    int until = near(step - pos0 % step), ucal = calib.x ? calib.y - (int)(pos0 % calib.y) : 0;
    const long long past = (c.h.try_add + c.h.try_rem) % c.M.nslide;
    Tally ty{0, 0, 0, past == 0 ? 0 : max(near(c.M.nslide) - near(c.M.nslide - past), 1)};
    int done = 0;
    while (done < todo) {
        if (!s_wenv.ready && !make_ready<NM>(c.ref())) break;
        int kind, out;
        one_move<NM>(c, ty, kind, out);
        // ctqmc_calibrate (CTQMC.F90:8128-8175): every calib.y moves, phase 1
        // (calib.x = 1) ends once the distance list is full, phase 2
        // (calib.x = 2) once every flavour has calib.z accepted pairs
        if (calib.x && --ucal == 0) {
            ucal = calib.y;
            if (calib_done<NM>(c.ref(), calib)) c.h.halt = HALT_DONE, s_wenv.ready = 0;
        }
        if (rec && lane_id() == 0) {
            w2d_move_record &r = rec[pos0 + done - rec_base];
            r.kind = kind;
            r.outcome = out;
            r.noper = c.h.nop;
            r.outer_sst = c.h.outer;
            r.window = c.h.wpos;
            r.trace_log = c.h.trace_log;
            r.trace_sign = c.h.trace_sign;
            r.det_log = c.h.det_log;
            r.det_sign = c.h.det_sign;
            r.cfgsign = c.h.cfgsign;
        }
        ++done;
        if (--until == 0) {
            until = every;
            if (ncorr > 0) measure<NM, SCORE>(c.ref());
            if (__hip_atomic_load(abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM))
                c.h.halt = HALT_ABORT, s_wenv.ready = 0;
        }
    }
    rng_close(c.rng);
    c.h.pos += done;
    c.h.moves += done;
    c.h.try_add += ty.add;
    c.h.try_rem += ty.rem;
    c.h.qn_rej += ty.qn;
    wsync();
    save_ctx(c, chain);
}

// d ln|det| / d theta and d ln|Tr| / d theta of one chain's configuration:
// out[2 t], out[2 t + 1]
template <int NM>
__global__ void __launch_bounds__(WAVE) dlogw_kernel(DevModel M, ChainLayout L, char *chains, int chain,
                                                       double *out)
{
    extern __shared__ __align__(16) char lds[];
    Ctx c = make_ctx<NM>(chains, chain, (CArgs)__builtin_amdgcn_kernarg_segment_ptr(), lds);
    score_pass(score_args(c, nullptr, nullptr), out, false);
}

// Copy every chain from layout A to layout B (larger capacity): header, random
// state, configuration, flavour lists, inverse blocks re-strided to B's
// leading dimension, trace caches and accumulators.  Work buffers are not
// copied (they hold nothing between moves).  Physical row / column slots stay
// valid since they are below A's capacity.
DEV void copy_words(char *dst, const char *src, long bytes)
{
    int *d = reinterpret_cast<int *>(dst);
    const int *s = reinterpret_cast<const int *>(src);
    for (long i = lane_id(); i < bytes / 4; i += WAVE) d[i] = s[i];
}

__global__ void __launch_bounds__(WAVE) migrate_kernel(ChainLayout A, ChainLayout B, const char *src, char *dst,
                                                       int nf, int nm, long accbytes)
{
    const int chain = blockIdx.x;
    const char *s = src + (long)chain * A.stride;
    char *d = dst + (long)chain * B.stride;
    copy_words(dst + B.hdrs + (long)chain * sizeof(ChainHdr), src + A.hdrs + (long)chain * sizeof(ChainHdr),
               sizeof(ChainHdr));
    copy_words(d + B.mt, s + A.mt, 624 * 4);
    copy_words(d + B.tau, s + A.tau, (long)A.cap * 8);
    copy_words(d + B.code, s + A.code, (long)A.cap * 4);
    for (int f = 0; f < nf; ++f) {
        copy_words(d + B.fc + (long)f * B.kcap * 8, s + A.fc + (long)f * A.kcap * 8, (long)A.kcap * 8);
        copy_words(d + B.fa + (long)f * B.kcap * 8, s + A.fa + (long)f * A.kcap * 8, (long)A.kcap * 8);
        copy_words(d + B.fcs + (long)f * B.kcap * 4, s + A.fcs + (long)f * A.kcap * 4, (long)A.kcap * 4);
        copy_words(d + B.fas + (long)f * B.kcap * 4, s + A.fas + (long)f * A.kcap * 4, (long)A.kcap * 4);
        const double *ms = reinterpret_cast<const double *>(s + A.minv) + (long)f * A.kcap * A.kcap;
        double *md = reinterpret_cast<double *>(d + B.minv) + (long)f * B.kcap * B.kcap;
        for (long e = lane_id(); e < (long)A.kcap * A.kcap; e += WAVE) {
            const long i = e % A.kcap, j = e / A.kcap;
            md[i + j * B.kcap] = ms[e];
        }
    }
    // boundary caches: as many as both layouts hold (a new window count
    // invalidates them anyway: the host sets cache_pos = -1)
    const long nbd = min(A.nbound, B.nbound);
    copy_words(d + B.kst, s + A.kst, (long)nm * nm * 8);
    copy_words(d + B.bnd, s + A.bnd, nbd * nm * nm * 8);
    copy_words(d + B.bndlog, s + A.bndlog, nbd * 8);
    copy_words(d + B.bndsst, s + A.bndsst, nbd * 4);
    copy_words(d + B.part, s + A.part, 2L * nm * 8 + 16);
    copy_words(d + B.gtau, s + A.gtau, accbytes);
}

// Launch order of the chains by expected cost: a counting sort of the chains
// by expansion order (nop >> shift, clamped to 1023), largest first, in one
// workgroup (LDS counters; order within a bucket is arbitrary: chains are
// independent, so their results do not depend on it).  A kernel rather than a
// host sort, so that it can sit in a captured graph between sweep launches.
constexpr int ORDER_BUCKETS = 1024;
__global__ void __launch_bounds__(1024) order_kernel(const ChainHdr *hdrs, int nc, int shift, int *order)
{
    __shared__ int cnt[ORDER_BUCKETS];
    const int t = threadIdx.x;
    cnt[t] = 0;
    __syncthreads();
    auto key = [&](int c) { return ORDER_BUCKETS - 1 - min(hdrs[c].nop >> shift, ORDER_BUCKETS - 1); };
    for (int c = t; c < nc; c += 1024) atomicAdd(&cnt[key(c)], 1);
    __syncthreads();
    if (t == 0) {   // exclusive scan (1024 entries)
        int run = 0;
        for (int b = 0; b < ORDER_BUCKETS; ++b) {
            const int x = cnt[b];
            cnt[b] = run;
            run += x;
        }
    }
    __syncthreads();
    for (int c = t; c < nc; c += 1024) order[atomicAdd(&cnt[key(c)], 1)] = c;
}

// MeasGiw (measure_giw_nfft, CTQMC.F90:1015-1059; the sum is the direct one of
// the NFFT fallback, Nfft_z.F90:64-90).  After a measurement, for every
// flavour f and n = 0..niw-1:
//   giw[chain][f][n] += cfgsign * sum_{a,c} M[c,a] exp(i w_n (tau_a - tau_c)),
// w_n = (2n+1) pi / beta, M the inverse hybridisation block (rows creators,
// columns annihilators, by physical slot), with the sign convention of the
// lookup path (CTQMC.F90:2403-2417 and :8816); negative frequencies are the
// complex conjugates.  The kernel follows every sweep launch of whole
// measurement intervals (the chain's state at the end of such a launch is the
// state it measured) and acts on the chains whose measurement count moved
// since its last visit: seen[chain][f] = {count at the last visit, G(i w)
// measurements made}; the host checks that the second equals the count.
// One workgroup per (chain, flavour).  A thread takes GIW_R consecutive
// frequencies; creators go in tiles of GIW_TC whose phases stay in registers,
// annihilators in tiles of GIW_TA with the M tile in LDS; the phase of the
// next frequency is one complex product with exp(2 pi i tau / beta).
constexpr int GIW_THREADS = 256, GIW_R = 4, GIW_TC = 8, GIW_TA = 64;

__global__ void __launch_bounds__(GIW_THREADS) giw_kernel(ChainLayout L, const char *chains, int nf, int niw,
                                                         double beta, double *giw, long long *seen)
{
    __shared__ double s_m[GIW_TA][GIW_TC];
    __shared__ double s_ct[GIW_TC], s_at[GIW_TA];
    __shared__ double2 s_cs[GIW_TC], s_as[GIW_TA];
    __shared__ int s_bad;
    const int chain = blockIdx.x, f = blockIdx.y, tid = threadIdx.x, nt = blockDim.x;
    // header fields written by the sweep kernels: device-coherent loads
    const ChainHdr *hp = reinterpret_cast<const ChainHdr *>(chains + L.hdrs) + chain;
    const long long cnt = __hip_atomic_load(&hp->cnt_meas, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int err = __hip_atomic_load(&hp->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    long long *sv = seen + 2 * ((long)chain * nf + f);
    const long long last = sv[0];
    if (err != 0 || cnt == last) return;   // uniform over the workgroup
    const int k = __hip_atomic_load(&hp->kf[f], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const double sg = __longlong_as_double(__hip_atomic_load(reinterpret_cast<const long long *>(&hp->cfgsign),
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (tid == 0) s_bad = (k < 0 || k > L.kcap) ? 1 : 0;
    __syncthreads();
    const int kk = s_bad ? 0 : k;
    const char *base = chains + (long)chain * L.stride;
    const double *tcl = reinterpret_cast<const double *>(base + L.fc) + (long)f * L.kcap;
    const double *tal = reinterpret_cast<const double *>(base + L.fa) + (long)f * L.kcap;
    const int *csl = reinterpret_cast<const int *>(base + L.fcs) + (long)f * L.kcap;
    const int *asl = reinterpret_cast<const int *>(base + L.fas) + (long)f * L.kcap;
    const double *Mf = reinterpret_cast<const double *>(base + L.minv) + (long)f * L.kcap * L.kcap;
    double *out = giw + ((long)chain * nf + f) * (long)niw * 2;
    const double ib = 1.0 / beta;
    for (int n0 = 0; n0 < niw; n0 += nt * GIW_R) {
        const int nb = n0 + tid * GIW_R;            // first frequency of this thread
        const double xb = 2.0 * nb + 1.0;           // w_nb tau / pi = xb * tau / beta
        double gr[GIW_R], gi[GIW_R];
#pragma unroll
        for (int r = 0; r < GIW_R; ++r) gr[r] = gi[r] = 0.0;
        for (int c0 = 0; c0 < kk; c0 += GIW_TC) {
            const int nc = min(GIW_TC, kk - c0);
            __syncthreads();
            if (tid < GIW_TC) {
                const double t = tid < nc ? tcl[c0 + tid] * ib : 0.0;
                double s, c;
                sincospi(2.0 * t, &s, &c);
                s_ct[tid] = t;
                s_cs[tid] = make_double2(c, s);
            }
            __syncthreads();
            // exp(-i w_n tau_c) for the thread's frequencies; zero past the tile
            double cr[GIW_R][GIW_TC], ci[GIW_R][GIW_TC];
#pragma unroll
            for (int j = 0; j < GIW_TC; ++j) {
                double s, c;
                sincospi(xb * s_ct[j], &s, &c);
                const double2 st = s_cs[j];
                const double on = j < nc ? 1.0 : 0.0;
                double pr = c * on, pi = -s * on;
#pragma unroll
                for (int r = 0; r < GIW_R; ++r) {
                    cr[r][j] = pr;
                    ci[r][j] = pi;
                    const double t = pr * st.x + pi * st.y;
                    pi = pi * st.x - pr * st.y;
                    pr = t;
                }
            }
            for (int a0 = 0; a0 < kk; a0 += GIW_TA) {
                const int na = min(GIW_TA, kk - a0);
                __syncthreads();
                for (int e = tid; e < GIW_TA * GIW_TC; e += nt) {
                    const int ai = e / GIW_TC, cj = e - ai * GIW_TC;
                    double v = 0.0;
                    if (ai < na && cj < nc) {
                        const int rs = csl[c0 + cj], cs = asl[a0 + ai];
                        if (rs >= 0 && rs < L.kcap && cs >= 0 && cs < L.kcap) v = Mf[rs + (long)cs * L.kcap];
                        else s_bad = 1;
                    }
                    s_m[ai][cj] = v;
                }
                for (int ai = tid; ai < GIW_TA; ai += nt) {
                    const double t = ai < na ? tal[a0 + ai] * ib : 0.0;
                    double s, c;
                    sincospi(2.0 * t, &s, &c);
                    s_at[ai] = t;
                    s_as[ai] = make_double2(c, s);
                }
                __syncthreads();
                for (int ai = 0; ai < na; ++ai) {
                    double ur[GIW_R], ui[GIW_R];
#pragma unroll
                    for (int r = 0; r < GIW_R; ++r) ur[r] = ui[r] = 0.0;
#pragma unroll
                    for (int j = 0; j < GIW_TC; ++j) {
                        const double m = s_m[ai][j];
#pragma unroll
                        for (int r = 0; r < GIW_R; ++r) {
                            ur[r] = fma(m, cr[r][j], ur[r]);
                            ui[r] = fma(m, ci[r][j], ui[r]);
                        }
                    }
                    double s, c;
                    sincospi(xb * s_at[ai], &s, &c);
                    const double2 st = s_as[ai];
#pragma unroll
                    for (int r = 0; r < GIW_R; ++r) {
                        gr[r] += c * ur[r] - s * ui[r];
                        gi[r] += c * ui[r] + s * ur[r];
                        const double t = c * st.x - s * st.y;
                        s = c * st.y + s * st.x;
                        c = t;
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < GIW_R; ++r) {
            const int n = nb + r;
            if (n < niw) {
                out[2 * n] += sg * gr[r];
                out[2 * n + 1] += sg * gi[r];
            }
        }
    }
    __syncthreads();
    if (tid == 0) {
        sv[0] = cnt;
        if (!s_bad && cnt == last + 1) sv[1] += 1;
    }
}

// Sum of the chains' arrays, element e of group g: group g holds chains
// [g nc / ng, (g+1) nc / ng) that have not stopped on an error (header err ==
// 0), chain c's array starts at `first` + c `stride` (bytes).  Grid: x over
// elements, y over groups; consecutive threads read consecutive doubles of one
// chain.  Bound by memory latency where groups are large: eight chains are in
// flight per thread, added in order (so the sum is the plain one over chains).
__global__ void __launch_bounds__(256) group_sum_kernel(const char *first, long stride, long nel, int nc, int ng,
                                                        const ChainHdr *hdrs, double *out)
{
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    const int g = blockIdx.y;
    if (e >= nel) return;
    const int c0 = (int)((long)g * nc / ng), c1 = (int)((long)(g + 1) * nc / ng);
    double acc = 0.0;
    for (int c = c0; c < c1; c += 8) {
        double v[8];
        int err[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int cc = min(c + u, c1 - 1);
            // the error flag is written by the sweep kernels: a device-coherent
            // load (a uniform address would otherwise go through the scalar cache)
            err[u] = __hip_atomic_load(&hdrs[cc].err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            v[u] = reinterpret_cast<const double *>(first + (long)cc * stride)[e];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c + u < c1 && err[u] == 0) acc += v[u];
    }
    out[(long)g * nel + e] = acc;
}

// Start of a warm-up or measurement call, one workgroup per chain: counters and
// position of the header (init_counters, CTQMC.F90:847), and the arrays that the
// call accumulates into.  measure: everything from gtau on but the unused part
// of the calibration list; else AccPair, over the bins of [0, beta]
// (CTQMC.F90:8199-8206).  On the device: reading and writing the headers from
// the host cost more than a short call's sampling.
__global__ void __launch_bounds__(256) begin_kernel(ChainLayout L, char *chains, int nf, int measure, int ntau,
                                                    double beta)
{
    const int c = blockIdx.x;
    char *base = chains + (long)c * L.stride;
    ChainHdr *x = reinterpret_cast<ChainHdr *>(chains + L.hdrs) + c;
    auto clear = [&](long from, long to) {
        double *p = reinterpret_cast<double *>(base + from);
        for (long i = threadIdx.x; i < (to - from) / 8; i += 256) p[i] = 0.0;
    };
    if (measure) {
        clear(L.gtau, L.aptau);
        clear(L.aptau, min(L.scsum, L.aptau + 8L * max(x->apt_n, 0)));
        clear(L.scsum, L.stride);
    } else {
        clear(L.accpair, L.accpair + 8L * nf * L.naccpair_cap);
    }
    if (threadIdx.x != 0) return;
    x->try_add = x->try_rem = x->try_glob = x->try_shift = 0;
    x->acc_add = x->acc_rem = x->acc_glob = x->acc_shift = 0;
    x->qn_rej = x->moves = 0;
    x->alg_flops = x->alg_bytes = 0.0;
    x->pos = 0;
    x->halt = HALT_NONE;
    x->apt_index = 1;
    if (measure) {
        x->meas_sign = 0.0;
        x->cnt_meas = 0;
    } else {
        x->naccpair = ntau;
        x->accpair_max = beta;
    }
}

// The header scalars of the same groups: sum of signs, measurements,
// accepted / tried moves of each kind, attempted and QN-rejected moves,
// algorithmic flops and bytes (scal[g][14]), and the chains summed (used[g]).
// One thread per group.
__global__ void __launch_bounds__(64) group_scalars_kernel(const ChainHdr *hdrs, int nc, int ng, double *scal,
                                                           int *used)
{
    const int g = blockIdx.x * 64 + threadIdx.x;
    if (g >= ng) return;
    const int c0 = (int)((long)g * nc / ng), c1 = (int)((long)(g + 1) * nc / ng);
    double S[14];
    for (int i = 0; i < 14; ++i) S[i] = 0.0;
    int n = 0;
    for (int c = c0; c < c1; ++c) {
        const ChainHdr &x = hdrs[c];
        if (x.err != 0) continue;
        S[0] += x.meas_sign, S[1] += (double)x.cnt_meas;
        S[2] += (double)x.acc_add, S[3] += (double)x.try_add;
        S[4] += (double)x.acc_rem, S[5] += (double)x.try_rem;
        S[6] += (double)x.acc_glob, S[7] += (double)x.try_glob;
        S[8] += (double)x.acc_shift, S[9] += (double)x.try_shift;
        S[10] += (double)x.moves, S[11] += (double)x.qn_rej;
        S[12] += x.alg_flops, S[13] += x.alg_bytes;
        ++n;
    }
    for (int i = 0; i < 14; ++i) scal[(long)g * 14 + i] = S[i];
    used[g] = n;
}

// Initial state of every chain: random stream of seed seed0 + chain, empty
// configuration, initial outer superstate drawn proportional to the empty traces
// (init_Trace, Trace.F90:640-670).  The stream is seeded here (mt19937's initial
// recurrence, uniform over the wave: 623 steps of four scalar instructions; the
// kernel takes 0.13 ms for 1024 2-orbital chains): drawn up on the host, its
// upload as a strided copy from pageable memory cost 2 ms of a create of 256
// chains.
template <int NM>
__global__ void __launch_bounds__(WAVE) init_kernel(DevModel M, ChainLayout L, char *chains, uint32_t seed0)
{
    extern __shared__ __align__(16) char lds[];
    Ctx c = make_ctx<NM>(chains, (int)blockIdx.x, (CArgs)__builtin_amdgcn_kernarg_segment_ptr(), lds);
    uint32_t x = seed0 + blockIdx.x;
    for (int i = 0; i < 624; ++i) {
        if (i > 0) x = 1812433253u * (x ^ (x >> 30)) + (uint32_t)i;
        if (lane_id() == 0) c.rng.mt[i] = x;
    }
    wsync();
    rng_open(c.rng);
    choose_outer<NM>(c);
    rng_close(c.rng);
    if (!(c.h.trace_log > -DBL_MAX)) c.h.err = 5;
    save_ctx(c, (int)blockIdx.x);
}

// Bytes of a chain's state that setconfig_kernel replaces: header, part traces,
// operators, flavour lists and the used corner of the inverses.
__host__ __device__ inline long held_bytes(const ChainHdr &x, int nf, int nm)
{
    long n = (long)sizeof(ChainHdr) + 16L * nm + 12L * x.nop;
    for (int f = 0; f < nf; ++f) n += (24L + 8L * x.kf[f]) * x.kf[f];
    return (n + 7) / 8 * 8;
}

// That state of the chains first, first + 1, ... to buf + at[i] (each held_bytes
// long), or (BACK) from there.  Grid: x over chains, y over flavours and, last,
// what belongs to none; a workgroup's copies are one to five round trips.
template <bool BACK>
__global__ void __launch_bounds__(256) hold_kernel(ChainLayout L, char *chains, int first, int nf, int nm, char *buf,
                                                   const long *at)
{
    const int chain = first + (int)blockIdx.x, f = blockIdx.y, t = threadIdx.x;
    char *base = chains + (long)chain * L.stride, *hdr = chains + L.hdrs + (long)chain * (long)sizeof(ChainHdr);
    char *b = buf + at[blockIdx.x];
    const ChainHdr &x = *reinterpret_cast<const ChainHdr *>(BACK ? b : hdr);
    // n words between the chain and the buffer
    auto move = [&](char *p, long n) {
        int *c = reinterpret_cast<int *>(p), *q = reinterpret_cast<int *>(b);
        for (long i = t; i < n; i += 256) (BACK ? c : q)[i] = (BACK ? q : c)[i];
        b += 4 * n;
    };
    if (f == nf) {
        move(hdr, sizeof(ChainHdr) / 4);
        move(base + L.part, 4L * nm);
        move(base + L.tau, 2L * x.nop);
        move(base + L.code, x.nop);
        return;
    }
    b += (long)sizeof(ChainHdr) + 16L * nm + 12L * x.nop;
    for (int g = 0; g < f; ++g) b += (24L + 8L * x.kf[g]) * x.kf[g];
    const int k = x.kf[f];
    const long fo = (long)f * L.kcap;
    move(base + L.fc + 8 * fo, 2L * k);
    move(base + L.fa + 8 * fo, 2L * k);
    move(base + L.fcs + 4 * fo, k);
    move(base + L.fas + 4 * fo, k);
    // columns of the inverse (in words: the buffer is aligned to four bytes here)
    int *M = reinterpret_cast<int *>(base + L.minv) + 2 * fo * L.kcap, *q = reinterpret_cast<int *>(b);
    for (int j = t / WAVE; j < k; j += 256 / WAVE)
        for (int i = t % WAVE; i < 2 * k; i += WAVE) {
            int &c = M[2L * j * L.kcap + i], &h = q[2L * j * k + i];
            (BACK ? c : h) = BACK ? h : c;
        }
}

// Configurations for chains first, first + 1, ...: operators off[i] .. off[i+1]
// of tau / code and outer superstate outer[i] for chain first + i; full trace,
// flavour lists, full inverses, sign (set_mc_config_from_arrays,
// Trace.F90:6872-7000).  One wave per chain, all chains at once.
template <int NM>
__global__ void __launch_bounds__(WAVE) setconfig_kernel(DevModel M, ChainLayout L, char *chains, int first,
                                                         const double *tau, const int *code, const int *off,
                                                         const int *outer)
{
    const int chain = first + (int)blockIdx.x;
    extern __shared__ __align__(16) char lds[];
    Ctx c = make_ctx<NM>(chains, chain, (CArgs)__builtin_amdgcn_kernarg_segment_ptr(), lds);
    const int o0 = off[blockIdx.x], n = off[blockIdx.x + 1] - o0;
    for (int j = lane_id(); j < n; j += WAVE) {
        c.tau[j] = tau[o0 + j];
        c.code[j] = code[o0 + j];
    }
    c.h.nop = n;
    c.h.outer = outer[blockIdx.x];
    c.h.err = 0;
    wsync();
    c.h.wpos = 0;
    set_window(c);
    const TraceVal T = full_trace<NM>(c, c.h.outer);
    if (T.S == 0.0 && !(T.lg > -DBL_MAX)) c.h.err = 5;   // W2D_ERR_ZERO_TRACE: broken quantum numbers
    keep_trace<NM>(c, T);
    rebuild_flavour_lists(c, c.fc, c.fa, c.h.kf, c.fcs, c.fas);
    double dl = 0.0, dsg = 1.0;
    for (int f = 0; f < c.M.nf; ++f) {
        const int k = c.h.kf[f];
        if (k == 0) continue;
        double l, sg;
        if (!delta_inverse<NM>(c, f, k, l, sg)) {
            c.h.err = ERR_SING;
            break;
        }
        dl += l;
        dsg *= sg;
    }
    c.h.det_log = dl;
    c.h.det_sign = dsg;
    c.h.cfgsign = -config_sign(c);
    c.h.cache_pos = -1;
    save_ctx(c, chain);
}

}  // namespace w2d
