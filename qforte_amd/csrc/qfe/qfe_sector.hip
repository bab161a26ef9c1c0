// Determinant-sector engine: UCC energies, adjoint gradients and pool
// gradients on the (N_alpha, N_beta) sector of the reference determinant, and
// the continuous-batching serving engine built on them.
//
// A UCC generator K = sum_t kappa_t P_t built from a fermionic excitation
// (JW of tau - tau^dag, ansatz.py:25-82 feeding trotterize) is a set of Pauli
// strings that share one X mask and commute, so the product of their
// exponentials that the reference applies (trotterization.py:29-35, one
// exponentiate_pauli_string per term) equals exp(theta K) exactly.  K maps a
// determinant j to j ^ x with weight alpha(j) = sum_t kappa_t (-1)^{j.z_t};
// for anti-Hermitian K, alpha(j) alpha(j ^ x) = -|alpha(j)|^2, so on every
// pair (j, j ^ x) exp(theta K) = cos(theta w) + sin(theta w) / w * K with
// w = |alpha(j)|: a rotation of determinant pairs.  Pairs never leave the
// sector when K conserves N_alpha and N_beta, so the state needs only
// C(norb, N_alpha) * C(norb, N_beta) amplitudes instead of 2^n.
//
// Writing z_t = z_0 ^ d_t, alpha(j) = s(j) A(j & m) with s(j) = (-1)^{j.z_0},
// m = x | (union of the d_t) and A(p) = sum_t kappa_t (-1)^{p.d_t}: the host
// tabulates A over the patterns p of m, checks anti-Hermiticity and sector
// conservation pattern by pattern, and emits one "entry" per active pattern
// pair (p, p ^ x).  The determinants of an entry are a product of an alpha
// string list and a beta string list (with partner ranks precomputed).
//
// <H> = sum_groups sum_{j, j^x in sector} conj(psi_j) psi_{j^x} T_g(j^x),
// T_g(j') = sum_{t in g} c_t (-1)^{j'.z_t}   (computer.cc:850-911 on the sector).
// For x != 0 the pairs (j, j^x) and (j^x, j) contribute complex-conjugate
// values (H_g is Hermitian), so only the half with the top bit of x clear in j
// is visited, with weight 2.  The pair space of every group is cut into work
// items of similar cost that run as independent workgroups over the chip.
//
// Layout: rank(j) = rank_alpha(alpha string) * D_beta + rank_beta(beta string),
// strings ranked in increasing numeric order; alpha = even bits, beta = odd
// bits (state_prep.py:5-11 occupation convention).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <unordered_map>
#include <vector>

#include "qfe_device.h"
#include "qfe_internal.h"

namespace qfe {
namespace {

struct SecStep {  // one run of commuting exponentials sharing an X mask
    uint32_t e_first, e_count;
    int32_t param;
    uint32_t gen;
    double scale;
};

struct SecEntry {  // one class of determinant pairs of a run
    uint64_t x, z0;
    uint32_t la_off, la_len, lb_off, lb_len;
    double w, inv_lb;
    double2 ulo, uhi;  // A(p_lo) / w, A(p_hi) / w
    uint32_t step;
};

struct SecGroup {  // Hamiltonian terms sharing an X mask, on sector pairs
    uint64_t x;
    uint32_t la_off, la_len, lb_off, lb_len;  // half lists (x != 0) or full lists (x == 0)
    uint32_t t_first, t_count;
    uint32_t xa, xb;                          // compressed flips
    double inv_lb, weight;
};

struct SecItem {  // groups [g0, g1) whole, or pairs [p0, p1) of group g0 when g1 == g0 + 1
    uint32_t g0, g1, p0, p1;
};

// ---- component tiles ----
// A segment is a run of consecutive generators.  The flips of its entries
// join alpha strings into components and beta strings likewise; a block is a
// union of whole components, so no pair of the segment leaves the tile
// (alpha block) x (beta block), and a workgroup applies the whole segment to
// its tile in LDS: one load and one store of the state per segment.
struct TileSeg {
    uint32_t nab, nbb;      // alpha and beta blocks
    uint32_t ablk, bblk;    // tix: first position of each block (nab + 1, nbb + 1 entries)
    uint32_t aperm, bperm;  // tix: string ranks, block by block
    uint32_t awb, bwb;      // tix: first word of each block (nab + 1, nbb + 1 entries)
    uint32_t atab, btab;    // ttab: [list * nab + block], [list * nbb + block]
};

struct TileRec {  // one entry in the program of a pass
    double w;
    double2 ulo, uhi;
    uint32_t entry, alist, blist, flags;
};
constexpr uint32_t kRecRot = 1;      // rotate (or un-rotate) the entry's pairs
constexpr uint32_t kRecOv = 2;       // add the pairs' overlaps
constexpr uint32_t kRecStepEnd = 4;  // the next record reads what this one wrote
constexpr uint32_t kRecGenEnd = 8;   // the overlap of a generator is complete

struct TileRun {  // one pass: the records [rec0, rec0 + nrec) over the tiles of a segment
    uint32_t seg, rec0, nrec, part;  // part: first partial sum (reverse sweep)
};

// The partial sums of the reverse sweep (one per wave of a tile and output) are
// kept for a window of consecutive passes and added up behind the last of
// them; the next window uses the same memory (see TileBuilder::most).
struct TileOut {  // output 0 is the energy, k + 1 generator k's overlap
    uint32_t out, r0, r1, add;  // its ranges tsum[r0 .. r1); add: an earlier window has a part of it
};
struct TileWindow {
    uint32_t pass, o0, o1, pad;  // last pass, outputs touts[o0 .. o1)
};

// A list word: local position of a string and of its partner in their block,
// and the parities of the entry's sign mask on both.
constexpr uint32_t kWordBits = 14, kWordPos = (1u << kWordBits) - 1u;

// ---- Hamiltonian rows: one workgroup per alpha string ---------------------------------
// H of a real template on one row of the sector (alpha string a, all beta
// strings, one per lane).  With a fixed, every coefficient that depends on a
// alone is one number for the whole row, and lists per string replace the scan
// over X masks:
//   alpha flips (and the diagonal): the terms of a flip merge by their beta Z
//     mask into cells, T(b) = sum_cells C_cell (-1)^{b & mu}, times a
//     coalesced row of psi;
//   beta flips: per pattern of the flipped bits the terms merge by the
//     remaining beta Z mask, times the row itself from LDS;
//   alpha and beta flips together: one number G[alpha flip][beta flip] per
//     pattern pair; rows of psi come through LDS four at a time, with every
//     sign folded into the staged row, the staged numbers or the lane's word.
// The merged numbers (M) are linear in the request's inputs and come from the
// prologue.  A 20-qubit row has 625 + 2 x 126 connected determinants; the term
// loops it replaces took 8 sign evaluations for each and tested all 2536 X
// masks per determinant: sigma of a 20-qubit request 2318 -> 133 us, of a
// 16-qubit one 2035 -> 64, energy items of an 8-qubit one 118 -> 15 (one
// request alone; latency and LDS gathers bound it).  Groups that do not fit
// this form (RowBuilder::fits) and complex templates stay with the term loops
// below.
struct RowFlip {  // an alpha flip of a row: partner rank and its cells
    uint32_t partner, cell0, ncell, pos;
};
struct RowPair {  // an alpha flip of a row that goes with beta flips
    uint32_t partner, fa, neg, pad;
};
struct RowTables {
    const uint32_t* chunk_off;  // chunks of row a: [chunk_off[a], chunk_off[a + 1])
    const uint4* chunks;        // (first flip, flips, first position, positions)
    const RowFlip* flips;       // padded to whole groups of kRowUnroll per chunk
    const uint32_t* pos_cell;   // cell of every position
    const uint32_t* amu;        // beta mask of every alpha cell
    const uint32_t* am;         // merged numbers of every alpha cell: [am[c], am[c + 1])
    const uint32_t* bmu;        // the same for beta cells
    const uint32_t* bm;
    const uint32_t* mmask;      // alpha sign mask of every merged number
    const uint32_t* b1;         // [k][Db] beta flips with one cell: partner | cell << 14 | sign << 31
    const uint2* b2;            // [k][Db] others: (partner, first cell | cells << 20)
    const uint32_t* pair_off;   // pair flips of row a, padded to whole groups of 4
    const RowPair* pairs;
    const uint32_t* words;      // [k][Db] beta flips of pairs: partner | flip << 14 | sign << 31
    const uint32_t* fb_mask;    // alpha sign mask of every beta flip
    const uint32_t* fa_mask;    // beta sign mask of every alpha flip
    const double* m;            // merged numbers of a fixed Hamiltonian
    const uint32_t *moff, *midx;  // or their inputs
    const double* mval;
    uint32_t nm, nbcell, nb1, nb2, nwords, nfb, gbase;
};
constexpr uint32_t kRowThreads = 256;
constexpr uint32_t kRowNone = 0xffffffffu;
constexpr uint32_t kRowCells = 512;   // alpha cells of a chunk
constexpr uint32_t kRowUnroll = 8;    // rows of psi in flight
constexpr uint32_t kRowCellBits = 17; // beta cells and flips per word

struct SecTables {  // device view of a template (lives in device memory)
    uint64_t D, ref_rank;
    uint32_t Da, Db;
    const uint64_t* afull;
    const uint64_t* bfull;
    const uint32_t* astr;
    const uint32_t* bstr;
    const int32_t* arank;  // 2^norb entries, -1 outside the sector
    const int32_t* brank;
    const int2* lists;
    const SecStep* steps;
    const SecEntry* entries;
    const SecGroup* groups;
    const SecItem* items;
    const uint32_t* gen_step;  // steps of generator k: [gen_step[k], gen_step[k+1])
    const uint64_t* tz;
    const double2* tph;    // phase of each term
    const void* tcoef;     // phase * coeff (fixed Hamiltonian), in the template's scalar type
    const uint64_t* map_off;
    const uint32_t* map_idx;
    const double2* map_val;
    const uint2* hchunks;  // groups [x, y) staged together by the sigma kernel
    const TileSeg* tsegs;
    const TileRun* tfwd;   // ansatz passes, in order
    const TileRun* trev;   // reverse-sweep passes, in order
    const TileRec* trec;
    const uint32_t* tix;   // block starts, permuted ranks and word starts of every segment
    const uint2* ttab;     // (offset, length) of every list in every block
    const uint32_t* twords;
    const uint2* tsum;     // ranges (first, count) of reverse-sweep partial sums
    const TileOut* touts;
    const TileWindow* twins;
    RowTables rows;
    uint32_t nsteps, nentries, ngroups, nterms, nitems, ngen, nhchunks, nwins;
    uint32_t nparts;  // energy partials: the work items', then one per row workgroup
    uint32_t nrows;   // row workgroups (0: every group is in the work items)
};

struct SlotDesc {
    const SecTables* t;
    void* psi;      // amplitudes: double2, or double for a real template
    void* sig;      // H psi (gradients only)
    double* hm;     // per-request merged numbers of the rows (null: t->rows.m)
    void* coef;     // per-request coefficients, same scalar type (null: t->tcoef)
    double2* cs;    // (cos, sin) per entry
    double* part;   // per work item energy partials
    double* gpart;  // reverse-sweep partial sums (gradients only)
    double* gacc;   // per generator <sigma|K|psi> (gradients only)
    const double* params;
    const double* inputs;
    double* out;
};

struct PoolOp {  // entries [e0, e1) of one pool operator
    uint32_t e0, e1;
};

constexpr uint32_t kTermLds = 1024;   // Hamiltonian terms of one group staged in LDS when they fit
constexpr int kUnroll = 4;            // independent pairs in flight per thread
constexpr int kItemThreads = 256;

__device__ __forceinline__ void divmod_u(uint32_t i, uint32_t d, double inv, uint32_t& q, uint32_t& r) {
    int64_t qq = (int64_t)((double)i * inv);
    int64_t rr = (int64_t)i - qq * (int64_t)d;
    if (rr < 0) {
        qq -= 1;
        rr += d;
    } else if (rr >= (int64_t)d) {
        qq += 1;
        rr -= d;
    }
    q = (uint32_t)qq;
    r = (uint32_t)rr;
}

// Largest s with prefix[s] <= b (prefix[0] = 0, n + 1 entries).
__device__ __forceinline__ uint32_t find_slot(const uint32_t* __restrict__ prefix, uint32_t n, uint32_t b) {
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (prefix[mid] <= b)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// The scalar type S of a template: double when every generator and every
// Hamiltonian coefficient is real (the state is then real throughout, as for
// every UCC ansatz over real orbitals), else double2.  Real templates move
// and multiply half as much; dropping exact zeros changes no bit of a result.
__device__ __forceinline__ double2 umul(double2 u, double2 v) { return cmul(u, v); }
__device__ __forceinline__ double umul(double2 u, double v) { return u.x * v; }
__device__ __forceinline__ double2 lincomb(double c, double2 a, double s, double2 h) {
    return make_double2(c * a.x + s * h.x, c * a.y + s * h.y);
}
__device__ __forceinline__ double lincomb(double c, double a, double s, double h) { return c * a + s * h; }
__device__ __forceinline__ double re_dot(double2 a, double2 b) { return a.x * b.x + a.y * b.y; }
__device__ __forceinline__ double re_dot(double a, double b) { return a * b; }
template <typename S>
__device__ __forceinline__ S real_amp(double v);
template <>
__device__ __forceinline__ double2 real_amp<double2>(double v) {
    return make_double2(v, 0.0);
}
template <>
__device__ __forceinline__ double real_amp<double>(double v) {
    return v;
}
__device__ __forceinline__ double2 to_complex(double2 v) { return v; }
__device__ __forceinline__ double2 to_complex(double v) { return make_double2(v, 0.0); }

// ---- 1. prologue: per-request Hamiltonian coefficients and rotation angles --------------
// `blocks` workgroups per request: a request's numbers are independent of each
// other.  Requests share grid x, since a launch of small ones holds more of
// them than the grid's second dimension does.
template <typename S>
__global__ __launch_bounds__(256) void k_sec_prologue(const SlotDesc* __restrict__ slots, int need_coef, uint32_t blocks) {
    const uint32_t slot = blockIdx.x / blocks;
    const SlotDesc sd = slots[slot];
    const SecTables* __restrict__ T = sd.t;
    const uint32_t i0 = (blockIdx.x - slot * blocks) * blockDim.x + threadIdx.x, step = blocks * blockDim.x;
    if (need_coef && sd.coef) {
        for (uint32_t k = i0; k < T->nterms; k += step) {
            double cr = 0.0, ci = 0.0;
            const uint64_t e1 = T->map_off[k + 1];
            for (uint64_t e = T->map_off[k]; e < e1; ++e) {
                const double v = sd.inputs[T->map_idx[e]];
                const double2 f = T->map_val[e];
                cr += f.x * v;
                ci += f.y * v;
            }
            if constexpr (sizeof(S) == sizeof(double))
                static_cast<double*>(sd.coef)[k] = T->tph[k].x * cr;
            else
                static_cast<double2*>(sd.coef)[k] = cmul(T->tph[k], make_double2(cr, ci));
        }
    }
    if (need_coef && sd.hm) {
        const RowTables& R = T->rows;
        for (uint32_t k = i0; k < R.nm; k += step) {
            double v = 0.0;
            const uint32_t e1 = R.moff[k + 1];
            for (uint32_t e = R.moff[k]; e < e1; ++e) v += R.mval[e] * sd.inputs[R.midx[e]];
            sd.hm[k] = v;
        }
    }
    for (uint32_t e = i0; e < T->nentries; e += step) {
        const SecEntry& en = T->entries[e];
        const SecStep& st = T->steps[en.step];
        double s, c;
        sincos(st.scale * sd.params[st.param] * en.w, &s, &c);
        sd.cs[e] = make_double2(c, s);
    }
}

// One pair (r1, r2) of an entry with old values (a, b), j1 the determinant
// of r1: psi_1' = c a + s s(j2) uhi b, psi_2' = c b + s s(j1) ulo a.  Every
// step-by-step kernel calls this; the tile passes apply the same formula.
template <typename S>
__device__ __forceinline__ void pair_rotate(S* __restrict__ psi, uint64_t r1, uint64_t r2, S a, S b, uint64_t j1, uint64_t x,
                                            uint64_t z0, double c, double s, double2 ulo, double2 uhi) {
    const double s1 = s * parity_sign(j1 & z0), s2 = s * parity_sign((j1 ^ x) & z0);
    psi[r1] = lincomb(c, a, s2, umul(uhi, b));
    psi[r2] = lincomb(c, b, s1, umul(ulo, a));
}

// <sigma|K|psi> contribution of one pair: (K psi)_1 = s(j2) w uhi psi_2,
// (K psi)_2 = s(j1) w ulo psi_1.
template <typename S>
__device__ __forceinline__ double pair_overlap(const SecEntry& en, uint64_t j1, S pa, S pb, S sa, S sb) {
    const double s1 = en.w * parity_sign(j1 & en.z0), s2 = en.w * parity_sign((j1 ^ en.x) & en.z0);
    return s2 * re_dot(sa, umul(en.uhi, pb)) + s1 * re_dot(sb, umul(en.ulo, pa));
}

__device__ __forceinline__ double2 conj_mul(double2 a, double2 b) { return cconjmul(a, b); }
__device__ __forceinline__ double conj_mul(double a, double b) { return a * b; }
__device__ __forceinline__ double re_mul(double2 a, double2 b) { return a.x * b.x - a.y * b.y; }
__device__ __forceinline__ double re_mul(double a, double b) { return a * b; }

// v with its sign bit flipped when neg = 1u << 31: adding flip_sign(c, neg) is
// bit-identical to fma(+-1.0, c, acc), with one integer op for the sign.
// Determinant indices and Z masks fit 32 bits (at most 32 qubits).
__device__ __forceinline__ double flip_sign(double v, uint32_t neg) {
    return __hiloint2double(__double2hiint(v) ^ (int)neg, __double2loint(v));
}
__device__ __forceinline__ void add_flipped(double2& t, double2 c, uint32_t neg) {
    t.x += flip_sign(c.x, neg);
    t.y += flip_sign(c.y, neg);
}
__device__ __forceinline__ void add_flipped(double& t, double c, uint32_t neg) { t += flip_sign(c, neg); }
// t += a b
__device__ __forceinline__ void add_mul(double2& t, double2 a, double2 b) {
    t.x += a.x * b.x - a.y * b.y;
    t.y += a.x * b.y + a.y * b.x;
}
__device__ __forceinline__ void add_mul(double& t, double a, double b) { t += a * b; }

// ---- 2. ansatz and reverse sweep: component tiles ---------------------------------------
constexpr uint32_t kRecChunk = 128;        // records staged in LDS at a time
constexpr uint32_t kTileWordsLds = 4096;   // list words of a tile staged in LDS when they fit

// A record as the tile's loop reads it: which pairs, and the factors of their
// rotation and overlap.
struct RecHead {
    uint32_t a_off, b_off, b_len, pairs, magic, flags;
    __device__ __forceinline__ RecHead uniform() const {  // every lane reads the same record
        auto u = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
        return RecHead{u(a_off), u(b_off), u(b_len), u(pairs), u(magic), u(flags)};
    }
};
template <typename S>
struct RecFactors {
    double c, s, w, ulo_x, ulo_y, uhi_x, uhi_y;
    __device__ void set(double c_, double s_, double w_, double2 ulo, double2 uhi) {
        c = c_;
        s = s_;
        w = w_;
        ulo_x = ulo.x;
        ulo_y = ulo.y;
        uhi_x = uhi.x;
        uhi_y = uhi.y;
    }
    // rotated pair from the old values; n1, n2: sign bits of the two directions
    __device__ __forceinline__ void rotate(S a, S b, uint32_t n1, uint32_t n2, S& ra, S& rb) const {
        ra = lincomb(c, a, flip_sign(s, n2), umul(make_double2(uhi_x, uhi_y), b));
        rb = lincomb(c, b, flip_sign(s, n1), umul(make_double2(ulo_x, ulo_y), a));
    }
    __device__ __forceinline__ double overlap(S a, S b, S ya, S yb, uint32_t n1, uint32_t n2) const {
        return flip_sign(w, n2) * re_dot(ya, umul(make_double2(uhi_x, uhi_y), b)) +
               flip_sign(w, n1) * re_dot(yb, umul(make_double2(ulo_x, ulo_y), a));
    }
};
// Real factors are +-1 and folded into sine and weight.
template <>
struct RecFactors<double> {
    double c, slo, shi, wlo, whi;
    __device__ void set(double c_, double s_, double w_, double2 ulo, double2 uhi) {
        c = c_;
        slo = s_ * ulo.x;
        shi = s_ * uhi.x;
        wlo = w_ * ulo.x;
        whi = w_ * uhi.x;
    }
    __device__ __forceinline__ void rotate(double a, double b, uint32_t n1, uint32_t n2, double& ra, double& rb) const {
        ra = lincomb(c, a, flip_sign(shi, n2), b);
        rb = lincomb(c, b, flip_sign(slo, n1), a);
    }
    __device__ __forceinline__ double overlap(double a, double b, double ya, double yb, uint32_t n1, uint32_t n2) const {
        return flip_sign(whi, n2) * (ya * b) + flip_sign(wlo, n1) * (yb * a);
    }
};
template <typename S>
struct LdsRec {
    RecFactors<S> f;
    RecHead head;
};

// i / d for i < 2^16, 0 < d < 2^16 by a multiplication: ceil(2^32 / d) (0 for d = 1).
__host__ __device__ __forceinline__ uint32_t div_magic(uint32_t d) { return d > 1 ? (uint32_t)((0x100000000ull + d - 1) / d) : 0u; }
__device__ __forceinline__ uint32_t div_by(uint32_t i, uint32_t magic) { return magic ? __umulhi(i, magic) : i; }

// One pass over the tiles of a segment, one workgroup of T threads per tile.
// MODE 0: the segment's rotations on psi (q = 0 starts from the reference);
// MODE 1: their inverses on sigma; MODE 2: the reverse sweep on psi and
// sigma: for each generator, last first, the tile's part of
// Re<sigma|K|psi>, then its inverse on both (q = 0 also adds Re<psi|sigma>).
// One workgroup used to walk all generators of a request, or one launch took
// each step of a lone large request: a step's pairs are few and its latency
// (a barrier and an LDS or L2 round trip, or a launch) was what counted.
// Tiles split the pairs of a step over many workgroups and keep many steps in
// one launch.
template <typename S, int T, int MODE>
__global__ __launch_bounds__(T) void k_sec_tile(const SlotDesc* __restrict__ slots, const uint32_t* __restrict__ prefix,
                                                uint32_t nslots, uint32_t q, uint32_t start) {
    extern __shared__ double2 tile_lds[];
    const uint32_t tid = threadIdx.x;
    const uint32_t slot = nslots == 1 ? 0u : find_slot(prefix, nslots, blockIdx.x);
    const uint32_t tile = nslots == 1 ? blockIdx.x : blockIdx.x - prefix[slot];
    const SlotDesc sd = slots[slot];
    const SecTables* __restrict__ Tb = sd.t;
    const TileRun run = (MODE == 2 ? Tb->trev : Tb->tfwd)[q];
    const TileSeg sg = Tb->tsegs[run.seg];
    const uint32_t* __restrict__ tix = Tb->tix;
    const uint32_t ab = tile / sg.nbb, bb = tile - ab * sg.nbb;
    const uint32_t a0 = tix[sg.ablk + ab], na = tix[sg.ablk + ab + 1] - a0;
    const uint32_t b0 = tix[sg.bblk + bb], nb = tix[sg.bblk + bb + 1] - b0;
    const uint32_t aw0 = tix[sg.awb + ab], naw = tix[sg.awb + ab + 1] - aw0;
    const uint32_t bw0 = tix[sg.bwb + bb], nbw = tix[sg.bwb + bb + 1] - bw0;
    const uint32_t n = na * nb, nmag = div_magic(nb), ntiles = sg.nab * sg.nbb;
    const uint32_t nrec = run.nrec, nchunk = nrec < kRecChunk ? nrec : kRecChunk;
    S* X = reinterpret_cast<S*>(tile_lds);
    S* Y = X + (MODE == 2 ? n : 0u);
    using Factors = RecFactors<S>;
    LdsRec<S>* recs = reinterpret_cast<LdsRec<S>*>(tile_lds + ((n * (MODE == 2 ? 2u : 1u) * sizeof(S) + 15) >> 4));
    uint32_t* lw = reinterpret_cast<uint32_t*>(recs + nchunk);
    const bool wlds = naw + nbw <= kTileWordsLds;
    S* __restrict__ gx = reinterpret_cast<S*>(MODE == 1 ? sd.sig : sd.psi);
    S* __restrict__ gy = reinterpret_cast<S*>(sd.sig);
    const uint64_t Db = Tb->Db;

    // records [c0, c0 + cnt) in the order of this pass; returns whether this
    // thread's records have pairs in the tile
    auto stage = [&](uint32_t c0, uint32_t cnt) {
        bool any = false;
        for (uint32_t r = tid; r < cnt; r += T) {
            const uint32_t at = MODE == 1 ? run.rec0 + nrec - 1 - (c0 + r) : run.rec0 + c0 + r;
            const TileRec tr = Tb->trec[at];
            const uint2 la = Tb->ttab[sg.atab + tr.alist * sg.nab + ab], lb = Tb->ttab[sg.btab + tr.blist * sg.nbb + bb];
            const double2 cs = sd.cs[tr.entry];
            LdsRec<S> o;
            o.f.set(cs.x, MODE == 0 ? cs.y : -cs.y, tr.w, tr.ulo, tr.uhi);
            o.head.a_off = la.x;
            o.head.b_off = lb.x;
            o.head.b_len = lb.y;
            o.head.pairs = la.y * lb.y;
            o.head.magic = div_magic(lb.y);
            o.head.flags = tr.flags;
            // last step first: a step ends before the record that ends the step before it
            if (MODE == 1) o.head.flags = kRecRot | (at > run.rec0 ? Tb->trec[at - 1].flags & kRecStepEnd : 0u);
            any |= o.head.pairs != 0;
            recs[r] = o;
        }
        return any;
    };
    bool any = stage(0, nchunk);
    if (wlds) {
        for (uint32_t i = tid; i < naw; i += T) lw[i] = Tb->twords[aw0 + i];
        for (uint32_t i = tid; i < nbw; i += T) lw[naw + i] = Tb->twords[bw0 + i];
    }
    // a tile without pairs keeps its amplitudes
    const bool idle = nrec <= kRecChunk && !__syncthreads_or(any) && !start;
    if (idle) {
        if (MODE == 2)
            for (uint32_t r = 0, k = 0; r < nrec; ++r)
                if (Tb->trec[run.rec0 + r].flags & kRecGenEnd) {
                    if ((tid & (kWave - 1)) == 0)
                        sd.gpart[run.part + (k * ntiles + tile) * (T / kWave) + tid / kWave] = 0.0;
                    ++k;
                }
        return;
    }
    double dot = 0.0;
    for (uint32_t i = tid; i < n; i += T) {
        const uint32_t la = div_by(i, nmag), lb = i - la * nb;
        const uint64_t r = (uint64_t)tix[sg.aperm + a0 + la] * Db + tix[sg.bperm + b0 + lb];
        if (MODE == 0 && start) {
            X[i] = real_amp<S>(r == Tb->ref_rank ? 1.0 : 0.0);
        } else {
            const S x = gx[r];
            X[i] = x;
            if (MODE == 2) {
                const S y = gy[r];
                Y[i] = y;
                dot += re_dot(x, y);
            }
        }
    }
    uint32_t part = MODE == 2 ? run.part + tile * (T / kWave) + tid / kWave : 0u;  // next partial sum of this wave
    const uint32_t pstep = ntiles * (T / kWave);
    if (MODE == 2 && start) {
        const double v = wave_sum_last(dot);
        if ((tid & (kWave - 1)) == kWave - 1) sd.gpart[part] = v;
        part += pstep;
    }
    __syncthreads();

    double acc = 0.0;
    auto words = [&](const RecHead& R, uint32_t i, uint32_t& wa, uint32_t& wb) {
        const uint32_t ia = div_by(i, R.magic), ib = i - ia * R.b_len;
        if (wlds) {
            wa = lw[R.a_off + ia];
            wb = lw[naw + R.b_off + ib];
        } else {
            wa = Tb->twords[aw0 + R.a_off + ia];
            wb = Tb->twords[bw0 + R.b_off + ib];
        }
    };
    auto pair = [&](const Factors& F, uint32_t flags, uint32_t wa, uint32_t wb) {
        const uint32_t l1 = (wa & kWordPos) * nb + (wb & kWordPos);
        const uint32_t l2 = ((wa >> kWordBits) & kWordPos) * nb + ((wb >> kWordBits) & kWordPos);
        const uint32_t sw = wa ^ wb;  // bit 30: the parity on the string pair, bit 31: on its partner
        const uint32_t n1 = (sw << 1) & 0x80000000u, n2 = sw & 0x80000000u;
        const S a = X[l1], b = X[l2];
        S ra, rb;
        if (MODE == 2) {
            const S ya = Y[l1], yb = Y[l2];
            if (flags & kRecOv) acc += F.overlap(a, b, ya, yb, n1, n2);
            if (flags & kRecRot) {
                F.rotate(a, b, n1, n2, ra, rb);
                X[l1] = ra;
                X[l2] = rb;
                F.rotate(ya, yb, n1, n2, ra, rb);
                Y[l1] = ra;
                Y[l2] = rb;
            }
        } else {
            F.rotate(a, b, n1, n2, ra, rb);
            X[l1] = ra;
            X[l2] = rb;
        }
    };
    for (uint32_t c0 = 0; c0 < nrec; c0 += kRecChunk) {
        const uint32_t cnt = nrec - c0 < kRecChunk ? nrec - c0 : kRecChunk;
        if (c0) {
            __syncthreads();
            stage(c0, cnt);
            __syncthreads();
        }
        // the record and first words of the next entry are read while the
        // current one is applied: they do not depend on its writes
        RecHead R = recs[0].head.uniform();
        Factors F = recs[0].f;
        uint32_t wa = 0, wb = 0;
        if (tid < R.pairs) words(R, tid, wa, wb);
        for (uint32_t r = 0; r < cnt; ++r) {
            const uint32_t nx = r + 1 < cnt ? r + 1 : r;
            const RecHead N = recs[nx].head.uniform();
            const Factors NF = recs[nx].f;
            uint32_t xa = 0, xb = 0;
            if (tid < N.pairs) words(N, tid, xa, xb);
            if (tid < R.pairs) pair(F, R.flags, wa, wb);
            for (uint32_t i = tid + T; i < R.pairs; i += T) {
                words(R, i, wa, wb);
                pair(F, R.flags, wa, wb);
            }
            if (MODE == 2 && (R.flags & kRecGenEnd)) {
                const double v = wave_sum_last(acc);
                if ((tid & (kWave - 1)) == kWave - 1) sd.gpart[part] = v;
                part += pstep;
                acc = 0.0;
            }
            if (R.flags & kRecStepEnd) __syncthreads();
            R = N;
            F = NF;
            wa = xa;
            wb = xb;
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < n; i += T) {
        const uint32_t la = div_by(i, nmag), lb = i - la * nb;
        const uint64_t r = (uint64_t)tix[sg.aperm + a0 + la] * Db + tix[sg.bperm + b0 + lb];
        gx[r] = X[i];
        if (MODE == 2) gy[r] = Y[i];
    }
}

// Sums of a window's partials in a fixed order, one wave per output: the
// window that ends with pass `pass` (a request that has none does nothing), or
// for kLastWindow every request's last one.
constexpr uint32_t kLastWindow = 0xffffffffu;
__global__ __launch_bounds__(256) void k_sec_tile_sum(const SlotDesc* __restrict__ slots, uint32_t pass) {
    const SlotDesc sd = slots[blockIdx.y];
    const SecTables* __restrict__ T = sd.t;
    uint32_t w = T->nwins - 1;
    if (pass != kLastWindow) {
        w = 0;
        while (w + 1 < T->nwins && T->twins[w].pass != pass) ++w;
        if (w + 1 == T->nwins) return;
    }
    const TileWindow W = T->twins[w];
    const uint32_t k = W.o0 + blockIdx.x * (256 / kWave) + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (k >= W.o1) return;
    const TileOut O = T->touts[k];
    double acc = 0.0;
    for (uint32_t r = O.r0; r < O.r1; ++r) {
        const uint2 range = T->tsum[r];
        for (uint32_t i = lane; i < range.y; i += kWave) acc += sd.gpart[range.x + i];
    }
    const double v = wave_sum_last(acc);
    if (lane == kWave - 1) {
        double* to = O.out ? sd.gacc + (O.out - 1) : sd.out;
        *to = O.add ? *to + v : v;
    }
}

// ---- 3. Hamiltonian rows (see RowTables) -------------------------------------------------
__device__ __forceinline__ uint32_t odd_sign(uint32_t v) { return (uint32_t)__popc(v) << 31; }

// ENERGY: partial sums psi . (H psi) into part[]; else sigma = H psi.
template <bool ENERGY>
__global__ __launch_bounds__(kRowThreads) void k_sec_rows(const SlotDesc* __restrict__ slots,
                                                          const uint32_t* __restrict__ prefix, uint32_t nslots) {
    extern __shared__ double2 row_lds[];
    __shared__ double2 red[16];
    const uint32_t tid = threadIdx.x, nt = blockDim.x;
    const uint32_t slot = nslots == 1 ? 0u : find_slot(prefix, nslots, blockIdx.x);
    const uint32_t at = nslots == 1 ? blockIdx.x : blockIdx.x - prefix[slot];
    const SlotDesc sd = slots[slot];
    const SecTables* __restrict__ T = sd.t;
    const RowTables& R = T->rows;
    const uint32_t Db = T->Db, ncol = (Db + nt - 1) / nt;
    const uint32_t ra = at / ncol, rb = (at - ra * ncol) * nt + tid;
    const bool live = rb < Db;
    const uint32_t rbs = live ? rb : 0u;
    const double* __restrict__ psi = static_cast<const double*>(sd.psi);
    const double* __restrict__ M = sd.hm ? sd.hm : R.m;
    const uint32_t sa = T->astr[ra], sb = T->bstr[rbs];
    // LDS: own row, beta cells, then alpha cells or the staged rows of a pair group
    double* own = reinterpret_cast<double*>(row_lds);
    double* cb = own + Db;
    double* ca = cb + R.nbcell + 1;
    uint32_t* cmu = reinterpret_cast<uint32_t*>(ca + kRowCells);
    double* buf = reinterpret_cast<double*>(row_lds + ((Db + R.nbcell + 2) >> 1));
    double* tab = buf + 4 * (size_t)Db;

    for (uint32_t i = tid; i < Db; i += nt) own[i] = psi[(uint64_t)ra * Db + i];
    auto merged = [&](uint32_t m0, uint32_t m1) {
        double v = 0.0;
        for (uint32_t m = m0; m < m1; ++m) v += flip_sign(M[m], odd_sign(sa & R.mmask[m]));
        return v;
    };
    for (uint32_t c = tid; c < R.nbcell; c += nt) cb[c] = merged(R.bm[c], R.bm[c + 1]);
    if (tid == 0) cb[R.nbcell] = 0.0;  // the cell of padding words
    __syncthreads();
    double acc = 0.0;

    // beta flips
    constexpr uint32_t kCell = (1u << kRowCellBits) - 1u;
    for (uint32_t k = 0; k < R.nb1; k += kRowUnroll) {
        uint32_t w[kRowUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kRowUnroll; ++u) w[u] = R.b1[(size_t)(k + u) * Db + rbs];
#pragma unroll
        for (uint32_t u = 0; u < kRowUnroll; ++u)
            acc += flip_sign(cb[(w[u] >> 14) & kCell], w[u] & 0x80000000u) * own[w[u] & 0x3fffu];
    }
    if (R.nb2) {
        uint2 w = R.b2[rbs];
        for (uint32_t k = 1; k <= R.nb2; ++k) {
            const uint2 next = R.b2[(size_t)(k < R.nb2 ? k : 0u) * Db + rbs];
            const uint32_t c0 = w.y & 0xfffffu, n = w.y >> 20;
            double t = 0.0;
            for (uint32_t c = c0; c < c0 + n; ++c) t += flip_sign(cb[c], odd_sign(sb & R.bmu[c]));
            acc += t * own[w.x];
            w = next;
        }
    }

    // alpha flips and the diagonal
    for (uint32_t ch = R.chunk_off[ra]; ch < R.chunk_off[ra + 1]; ++ch) {
        const uint4 cd = R.chunks[ch];
        if (ch != R.chunk_off[ra]) __syncthreads();
        for (uint32_t p = tid; p < cd.w; p += nt) {
            const uint32_t c = R.pos_cell[cd.z + p];
            ca[p] = merged(R.am[c], R.am[c + 1]);
            cmu[p] = R.amu[c];
        }
        __syncthreads();
        for (uint32_t f = 0; f < cd.y; f += kRowUnroll) {
            double v[kRowUnroll];
#pragma unroll
            for (uint32_t u = 0; u < kRowUnroll; ++u) v[u] = psi[(uint64_t)R.flips[cd.x + f + u].partner * Db + rbs];
#pragma unroll
            for (uint32_t u = 0; u < kRowUnroll; ++u) {
                const RowFlip fl = R.flips[cd.x + f + u];
                double t = 0.0;
                for (uint32_t p = fl.pos; p < fl.pos + fl.ncell; ++p) t += flip_sign(ca[p], odd_sign(sb & cmu[p]));
                acc += t * v[u];
            }
        }
    }

    // alpha and beta flips together, four alpha flips at a time
    for (uint32_t p0 = R.pair_off[ra]; p0 < R.pair_off[ra + 1]; p0 += 4) {
        __syncthreads();
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const RowPair pr = R.pairs[p0 + q];
            const bool on = pr.partner != kRowNone;
            const uint32_t rm = on ? R.fa_mask[pr.fa] : 0u;
            for (uint32_t i = tid; i < Db; i += nt)
                buf[4 * i + q] = on ? flip_sign(psi[(uint64_t)pr.partner * Db + i], odd_sign(T->bstr[i] & rm)) : 0.0;
            const double* __restrict__ g = M + R.gbase + (size_t)(on ? pr.fa : 0u) * R.nfb;
            if (tid == 0) tab[4 * R.nfb + q] = 0.0;  // the flip of padding words
            for (uint32_t i = tid; i < R.nfb; i += nt)
                tab[4 * i + q] = on ? flip_sign(g[i], odd_sign(sa & R.fb_mask[i]) ^ pr.neg) : 0.0;
        }
        __syncthreads();
        for (uint32_t k = 0; k < R.nwords; k += 4) {
            uint32_t w[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) w[u] = R.words[(size_t)(k + u) * Db + rbs];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const double2* x = reinterpret_cast<const double2*>(buf + 4 * (w[u] & 0x3fffu));
                const double2* g = reinterpret_cast<const double2*>(tab + 4 * ((w[u] >> 14) & kCell));
                const double2 x0 = x[0], x1 = x[1], g0 = g[0], g1 = g[1];
                acc += flip_sign((g0.x * x0.x + g0.y * x0.y) + (g1.x * x1.x + g1.y * x1.y), w[u] & 0x80000000u);
            }
        }
    }
    if (ENERGY) {
        const double2 tot = block_sum(make_double2(live ? acc * own[rbs] : 0.0, 0.0), red);
        if (tid == 0) sd.part[T->nitems + at] = tot.x;
    } else if (live) {
        static_cast<double*>(sd.sig)[(uint64_t)ra * Db + rb] = acc;
    }
}

// ---- 4. energy work items: one workgroup per (request, item) ---------------------------
template <typename S>
__global__ __launch_bounds__(kItemThreads) void k_sec_energy(const SlotDesc* __restrict__ slots,
                                                             const uint32_t* __restrict__ prefix, uint32_t nslots) {
    __shared__ uint32_t tz_s[kTermLds];
    __shared__ S c_s[kTermLds];
    __shared__ double2 red[16];
    const uint32_t slot = find_slot(prefix, nslots, blockIdx.x);
    const SlotDesc sd = slots[slot];
    const SecTables* __restrict__ T = sd.t;
    const SecItem it = T->items[blockIdx.x - prefix[slot]];
    const S* __restrict__ coef = static_cast<const S*>(sd.coef ? sd.coef : T->tcoef);
    const S* __restrict__ psi = static_cast<const S*>(sd.psi);
    const uint32_t tid = threadIdx.x;
    const uint64_t Db = T->Db;
    const bool whole = it.g1 != it.g0 + 1;
    double acc = 0.0;
    for (uint32_t g = it.g0; g < it.g1; ++g) {
        const SecGroup& gr = T->groups[g];
        const uint32_t t0 = gr.t_first, nt = gr.t_count;
        const bool lds = nt <= kTermLds;
        if (lds) {
            __syncthreads();
            for (uint32_t k = tid; k < nt; k += kItemThreads) {
                tz_s[k] = (uint32_t)T->tz[t0 + k];
                c_s[k] = coef[t0 + k];
            }
            __syncthreads();
        }
        const uint32_t lb = gr.lb_len;
        const uint32_t p0 = whole ? 0u : it.p0, p1 = whole ? gr.la_len * lb : it.p1;
        const uint32_t x = (uint32_t)gr.x;
        double gacc = 0.0;
        for (uint32_t i0 = p0 + tid; i0 < p1; i0 += kUnroll * kItemThreads) {
            uint32_t j2[kUnroll];
            S v[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const uint32_t i = i0 + u * kItemThreads;
                j2[u] = 0;
                v[u] = real_amp<S>(0.0);
                if (i < p1) {
                    uint32_t ia, ib;
                    divmod_u(i, lb, gr.inv_lb, ia, ib);
                    const int2 pa = T->lists[gr.la_off + ia];
                    const int2 pb = T->lists[gr.lb_off + ib];
                    j2[u] = (uint32_t)(T->afull[pa.x] | T->bfull[pb.x]) ^ x;
                    v[u] = conj_mul(psi[(uint64_t)pa.x * Db + (uint64_t)pb.x], psi[(uint64_t)pa.y * Db + (uint64_t)pb.y]);
                }
            }
            S tr[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) tr[u] = real_amp<S>(0.0);
            for (uint32_t t = 0; t < nt; ++t) {
                const uint32_t z = lds ? tz_s[t] : (uint32_t)T->tz[t0 + t];
                const S c = lds ? c_s[t] : coef[t0 + t];
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) {
                    const uint32_t neg = (uint32_t)__popc(j2[u] & z) << 31;
                    add_flipped(tr[u], c, neg);
                }
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) gacc += re_mul(v[u], tr[u]);
        }
        acc += gr.weight * gacc;
    }
    const double2 tot = block_sum(make_double2(acc, 0.0), red);
    if (tid == 0) sd.part[blockIdx.x - prefix[slot]] = tot.x;
}

// ---- 5. per-request sum of the item partials in a fixed order ---------------------------
__global__ __launch_bounds__(256) void k_sec_sum(const SlotDesc* __restrict__ slots) {
    __shared__ double2 red[16];
    const SlotDesc sd = slots[blockIdx.x];
    const uint32_t n = sd.t->nparts;
    double acc = 0.0;
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) acc += sd.part[k];
    const double2 tot = block_sum(make_double2(acc, 0.0), red);
    if (threadIdx.x == 0) *sd.out = tot.x;
}

// ---- gradients ---------------------------------------------------------------------------
// sigma = H psi, output-centric: each determinant gathers from every group
// whose flip keeps it in the sector.
constexpr uint32_t kHpsiGroups = 256;  // group headers staged per chunk
constexpr uint32_t kHpsiTerms = 1024;  // terms staged per chunk (larger chunks read terms from memory)

// PER determinants per thread: each staged term is read once for all of them
// (batched launches use 4; a single request keeps 1 so it fills the chip).
template <typename S, int PER>
__global__ __launch_bounds__(256) void k_sec_hpsi(const SlotDesc* __restrict__ slots) {
    constexpr int kHpsiPer = PER;
    constexpr uint32_t kHpsiSpan = 256 * PER;  // determinants per block
    __shared__ uint4 hdr[kHpsiGroups];  // xa, xb, first term, term count
    __shared__ uint32_t gx[kHpsiGroups];
    __shared__ uint32_t tzs[kHpsiTerms];
    __shared__ S cfs[kHpsiTerms];
    const SlotDesc sd = slots[blockIdx.y];
    const SecTables* __restrict__ T = sd.t;
    if ((uint64_t)blockIdx.x * kHpsiSpan >= T->D) return;  // the whole block: a smaller request of the launch
    uint32_t sa[kHpsiPer], sb[kHpsiPer];
    uint32_t j[kHpsiPer];
    bool live[kHpsiPer];
    S sr[kHpsiPer];
#pragma unroll
    for (int q = 0; q < kHpsiPer; ++q) {
        const uint64_t r = (uint64_t)blockIdx.x * kHpsiSpan + (uint64_t)q * 256 + threadIdx.x;
        live[q] = r < T->D;  // every thread stays for the staging barriers
        const uint32_t ra = live[q] ? (uint32_t)(r / T->Db) : 0u, rb = live[q] ? (uint32_t)(r % T->Db) : 0u;
        sa[q] = T->astr[ra];
        sb[q] = T->bstr[rb];
        j[q] = (uint32_t)(T->afull[ra] | T->bfull[rb]);
        sr[q] = T->nrows && live[q] ? static_cast<const S*>(sd.sig)[r] : real_amp<S>(0.0);  // the rows' part
    }
    const S* __restrict__ coef = static_cast<const S*>(sd.coef ? sd.coef : T->tcoef);
    for (uint32_t c = 0; c < T->nhchunks; ++c) {
        const uint2 ch = T->hchunks[c];
        const uint32_t t0 = T->groups[ch.x].t_first;
        const uint32_t t1 = T->groups[ch.y - 1].t_first + T->groups[ch.y - 1].t_count;
        const bool tl = t1 - t0 <= kHpsiTerms;
        __syncthreads();
        for (uint32_t g = ch.x + threadIdx.x; g < ch.y; g += blockDim.x) {
            const SecGroup& gr = T->groups[g];
            hdr[g - ch.x] = make_uint4(gr.xa, gr.xb, gr.t_first, gr.t_count);
            gx[g - ch.x] = (uint32_t)gr.x;
        }
        if (tl)
            for (uint32_t t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
                tzs[t - t0] = (uint32_t)T->tz[t];
                cfs[t - t0] = coef[t];
            }
        __syncthreads();
        for (uint32_t g = 0; g < ch.y - ch.x; ++g) {
            const uint4 h = hdr[g];
            const int pa = __popc(h.x), pb = __popc(h.y);
            bool on[kHpsiPer];
            bool any = false;
#pragma unroll
            for (int q = 0; q < kHpsiPer; ++q) {
                on[q] = live[q] && 2 * __popc(sa[q] & h.x) == pa && 2 * __popc(sb[q] & h.y) == pb;
                any |= on[q];
            }
            if (!any) continue;
            uint32_t j2[kHpsiPer];
            S tr[kHpsiPer];
#pragma unroll
            for (int q = 0; q < kHpsiPer; ++q) {
                j2[q] = j[q] ^ gx[g];
                tr[q] = real_amp<S>(0.0);
            }
            for (uint32_t t = h.z; t < h.z + h.w; ++t) {
                const uint32_t z = tl ? tzs[t - t0] : (uint32_t)T->tz[t];
                const S cf = tl ? cfs[t - t0] : coef[t];
#pragma unroll
                for (int q = 0; q < kHpsiPer; ++q) {
                    const uint32_t neg = (uint32_t)__popc(j2[q] & z) << 31;
                    add_flipped(tr[q], cf, neg);
                }
            }
#pragma unroll
            for (int q = 0; q < kHpsiPer; ++q) {
                if (!on[q]) continue;
                const uint64_t r2 = (uint64_t)T->arank[sa[q] ^ h.x] * T->Db + (uint64_t)T->brank[sb[q] ^ h.y];
                add_mul(sr[q], tr[q], static_cast<const S*>(sd.psi)[r2]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kHpsiPer; ++q) {
        const uint64_t r = (uint64_t)blockIdx.x * kHpsiSpan + (uint64_t)q * 256 + threadIdx.x;
        if (live[q]) static_cast<S*>(sd.sig)[r] = sr[q];
    }
}

// Pool gradients: 2 Re<H psi|A_k psi> for the operators of one batch, one
// workgroup per operator (entries and lists of the pool's own tables).
template <typename S>
__global__ __launch_bounds__(256) void k_sec_pool(const SecTables* __restrict__ T, const SecEntry* __restrict__ pe,
                                                  const int2* __restrict__ plists, const PoolOp* __restrict__ ops,
                                                  const S* __restrict__ sig, const S* __restrict__ psi,
                                                  double* __restrict__ out) {
    __shared__ double2 red[16];
    const PoolOp op = ops[blockIdx.x];
    const uint64_t Db = T->Db;
    double acc = 0.0;
    for (uint32_t e = op.e0; e < op.e1; ++e) {
        const SecEntry en = pe[e];
        const uint32_t lb = en.lb_len, total = en.la_len * lb;
        for (uint32_t i = threadIdx.x; i < total; i += blockDim.x) {
            uint32_t ia, ib;
            divmod_u(i, lb, en.inv_lb, ia, ib);
            const int2 pa = plists[en.la_off + ia];
            const int2 pb = plists[en.lb_off + ib];
            const uint64_t r1 = (uint64_t)pa.x * Db + (uint64_t)pb.x, r2 = (uint64_t)pa.y * Db + (uint64_t)pb.y;
            const uint64_t j1 = T->afull[pa.x] | T->bfull[pb.x];
            acc += pair_overlap(en, j1, psi[r1], psi[r2], sig[r1], sig[r2]);
        }
    }
    const double2 tot = block_sum(make_double2(acc, 0.0), red);
    if (threadIdx.x == 0) out[blockIdx.x] = 2.0 * tot.x;
}

// ---- one launch per step (captured for the audit) -----------------------------------------
// The evaluation as a chain of kernels, one step (or generator) each over the
// whole grid: what qfe_template_graph_audit captures and checks node by node.
// No result comes from it: every evaluation takes the tile passes above.
// Pair t of a step is taken in entry order.
constexpr int kWideTPB = 256;

__device__ __forceinline__ bool step_pair(const SecTables* __restrict__ T, uint32_t e, uint32_t e_end, uint32_t t,
                                          uint32_t& entry, uint32_t& idx) {
    for (; e < e_end; ++e) {
        const uint32_t cnt = T->entries[e].la_len * T->entries[e].lb_len;
        if (t < cnt) {
            entry = e;
            idx = t;
            return true;
        }
        t -= cnt;
    }
    return false;
}

__device__ __forceinline__ void pair_of(const SecTables* __restrict__ T, const SecEntry& en, uint32_t i, uint64_t& r1,
                                        uint64_t& r2, uint64_t& j1) {
    uint32_t ia, ib;
    divmod_u(i, en.lb_len, en.inv_lb, ia, ib);
    const int2 pa = T->lists[en.la_off + ia];
    const int2 pb = T->lists[en.lb_off + ib];
    r1 = (uint64_t)pa.x * T->Db + (uint64_t)pb.x;
    r2 = (uint64_t)pa.y * T->Db + (uint64_t)pb.y;
    j1 = T->afull[pa.x] | T->bfull[pb.x];
}

// Rotate the pairs of step `step` by (c, s) (inverse: (c, -s)); `both` also rotates sigma.
template <typename S>
__global__ __launch_bounds__(kWideTPB) void k_sec_step(const SlotDesc* __restrict__ slots, uint32_t step, int inverse,
                                                       int both) {
    const SlotDesc sd = slots[0];
    const SecTables* __restrict__ T = sd.t;
    const SecStep st = T->steps[step];
    uint32_t e, i;
    if (!step_pair(T, st.e_first, st.e_first + st.e_count, blockIdx.x * kWideTPB + threadIdx.x, e, i)) return;
    const SecEntry& en = T->entries[e];
    const double2 cs = sd.cs[e];
    const double sn = inverse ? -cs.y : cs.y;
    uint64_t r1, r2, j1;
    pair_of(T, en, i, r1, r2, j1);
    S *psi = static_cast<S*>(sd.psi), *sig = static_cast<S*>(sd.sig);
    pair_rotate(psi, r1, r2, psi[r1], psi[r2], j1, en.x, en.z0, cs.x, sn, en.ulo, en.uhi);
    if (both) pair_rotate(sig, r1, r2, sig[r1], sig[r2], j1, en.x, en.z0, cs.x, sn, en.ulo, en.uhi);
}


// Generator with one step: its overlap and its un-rotation of psi and sigma
// read the same four old values of each pair, so one pass does both.
// partial[blockIdx.x] receives the block's overlap sum.
template <typename S>
__global__ __launch_bounds__(kWideTPB) void k_sec_genrev(const SlotDesc* __restrict__ slots, uint32_t step,
                                                         double* __restrict__ partial) {
    __shared__ double2 red[16];
    const SlotDesc sd = slots[0];
    const SecTables* __restrict__ T = sd.t;
    const SecStep st = T->steps[step];
    double acc = 0.0;
    uint32_t e, i;
    if (step_pair(T, st.e_first, st.e_first + st.e_count, blockIdx.x * kWideTPB + threadIdx.x, e, i)) {
        const SecEntry& en = T->entries[e];
        const double2 cs = sd.cs[e];
        uint64_t r1, r2, j1;
        pair_of(T, en, i, r1, r2, j1);
        S *psi = static_cast<S*>(sd.psi), *sig = static_cast<S*>(sd.sig);
        const S pa = psi[r1], pb = psi[r2], sa = sig[r1], sb = sig[r2];
        acc = pair_overlap(en, j1, pa, pb, sa, sb);
        pair_rotate(psi, r1, r2, pa, pb, j1, en.x, en.z0, cs.x, -cs.y, en.ulo, en.uhi);
        pair_rotate(sig, r1, r2, sa, sb, j1, en.x, en.z0, cs.x, -cs.y, en.ulo, en.uhi);
    }
    const double2 tot = block_sum(make_double2(acc, 0.0), red);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot.x;
}

// Generator with several steps: the overlap over all of its entries first
// (steps [s0, s1), their entries contiguous), un-rotation by k_sec_step after.
template <typename S>
__global__ __launch_bounds__(kWideTPB) void k_sec_genov(const SlotDesc* __restrict__ slots, uint32_t s0, uint32_t s1,
                                                        double* __restrict__ partial) {
    __shared__ double2 red[16];
    const SlotDesc sd = slots[0];
    const SecTables* __restrict__ T = sd.t;
    const uint32_t e0 = T->steps[s0].e_first, e1 = T->steps[s1 - 1].e_first + T->steps[s1 - 1].e_count;
    double acc = 0.0;
    uint32_t e, i;
    if (step_pair(T, e0, e1, blockIdx.x * kWideTPB + threadIdx.x, e, i)) {
        const SecEntry& en = T->entries[e];
        uint64_t r1, r2, j1;
        pair_of(T, en, i, r1, r2, j1);
        const S *psi = static_cast<const S*>(sd.psi), *sig = static_cast<const S*>(sd.sig);
        acc = pair_overlap(en, j1, psi[r1], psi[r2], sig[r1], sig[r2]);
    }
    const double2 tot = block_sum(make_double2(acc, 0.0), red);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot.x;
}

// Re<psi|sigma> block partials (the energy of the gradient path).
template <typename S>
__global__ __launch_bounds__(kWideTPB) void k_sec_edot(const SlotDesc* __restrict__ slots, double* __restrict__ partial) {
    __shared__ double2 red[16];
    const SlotDesc sd = slots[0];
    const uint64_t D = sd.t->D;
    const uint64_t r = (uint64_t)blockIdx.x * kWideTPB + threadIdx.x;
    double e = 0.0;
    if (r < D) e = re_dot(static_cast<const S*>(sd.psi)[r], static_cast<const S*>(sd.sig)[r]);
    const double2 tot = block_sum(make_double2(e, 0.0), red);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot.x;
}

// Fixed-order sums: out = sum of partial[seg[0]], gacc[k] = sum of partial[seg[k + 1]].
__global__ __launch_bounds__(kWideTPB) void k_sec_wsum(const SlotDesc* __restrict__ slots, const double* __restrict__ partial,
                                                       const uint2* __restrict__ seg, uint32_t nseg) {
    const uint32_t k = blockIdx.x * kWideTPB + threadIdx.x;
    if (k >= nseg) return;
    const uint2 sg = seg[k];
    double acc = 0.0;
    for (uint32_t q = 0; q < sg.y; ++q) acc += partial[sg.x + q];
    if (k == 0)
        *slots[0].out = acc;
    else
        slots[0].gacc[k - 1] = acc;
}

// The reference determinant (grid over the sector).
template <typename S>
__global__ __launch_bounds__(kWideTPB) void k_sec_ref(const SlotDesc* __restrict__ slots) {
    const SlotDesc sd = slots[0];
    const uint64_t r = (uint64_t)blockIdx.x * kWideTPB + threadIdx.x;
    if (r < sd.t->D) static_cast<S*>(sd.psi)[r] = real_amp<S>(r == sd.t->ref_rank ? 1.0 : 0.0);
}

// out[i] = sigma[rank[i]] (PQE residual amplitudes).
template <typename S>
__global__ void k_sec_gather(const SlotDesc* __restrict__ slots, const uint64_t* __restrict__ rank, uint64_t count,
                             double2* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) out[i] = to_complex(static_cast<const S*>(slots[0].sig)[rank[i]]);
}

// Scatter a sector state into a zeroed full state.
template <typename S>
__global__ void k_sector_scatter(const S* __restrict__ psi, uint64_t D, uint32_t Db, const uint64_t* __restrict__ afull,
                                 const uint64_t* __restrict__ bfull, double2* __restrict__ out) {
    const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= D) return;
    out[afull[r / Db] | bfull[r % Db]] = to_complex(psi[r]);
}

constexpr size_t kRowLdsMax = 64 << 10;   // dynamic LDS of a row workgroup
constexpr uint64_t kRowLists = 1ull << 22;  // flips over all rows of a template

// Serving lanes by size tier: a sector state of up to 40 KiB with its string
// tables, one that fits a workgroup's LDS, a larger one.
constexpr size_t kTier0Lds = 40 << 10;
constexpr uint32_t kTableLds = 1024;

// Tile shape.  Larger tiles take fewer passes but longer chains of steps per
// workgroup.  20-qubit residuals / 16-qubit gradient / 512 mixed energies / 128
// mixed gradients (us): 64 threads and 512 amplitudes 1489 / 621 / 8867 / 6602,
// 64 and 1024 1368 / 634 / 8165 / 5942, 128 and 1024 1247 / 556 / 7982 / 5620,
// 256 and 1024 1213 / 540 / 8841 / 6355, 128 and 2048 1274 / 610 / 7595 / 5377,
// 256 and 2048 1219 / 596 / 7531 / 5242: lone requests and batches differ.
constexpr int kTileThreads = 128;
constexpr uint64_t kTileAmps = 1024;  // amplitudes of a tile

// ---- host-side construction -------------------------------------------------------------

// The bits of one spin (2 i + parity) together, and apart again; norb <= 16.
inline uint32_t compress(uint64_t v, int parity, int norb) {
    uint32_t x = (uint32_t)(v >> parity) & 0x55555555u;
    x = (x | (x >> 1)) & 0x33333333u;
    x = (x | (x >> 2)) & 0x0f0f0f0fu;
    x = (x | (x >> 4)) & 0x00ff00ffu;
    return (x | (x >> 8)) & ((1u << norb) - 1u);
}
inline uint64_t spread(uint32_t v, int parity, int norb) {
    uint32_t x = v & ((1u << norb) - 1u);
    x = (x | (x << 8)) & 0x00ff00ffu;
    x = (x | (x << 4)) & 0x0f0f0f0fu;
    x = (x | (x << 2)) & 0x33333333u;
    x = (x | (x << 1)) & 0x55555555u;
    return (uint64_t)x << parity;
}
inline int popc32(uint32_t v) { return __builtin_popcount(v); }
inline int popc64(uint64_t v) { return __builtin_popcountll(v); }
inline double2 cplx_mul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
inline double cplx_abs(double2 a) { return std::hypot(a.x, a.y); }
inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct Space {
    int norb = 0;
    std::vector<uint32_t> str[2];
    std::vector<int32_t> rank[2];
    void build(int nb, int na_, int nb_) {
        norb = nb;
        const int ne[2] = {na_, nb_};
        for (int s = 0; s < 2; ++s) {
            str[s].clear();
            rank[s].assign((size_t)1 << norb, -1);
            for (uint32_t v = 0; v < (1u << norb); ++v)
                if (popc32(v) == ne[s]) {
                    rank[s][v] = (int32_t)str[s].size();
                    str[s].push_back(v);
                }
        }
    }
};

// Lists of (rank, partner rank) string pairs.  kind 0: (a & mask) == pattern;
// kind 1: popcount(a & mask) == popcount(mask) / 2; kind 2: kind 1 and
// (a & clear) == 0.  The partner is a ^ flip.
struct ListPool {
    std::vector<int2> pool;
    struct Key {
        int s, kind;
        uint32_t mask, pattern, flip;
        bool operator==(const Key& o) const {
            return s == o.s && kind == o.kind && mask == o.mask && pattern == o.pattern && flip == o.flip;
        }
    };
    struct Hash {
        size_t operator()(const Key& k) const {
            const uint64_t a = ((uint64_t)k.mask << 32) | k.pattern, b = ((uint64_t)k.flip << 8) | (uint32_t)(k.s * 4 + k.kind);
            return (size_t)((a * 0x9E3779B97F4A7C15ull) ^ ((b * 0xC2B2AE3D27D4EB4Full) >> 17));
        }
    };
    std::unordered_map<Key, std::pair<uint32_t, uint32_t>, Hash> index;
    std::pair<uint32_t, uint32_t> get(const Space& sp, int s, int kind, uint32_t mask, uint32_t pattern, uint32_t flip) {
        const Key key{s, kind, mask, pattern, flip};
        auto it = index.find(key);
        if (it != index.end()) return it->second;
        const uint32_t off = (uint32_t)pool.size();
        for (size_t r = 0; r < sp.str[s].size(); ++r) {
            const uint32_t a = sp.str[s][r];
            bool ok;
            if (kind == 0)
                ok = (a & mask) == pattern;
            else
                ok = 2 * popc32(a & mask) == popc32(mask) && (kind == 1 || (a & pattern) == 0);
            if (!ok) continue;
            const int32_t partner = sp.rank[s][a ^ flip];
            if (partner < 0) continue;
            pool.push_back(make_int2((int)r, partner));
        }
        auto v = std::make_pair(off, (uint32_t)pool.size() - off);
        index.emplace(key, v);
        return v;
    }
};

// Split generator k (terms [b, e)) into runs and entries; appends to steps
// and entries.  Used for ansatz generators and for pool operators.
int build_runs(const Space& sp, ListPool& lp, int norb, uint64_t lim, const qfe_pauli* terms, uint64_t b, uint64_t e,
               int32_t param, double scale, uint32_t gen, std::vector<SecStep>& steps, std::vector<SecEntry>& entries,
               const char* who) {
    std::vector<std::pair<uint64_t, double2>> A;
    std::vector<double2> kap;
    while (b < e) {
        const uint64_t x = terms[b].x, z0 = terms[b].z;
        uint64_t r = b;
        while (r < e && terms[r].x == x && (popc64(x & (terms[r].z ^ z0)) & 1) == 0) ++r;
        uint64_t m = x;
        for (uint64_t k = b; k < r; ++k) {
            if ((terms[k].x | terms[k].z) & ~lim) return fail(QFE_ERR_ARG, std::string(who) + ": term acts on a qubit out of range");
            m |= terms[k].z ^ z0;
        }
        if (popc64(m) > 20) return fail(QFE_ERR_ARG, std::string(who) + ": a run of commuting terms spans more than 20 qubits");
        double scale_abs = 0.0;
        kap.assign(r - b, make_double2(0.0, 0.0));
        for (uint64_t k = b; k < r; ++k) {
            // exp(theta * coeff * P) with coeff purely imaginary, as the full-space program applies it
            kap[k - b] = cplx_mul(make_double2(0.0, terms[k].coeff.im), make_double2(terms[k].phase.re, terms[k].phase.im));
            scale_abs += cplx_abs(kap[k - b]);
        }
        const double tol = 1e-13 * (scale_abs > 0 ? scale_abs : 1.0);
        // A(p) over the submasks p of m, ascending, where it is not zero
        A.clear();
        for (uint64_t p = 0;;) {
            double2 s = make_double2(0.0, 0.0);
            for (uint64_t k = b; k < r; ++k) {
                const double sg = (popc64(p & (terms[k].z ^ z0)) & 1) ? -1.0 : 1.0;
                s.x += sg * kap[k - b].x;
                s.y += sg * kap[k - b].y;
            }
            if (std::fabs(s.x) > tol || std::fabs(s.y) > tol || cplx_abs(s) > tol) A.emplace_back(p, s);
            if (p == m) break;
            p = (p - m) & m;  // the next submask
        }
        if (x == 0 && !A.empty()) return fail(QFE_ERR_ARG, std::string(who) + ": diagonal runs are not supported on the sector");
        SecStep st{};
        st.e_first = (uint32_t)entries.size();
        st.param = param;
        st.scale = scale;
        st.gen = gen;
        const double sx = (popc64(x & z0) & 1) ? -1.0 : 1.0;
        for (const auto& kv : A) {
            const uint64_t plo = kv.first, phi = plo ^ x;
            const auto it = std::lower_bound(A.begin(), A.end(), phi, [](const std::pair<uint64_t, double2>& u, uint64_t v) { return u.first < v; });
            if (it == A.end() || it->first != phi) return fail(QFE_ERR_ARG, std::string(who) + ": a run is not anti-Hermitian");
            if (plo > phi) continue;
            const double2 alo = kv.second, ahi = it->second;
            const double w = cplx_abs(alo);
            const double2 prod = cplx_mul(alo, ahi);
            if (std::fabs(sx * prod.x + w * w) > 1e-12 * w * w || std::fabs(prod.y) > 1e-12 * w * w)
                return fail(QFE_ERR_ARG, std::string(who) + ": a run is not anti-Hermitian");
            const uint32_t pa = compress(plo, 0, norb), pb = compress(plo, 1, norb);
            const uint32_t qa = compress(phi, 0, norb), qb = compress(phi, 1, norb);
            if (popc32(pa) != popc32(qa) || popc32(pb) != popc32(qb))
                return fail(QFE_ERR_ARG, std::string(who) + ": a run does not conserve the alpha and beta particle numbers");
            const uint32_t ma = compress(m, 0, norb), mb = compress(m, 1, norb);
            const uint32_t xa = compress(x, 0, norb), xb = compress(x, 1, norb);
            auto la = lp.get(sp, 0, 0, ma, pa, xa);
            auto lb = lp.get(sp, 1, 0, mb, pb, xb);
            if (!la.second || !lb.second) continue;
            SecEntry en{};
            en.x = x;
            en.z0 = z0;
            en.la_off = la.first;
            en.la_len = la.second;
            en.lb_off = lb.first;
            en.lb_len = lb.second;
            en.w = w;
            en.inv_lb = 1.0 / (double)lb.second;
            en.ulo = make_double2(alo.x / w, alo.y / w);
            en.uhi = make_double2(ahi.x / w, ahi.y / w);
            en.step = (uint32_t)steps.size();
            entries.push_back(en);
        }
        st.e_count = (uint32_t)entries.size() - st.e_first;
        if (st.e_count) steps.push_back(st);
        b = r;
    }
    return QFE_OK;
}

struct TileLaunch {  // host view of a pass: its grid and dynamic LDS
    uint32_t tiles, lds;
};

// Union-find over the strings of one spin.
struct Components {
    std::vector<uint32_t> parent, size;
    uint32_t largest = 1;
    explicit Components(uint32_t n) : parent(n), size(n, 1) {
        for (uint32_t i = 0; i < n; ++i) parent[i] = i;
    }
    uint32_t find(uint32_t v) {
        while (parent[v] != v) v = parent[v] = parent[parent[v]];
        return v;
    }
    void join(uint32_t a, uint32_t b) {
        a = find(a);
        b = find(b);
        if (a == b) return;
        if (size[a] < size[b]) std::swap(a, b);
        parent[b] = a;
        size[a] += size[b];
        largest = std::max(largest, size[a]);
    }
};

// Builds the component tiles of a template (see TileSeg).
struct TileBuilder {
    const Space& sp;
    const ListPool& lp;
    const std::vector<SecStep>& steps;
    const std::vector<SecEntry>& entries;
    std::vector<TileSeg> segs;
    std::vector<TileRun> fwd, rev;
    std::vector<TileLaunch> lfwd, lrev;
    std::vector<TileRec> recs;
    std::vector<uint32_t> tix, words;
    std::vector<uint2> tab, sum;
    std::vector<TileOut> outs;
    std::vector<TileWindow> wins;
    int norb;
    bool real;  // amplitudes are doubles
    // Partial sums of a window: 2 MB, which holds a whole sweep up to about 20
    // qubits; on larger sectors the bytes that a real request's two states save
    // against a complex one's (a complex one takes 1/16 on top), at most 256
    // MB.  All at once they took 15 GB at 32 qubits (8, 8) beside states of
    // 2.6 GB, and more than 2^32 numbers from 13.4 thousand generators on.
    const uint64_t most;

    TileBuilder(const Space& s, const ListPool& l, const std::vector<SecStep>& st, const std::vector<SecEntry>& en, size_t ngen,
                int norb_, bool real_)
        : sp(s), lp(l), steps(st), entries(en), norb(norb_), real(real_), most(window((uint64_t)s.str[0].size() * s.str[1].size(), real_)),
          seen(ngen + 1, 0) {}
    static uint64_t window(uint64_t D, bool real) {
        return std::min<uint64_t>(1u << 25, std::max<uint64_t>(1u << 18, real ? 2 * D : D / 4));
    }
    uint32_t parts = 0, peak = 0;            // of the open window, of all
    std::map<uint32_t, std::vector<uint2>> ranges;  // of the open window's outputs
    std::vector<char> seen;                  // outputs of earlier windows

    void join_step(uint32_t s, Components& a, Components& b) const {
        for (uint32_t e = steps[s].e_first; e < steps[s].e_first + steps[s].e_count; ++e) {
            for (uint32_t i = 0; i < entries[e].la_len; ++i) {
                const int2 v = lp.pool[entries[e].la_off + i];
                a.join((uint32_t)v.x, (uint32_t)v.y);
            }
            for (uint32_t i = 0; i < entries[e].lb_len; ++i) {
                const int2 v = lp.pool[entries[e].lb_off + i];
                b.join((uint32_t)v.x, (uint32_t)v.y);
            }
        }
    }

    // Whole components into blocks of at most `most` strings, largest
    // components first; ranks ascending within a block.
    static std::vector<std::vector<uint32_t>> pack(Components& c, uint32_t most) {
        const uint32_t n = (uint32_t)c.parent.size();
        std::vector<std::vector<uint32_t>> comp(n), blocks;
        for (uint32_t i = 0; i < n; ++i) comp[c.find(i)].push_back(i);
        std::vector<uint32_t> order;
        for (uint32_t i = 0; i < n; ++i)
            if (!comp[i].empty()) order.push_back(i);
        std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) {
            return comp[x].size() != comp[y].size() ? comp[x].size() > comp[y].size() : comp[x][0] < comp[y][0];
        });
        std::vector<size_t> open;  // blocks with room
        for (uint32_t k : order) {
            size_t at = blocks.size();
            for (size_t i = 0; i < open.size(); ++i)
                if (blocks[open[i]].size() + comp[k].size() <= most) {
                    at = open[i];
                    break;
                }
            if (at == blocks.size()) {
                blocks.emplace_back();
                open.push_back(at);
                if (open.size() > 8) open.erase(open.begin());
            }
            blocks[at].insert(blocks[at].end(), comp[k].begin(), comp[k].end());
        }
        for (auto& b : blocks) std::sort(b.begin(), b.end());
        return blocks;
    }

    // One spin of a segment: blocks, permuted ranks and list words.
    struct Side {
        uint32_t nblk = 0, blk = 0, perm = 0, wb = 0, tab = 0;
        std::vector<uint32_t> len, nword;                     // strings and words of each block
        std::map<std::pair<uint32_t, uint32_t>, uint32_t> id;  // (list offset, sign mask) -> list
    };
    Side build_side(int s, Components& c, uint32_t most, uint32_t s0, uint32_t s1) {
        Side d;
        const auto blocks = pack(c, most);
        d.nblk = (uint32_t)blocks.size();
        std::vector<uint32_t> where(c.parent.size()), local(c.parent.size());
        d.blk = (uint32_t)tix.size();
        uint32_t at = 0;
        for (const auto& b : blocks) {
            tix.push_back(at);
            at += (uint32_t)b.size();
            d.len.push_back((uint32_t)b.size());
        }
        tix.push_back(at);
        d.perm = (uint32_t)tix.size();
        for (uint32_t k = 0; k < d.nblk; ++k)
            for (uint32_t i = 0; i < blocks[k].size(); ++i) {
                tix.push_back(blocks[k][i]);
                where[blocks[k][i]] = k;
                local[blocks[k][i]] = i;
            }
        struct List {
            uint32_t off, len, z;
        };
        std::vector<List> lists;
        for (uint32_t e = steps_begin(s0); e < steps_begin(s1); ++e) {
            const SecEntry& en = entries[e];
            const uint32_t off = s ? en.lb_off : en.la_off, len = s ? en.lb_len : en.la_len;
            const uint32_t z = compress(en.z0, s, norb);
            if (d.id.emplace(std::make_pair(off, z), (uint32_t)lists.size()).second) lists.push_back({off, len, z});
        }
        std::vector<std::vector<uint32_t>> bw(d.nblk);
        d.tab = (uint32_t)tab.size();
        tab.resize(tab.size() + lists.size() * d.nblk, make_uint2(0, 0));
        for (size_t l = 0; l < lists.size(); ++l) {
            uint2* row = tab.data() + d.tab + l * d.nblk;
            for (uint32_t k = 0; k < d.nblk; ++k) row[k].x = (uint32_t)bw[k].size();
            for (uint32_t i = 0; i < lists[l].len; ++i) {
                const int2 v = lp.pool[lists[l].off + i];
                const uint32_t k = where[v.x];
                const uint32_t p1 = popc32(sp.str[s][v.x] & lists[l].z) & 1, p2 = popc32(sp.str[s][v.y] & lists[l].z) & 1;
                bw[k].push_back(local[v.x] | (local[v.y] << kWordBits) | (p1 << 30) | (p2 << 31));
                ++row[k].y;
            }
        }
        d.wb = (uint32_t)tix.size();
        for (uint32_t k = 0; k < d.nblk; ++k) {
            tix.push_back((uint32_t)words.size());
            words.insert(words.end(), bw[k].begin(), bw[k].end());
            d.nword.push_back((uint32_t)bw[k].size());
        }
        tix.push_back((uint32_t)words.size());
        return d;
    }
    uint32_t steps_begin(uint32_t s) const { return s < steps.size() ? steps[s].e_first : (uint32_t)entries.size(); }

    void add_run(std::vector<TileRun>& runs, std::vector<TileLaunch>& launches, const Side& a, const Side& b, uint32_t seg,
                 uint32_t rec0, int states) {
        TileRun r{seg, rec0, (uint32_t)recs.size() - rec0, parts};
        uint32_t lds = 0;
        const size_t amp = real ? sizeof(double) : sizeof(double2);
        const uint32_t chunk = std::min(r.nrec, kRecChunk) * (uint32_t)(real ? sizeof(LdsRec<double>) : sizeof(LdsRec<double2>));
        for (uint32_t i = 0; i < a.nblk; ++i)
            for (uint32_t j = 0; j < b.nblk; ++j) {
                const uint32_t w = a.nword[i] + b.nword[j];
                const uint32_t amps = (uint32_t)(((size_t)a.len[i] * b.len[j] * states * amp + 15) & ~(size_t)15);
                lds = std::max(lds, amps + chunk + (w <= kTileWordsLds ? 4 * w : 0u));
            }
        runs.push_back(r);
        launches.push_back(TileLaunch{a.nblk * b.nblk, lds});
    }

    // Steps [s0, s1) as one segment.  gens: (first step, last step) of its
    // generators, last generator first, for the reverse sweep.
    void add_segment(uint32_t s0, uint32_t s1, Components& ca, Components& cb) {
        uint32_t la = ca.largest, lb = cb.largest;
        const uint32_t Da = (uint32_t)ca.parent.size(), Db = (uint32_t)cb.parent.size();
        for (;;) {  // fill the tile: beta first, whose ranks are contiguous in memory
            if (lb < Db && (uint64_t)la * lb * 2 <= kTileAmps)
                lb = std::min(lb * 2, Db);
            else if (la < Da && (uint64_t)la * lb * 2 <= kTileAmps)
                la = std::min(la * 2, Da);
            else
                break;
        }
        side[0].push_back(build_side(0, ca, la, s0, s1));
        side[1].push_back(build_side(1, cb, lb, s0, s1));
        const Side &a = side[0].back(), &b = side[1].back();
        segs.push_back(TileSeg{a.nblk, b.nblk, a.blk, b.blk, a.perm, b.perm, a.wb, b.wb, a.tab, b.tab});
        seg_steps.push_back({s0, s1});
        const uint32_t rec0 = (uint32_t)recs.size();
        for (uint32_t s = s0; s < s1; ++s) add_step(segs.size() - 1, s, kRecRot);
        add_run(fwd, lfwd, a, b, (uint32_t)segs.size() - 1, rec0, 1);
    }
    std::vector<Side> side[2];
    std::vector<std::pair<uint32_t, uint32_t>> seg_steps;

    void add_step(size_t seg, uint32_t s, uint32_t flags) {
        for (uint32_t e = steps[s].e_first; e < steps[s].e_first + steps[s].e_count; ++e) {
            const SecEntry& en = entries[e];
            TileRec r{};
            r.w = en.w;
            r.ulo = en.ulo;
            r.uhi = en.uhi;
            r.entry = e;
            r.alist = side[0][seg].id.at({en.la_off, compress(en.z0, 0, norb)});
            r.blist = side[1][seg].id.at({en.lb_off, compress(en.z0, 1, norb)});
            r.flags = flags | (e + 1 == steps[s].e_first + steps[s].e_count ? kRecStepEnd : 0u);
            recs.push_back(r);
        }
    }

    // Partial sums of one output of a pass over a segment.
    uint32_t per_out(uint32_t seg) const { return side[0][seg].nblk * side[1][seg].nblk * (kTileThreads / 64); }

    // One reverse-sweep pass over a segment: its records are recs[rec0..]; the
    // generators it completes are `gens` in order.
    void add_reverse(uint32_t seg, uint32_t rec0, const std::vector<uint32_t>& gens) {
        const uint32_t per = per_out(seg);
        if (parts && parts + (uint64_t)per * gens.size() > most) close_window();
        add_run(rev, lrev, side[0][seg], side[1][seg], seg, rec0, 2);
        auto add = [&](uint32_t out) {
            ranges[out].push_back(make_uint2(parts, per));
            parts += per;
        };
        if (rev.size() == 1) add(0);
        for (uint32_t g : gens) add(g + 1);
        peak = std::max(peak, parts);
    }
    void close_window() {
        const uint32_t o0 = (uint32_t)outs.size();
        for (const auto& r : ranges) {
            const uint32_t r0 = (uint32_t)sum.size();
            sum.insert(sum.end(), r.second.begin(), r.second.end());
            outs.push_back(TileOut{r.first, r0, (uint32_t)sum.size(), (uint32_t)seen[r.first]});
            seen[r.first] = 1;
        }
        wins.push_back(TileWindow{(uint32_t)rev.size() - 1, o0, (uint32_t)outs.size(), 0});
        ranges.clear();
        parts = 0;
    }

    void build(const std::vector<uint32_t>& gen_step) {
        const uint32_t ngen = (uint32_t)gen_step.size() - 1;
        const uint32_t Da = (uint32_t)sp.str[0].size(), Db = (uint32_t)sp.str[1].size();
        struct Part {  // generators [g0, g1) in one segment, or a generator too wide for one
            uint32_t g0, g1, seg0, seg1;
        };
        std::vector<Part> plan;
        // grow segments by generators (by steps inside a generator that is too wide)
        auto grow = [&](uint32_t u0, uint32_t u1, auto first_step) {
            uint32_t u = u0;
            while (u < u1) {
                Components ca(Da), cb(Db);
                uint32_t v = u;
                while (v < u1) {
                    Components ta = ca, tb = cb;
                    for (uint32_t s = first_step(v); s < first_step(v + 1); ++s) join_step(s, ta, tb);
                    if (v > u && (uint64_t)ta.largest * tb.largest > kTileAmps) break;
                    const bool wide = (uint64_t)ta.largest * tb.largest > kTileAmps;
                    ca = std::move(ta);
                    cb = std::move(tb);
                    ++v;
                    if (wide) break;
                }
                if ((uint64_t)ca.largest * cb.largest > kTileAmps) return std::make_pair(u, v);
                add_segment(first_step(u), first_step(v), ca, cb);
                u = v;
                if (on_segment) on_segment(v);
            }
            return std::make_pair(u1, u1);
        };
        uint32_t g = 0;
        while (g < ngen) {
            uint32_t start = g;
            on_segment = [&](uint32_t v) {
                plan.push_back({start, v, (uint32_t)segs.size() - 1, (uint32_t)segs.size()});
                start = v;
            };
            const auto stop = grow(g, ngen, [&](uint32_t k) { return gen_step[k]; });
            on_segment = nullptr;
            g = stop.first;
            if (g >= ngen) break;
            const uint32_t seg0 = (uint32_t)segs.size();  // generator g alone is too wide: segments of its steps
            grow(gen_step[g], gen_step[g + 1], [](uint32_t k) { return k; });
            plan.push_back({g, g + 1, seg0, (uint32_t)segs.size()});
            ++g;
        }
        if (segs.empty()) {  // no generator: one pass still writes the reference and one adds up the energy
            Components ca(Da), cb(Db);
            add_segment((uint32_t)steps.size(), (uint32_t)steps.size(), ca, cb);
            plan.push_back({0, 0, 0, 1});
        }
        for (size_t i = plan.size(); i-- > 0;) {
            const Part& p = plan[i];
            if (p.seg1 == p.seg0 + 1) {
                uint32_t rec0 = (uint32_t)recs.size();
                std::vector<uint32_t> gens;
                for (uint32_t k = p.g1; k-- > p.g0;) {
                    const uint32_t s0 = gen_step[k], s1 = gen_step[k + 1];
                    if (s0 == s1) continue;
                    // a pass's own sums (the first has the energy's too) fit a window
                    if (!gens.empty() && (gens.size() + 1 + rev.empty()) * (uint64_t)per_out(p.seg0) > most) {
                        add_reverse(p.seg0, rec0, gens);
                        rec0 = (uint32_t)recs.size();
                        gens.clear();
                    }
                    gens.push_back(k);
                    if (s1 == s0 + 1) {  // one step: a pair's four old values give its overlap and both un-rotated pairs
                        add_step(p.seg0, s0, kRecRot | kRecOv);
                        recs.back().flags |= kRecGenEnd;
                        continue;
                    }
                    const size_t first = recs.size();
                    for (uint32_t s = s0; s < s1; ++s) add_step(p.seg0, s, kRecOv);
                    for (size_t r = first; r < recs.size(); ++r) recs[r].flags &= ~kRecStepEnd;
                    recs.back().flags |= kRecGenEnd | kRecStepEnd;
                    for (uint32_t s = s1; s-- > s0;) add_step(p.seg0, s, kRecRot);
                }
                add_reverse(p.seg0, rec0, gens);
                continue;
            }
            // a generator over several segments: its whole overlap before any un-rotation
            for (uint32_t sgm = p.seg0; sgm < p.seg1; ++sgm) {
                const uint32_t rec0 = (uint32_t)recs.size();
                for (uint32_t s = seg_steps[sgm].first; s < seg_steps[sgm].second; ++s) add_step(sgm, s, kRecOv);
                recs.back().flags |= kRecGenEnd;
                add_reverse(sgm, rec0, {p.g0});
            }
            for (uint32_t sgm = p.seg1; sgm-- > p.seg0;) {
                const uint32_t rec0 = (uint32_t)recs.size();
                for (uint32_t s = seg_steps[sgm].second; s-- > seg_steps[sgm].first;) add_step(sgm, s, kRecRot);
                add_reverse(sgm, rec0, {});
            }
        }
        for (uint32_t k = 0; k < seen.size(); ++k)
            if (!seen[k]) (void)ranges[k];  // a generator without pairs: a sum of nothing
        close_window();
    }
    std::function<void(uint32_t)> on_segment;
};

// Builds the row tables of a real template (see k_sec_rows).
struct RowBuilder {
    const Space& sp;
    int norb;
    std::vector<uint32_t> chunk_off{0}, pos_cell, amu, am{0}, bmu, bm{0}, mmask, b1, pair_off{0}, words, fb_mask, fa_mask;
    std::vector<uint4> chunks;
    std::vector<uint2> b2;
    std::vector<RowFlip> flips;
    std::vector<RowPair> pairs;
    std::vector<uint2> mrow;                          // terms of every merged number: [x, x + y) of
    std::vector<std::pair<uint32_t, double>> mterm;   // (term, sign)
    uint32_t nb1 = 0, nb2 = 0, nwords = 0, nfa = 0, nfb = 0, gbase = 0;

    struct Term {
        uint32_t za, zb, k;
    };
    struct Group {
        uint64_t x;
        uint32_t xa, xb;
        std::vector<Term> terms;
    };
    explicit RowBuilder(const Space& s, int norb_) : sp(s), norb(norb_) {}

    static uint32_t parity(uint32_t v) { return (uint32_t)__builtin_popcount(v) & 1u; }
    // Qubits strictly between the first and second, third and fourth ... set bits of x.
    static uint64_t between(uint64_t x) {
        uint64_t r = 0;
        while (x) {
            const int lo = __builtin_ctzll(x);
            x &= x - 1;
            if (!x) break;
            const int hi = __builtin_ctzll(x);
            x &= x - 1;
            r |= ((1ull << hi) - 1ull) & ~((2ull << lo) - 1ull);
        }
        return r;
    }
    // Whether a group has the form the rows take: flips of one spin (or none)
    // always; flips of both spins when all its terms share the sign mask
    // outside x and it is the product of the two flips' Jordan-Wigner strings.
    bool fits(const Group& g) const {
        if (!g.xa && !g.xb) return cells_of(g) <= kRowCells;
        if (!g.xa || !g.xb) return popc32(g.xa | g.xb) <= 8 && g.terms.size() <= 256;
        if (popc32(g.xa) > 4 || popc32(g.xb) > 4) return false;
        const uint64_t j = (between(spread(g.xa, 0, norb)) ^ between(spread(g.xb, 1, norb))) & ~g.x;
        const uint32_t ja = compress(j, 0, norb), jb = compress(j, 1, norb);
        for (const Term& t : g.terms)
            if ((t.za & ~g.xa) != ja || (t.zb & ~g.xb) != jb) return false;
        return true;
    }
    static size_t cells_of(const Group& g) {
        std::vector<uint32_t> m;
        for (const Term& t : g.terms) m.push_back(t.zb);
        std::sort(m.begin(), m.end());
        return (size_t)(std::unique(m.begin(), m.end()) - m.begin());
    }
    static std::vector<uint32_t> patterns(uint32_t x) {  // half of the bits of x set, ascending
        std::vector<uint32_t> out;
        for (uint32_t p = 0;; p = (p - x) & x) {
            if (2 * popc32(p) == popc32(x)) out.push_back(p);
            if (p == x) break;
        }
        return out;
    }
    static bool flips_in(uint32_t v, uint32_t x) { return 2 * popc32(v & x) == popc32(x); }

    // A flip of one spin by the pattern of the partner's flipped bits: what
    // belongs to each (cells of a group, or numbers first, first + 1, ...).
    struct Flip {
        uint32_t x, first;
        std::vector<uint32_t> pat;
        std::vector<std::pair<uint32_t, uint32_t>> cells;  // (first cell, cells)
        size_t at(uint32_t to) const { return (size_t)(std::lower_bound(pat.begin(), pat.end(), to & x) - pat.begin()); }
    };

    // Cells of a group for every pattern of the flipped bits of spin s: terms
    // merged by the beta mask, then by the alpha mask.
    Flip add_cells(const Group& g, int s, std::vector<uint32_t>& mu, std::vector<uint32_t>& m) {
        Flip f{s ? g.xb : g.xa, 0, patterns(s ? g.xb : g.xa), {}};
        // masks outside the flipped bits, which the pattern does not change
        struct Key {
            uint32_t b, a, t;
        };
        std::vector<Key> key;
        for (uint32_t t = 0; t < g.terms.size(); ++t)
            key.push_back(s ? Key{g.terms[t].zb & ~g.xb, g.terms[t].za, t} : Key{g.terms[t].zb, g.terms[t].za & ~g.xa, t});
        std::sort(key.begin(), key.end(), [](const Key& u, const Key& v) { return u.b != v.b ? u.b < v.b : u.a != v.a ? u.a < v.a : u.t < v.t; });
        for (uint32_t p : f.pat) {
            const uint32_t c0 = (uint32_t)mu.size();
            for (size_t i = 0; i < key.size(); ++i) {
                const bool cell = i == 0 || key[i].b != key[i - 1].b;
                if (cell) {
                    if (i) m.push_back((uint32_t)mrow.size());
                    mu.push_back(key[i].b);
                }
                if (cell || key[i].a != key[i - 1].a) {
                    mmask.push_back(key[i].a);
                    mrow.push_back(make_uint2((uint32_t)mterm.size(), 0));
                }
                const Term& t = g.terms[key[i].t];
                mterm.push_back({t.k, parity(p & (s ? t.zb : t.za)) ? -1.0 : 1.0});
                ++mrow.back().y;
            }
            if (!key.empty()) m.push_back((uint32_t)mrow.size());
            f.cells.push_back({c0, (uint32_t)mu.size() - c0});
        }
        return f;
    }

    // LDS of a row workgroup.
    size_t lds() const {
        const size_t Db = sp.str[1].size(), nb = bmu.size();
        const size_t a = kRowCells * 12 + 16, ab = nwords ? 32 * (Db + nfb + 1) : 0;
        return ((Db + nb + 2) / 2) * 16 + std::max(a, ab);
    }

    void build(const std::vector<Group>& groups) {
        const auto &as = sp.str[0], &bs = sp.str[1];
        const uint32_t Da = (uint32_t)as.size(), Db = (uint32_t)bs.size();
        auto rank = [&](int s, uint32_t v) { return (uint32_t)sp.rank[s][v]; };
        // alpha flips and the diagonal
        std::vector<Flip> af, bf;
        for (const Group& g : groups)
            if (!g.xb) af.push_back(add_cells(g, 0, amu, am));
        for (uint32_t ra = 0; ra < Da; ++ra) {
            uint4 cd = make_uint4((uint32_t)flips.size(), 0, (uint32_t)pos_cell.size(), 0);
            auto close = [&]() {
                if (flips.size() == cd.x) return;
                while ((flips.size() - cd.x) % kRowUnroll) flips.push_back(RowFlip{ra, 0, 0, 0});
                cd.y = (uint32_t)flips.size() - cd.x;
                chunks.push_back(cd);
                cd = make_uint4((uint32_t)flips.size(), 0, (uint32_t)pos_cell.size(), 0);
            };
            for (const Flip& f : af) {
                if (!flips_in(as[ra], f.x)) continue;
                const uint32_t to = as[ra] ^ f.x;
                const auto c = f.cells[f.at(to)];
                if (cd.w + c.second > kRowCells) close();
                flips.push_back(RowFlip{rank(0, to), c.first, c.second, cd.w});
                for (uint32_t k = 0; k < c.second; ++k) pos_cell.push_back(c.first + k);
                cd.w += c.second;
            }
            close();
            chunk_off.push_back((uint32_t)chunks.size());
        }
        // beta flips
        bm[0] = (uint32_t)mrow.size();
        for (const Group& g : groups)
            if (!g.xa && g.xb) bf.push_back(add_cells(g, 1, bmu, bm));
        std::vector<std::vector<uint32_t>> l1(Db);
        std::vector<std::vector<uint2>> l2(Db);
        for (uint32_t rb = 0; rb < Db; ++rb) {
            for (const Flip& f : bf) {
                if (!flips_in(bs[rb], f.x)) continue;
                const uint32_t to = bs[rb] ^ f.x;
                const auto c = f.cells[f.at(to)];
                if (c.second == 1)
                    l1[rb].push_back(rank(1, to) | (c.first << 14) | (parity(bs[rb] & bmu[c.first]) << 31));
                else
                    l2[rb].push_back(make_uint2(rank(1, to), c.first | (c.second << 20)));
            }
            nb1 = std::max(nb1, (uint32_t)l1[rb].size());
            nb2 = std::max(nb2, (uint32_t)l2[rb].size());
        }
        // padding words point at a cell (below: a flip) that is zero
        nb1 = (nb1 + kRowUnroll - 1) / kRowUnroll * kRowUnroll;
        b1.assign((size_t)nb1 * Db, (uint32_t)bmu.size() << 14);
        b2.assign((size_t)nb2 * Db, make_uint2(0, 0));
        for (uint32_t rb = 0; rb < Db; ++rb) {
            for (size_t k = 0; k < l1[rb].size(); ++k) b1[k * Db + rb] = l1[rb][k];
            for (size_t k = 0; k < l2[rb].size(); ++k) b2[k * Db + rb] = l2[rb][k];
        }
        // both: flips (mask, pattern of the partner) of each spin, and the table over them
        auto flips_of = [&](int s, uint32_t& count, std::vector<uint32_t>& mask) {
            std::vector<uint32_t> xs;
            for (const Group& g : groups)
                if (g.xa && g.xb) xs.push_back(s ? g.xb : g.xa);
            std::sort(xs.begin(), xs.end());
            xs.erase(std::unique(xs.begin(), xs.end()), xs.end());
            std::vector<Flip> out;
            for (uint32_t x : xs) {
                out.push_back(Flip{x, count, patterns(x), {}});
                count += (uint32_t)out.back().pat.size();
                mask.resize(count, compress(between(spread(x, s, norb)), 1 - s, norb));
            }
            return out;
        };
        const std::vector<Flip> fa = flips_of(0, nfa, fa_mask), fb = flips_of(1, nfb, fb_mask);
        auto find = [](const std::vector<Flip>& f, uint32_t x) -> const Flip& {
            return *std::lower_bound(f.begin(), f.end(), x, [](const Flip& u, uint32_t v) { return u.x < v; });
        };
        gbase = (uint32_t)mrow.size();
        mrow.resize(mrow.size() + (size_t)nfa * nfb, make_uint2(0, 0));
        mmask.resize(mrow.size(), 0u);
        for (const Group& g : groups) {
            if (!g.xa || !g.xb) continue;
            const Flip &u = find(fa, g.xa), &v = find(fb, g.xb);
            const uint32_t jba = compress(between(spread(g.xb, 1, norb)), 0, norb);
            const uint32_t jab = compress(between(spread(g.xa, 0, norb)), 1, norb);
            for (size_t i = 0; i < u.pat.size(); ++i)
                for (size_t k = 0; k < v.pat.size(); ++k) {
                    const uint32_t pa = u.pat[i], pb = v.pat[k];
                    // the strings' bits on the flipped qubits of the other spin depend on the patterns alone
                    const uint32_t c = parity((g.xa ^ pa) & jba) ^ parity(pb & jab);
                    mrow[gbase + (u.first + i) * nfb + v.first + k] = make_uint2((uint32_t)mterm.size(), (uint32_t)g.terms.size());
                    for (const Term& t : g.terms) mterm.push_back({t.k, (c ^ parity(pa & t.za) ^ parity(pb & t.zb)) ? -1.0 : 1.0});
                }
        }
        std::vector<uint32_t> ja, jb;  // a flip's own string
        for (const Flip& f : fa) ja.push_back(compress(between(spread(f.x, 0, norb)), 0, norb) & ~f.x);
        for (const Flip& f : fb) jb.push_back(compress(between(spread(f.x, 1, norb)), 1, norb) & ~f.x);
        for (uint32_t ra = 0; ra < Da; ++ra) {
            for (size_t i = 0; i < fa.size(); ++i) {
                if (!flips_in(as[ra], fa[i].x)) continue;
                const uint32_t to = as[ra] ^ fa[i].x;
                pairs.push_back(RowPair{rank(0, to), fa[i].first + (uint32_t)fa[i].at(to), parity(as[ra] & ja[i]) << 31, 0});
            }
            while ((pairs.size() - pair_off.back()) % 4) pairs.push_back(RowPair{kRowNone, 0, 0, 0});
            pair_off.push_back((uint32_t)pairs.size());
        }
        std::vector<std::vector<uint32_t>> lw(Db);
        for (uint32_t rb = 0; rb < Db; ++rb) {
            for (size_t i = 0; i < fb.size(); ++i) {
                if (!flips_in(bs[rb], fb[i].x)) continue;
                const uint32_t to = bs[rb] ^ fb[i].x;
                lw[rb].push_back(rank(1, to) | ((fb[i].first + (uint32_t)fb[i].at(to)) << 14) | (parity(bs[rb] & jb[i]) << 31));
            }
            nwords = std::max(nwords, (uint32_t)lw[rb].size());
        }
        nwords = (nwords + 3) / 4 * 4;
        words.assign((size_t)nwords * Db, nfb << 14);
        for (uint32_t rb = 0; rb < Db; ++rb)
            for (size_t k = 0; k < lw[rb].size(); ++k) words[k * Db + rb] = lw[rb][k];
        if (!nwords) pair_off.assign(Da + 1, 0);
    }
};

// Packs host arrays into one device allocation at 256-byte offsets.
struct Packer {
    struct Piece {
        const void* src;
        size_t bytes, off;
    };
    std::vector<Piece> pieces;
    size_t total;
    explicit Packer(size_t head) : total(align256(head)) {}
    size_t add(const void* src, size_t bytes) {
        pieces.push_back({src, bytes, total});
        total += align256(bytes ? bytes : 1);
        return pieces.size() - 1;
    }
    void fill(char* img) const {
        for (const auto& p : pieces)
            if (p.bytes) std::memcpy(img + p.off, p.src, p.bytes);
    }
};

}  // namespace
}  // namespace qfe

using namespace qfe;

struct qfe_template_s {
    int n = 0, norb = 0;
    uint64_t D = 0;
    uint32_t Da = 0, Db = 0;
    uint64_t nparam = 0, ninputs = 0, ngen = 0;
    std::vector<int32_t> gparam;
    std::vector<double> gscale;
    uint32_t nterms = 0, nentries = 0, nitems = 0, nrows = 0, nm = 0;
    size_t row_lds = 0;    // dynamic LDS of a row workgroup
    bool has_map = false;
    bool real = false;     // scalar type of the state and the coefficients (see umul)
    size_t amp() const { return real ? sizeof(double) : sizeof(double2); }
    uint64_t cost = 0;     // work estimate for ordering slots in a launch
    int tier = 2;          // ansatz launch shape
    std::vector<TileLaunch> fwd, rev;  // tile passes of the ansatz and of the reverse sweep
    std::vector<TileWindow> wins;      // windows of the reverse sweep's partial sums
    Space sp;              // host copy of the string space (pool operators)
    void* dev = nullptr;   // all tables
    SecTables* dt = nullptr;
    const uint64_t* afull = nullptr;
    const uint64_t* bfull = nullptr;
    // per-request device bytes: psi, coef, cs, part (energy); + sig, gacc (gradient)
    size_t off_psi = 0, off_coef = 0, off_cs = 0, off_part = 0, off_sig = 0, off_gacc = 0, off_gpart = 0, off_hm = 0;
    size_t work_bytes = 0, grad_bytes = 0, io_count = 0, request_bytes = 0, grad_request_bytes = 0;
    size_t grad_least_bytes = 0;  // without the partial sums, which no budget is refused for
    void* arena = nullptr;  // single-request arena: [desc][out][prefix][io][work, with gradient parts from the first call that has them]
    size_t arena_bytes = 0;
    // step-by-step sequence (large sectors, for the audit only, which allocates
    // it): host step structure and device [segments (uint2 x (ngen + 1))][block partials]
    std::vector<uint32_t> h_gen_step, step_pairs;
    std::vector<uint2> wide_seg;  // (first partial, count): the energy, then generator k
    uint32_t wide_parts = 0;
    void* wide = nullptr;
    // captured single-request sequences (energy, gradient) and their pinned
    // host block: [request head as uploaded][energy][generator overlaps]
    hipGraph_t graph[2] = {nullptr, nullptr};
    hipGraphExec_t gexec[2] = {nullptr, nullptr};
    void* gpin = nullptr;
    // host-side audit of each captured sequence: nodes, kernel nodes, kernel
    // nodes whose arguments were compared, memcpy nodes whose parameters were compared
    uint64_t audit[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
};

namespace qfe {
namespace {

// Row lists are worth their tables unless the sector is enormous.
bool rows_worth(const RowBuilder& b, const std::vector<RowBuilder::Group>& groups) {
    if (groups.empty() || b.sp.str[1].size() > (1u << 14)) return false;
    uint64_t flips = 0;
    for (const auto& g : groups) flips += g.xb ? 0 : b.sp.str[0].size();
    return flips <= kRowLists;
}

int template_build(qfe_template t, int n, uint64_t ref, const qfe_pauli* gen_terms, const uint64_t* gen_off, uint64_t ngen,
                   const int32_t* gen_param, const double* gen_scale, uint64_t nparam, const qfe_pauli* ham, uint64_t nham,
                   const uint64_t* map_off, const uint32_t* map_idx, const qfe_c64* map_val, uint64_t ninputs) {
    if (n < 2 || n > 32 || (n & 1)) return fail(QFE_ERR_ARG, "qfe_template_create: nqubit must be even and in [2, 32]");
    const int norb = n / 2;
    const uint64_t lim = (1ull << n) - 1ull;
    if (ref & ~lim) return fail(QFE_ERR_ARG, "qfe_template_create: reference index out of range");
    const uint32_t refa = compress(ref, 0, norb), refb = compress(ref, 1, norb);
    Space& sp = t->sp;
    sp.build(norb, popc32(refa), popc32(refb));
    ListPool lp;
    t->n = n;
    t->norb = norb;
    t->Da = (uint32_t)sp.str[0].size();
    t->Db = (uint32_t)sp.str[1].size();
    t->D = (uint64_t)t->Da * t->Db;
    t->nparam = nparam;
    t->ninputs = ninputs;
    t->ngen = ngen;
    t->gparam.assign(gen_param, gen_param + ngen);
    t->gscale.assign(gen_scale, gen_scale + ngen);
    const uint64_t ref_rank = (uint64_t)sp.rank[0][refa] * t->Db + (uint64_t)sp.rank[1][refb];

    std::vector<SecStep> steps;
    std::vector<SecEntry> entries;
    std::vector<uint32_t> gen_step{0};
    for (uint64_t g = 0; g < ngen; ++g) {
        if (gen_off[g + 1] < gen_off[g]) return fail(QFE_ERR_ARG, "qfe_template_create: generator offsets must not decrease");
        if (gen_param[g] < 0 || (uint64_t)gen_param[g] >= nparam)
            return fail(QFE_ERR_ARG, "qfe_template_create: generator parameter index out of range");
        int rc = build_runs(sp, lp, norb, lim, gen_terms, gen_off[g], gen_off[g + 1], gen_param[g], gen_scale[g],
                            (uint32_t)g, steps, entries, "qfe_template_create");
        if (rc) return rc;
        gen_step.push_back((uint32_t)steps.size());
    }

    t->has_map = map_off != nullptr;
    // Hamiltonian terms by X mask (first appearance).  A flip connects
    // determinants of the sector when each spin has room for it: half of its
    // bits occupied, half empty.  The other masks are read by nothing.
    struct Mask {
        uint64_t x;
        const uint64_t *first, *last;  // its terms
        const uint64_t* begin() const { return first; }
        const uint64_t* end() const { return last; }
        bool in_rows;
    };
    std::vector<Mask> masks;
    std::vector<uint64_t> members;
    {
        const int ne[2] = {popc32(refa), popc32(refb)};
        auto connects = [&](uint64_t x) {
            for (int s = 0; s < 2; ++s) {
                const int m = popc32(compress(x, s, norb));
                if ((m & 1) || m / 2 > ne[s] || m / 2 > norb - ne[s]) return false;
            }
            return true;
        };
        // mask of every term (open addressing), then the terms to their places
        size_t cap = 16;
        while (cap < 2 * nham) cap <<= 1;
        std::vector<uint32_t> slot(cap, 0), of(nham), count;  // slot: mask + 1
        std::vector<uint64_t> xs;
        for (uint64_t k = 0; k < nham; ++k) {
            if ((ham[k].x | ham[k].z) & ~lim)
                return fail(QFE_ERR_ARG, "qfe_template_create: Hamiltonian term acts on a qubit out of range");
            size_t h = (size_t)((ham[k].x * 0x9E3779B97F4A7C15ull) >> 20) & (cap - 1);
            while (slot[h] && xs[slot[h] - 1] != ham[k].x) h = (h + 1) & (cap - 1);
            if (!slot[h]) {
                xs.push_back(ham[k].x);
                count.push_back(0);
                slot[h] = (uint32_t)xs.size();
            }
            of[k] = slot[h] - 1;
            count[of[k]]++;
        }
        std::vector<uint64_t> at(xs.size() + 1, 0);
        for (size_t m = 0; m < xs.size(); ++m) at[m + 1] = at[m] + count[m];
        members.resize(nham);
        for (uint64_t k = nham; k-- > 0;) members[at[of[k]] + --count[of[k]]] = k;
        for (size_t m = 0; m < xs.size(); ++m)
            if (connects(xs[m])) masks.push_back(Mask{xs[m], members.data() + at[m], members.data() + at[m + 1], false});
    }
    // the map of every such term, before anything reads it
    if (map_off)
        for (const Mask& m : masks)
            for (uint64_t k : m) {
                if (map_off[k + 1] < map_off[k]) return fail(QFE_ERR_ARG, "qfe_template_create: map offsets must not decrease");
                for (uint64_t e = map_off[k]; e < map_off[k + 1]; ++e)
                    if (map_idx[e] >= ninputs) return fail(QFE_ERR_ARG, "qfe_template_create: map index out of range");
            }
    t->real = true;
    for (const auto& en : entries) t->real = t->real && en.ulo.y == 0.0 && en.uhi.y == 0.0;
    for (const Mask& m : masks)
        for (uint64_t k : m) {
            if (!t->has_map) {
                t->real = t->real && cplx_mul(make_double2(ham[k].phase.re, ham[k].phase.im),
                                              make_double2(ham[k].coeff.re, ham[k].coeff.im)).y == 0.0;
                continue;
            }
            t->real = t->real && ham[k].phase.im == 0.0;
            for (uint64_t e = map_off[k]; e < map_off[k + 1]; ++e) t->real = t->real && map_val[e].im == 0.0;
        }
    RowBuilder rowb(sp, norb);

    std::vector<SecGroup> groups;
    std::vector<uint64_t> tz;
    std::vector<double2> tph, tcoef;
    std::vector<uint64_t> moff{0};
    std::vector<uint32_t> midx;
    std::vector<double2> mval;
    {
        // groups that the rows take, in a real template
        std::vector<RowBuilder::Group> rgroups;
        std::vector<uint32_t> taken;  // their masks
        for (uint32_t i = 0; t->real && i < masks.size(); ++i) {
            const uint64_t x = masks[i].x;
            RowBuilder::Group g{x, compress(x, 0, norb), compress(x, 1, norb), {}};
            g.terms.reserve((size_t)(masks[i].last - masks[i].first));
            for (uint64_t k : masks[i]) g.terms.push_back({compress(ham[k].z, 0, norb), compress(ham[k].z, 1, norb), (uint32_t)k});
            if (!rowb.fits(g)) continue;
            rgroups.push_back(std::move(g));
            taken.push_back(i);
        }
        if (rows_worth(rowb, rgroups)) {
            rowb.build(rgroups);
            if (rowb.lds() <= kRowLdsMax && rowb.bmu.size() < (1u << kRowCellBits) - 1 && rowb.nfb < (1u << kRowCellBits) - 1) {
                for (uint32_t i : taken) masks[i].in_rows = true;
                t->row_lds = rowb.lds();
                t->nrows = t->Da * ((t->Db + kRowThreads - 1) / kRowThreads);
                t->nm = (uint32_t)rowb.mrow.size();
            }
        }
        for (const Mask& m : masks) {
            if (m.in_rows) continue;
            const uint64_t x = m.x;
            const uint32_t xa = compress(x, 0, norb), xb = compress(x, 1, norb);
            SecGroup gr{};
            gr.x = x;
            gr.xa = xa;
            gr.xb = xb;
            std::pair<uint32_t, uint32_t> la, lb;
            if (x == 0) {
                la = lp.get(sp, 0, 1, 0, 0, 0);
                lb = lp.get(sp, 1, 1, 0, 0, 0);
                gr.weight = 1.0;
            } else {
                // visit the half of the pairs with the top bit of x clear, weight 2
                const int hb = 63 - __builtin_clzll(x);
                const uint32_t clear = 1u << (hb / 2);
                if ((hb & 1) == 0) {
                    la = lp.get(sp, 0, 2, xa, clear, xa);
                    lb = lp.get(sp, 1, 1, xb, 0, xb);
                } else {
                    la = lp.get(sp, 0, 1, xa, 0, xa);
                    lb = lp.get(sp, 1, 2, xb, clear, xb);
                }
                gr.weight = 2.0;
            }
            gr.la_off = la.first;
            gr.la_len = la.second;
            gr.lb_off = lb.first;
            gr.lb_len = lb.second;
            gr.inv_lb = 1.0 / (double)lb.second;
            gr.t_first = (uint32_t)tz.size();
            for (uint64_t k : m) {
                tz.push_back(ham[k].z);
                const double2 ph = make_double2(ham[k].phase.re, ham[k].phase.im);
                tph.push_back(ph);
                tcoef.push_back(cplx_mul(ph, make_double2(ham[k].coeff.re, ham[k].coeff.im)));
                if (map_off) {
                    for (uint64_t e = map_off[k]; e < map_off[k + 1]; ++e) {
                        midx.push_back(map_idx[e]);
                        mval.push_back(make_double2(map_val[e].re, map_val[e].im));
                    }
                    moff.push_back(midx.size());
                }
            }
            gr.t_count = (uint32_t)tz.size() - gr.t_first;
            groups.push_back(gr);
        }
    }
    // work items of similar cost (pairs x (terms + 4)): small groups merge,
    // large groups split into pair ranges
    std::vector<SecItem> items;
    {
        const uint64_t target = 1ull << 18;
        uint32_t g = 0;
        while (g < groups.size()) {
            const uint64_t pairs = (uint64_t)groups[g].la_len * groups[g].lb_len;
            const uint64_t per = groups[g].t_count + 4;
            if (pairs * per >= target) {
                uint64_t chunk = std::max<uint64_t>(2048, target / per);
                chunk = (chunk + 255) & ~255ull;
                for (uint64_t p = 0; p < pairs; p += chunk)
                    items.push_back(SecItem{g, g + 1, (uint32_t)p, (uint32_t)std::min(pairs, p + chunk)});
                ++g;
                continue;
            }
            uint32_t g1 = g;
            uint64_t cost = 0;
            while (g1 < groups.size()) {
                const uint64_t c = (uint64_t)groups[g1].la_len * groups[g1].lb_len * (groups[g1].t_count + 4);
                if (g1 > g && (cost + c > target || c >= target)) break;
                cost += c;
                ++g1;
            }
            // a single small group is "whole" only when g1 != g + 1; give it its full pair range instead
            if (g1 == g + 1)
                items.push_back(SecItem{g, g + 1, 0, (uint32_t)((uint64_t)groups[g].la_len * groups[g].lb_len)});
            else
                items.push_back(SecItem{g, g1, 0, 0});
            g = g1;
        }
    }
    t->h_gen_step = gen_step;
    t->step_pairs.assign(steps.size(), 0);
    for (size_t k = 0; k < steps.size(); ++k)
        for (uint32_t e = steps[k].e_first; e < steps[k].e_first + steps[k].e_count; ++e)
            t->step_pairs[k] += entries[e].la_len * entries[e].lb_len;
    // sigma-kernel chunks: up to kHpsiGroups groups and kHpsiTerms terms each
    std::vector<uint2> hchunks;
    for (uint32_t g = 0; g < groups.size();) {
        uint32_t g1 = g + 1;
        uint32_t terms = groups[g].t_count;
        while (g1 < groups.size() && g1 - g < kHpsiGroups && terms + groups[g1].t_count <= kHpsiTerms)
            terms += groups[g1++].t_count;
        hchunks.push_back(make_uint2(g, g1));
        g = g1;
    }
    t->nterms = (uint32_t)tz.size();
    t->nentries = (uint32_t)entries.size();
    t->nitems = (uint32_t)items.size();

    uint64_t cost = t->D;
    for (const auto& en : entries) cost += (uint64_t)en.la_len * en.lb_len * 4;
    for (const auto& gr : groups) cost += (uint64_t)gr.la_len * gr.lb_len * (2 + gr.t_count);
    if (t->nrows) cost += t->D * (rowb.nb1 + 8 * rowb.nb2 + (rowb.flips.size() + rowb.pairs.size() * (uint64_t)rowb.nwords) / t->Da);
    t->cost = cost;

    {  // serving tier
        int dev = 0, max_lds = 0;
        (void)hipGetDevice(&dev);
        if (hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) max_lds = 65536;
        const size_t tab = ((uint64_t)t->Da + t->Db) <= kTableLds ? ((uint64_t)t->Da + t->Db) * 8 : 0;
        const size_t with_psi = t->D * sizeof(double2) + tab;
        t->tier = with_psi <= kTier0Lds ? 0 : (with_psi + 1024 <= (size_t)max_lds ? 1 : 2);
    }

    std::vector<uint64_t> af(t->Da), bf(t->Db);
    for (uint32_t a = 0; a < t->Da; ++a) af[a] = spread(sp.str[0][a], 0, norb);
    for (uint32_t b2 = 0; b2 < t->Db; ++b2) bf[b2] = spread(sp.str[1][b2], 1, norb);
    std::vector<double> tcoef_real;
    if (t->real)
        for (const auto& v : tcoef) tcoef_real.push_back(v.x);
    TileBuilder tb(sp, lp, steps, entries, ngen, norb, t->real);
    tb.build(gen_step);
    t->fwd = tb.lfwd;
    t->rev = tb.lrev;
    t->wins = tb.wins;
    // merged numbers of the rows: from the inputs, or constants
    std::vector<double> rm, rmval;
    std::vector<uint32_t> rmoff{0}, rmidx;
    if (t->nrows) {
        struct Part {
            uint32_t input, order;
            double v;
        };
        std::vector<Part> in;
        for (const uint2& row : rowb.mrow) {
            in.clear();
            double v = 0.0;
            for (uint32_t i = row.x; i < row.x + row.y; ++i) {
                const auto& tk = rowb.mterm[i];
                const qfe_pauli& h = ham[tk.first];
                if (t->has_map)
                    for (uint64_t e = map_off[tk.first]; e < map_off[tk.first + 1]; ++e)
                        in.push_back(Part{map_idx[e], (uint32_t)in.size(), tk.second * h.phase.re * map_val[e].re});
                else
                    v += tk.second * (h.phase.re * h.coeff.re - h.phase.im * h.coeff.im);
            }
            std::sort(in.begin(), in.end(), [](const Part& a, const Part& b) { return a.input != b.input ? a.input < b.input : a.order < b.order; });
            for (size_t i = 0; i < in.size();) {
                const uint32_t idx = in[i].input;
                double sum = 0.0;
                for (; i < in.size() && in[i].input == idx; ++i) sum += in[i].v;
                if (sum == 0.0) continue;
                rmidx.push_back(idx);
                rmval.push_back(sum);
            }
            rmoff.push_back((uint32_t)rmidx.size());
            if (!t->has_map) rm.push_back(v);
        }
    }
    const RowBuilder none(sp, norb);
    const RowBuilder& rows = t->nrows ? rowb : none;
    Packer pk(sizeof(SecTables));
    const size_t i_af = pk.add(af.data(), af.size() * 8), i_bf = pk.add(bf.data(), bf.size() * 8);
    const size_t i_as = pk.add(sp.str[0].data(), sp.str[0].size() * 4), i_bs = pk.add(sp.str[1].data(), sp.str[1].size() * 4);
    const size_t i_ar = pk.add(sp.rank[0].data(), sp.rank[0].size() * 4), i_br = pk.add(sp.rank[1].data(), sp.rank[1].size() * 4);
    const size_t i_l = pk.add(lp.pool.data(), lp.pool.size() * sizeof(int2));
    const size_t i_st = pk.add(steps.data(), steps.size() * sizeof(SecStep));
    const size_t i_en = pk.add(entries.data(), entries.size() * sizeof(SecEntry));
    const size_t i_gr = pk.add(groups.data(), groups.size() * sizeof(SecGroup));
    const size_t i_it = pk.add(items.data(), items.size() * sizeof(SecItem));
    const size_t i_gs = pk.add(gen_step.data(), gen_step.size() * 4);
    const size_t i_tz = pk.add(tz.data(), tz.size() * 8);
    const size_t i_tph = pk.add(tph.data(), tph.size() * sizeof(double2));
    const size_t i_tc = t->real ? pk.add(tcoef_real.data(), tcoef_real.size() * 8) : pk.add(tcoef.data(), tcoef.size() * sizeof(double2));
    const size_t i_mo = pk.add(moff.data(), moff.size() * 8);
    const size_t i_mi = pk.add(midx.data(), midx.size() * 4);
    const size_t i_mv = pk.add(mval.data(), mval.size() * sizeof(double2));
    const size_t i_hc = pk.add(hchunks.data(), hchunks.size() * sizeof(uint2));
    const size_t i_ts = pk.add(tb.segs.data(), tb.segs.size() * sizeof(TileSeg));
    const size_t i_tf = pk.add(tb.fwd.data(), tb.fwd.size() * sizeof(TileRun));
    const size_t i_tr = pk.add(tb.rev.data(), tb.rev.size() * sizeof(TileRun));
    const size_t i_tc2 = pk.add(tb.recs.data(), tb.recs.size() * sizeof(TileRec));
    const size_t i_tx = pk.add(tb.tix.data(), tb.tix.size() * 4);
    const size_t i_tt = pk.add(tb.tab.data(), tb.tab.size() * sizeof(uint2));
    const size_t i_tw = pk.add(tb.words.data(), tb.words.size() * 4);
    const size_t i_tu = pk.add(tb.sum.data(), tb.sum.size() * sizeof(uint2));
    const size_t i_to = pk.add(tb.outs.data(), tb.outs.size() * sizeof(TileOut));
    const size_t i_tv = pk.add(tb.wins.data(), tb.wins.size() * sizeof(TileWindow));
    auto add_all = [&](const auto& v) { return pk.add(v.data(), v.size() * sizeof(v[0])); };
    const size_t r_chunk_off = add_all(rows.chunk_off);
    const size_t r_chunks = add_all(rows.chunks);
    const size_t r_flips = add_all(rows.flips);
    const size_t r_pos_cell = add_all(rows.pos_cell);
    const size_t r_amu = add_all(rows.amu);
    const size_t r_am = add_all(rows.am);
    const size_t r_bmu = add_all(rows.bmu);
    const size_t r_bm = add_all(rows.bm);
    const size_t r_mmask = add_all(rows.mmask);
    const size_t r_b1 = add_all(rows.b1);
    const size_t r_b2 = add_all(rows.b2);
    const size_t r_pair_off = add_all(rows.pair_off);
    const size_t r_pairs = add_all(rows.pairs);
    const size_t r_words = add_all(rows.words);
    const size_t r_fb_mask = add_all(rows.fb_mask);
    const size_t r_fa_mask = add_all(rows.fa_mask);
    const size_t r_m = add_all(rm), r_moff = add_all(rmoff), r_midx = add_all(rmidx), r_mval = add_all(rmval);
    QFE_HIP(device_malloc(&t->dev, pk.total));
    char* base = (char*)t->dev;
    auto at = [&](size_t i) { return base + pk.pieces[i].off; };
    SecTables h{};
    h.D = t->D;
    h.ref_rank = ref_rank;
    h.Da = t->Da;
    h.Db = t->Db;
    h.afull = (const uint64_t*)at(i_af);
    h.bfull = (const uint64_t*)at(i_bf);
    h.astr = (const uint32_t*)at(i_as);
    h.bstr = (const uint32_t*)at(i_bs);
    h.arank = (const int32_t*)at(i_ar);
    h.brank = (const int32_t*)at(i_br);
    h.lists = (const int2*)at(i_l);
    h.steps = (const SecStep*)at(i_st);
    h.entries = (const SecEntry*)at(i_en);
    h.groups = (const SecGroup*)at(i_gr);
    h.items = (const SecItem*)at(i_it);
    h.gen_step = (const uint32_t*)at(i_gs);
    h.tz = (const uint64_t*)at(i_tz);
    h.tph = (const double2*)at(i_tph);
    h.tcoef = at(i_tc);
    h.map_off = t->has_map ? (const uint64_t*)at(i_mo) : nullptr;
    h.map_idx = (const uint32_t*)at(i_mi);
    h.map_val = (const double2*)at(i_mv);
    h.hchunks = (const uint2*)at(i_hc);
    h.nhchunks = (uint32_t)hchunks.size();
    h.tsegs = (const TileSeg*)at(i_ts);
    h.tfwd = (const TileRun*)at(i_tf);
    h.trev = (const TileRun*)at(i_tr);
    h.trec = (const TileRec*)at(i_tc2);
    h.tix = (const uint32_t*)at(i_tx);
    h.ttab = (const uint2*)at(i_tt);
    h.twords = (const uint32_t*)at(i_tw);
    h.tsum = (const uint2*)at(i_tu);
    h.touts = (const TileOut*)at(i_to);
    h.twins = (const TileWindow*)at(i_tv);
    h.nwins = (uint32_t)tb.wins.size();
    h.rows.chunk_off = (const uint32_t*)at(r_chunk_off);
    h.rows.chunks = (const uint4*)at(r_chunks);
    h.rows.flips = (const RowFlip*)at(r_flips);
    h.rows.pos_cell = (const uint32_t*)at(r_pos_cell);
    h.rows.amu = (const uint32_t*)at(r_amu);
    h.rows.am = (const uint32_t*)at(r_am);
    h.rows.bmu = (const uint32_t*)at(r_bmu);
    h.rows.bm = (const uint32_t*)at(r_bm);
    h.rows.mmask = (const uint32_t*)at(r_mmask);
    h.rows.b1 = (const uint32_t*)at(r_b1);
    h.rows.b2 = (const uint2*)at(r_b2);
    h.rows.pair_off = (const uint32_t*)at(r_pair_off);
    h.rows.pairs = (const RowPair*)at(r_pairs);
    h.rows.words = (const uint32_t*)at(r_words);
    h.rows.fb_mask = (const uint32_t*)at(r_fb_mask);
    h.rows.fa_mask = (const uint32_t*)at(r_fa_mask);
    h.rows.m = (const double*)at(r_m);
    h.rows.moff = (const uint32_t*)at(r_moff);
    h.rows.midx = (const uint32_t*)at(r_midx);
    h.rows.mval = (const double*)at(r_mval);
    h.rows.nm = t->nm;
    h.rows.nbcell = (uint32_t)rows.bmu.size();
    h.rows.nb1 = rows.nb1;
    h.rows.nb2 = rows.nb2;
    h.rows.nwords = rows.nwords;
    h.rows.nfb = rows.nfb;
    h.rows.gbase = rows.gbase;
    h.nrows = t->nrows;
    h.nparts = t->nitems + t->nrows;
    h.nsteps = (uint32_t)steps.size();
    h.nentries = (uint32_t)entries.size();
    h.ngroups = (uint32_t)groups.size();
    h.nterms = (uint32_t)tz.size();
    h.nitems = (uint32_t)items.size();
    h.ngen = (uint32_t)ngen;
    std::vector<char> img(pk.total, 0);
    pk.fill(img.data());
    std::memcpy(img.data(), &h, sizeof(h));
    QFE_HIP(hipMemcpy(t->dev, img.data(), pk.total, hipMemcpyHostToDevice));
    t->dt = (SecTables*)t->dev;
    t->afull = h.afull;
    t->bfull = h.bfull;

    // per-request layout: energy parts first, gradient parts after
    size_t o = 0;
    t->off_psi = o;
    o += align256(t->D * t->amp());
    t->off_coef = o;
    if (t->has_map) o += align256((size_t)t->nterms * t->amp());
    t->off_hm = o;
    if (t->has_map) o += align256((size_t)t->nm * 8);
    t->off_cs = o;
    o += align256((size_t)t->nentries * sizeof(double2) + 16);
    t->off_part = o;
    o += align256((size_t)(t->nitems + t->nrows) * 8 + 8);
    t->work_bytes = o;
    t->off_sig = o;
    o += align256(t->D * t->amp());
    t->off_gacc = o;
    o += align256(ngen * 8 + 8);
    t->off_gpart = o;
    const size_t sums = align256((size_t)tb.peak * 8);
    o += sums;
    t->grad_bytes = o;
    t->io_count = nparam + ninputs;
    t->request_bytes = t->work_bytes + align256(t->io_count * 8 + 8) + sizeof(SlotDesc);
    t->grad_request_bytes = t->grad_bytes + align256(t->io_count * 8 + 8) + sizeof(SlotDesc) + ngen * 8;
    t->grad_least_bytes = t->grad_request_bytes - sums;
    return QFE_OK;
}

SlotDesc make_slot(qfe_template t, char* work, const double* io, double* out, bool grad) {
    SlotDesc d{};
    d.t = t->dt;
    d.psi = work + t->off_psi;
    d.coef = t->has_map ? work + t->off_coef : nullptr;
    d.hm = t->has_map && t->nrows ? (double*)(work + t->off_hm) : nullptr;
    d.cs = (double2*)(work + t->off_cs);
    d.part = (double*)(work + t->off_part);
    d.sig = grad ? work + t->off_sig : nullptr;
    d.gacc = grad ? (double*)(work + t->off_gacc) : nullptr;
    d.gpart = grad ? (double*)(work + t->off_gpart) : nullptr;
    d.params = io;
    d.inputs = io + t->nparam;
    d.out = out;
    return d;
}

// f(S{}) with the scalar type of a template.
template <typename F>
auto with_scalar(const qfe_template_s* t, F&& f) {
    return t->real ? f(double{}) : f(double2{});
}

// The passes of one direction over k requests of one scalar type: launch q runs pass q of every
// request that has one.  prefix: tile prefix of every launch (k + 1 entries
// each, from pass_prefix); null for a single request.
template <int MODE>
int launch_tiles(const std::vector<qfe_template>& ts, const SlotDesc* d, const uint32_t* prefix, hipStream_t st) {
    const uint32_t k = (uint32_t)ts.size();
    size_t npass = 0;
    for (const auto& t : ts) npass = std::max(npass, (MODE == 2 ? t->rev : t->fwd).size());
    for (size_t i = 0; i < npass; ++i) {
        const size_t q = MODE == 1 ? npass - 1 - i : i;
        uint64_t tiles = 0;
        uint32_t lds = 0;
        for (const auto& t : ts) {
            const auto& runs = MODE == 2 ? t->rev : t->fwd;
            if (q >= runs.size()) continue;
            tiles += runs[q].tiles;
            lds = std::max(lds, runs[q].lds);
        }
        if (tiles >= (1ull << 31)) return fail(QFE_ERR_ARG, "qfe_template: too many tiles in one launch");
        with_scalar(ts[0], [&](auto z) {
            hipLaunchKernelGGL((k_sec_tile<decltype(z), kTileThreads, MODE>), dim3((unsigned)tiles), dim3(kTileThreads), lds, st,
                               d, prefix ? prefix + q * (k + 1) : nullptr, k, (uint32_t)q, (uint32_t)(MODE != 1 && q == 0));
        });
        QFE_HIP(hipGetLastError());
        if (MODE != 2) continue;
        uint32_t outs = 0;  // of the windows that end here, but for every request's last
        for (const auto& t : ts)
            for (size_t w = 0; w + 1 < t->wins.size(); ++w)
                if (t->wins[w].pass == q) outs = std::max(outs, t->wins[w].o1 - t->wins[w].o0);
        if (outs) {
            hipLaunchKernelGGL(k_sec_tile_sum, dim3((outs + 3) / 4, k), dim3(256), 0, st, d, (uint32_t)q);
            QFE_HIP(hipGetLastError());
        }
    }
    return QFE_OK;
}

// Tile prefixes of every pass of one direction over k requests.
void pass_prefix(const std::vector<qfe_template>& ts, bool rev, std::vector<uint32_t>& out) {
    size_t npass = 0;
    for (const auto& t : ts) npass = std::max(npass, (rev ? t->rev : t->fwd).size());
    for (size_t q = 0; q < npass; ++q) {
        uint32_t at = 0;
        for (const auto& t : ts) {
            const auto& runs = rev ? t->rev : t->fwd;
            out.push_back(at);
            if (q < runs.size()) at += runs[q].tiles;
        }
        out.push_back(at);
    }
}

int launch_prologue(const std::vector<qfe_template>& ts, const SlotDesc* d, int need_coef, hipStream_t st) {
    uint32_t most = 1;
    for (const auto& t : ts) most = std::max(most, std::max(t->nentries, need_coef ? std::max(t->nterms, t->nm) : 0u));
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((most + 255) / 256, ((1ull << 31) - 1) / ts.size());
    with_scalar(ts[0], [&](auto z) {
        hipLaunchKernelGGL(k_sec_prologue<decltype(z)>, dim3(blocks * (unsigned)ts.size()), dim3(256), 0, st, d, need_coef, blocks);
    });
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

// The row workgroups of k requests (prefix: row prefix, null for one request).
int launch_rows(const std::vector<qfe_template>& ts, const SlotDesc* d, const uint32_t* prefix, bool energy, hipStream_t st) {
    uint64_t rows = 0;
    uint32_t Db = 1;
    size_t lds = 0;
    for (const auto& t : ts) {
        rows += t->nrows;
        Db = std::max(Db, t->Db);
        lds = std::max(lds, t->row_lds);
    }
    if (!rows) return QFE_OK;
    if (rows >= (1ull << 31)) return fail(QFE_ERR_ARG, "qfe_template: too many rows in one launch");
    const unsigned threads = std::min(kRowThreads, (Db + 63u) & ~63u);  // a row of at most 256 strings is one workgroup
    if (energy)
        hipLaunchKernelGGL(k_sec_rows<true>, dim3((unsigned)rows), dim3(threads), lds, st, d, prefix, (uint32_t)ts.size());
    else
        hipLaunchKernelGGL(k_sec_rows<false>, dim3((unsigned)rows), dim3(threads), lds, st, d, prefix, (uint32_t)ts.size());
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

// sigma = H psi: the rows, then the groups that they do not take (grid y = request).
int launch_sigma(const std::vector<qfe_template>& ts, const SlotDesc* ddesc, const uint32_t* rowprefix, hipStream_t st) {
    const unsigned k = (unsigned)ts.size();
    uint64_t D = 1;
    bool rest = false;
    for (const auto& t : ts) {
        D = std::max(D, t->D);
        rest = rest || t->nitems || !t->nrows;
    }
    int rc = launch_rows(ts, ddesc, rowprefix, false, st);
    if (rc || !rest) return rc;
    with_scalar(ts[0], [&](auto z) {
        using S = decltype(z);
        if (k == 1)
            hipLaunchKernelGGL((k_sec_hpsi<S, 1>), dim3((unsigned)((D + 255) / 256), k), dim3(256), 0, st, ddesc);
        else
            hipLaunchKernelGGL((k_sec_hpsi<S, 4>), dim3((unsigned)((D + 1023) / 1024), k), dim3(256), 0, st, ddesc);
    });
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

// Prefixes of a launch over several requests, on the device (null for one request).
struct Prefixes {
    const uint32_t *items, *fwd, *rows, *rev;
};

// Energy of k requests: prologue, ansatz, rows and items, sums.
int launch_energy(const std::vector<qfe_template>& ts, const SlotDesc* ddesc, const Prefixes& pre, uint32_t total_items,
                  hipStream_t st) {
    const unsigned k = (unsigned)ts.size();
    int rc = launch_prologue(ts, ddesc, 1, st);
    if (!rc) rc = launch_tiles<0>(ts, ddesc, pre.fwd, st);
    if (!rc) rc = launch_rows(ts, ddesc, pre.rows, true, st);
    if (rc) return rc;
    if (total_items) {
        with_scalar(ts[0], [&](auto z) {
            hipLaunchKernelGGL(k_sec_energy<decltype(z)>, dim3(total_items), dim3(kItemThreads), 0, st, ddesc, pre.items, (uint32_t)k);
        });
        QFE_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_sec_sum, dim3(k), dim3(256), 0, st, ddesc);
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

// psi = U|ref> and sigma = H psi of k requests.
int launch_psi_sigma(const std::vector<qfe_template>& ts, const SlotDesc* ddesc, const Prefixes& pre, hipStream_t st) {
    int rc = launch_prologue(ts, ddesc, 1, st);
    if (!rc) rc = launch_tiles<0>(ts, ddesc, pre.fwd, st);
    return rc ? rc : launch_sigma(ts, ddesc, pre.rows, st);
}

// Energy and adjoint gradient of k requests.
int launch_gradient(const std::vector<qfe_template>& ts, const SlotDesc* ddesc, const Prefixes& pre, hipStream_t st) {
    int rc = launch_psi_sigma(ts, ddesc, pre, st);
    if (!rc) rc = launch_tiles<2>(ts, ddesc, pre.rev, st);
    if (rc) return rc;
    uint32_t outs = 1;
    for (const auto& t : ts) outs = std::max(outs, t->wins.back().o1 - t->wins.back().o0);
    hipLaunchKernelGGL(k_sec_tile_sum, dim3((outs + 3) / 4, (unsigned)ts.size()), dim3(256), 0, st, ddesc, kLastWindow);
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

// ---- step-by-step sequences (tier 2, captured for the audit) ------------------------------
uint32_t wide_blocks(uint64_t items) { return (uint32_t)((items + kWideTPB - 1) / kWideTPB); }

// U|ref>: the reference determinant, then one launch per step.
template <typename S>
int wide_ansatz(qfe_template t, const SlotDesc* d, hipStream_t st) {
    hipLaunchKernelGGL(k_sec_ref<S>, dim3(wide_blocks(t->D)), dim3(kWideTPB), 0, st, d);
    QFE_HIP(hipGetLastError());
    for (uint32_t k = 0; k < (uint32_t)t->step_pairs.size(); ++k) {
        if (!t->step_pairs[k]) continue;
        hipLaunchKernelGGL(k_sec_step<S>, dim3(wide_blocks(t->step_pairs[k])), dim3(kWideTPB), 0, st, d, k, 0, 0);
        QFE_HIP(hipGetLastError());
    }
    return QFE_OK;
}

// Energy: prologue, ansatz, work items, sum (the items and sum kernels of the batched path).
template <typename S>
int wide_energy(qfe_template t, const SlotDesc* d, const uint32_t* dprefix, hipStream_t st) {
    int rc = launch_prologue({t}, d, 1, st);
    if (!rc) rc = wide_ansatz<S>(t, d, st);
    if (!rc) rc = launch_rows({t}, d, nullptr, true, st);
    if (rc) return rc;
    if (t->nitems) {
        hipLaunchKernelGGL(k_sec_energy<S>, dim3(t->nitems), dim3(kItemThreads), 0, st, d, dprefix, 1u);
        QFE_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_sec_sum, dim3(1), dim3(256), 0, st, d);
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

// psi and sigma = H psi (pool gradients and the gradient below).
template <typename S>
int wide_psi_sigma(qfe_template t, const SlotDesc* d, hipStream_t st) {
    int rc = launch_prologue({t}, d, 1, st);
    if (!rc) rc = wide_ansatz<S>(t, d, st);
    return rc ? rc : launch_sigma({t}, d, nullptr, st);
}

// Energy and generator overlaps: E = Re<psi|sigma>, then for k = M-1 .. 0 the
// overlap of generator k and its un-rotation on psi and sigma; fixed-order sums.
template <typename S>
int wide_gradient(qfe_template t, const SlotDesc* d, hipStream_t st) {
    int rc = wide_psi_sigma<S>(t, d, st);
    if (rc) return rc;
    const size_t seg_bytes = align256(t->wide_seg.size() * sizeof(uint2));
    double* part = (double*)((char*)t->wide + seg_bytes);
    hipLaunchKernelGGL(k_sec_edot<S>, dim3(t->wide_seg[0].y), dim3(kWideTPB), 0, st, d, part + t->wide_seg[0].x);
    QFE_HIP(hipGetLastError());
    for (uint32_t k = (uint32_t)t->ngen; k-- > 0;) {
        const uint2 sg = t->wide_seg[k + 1];
        if (!sg.y) continue;
        const uint32_t s0 = t->h_gen_step[k], s1 = t->h_gen_step[k + 1];
        if (s1 == s0 + 1) {
            hipLaunchKernelGGL(k_sec_genrev<S>, dim3(sg.y), dim3(kWideTPB), 0, st, d, s0, part + sg.x);
            QFE_HIP(hipGetLastError());
            continue;
        }
        hipLaunchKernelGGL(k_sec_genov<S>, dim3(sg.y), dim3(kWideTPB), 0, st, d, s0, s1, part + sg.x);
        QFE_HIP(hipGetLastError());
        for (uint32_t sdx = s1; sdx-- > s0;) {
            if (!t->step_pairs[sdx]) continue;
            hipLaunchKernelGGL(k_sec_step<S>, dim3(wide_blocks(t->step_pairs[sdx])), dim3(kWideTPB), 0, st, d, sdx, 1, 1);
            QFE_HIP(hipGetLastError());
        }
    }
    const uint32_t nseg = (uint32_t)t->wide_seg.size();
    hipLaunchKernelGGL(k_sec_wsum, dim3(wide_blocks(nseg)), dim3(kWideTPB), 0, st, d, (const double*)part,
                       (const uint2*)t->wide, nseg);
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

// Single request on the library stream.  Arena: [desc 256][out 256][prefix 256][io][work + gradient parts].
struct Single {
    SlotDesc* ddesc;
    double* dout;
    uint32_t* dprefix;
    char* work;
};

size_t single_head(qfe_template t) { return 768 + align256(t->io_count * 8 + 8); }

// The arena of single requests; it grows when the first gradient parts are asked for.
int single_arena(qfe_template t, bool grad) {
    const size_t need = single_head(t) + (grad ? t->grad_bytes : t->work_bytes);
    if (t->arena_bytes >= need) return QFE_OK;
    if (t->arena) {
        QFE_HIP(hipStreamSynchronize(ctx().stream));
        QFE_HIP(hipFree(t->arena));
        t->arena = nullptr;
        t->arena_bytes = 0;
    }
    QFE_HIP(device_malloc(&t->arena, need));
    t->arena_bytes = need;
    return QFE_OK;
}

int single_setup(qfe_template t, const double* params, const double* inputs, bool grad, Single& S) {
    const size_t head = single_head(t);
    int rc = single_arena(t, grad);
    if (rc) return rc;
    char* dev = (char*)t->arena;
    S.ddesc = (SlotDesc*)dev;
    S.dout = (double*)(dev + 256);
    S.dprefix = (uint32_t*)(dev + 512);
    S.work = dev + head;
    void* host = nullptr;
    rc = staging_begin(head, &host);
    if (rc) return rc;
    char* h = (char*)host;
    SlotDesc d = make_slot(t, S.work, (const double*)(dev + 768), S.dout, grad);
    std::memcpy(h, &d, sizeof(d));
    const uint32_t pre[2] = {0, t->nitems};
    std::memcpy(h + 512, pre, sizeof(pre));
    if (t->nparam) std::memcpy(h + 768, params, t->nparam * 8);
    if (t->ninputs) std::memcpy(h + 768 + t->nparam * 8, inputs, t->ninputs * 8);
    return staging_commit(dev, head);
}

int fetch_doubles(const double* dev, size_t count, double* host) {
    void* pin = nullptr;
    int rc = pinned_reserve(count * 8 + 8, &pin);
    if (rc) return rc;
    QFE_HIP(hipMemcpyAsync(pin, dev, count * 8, hipMemcpyDeviceToHost, ctx().stream));
    QFE_HIP(hipStreamSynchronize(ctx().stream));
    std::memcpy(host, pin, count * 8);
    return QFE_OK;
}

// grad[p] = sum over generators k with parameter p of 2 scale_k <sigma_k|K_k|psi_k>.
void gradient_from_overlaps(qfe_template t, const double* acc, double* grad) {
    for (uint64_t i = 0; i < t->nparam; ++i) grad[i] = 0.0;
    for (uint64_t k = 0; k < t->ngen; ++k) grad[t->gparam[k]] += 2.0 * t->gscale[k] * acc[k];
}

// psi = U|ref> and sigma = H psi for one request (pool gradients).
int single_psi_sigma(qfe_template t, const double* params, const double* inputs, Single& S) {
    int rc = single_setup(t, params, inputs, true, S);
    return rc ? rc : launch_psi_sigma({t}, S.ddesc, Prefixes{}, ctx().stream);
}

// ---- captured single-request sequences (large sectors) ----------------------------------
// The step-by-step sequence as one hipGraph per template.  The first node
// uploads the whole request head (descriptor, prefix, amplitudes, inputs) from
// the template's pinned block; the last nodes copy the energy (and the
// generator overlaps) back into the same block.

// ---- host-side audit of a captured sequence ---------------------------------------------
// After instantiation every node of a template graph is compared with the
// sequence the template's structure fixes, computed here independently of the
// wide_* launchers: the graph must be one chain from its root; each node must
// be the expected memcpy (addresses and size inside the arena and the pinned
// block) or the expected kernel with a non-zero grid and a block of at most
// 1024 threads, every scalar argument equal to the expected one and every
// pointer argument equal to the expected address (partial-sum pointers with
// their whole grid inside the partial array); the uploaded descriptor's
// pointers must lie inside the arena.  A mismatch fails graph_build with
// QFE_ERR_STATE and the graph is not kept, so nothing malformed is launched.
struct GraphAudit {
    uint64_t nodes = 0, kernels = 0, kernels_checked = 0, copies_checked = 0;
};

struct NodeExpect {
    bool copy = false;
    const void* func = nullptr;
    unsigned grid = 0, block = 0;
    std::vector<std::vector<char>> args;  // expected bytes of each argument
    const void* dst = nullptr;
    const void* src = nullptr;
    size_t bytes = 0;
};

template <typename... A>
NodeExpect expect_kernel(const void* func, uint64_t grid, unsigned block, A... a) {
    NodeExpect e;
    e.func = func;
    e.grid = grid > 0x7fffffffull ? 0u : (unsigned)grid;  // out of range: fails the non-zero grid check
    e.block = block;
    (e.args.push_back(std::vector<char>((const char*)&a, (const char*)&a + sizeof(A))), ...);
    return e;
}

NodeExpect expect_copy(const void* dst, const void* src, size_t bytes) {
    NodeExpect e;
    e.copy = true;
    e.dst = dst;
    e.src = src;
    e.bytes = bytes;
    return e;
}

template <typename S>
void expected_nodes(qfe_template t, int grad, std::vector<NodeExpect>& out) {
    const size_t head = single_head(t);
    char* dev = (char*)t->arena;
    char* pin = (char*)t->gpin;
    const SlotDesc* d = (const SlotDesc*)dev;
    const auto KB = [](uint64_t items) { return (items + kWideTPB - 1) / kWideTPB; };
    out.clear();
    out.push_back(expect_copy(dev, pin, head));
    const uint64_t pro = KB(std::max(std::max(t->nentries, 1u), std::max(t->nterms, t->nm)));
    out.push_back(expect_kernel((const void*)&k_sec_prologue<S>, pro, 256, d, (int)1, (uint32_t)pro));
    out.push_back(expect_kernel((const void*)&k_sec_ref<S>, KB(t->D), kWideTPB, d));
    for (uint32_t k = 0; k < (uint32_t)t->step_pairs.size(); ++k)
        if (t->step_pairs[k])
            out.push_back(expect_kernel((const void*)&k_sec_step<S>, KB(t->step_pairs[k]), kWideTPB, d, k, (int)0, (int)0));
    if (t->nrows)
        out.push_back(expect_kernel(grad ? (const void*)&k_sec_rows<false> : (const void*)&k_sec_rows<true>, t->nrows,
                                    std::min(kRowThreads, (t->Db + 63u) & ~63u), d, (const uint32_t*)nullptr, (uint32_t)1));
    if (!grad) {
        if (t->nitems)
            out.push_back(expect_kernel((const void*)&k_sec_energy<S>, t->nitems, kItemThreads, d,
                                        (const uint32_t*)(dev + 512), (uint32_t)1));
        out.push_back(expect_kernel((const void*)&k_sec_sum, 1, 256, d));
        out.push_back(expect_copy(pin + head, dev + 256, 8));
        return;
    }
    if (t->nitems || !t->nrows) out.push_back(expect_kernel((const void*)&k_sec_hpsi<S, 1>, (t->D + 255) / 256, 256, d));
    double* part = (double*)((char*)t->wide + align256(t->wide_seg.size() * sizeof(uint2)));
    out.push_back(expect_kernel((const void*)&k_sec_edot<S>, t->wide_seg[0].y, kWideTPB, d, part + t->wide_seg[0].x));
    for (uint32_t k = (uint32_t)t->ngen; k-- > 0;) {
        const uint2 sg = t->wide_seg[k + 1];
        if (!sg.y) continue;
        const uint32_t s0 = t->h_gen_step[k], s1 = t->h_gen_step[k + 1];
        if (s1 == s0 + 1) {
            out.push_back(expect_kernel((const void*)&k_sec_genrev<S>, sg.y, kWideTPB, d, s0, part + sg.x));
            continue;
        }
        out.push_back(expect_kernel((const void*)&k_sec_genov<S>, sg.y, kWideTPB, d, s0, s1, part + sg.x));
        for (uint32_t sdx = s1; sdx-- > s0;)
            if (t->step_pairs[sdx])
                out.push_back(expect_kernel((const void*)&k_sec_step<S>, KB(t->step_pairs[sdx]), kWideTPB, d, sdx, (int)1, (int)1));
    }
    const uint32_t nseg = (uint32_t)t->wide_seg.size();
    out.push_back(expect_kernel((const void*)&k_sec_wsum, KB(nseg), kWideTPB, d, (const double*)part,
                                (const uint2*)t->wide, nseg));
    out.push_back(expect_copy(pin + head, dev + 256, 8));
    if (t->ngen) out.push_back(expect_copy(pin + head + 8, dev + head + t->off_gacc, t->ngen * 8));
}

bool inside(const void* p, size_t bytes, const void* base, size_t cap) {
    const uintptr_t a = (uintptr_t)p, b = (uintptr_t)base;
    return a >= b && bytes <= cap && a - b <= cap - bytes;
}

int audit_fail(int grad, size_t node, const std::string& what) {
    return fail(QFE_ERR_STATE, std::string("qfe_template: captured ") + (grad ? "gradient" : "energy") + " sequence, node " +
                                   std::to_string(node) + ": " + what);
}

int audit_graph(qfe_template t, hipGraph_t g, int grad, GraphAudit& A) {
    const size_t head = single_head(t);
    const size_t arena_bytes = head + t->grad_bytes, pin_bytes = head + 8 * (t->ngen + 2);
    const char* dev = (const char*)t->arena;
    // descriptor as the first node uploads it
    SlotDesc d;
    std::memcpy(&d, t->gpin, sizeof(d));
    const char* work = dev + head;
    auto in_work = [&](const void* p, size_t bytes) { return p && inside(p, bytes, work, t->grad_bytes); };
    if (d.t != t->dt || d.out != (double*)(dev + 256) || !in_work(d.psi, t->D * t->amp()) ||
        !in_work(d.sig, t->D * t->amp()) || !in_work(d.cs, (size_t)t->nentries * sizeof(double2)) ||
        !in_work(d.part, (size_t)(t->nitems + t->nrows) * 8) || !in_work(d.gacc, t->ngen * 8) ||
        (t->has_map && !in_work(d.coef, (size_t)t->nterms * t->amp())) || (d.hm && !in_work(d.hm, (size_t)t->nm * 8)) ||
        !inside(d.params, t->io_count * 8, dev + 768, head - 768))
        return audit_fail(grad, 0, "descriptor pointer outside the arena");
    std::vector<NodeExpect> want;
    with_scalar(t, [&](auto z) { expected_nodes<decltype(z)>(t, grad, want); });
    size_t nroot = 0;
    QFE_HIP(hipGraphGetRootNodes(g, nullptr, &nroot));
    if (nroot != 1) return audit_fail(grad, 0, std::to_string(nroot) + " root nodes (expected one chain)");
    hipGraphNode_t node = nullptr;
    QFE_HIP(hipGraphGetRootNodes(g, &node, &nroot));
    const double* part_lo = (const double*)((const char*)t->wide + align256(t->wide_seg.size() * sizeof(uint2)));
    const double* part_hi = part_lo + t->wide_parts;
    A = GraphAudit{};
    for (size_t i = 0;; ++i) {
        if (i >= want.size()) return audit_fail(grad, i, "more nodes than the sequence has launches");
        const NodeExpect& w = want[i];
        hipGraphNodeType type;
        QFE_HIP(hipGraphNodeGetType(node, &type));
        if (w.copy) {
            if (type != hipGraphNodeTypeMemcpy) return audit_fail(grad, i, "expected a memcpy node");
            // the expected copy itself must stay inside the arena and the pinned block
            const bool up = w.dst == t->arena;
            if (up ? !(inside(w.dst, w.bytes, t->arena, arena_bytes) && inside(w.src, w.bytes, t->gpin, pin_bytes))
                   : !(inside(w.src, w.bytes, t->arena, arena_bytes) && inside(w.dst, w.bytes, t->gpin, pin_bytes)))
                return audit_fail(grad, i, "memcpy outside the arena or the pinned block");
            hipMemcpy3DParms p{};
            // a runtime that does not read back captured 1D copies returns null pointers: shape unchecked
            if (hipGraphMemcpyNodeGetParams(node, &p) == hipSuccess && (p.dstPtr.ptr || p.srcPtr.ptr)) {
                // a captured 1D copy reads back as a width-only extent of `bytes`
                const size_t bytes = p.extent.width * std::max<size_t>(1, p.extent.height) * std::max<size_t>(1, p.extent.depth);
                if (p.dstPtr.ptr != w.dst || p.srcPtr.ptr != w.src || bytes != w.bytes)
                    return audit_fail(grad, i, "memcpy addresses or size differ from the sequence");
                ++A.copies_checked;
            }
        } else {
            if (type != hipGraphNodeTypeKernel) return audit_fail(grad, i, "expected a kernel node");
            hipKernelNodeParams p{};
            QFE_HIP(hipGraphKernelNodeGetParams(node, &p));
            if (p.func != w.func) return audit_fail(grad, i, "kernel differs from the sequence");
            if (p.gridDim.x == 0 || p.gridDim.y != 1 || p.gridDim.z != 1 || w.grid == 0)
                return audit_fail(grad, i, "zero or out-of-range grid");
            if (p.blockDim.x == 0 || p.blockDim.x > 1024 || p.blockDim.y != 1 || p.blockDim.z != 1)
                return audit_fail(grad, i, "block outside 1..1024 threads");
            if (p.gridDim.x != w.grid || p.blockDim.x != w.block)
                return audit_fail(grad, i, "launch shape differs from the sequence (grid " + std::to_string(p.gridDim.x) +
                                               ", expected " + std::to_string(w.grid) + ")");
            ++A.kernels;
            // a runtime that keeps no argument copies leaves kernelParams null: shape checked only
            for (size_t a = 0; p.kernelParams && a < w.args.size(); ++a) {
                if (!p.kernelParams[a] || std::memcmp(p.kernelParams[a], w.args[a].data(), w.args[a].size()))
                    return audit_fail(grad, i, "argument " + std::to_string(a) + " differs from the sequence");
                if (w.args[a].size() == sizeof(void*) && w.func != (const void*)&k_sec_wsum) {
                    const double* q;
                    std::memcpy(&q, w.args[a].data(), sizeof(q));
                    // a partial-sum pointer covers one double per workgroup of its launch
                    if (q >= part_lo && q <= part_hi && q + p.gridDim.x > part_hi)
                        return audit_fail(grad, i, "partial sums past the end of the partial array");
                }
            }
            if (p.kernelParams) ++A.kernels_checked;
        }
        size_t ndep = 0;
        QFE_HIP(hipGraphNodeGetDependentNodes(node, nullptr, &ndep));
        if (ndep == 0) {
            if (i + 1 != want.size()) return audit_fail(grad, i, "chain ends before the sequence does");
            A.nodes = i + 1;
            break;
        }
        if (ndep != 1) return audit_fail(grad, i, "node with " + std::to_string(ndep) + " dependents (expected one chain)");
        QFE_HIP(hipGraphNodeGetDependentNodes(node, &node, &ndep));
    }
    return QFE_OK;
}

int graph_build(qfe_template t, int grad) {
    const size_t head = single_head(t);
    int rc = single_arena(t, true);  // of its final size: the captured addresses stay valid
    if (rc) return rc;
    if (!t->wide) {  // partial-sum segments of the step-by-step reverse sweep
        t->wide_seg.assign(1, make_uint2(0, wide_blocks(t->D)));
        uint64_t at = wide_blocks(t->D);
        for (uint64_t k = 0; k < t->ngen; ++k) {
            uint64_t pairs = 0;
            for (uint32_t s = t->h_gen_step[k]; s < t->h_gen_step[k + 1]; ++s) pairs += t->step_pairs[s];
            t->wide_seg.push_back(make_uint2((uint32_t)at, wide_blocks(pairs)));
            at += wide_blocks(pairs);
            if (at >= (1ull << 31)) return fail(QFE_ERR_ARG, "qfe_template_graph_audit: too many partial sums in one sequence");
        }
        t->wide_parts = (uint32_t)at;
        const size_t seg_bytes = align256(t->wide_seg.size() * sizeof(uint2));
        QFE_HIP(device_malloc(&t->wide, seg_bytes + at * 8 + 8));
        QFE_HIP(hipMemcpy(t->wide, t->wide_seg.data(), t->wide_seg.size() * sizeof(uint2), hipMemcpyHostToDevice));
    }
    if (!t->gpin) QFE_HIP(hipHostMalloc(&t->gpin, head + 8 * (t->ngen + 2), hipHostMallocDefault));
    char* dev = (char*)t->arena;
    char* pin = (char*)t->gpin;
    const SlotDesc* ddesc = (const SlotDesc*)dev;
    double* dout = (double*)(dev + 256);
    // descriptor with the gradient parts (the energy sequence ignores them) and the one-slot prefix
    SlotDesc d = make_slot(t, dev + head, (const double*)(dev + 768), dout, true);
    std::memcpy(pin, &d, sizeof(d));
    const uint32_t pre[2] = {0, t->nitems};
    std::memcpy(pin + 512, pre, sizeof(pre));
    hipStream_t st = ctx().stream;
    QFE_HIP(hipStreamSynchronize(st));
    QFE_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
    auto record = [&]() -> int {
        QFE_HIP(hipMemcpyAsync(dev, pin, head, hipMemcpyHostToDevice, st));
        int r = with_scalar(t, [&](auto z) {
            using S = decltype(z);
            return grad ? wide_gradient<S>(t, ddesc, st) : wide_energy<S>(t, ddesc, (const uint32_t*)(dev + 512), st);
        });
        if (r) return r;
        QFE_HIP(hipMemcpyAsync(pin + head, dout, 8, hipMemcpyDeviceToHost, st));
        if (grad && t->ngen)
            QFE_HIP(hipMemcpyAsync(pin + head + 8, dev + head + t->off_gacc, t->ngen * 8, hipMemcpyDeviceToHost, st));
        return QFE_OK;
    };
    rc = record();
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(st, &g);
    if (!rc && e != hipSuccess) rc = hip_fail(e, "qfe_template: end capture");
    if (!rc) {
        const hipError_t ie = hipGraphInstantiate(&t->gexec[grad], g, nullptr, nullptr, 0);
        if (ie != hipSuccess) rc = hip_fail(ie, "qfe_template: instantiate");
    }
    if (!rc) {
        GraphAudit A;
        rc = audit_graph(t, g, grad, A);
        if (!rc) {
            t->audit[grad][0] = A.nodes;
            t->audit[grad][1] = A.kernels;
            t->audit[grad][2] = A.kernels_checked;
            t->audit[grad][3] = A.copies_checked;
        }
    }
    if (rc) {
        if (t->gexec[grad]) (void)hipGraphExecDestroy(t->gexec[grad]);
        if (g) (void)hipGraphDestroy(g);
        t->gexec[grad] = nullptr;
        return rc;
    }
    t->graph[grad] = g;
    return QFE_OK;
}

}  // namespace
}  // namespace qfe

// ---- serving engine -----------------------------------------------------------------------

namespace {

struct Request {
    uint64_t id;
    qfe_template t;
    std::vector<double> params, inputs;
};

struct Lane {
    hipStream_t stream = nullptr;
    hipEvent_t done = nullptr;
    void* dev = nullptr;
    size_t dev_cap = 0;
    void* up = nullptr;
    size_t up_cap = 0;
    double* out = nullptr;
    size_t out_cap = 0;
    std::vector<uint64_t> ids;  // in slot order
    std::vector<qfe_template> ts;
    std::vector<size_t> goff;  // gradient launches: each request's first overlap after the k energies
    bool busy = false;
    bool grad = false;
    int tier = 0;
    uint64_t seq = 0;  // launch order
};

}  // namespace

struct qfe_batch_s {
    uint64_t budget = 0;
    int max_active = 0;
    uint64_t next_id = 1;
    uint64_t active = 0;
    uint64_t seq = 0;
    std::deque<Request> queue[3];   // energy requests, one queue per ansatz tier
    std::deque<Request> gqueue[3];  // energy + gradient requests
    std::vector<Lane> lanes;
    std::deque<std::pair<uint64_t, double>> done;
    std::unordered_map<uint64_t, std::vector<double>> grads;  // completed gradients not yet taken
};

namespace {

// Requests of different tiers never share a launch, so small requests do not
// wait for the longest request of a mixed launch (nor, in tier 2, requests of
// different sector dimensions).  One lane per tier: tier 0
// on the library stream, tiers 1 and 2 on two streams the library creates once
// and every engine shares.  With the null stream (synchronous copies, torch)
// these are four streams, HIP's default four hardware queues per process, so
// no lane shares a queue with another.  Streams that share a queue run one
// kernel at a time between them: with a third lane stream of its own (five
// streams on four queues) the 16-qubit requests of tier 1 waited behind the
// tier-2 launches (p50 13.6 ms at half load, 1.2 ms without), and two lanes
// per tier (six lane streams) gave 13.4 ms p50 over all classes.  Letting two
// lanes take tier-1 and tier-2 launches by age instead (one dimension never on
// both) brought the 18-qubit p50 from 7.7 to 3.6 ms but the 16-qubit one from
// 1.2 to 2.5 ms, and two concurrent tier-2 launches slowed the tier-0 lane:
// 21.2K instead of 21.7K energies/s, p50 45 instead of 3 ms at 1.5x load.
constexpr int kLanesPerTier = 1;
constexpr int kLanes = 3 * kLanesPerTier;

hipStream_t g_lane_stream[kLanes] = {};

int lane_stream(int i, hipStream_t* out) {
    if (i == 0) {  // the tier-0 lane runs on the library stream
        *out = ctx().stream;
        return QFE_OK;
    }
    if (!g_lane_stream[i]) QFE_HIP(hipStreamCreateWithFlags(&g_lane_stream[i], hipStreamNonBlocking));
    *out = g_lane_stream[i];
    return QFE_OK;
}
// A launch admits requests up to this footprint even under a larger budget:
// the requests' states then stay in the 256 MB last-level cache while their
// per-step gathers run (4096 mixed 8-20 qubit requests: 19.5K -> 21.8K
// energies/s and 6.5K -> 7.0K gradients/s against a 64 GiB share).
constexpr uint64_t kLaunchFootprint = 256ull << 20;

template <typename T>
int grow_device(void*& p, size_t& cap, size_t need) {
    if (cap >= need) return QFE_OK;
    if (p) QFE_HIP(hipFree(p));
    p = nullptr;
    cap = 0;
    QFE_HIP(device_malloc(&p, need + need / 4));
    cap = need + need / 4;
    return QFE_OK;
}

int grow_pinned(void*& p, size_t& cap, size_t need) {
    if (cap >= need) return QFE_OK;
    if (p) QFE_HIP(hipHostFree(p));
    p = nullptr;
    cap = 0;
    QFE_HIP(hipHostMalloc(&p, need + need / 4, hipHostMallocDefault));
    cap = need + need / 4;
    return QFE_OK;
}

// Largest launch of gradient requests (the sigma kernel's grid y is the request).
constexpr size_t kMaxGradLaunch = 65535;

int lane_start(qfe_batch b, Lane& L, bool grad, const std::vector<Request>& take);

int lane_launch(qfe_batch b, Lane& L) {
    // a launch holds one kind: the kind whose oldest queued request arrived first
    std::deque<Request>& qe = b->queue[L.tier];
    std::deque<Request>& qg = b->gqueue[L.tier];
    const bool grad = qe.empty() || (!qg.empty() && qg.front().id < qe.front().id);
    std::deque<Request>& queue = grad ? qg : qe;
    // admit from the front of the queue while the footprint fits this lane's
    // share.  A tier-2 launch holds requests of one sector dimension, that of
    // its oldest request: a launch ends with its largest request, and the
    // shorter ones would wait for it; requests of other dimensions keep their
    // place in the queue.
    const uint64_t share = std::min<uint64_t>(b->budget / kLanes, kLaunchFootprint);
    const bool one_dim = L.tier == 2;
    const uint64_t dim0 = queue.front().t->D;
    const bool real0 = queue.front().t->real;  // a launch holds one scalar type
    std::vector<Request> take;
    std::vector<Request> skipped;
    uint64_t foot = 0;
    while (!queue.empty() && (int64_t)(b->active + take.size()) < b->max_active &&
           (!grad || take.size() < kMaxGradLaunch)) {
        if ((one_dim && queue.front().t->D != dim0) || queue.front().t->real != real0) {
            skipped.push_back(std::move(queue.front()));
            queue.pop_front();
            continue;
        }
        const uint64_t f = grad ? queue.front().t->grad_request_bytes : queue.front().t->request_bytes;
        if (!take.empty() && foot + f > share) break;
        foot += f;
        take.push_back(std::move(queue.front()));
        queue.pop_front();
    }
    for (size_t i = skipped.size(); i-- > 0;) queue.push_front(std::move(skipped[i]));
    if (take.empty()) return QFE_OK;
    // heaviest requests first, so their workgroups start first
    std::stable_sort(take.begin(), take.end(), [](const Request& x, const Request& y) { return x.t->cost > y.t->cost; });
    const int rc = lane_start(b, L, grad, take);
    if (rc) {  // no request is lost: they keep their places for a later step
        for (Request& r : take) queue.push_front(std::move(r));
        std::sort(queue.begin(), queue.end(), [](const Request& x, const Request& y) { return x.id < y.id; });
    }
    return rc;
}

int lane_start(qfe_batch b, Lane& L, bool grad, const std::vector<Request>& take) {
    const size_t k = take.size();
    size_t io_total = 0, work_total = 0, gtotal = 0;
    uint64_t items = 0;
    std::vector<qfe_template> ts(k);
    for (size_t i = 0; i < k; ++i) {
        ts[i] = take[i].t;
        io_total += ts[i]->io_count;
        work_total += grad ? ts[i]->grad_bytes : ts[i]->work_bytes;
        items += ts[i]->nitems;
        if (grad) gtotal += ts[i]->ngen;
    }
    if (items >= (1ull << 31)) return fail(QFE_ERR_ARG, "qfe_batch: too many work items in one launch");
    // results: k energies, then the generator overlaps of every gradient request
    const size_t nres = k + gtotal;
    const size_t o_out = align256(k * sizeof(SlotDesc));
    const size_t o_pre = o_out + align256(nres * 8);
    std::vector<uint32_t> tpre;  // tile prefixes: the ansatz passes, then the reverse sweep's
    pass_prefix(ts, false, tpre);
    const size_t nfwd = tpre.size();
    uint32_t row_at = 0;  // row workgroups
    for (size_t i = 0; i <= k; ++i) {
        tpre.push_back(row_at);
        if (i < k) row_at += ts[i]->nrows;
    }
    const size_t nrow = tpre.size();
    if (grad) pass_prefix(ts, true, tpre);
    const size_t o_tpre = o_pre + align256((k + 1) * 4);
    const size_t o_io = o_tpre + align256(tpre.size() * 4);
    const size_t head = o_io + align256(io_total * 8 + 8);
    const size_t need = head + work_total;
    int rc = grow_device<char>(L.dev, L.dev_cap, need);
    if (!rc) rc = grow_pinned(L.up, L.up_cap, head);
    if (!rc) {
        void* p = L.out;
        size_t cap = L.out_cap * 8;
        rc = grow_pinned(p, cap, nres * 8 + 8);
        L.out = (double*)p;
        L.out_cap = cap / 8;
    }
    if (rc) return rc;
    char* dev = (char*)L.dev;
    char* up = (char*)L.up;
    double* dout = (double*)(dev + o_out);
    uint32_t* hpre = (uint32_t*)(up + o_pre);
    size_t io_pos = 0, work_pos = head, gpos = k;
    uint32_t acc_items = 0;
    L.ids.clear();
    L.goff.clear();
    for (size_t i = 0; i < k; ++i) {
        qfe_template t = ts[i];
        const double* dio = (const double*)(dev + o_io) + io_pos;
        double* hio = (double*)(up + o_io) + io_pos;
        SlotDesc d = make_slot(t, dev + work_pos, dio, dout + i, grad);
        if (grad) {
            d.gacc = dout + gpos;
            L.goff.push_back(gpos);
            gpos += t->ngen;
        }
        std::memcpy(up + i * sizeof(SlotDesc), &d, sizeof(d));
        if (t->nparam) std::memcpy(hio, take[i].params.data(), t->nparam * 8);
        if (t->ninputs) std::memcpy(hio + t->nparam, take[i].inputs.data(), t->ninputs * 8);
        hpre[i] = acc_items;
        acc_items += t->nitems;
        io_pos += t->io_count;
        work_pos += grad ? t->grad_bytes : t->work_bytes;
        L.ids.push_back(take[i].id);
    }
    hpre[k] = acc_items;
    std::memcpy(up + o_tpre, tpre.data(), tpre.size() * 4);
    const uint32_t* dtpre = (const uint32_t*)(dev + o_tpre);
    const Prefixes pre{(const uint32_t*)(dev + o_pre), dtpre, dtpre + nfwd, dtpre + nrow};
    QFE_HIP(hipMemcpyAsync(dev, up, head, hipMemcpyHostToDevice, L.stream));
    if (grad)
        rc = launch_gradient(ts, (const SlotDesc*)dev, pre, L.stream);
    else
        rc = launch_energy(ts, (const SlotDesc*)dev, pre, acc_items, L.stream);
    if (rc) return rc;
    QFE_HIP(hipMemcpyAsync(L.out, dout, nres * 8, hipMemcpyDeviceToHost, L.stream));
    QFE_HIP(hipEventRecord(L.done, L.stream));
    L.ts = std::move(ts);
    L.grad = grad;
    L.busy = true;
    L.seq = ++b->seq;
    b->active += k;
    return QFE_OK;
}

void retire(qfe_batch b, Lane& L) {
    for (size_t i = 0; i < L.ids.size(); ++i) b->done.emplace_back(L.ids[i], L.out[i]);
    if (L.grad)
        for (size_t i = 0; i < L.ids.size(); ++i) {
            std::vector<double> g(L.ts[i]->nparam);
            gradient_from_overlaps(L.ts[i], L.out + L.goff[i], g.data());
            b->grads[L.ids[i]] = std::move(g);
        }
    b->active -= L.ids.size();
    L.ids.clear();
    L.busy = false;
}

// Retire every finished launch; with wait_oldest, first block on the oldest
// launch still running.
int collect(qfe_batch b, bool wait_oldest) {
    if (wait_oldest) {
        Lane* oldest = nullptr;
        for (auto& L : b->lanes)
            if (L.busy && (!oldest || L.seq < oldest->seq)) oldest = &L;
        if (oldest) {
            QFE_HIP(hipEventSynchronize(oldest->done));
            retire(b, *oldest);
        }
    }
    for (auto& L : b->lanes) {
        if (!L.busy) continue;
        const hipError_t q = hipEventQuery(L.done);
        if (q == hipErrorNotReady) continue;
        if (q != hipSuccess) return hip_fail(q, "qfe_batch: launch completion");
        retire(b, L);
    }
    return QFE_OK;
}

Request make_request(qfe_batch b, qfe_template t, const double* params, const double* inputs) {
    Request r;
    r.id = b->next_id++;
    r.t = t;
    r.params.assign(params, params + t->nparam);
    if (t->ninputs) r.inputs.assign(inputs, inputs + t->ninputs);
    return r;
}

bool any_busy(qfe_batch b) {
    for (const auto& L : b->lanes)
        if (L.busy) return true;
    return false;
}

int fill_lanes(qfe_batch b) {
    for (auto& L : b->lanes) {
        if (L.busy || (b->queue[L.tier].empty() && b->gqueue[L.tier].empty())) continue;
        int rc = lane_launch(b, L);
        if (rc) return rc;
    }
    return QFE_OK;
}

int hand_out(qfe_batch b, uint64_t* ids, double* es, uint64_t cap, uint64_t* nd) {
    uint64_t k = 0;
    while (k < cap && !b->done.empty()) {
        ids[k] = b->done.front().first;
        es[k] = b->done.front().second;
        b->done.pop_front();
        ++k;
    }
    *nd = k;
    return QFE_OK;
}

}  // namespace

extern "C" {

int qfe_template_create(int nqubit, uint64_t ref_index, const qfe_pauli* gen_terms, const uint64_t* gen_offsets,
                        uint64_t ngen, const int32_t* gen_param, const double* gen_scale, uint64_t nparam,
                        const qfe_pauli* ham_terms, uint64_t nham, const uint64_t* map_offsets,
                        const uint32_t* map_index, const qfe_c64* map_value, uint64_t ninputs, qfe_template* out) {
    if (!out || !gen_offsets || (ngen && (!gen_terms || !gen_param || !gen_scale)) || (nham && !ham_terms))
        return fail(QFE_ERR_ARG, "qfe_template_create: null argument");
    if (map_offsets && (!map_index || !map_value) && map_offsets[nham] > 0)
        return fail(QFE_ERR_ARG, "qfe_template_create: null map arrays");
    if (!map_offsets && ninputs) return fail(QFE_ERR_ARG, "qfe_template_create: inputs need a coefficient map");
    int rc = ensure_init();
    if (rc) return rc;
    qfe_template t = new qfe_template_s();
    rc = template_build(t, nqubit, ref_index, gen_terms, gen_offsets, ngen, gen_param, gen_scale, nparam, ham_terms, nham,
                        map_offsets, map_index, map_value, ninputs);
    if (rc) {
        qfe_template_destroy(t);
        return rc;
    }
    *out = t;
    return QFE_OK;
}

int qfe_template_destroy(qfe_template t) {
    if (!t) return QFE_OK;
    if (ctx().ready) (void)hipStreamSynchronize(ctx().stream);
    if (t->dev) (void)hipFree(t->dev);
    if (t->arena) (void)hipFree(t->arena);
    if (t->wide) (void)hipFree(t->wide);
    for (int k = 0; k < 2; ++k) {
        if (t->gexec[k]) (void)hipGraphExecDestroy(t->gexec[k]);
        if (t->graph[k]) (void)hipGraphDestroy(t->graph[k]);
    }
    if (t->gpin) (void)hipHostFree(t->gpin);
    delete t;
    return QFE_OK;
}

int qfe_template_info(qfe_template t, uint64_t* sector_dim, uint64_t* request_bytes) {
    if (!t) return fail(QFE_ERR_ARG, "qfe_template_info: invalid handle");
    if (sector_dim) *sector_dim = t->D;
    if (request_bytes) *request_bytes = t->request_bytes;
    return QFE_OK;
}

int qfe_template_graph_audit(qfe_template t, int gradient, uint64_t* out4) {
    if (!t || !out4 || (gradient != 0 && gradient != 1)) return fail(QFE_ERR_ARG, "qfe_template_graph_audit: invalid argument");
    for (int k = 0; k < 4; ++k) out4[k] = 0;
    if (t->tier != 2) return QFE_OK;  // one-workgroup sequences are launched directly, never captured
    if (!t->gexec[gradient]) {
        int rc = graph_build(t, gradient);
        if (rc) return rc;
    }
    for (int k = 0; k < 4; ++k) out4[k] = t->audit[gradient][k];
    return QFE_OK;
}

int qfe_template_energy(qfe_template t, const double* params, const double* inputs, double* energy) {
    if (!t || !energy || (t->nparam && !params) || (t->ninputs && !inputs))
        return fail(QFE_ERR_ARG, "qfe_template_energy: null argument");
    Single S;
    int rc = single_setup(t, params, inputs, false, S);
    if (rc) return rc;
    rc = launch_energy({t}, S.ddesc, Prefixes{S.dprefix, nullptr, nullptr, nullptr}, t->nitems, ctx().stream);
    if (rc) return rc;
    return fetch_doubles(S.dout, 1, energy);
}

int qfe_template_prepare(qfe_template t, const double* params, qfe_state out) {
    if (!t || !out || (t->nparam && !params)) return fail(QFE_ERR_ARG, "qfe_template_prepare: null argument");
    if (out->n != t->n) return fail(QFE_ERR_ARG, "qfe_template_prepare: state has the wrong number of qubits");
    std::vector<double> zeros(t->ninputs + 1, 0.0);
    Single S;
    int rc = single_setup(t, params, zeros.data(), false, S);
    if (rc) return rc;
    hipStream_t st = ctx().stream;
    rc = launch_prologue({t}, S.ddesc, 0, st);
    if (!rc) rc = launch_tiles<0>({t}, S.ddesc, nullptr, st);
    if (!rc) rc = launch_zero(out->d, out->N, st);
    if (rc) return rc;
    with_scalar(t, [&](auto z) {
        using A = decltype(z);
        hipLaunchKernelGGL(k_sector_scatter<A>, dim3((unsigned)((t->D + 255) / 256)), dim3(256), 0, st,
                           (const A*)(S.work + t->off_psi), t->D, t->Db, t->afull, t->bfull, out->d);
    });
    QFE_HIP(hipGetLastError());
    return QFE_OK;
}

int qfe_template_gradient(qfe_template t, const double* params, const double* inputs, double* grad, double* energy) {
    if (!t || !grad || (t->nparam && !params) || (t->ninputs && !inputs))
        return fail(QFE_ERR_ARG, "qfe_template_gradient: null argument");
    std::vector<double> acc(t->ngen + 1);
    Single S;
    int rc = single_setup(t, params, inputs, true, S);
    if (!rc) rc = launch_gradient({t}, S.ddesc, Prefixes{}, ctx().stream);
    if (rc) return rc;
    rc = fetch_doubles((const double*)(S.work + t->off_gacc), t->ngen, acc.data());
    if (!rc) rc = fetch_doubles(S.dout, 1, &acc[t->ngen]);
    if (rc) return rc;
    gradient_from_overlaps(t, acc.data(), grad);
    if (energy) *energy = acc[t->ngen];
    return QFE_OK;
}

int qfe_template_residuals(qfe_template t, const double* params, const double* inputs, const uint64_t* idx,
                           uint64_t count, qfe_c64* out) {
    if (!t || (count && (!idx || !out)) || (t->nparam && !params) || (t->ninputs && !inputs))
        return fail(QFE_ERR_ARG, "qfe_template_residuals: null argument");
    std::vector<uint64_t> rank(count);
    for (uint64_t i = 0; i < count; ++i) {
        if (idx[i] >> t->n) return fail(QFE_ERR_ARG, "qfe_template_residuals: basis index out of range");
        const int32_t ra = t->sp.rank[0][compress(idx[i], 0, t->norb)];
        const int32_t rb = t->sp.rank[1][compress(idx[i], 1, t->norb)];
        if (ra < 0 || rb < 0) return fail(QFE_ERR_ARG, "qfe_template_residuals: basis index outside the sector");
        rank[i] = (uint64_t)ra * t->Db + (uint64_t)rb;
    }
    // sigma = H U|ref>, then U^dag on sigma: every step inverted, last step first
    Single S;
    int rc = single_psi_sigma(t, params, inputs, S);
    if (rc) return rc;
    hipStream_t st = ctx().stream;
    rc = launch_tiles<1>({t}, S.ddesc, nullptr, st);
    if (rc) return rc;
    if (!count) return QFE_OK;
    void* scratch = nullptr;
    const size_t o_out = align256(count * 8);
    rc = scratch_reserve(o_out + count * sizeof(double2), &scratch);
    if (rc) return rc;
    QFE_HIP(hipMemcpyAsync(scratch, rank.data(), count * 8, hipMemcpyHostToDevice, st));
    double2* dres = (double2*)((char*)scratch + o_out);
    with_scalar(t, [&](auto z) {
        hipLaunchKernelGGL(k_sec_gather<decltype(z)>, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, S.ddesc,
                           (const uint64_t*)scratch, count, dres);
    });
    QFE_HIP(hipGetLastError());
    QFE_HIP(hipMemcpyAsync(out, dres, count * sizeof(double2), hipMemcpyDeviceToHost, st));
    QFE_HIP(hipStreamSynchronize(st));
    return QFE_OK;
}

// Largest tables of a pool-gradient call that go through the kept scratch and
// staging: an allocation and its release cost the 14-qubit call (0.4 MiB) more
// than its kernel, and nothing next to tables above this.
constexpr size_t kPoolKeep = 16u << 20;

int qfe_template_pool_gradients(qfe_template t, const double* params, const double* inputs, const qfe_pauli* pool_terms,
                                const uint64_t* op_offsets, uint64_t nops, uint64_t batch, double* grads) {
    if (!t || (nops && (!pool_terms || !op_offsets || !grads)) || (t->nparam && !params) || (t->ninputs && !inputs))
        return fail(QFE_ERR_ARG, "qfe_template_pool_gradients: null argument");
    (void)batch;
    // pool operators as pair rotations on the template's sector
    ListPool lp;
    std::vector<SecStep> steps;
    std::vector<SecEntry> entries;
    std::vector<PoolOp> ops(nops);
    const uint64_t lim = (1ull << t->n) - 1ull;
    for (uint64_t o = 0; o < nops; ++o) {
        if (op_offsets[o + 1] < op_offsets[o]) return fail(QFE_ERR_ARG, "qfe_template_pool_gradients: offsets must not decrease");
        ops[o].e0 = (uint32_t)entries.size();
        int rc = build_runs(t->sp, lp, t->norb, lim, pool_terms, op_offsets[o], op_offsets[o + 1], 0, 1.0, (uint32_t)o, steps,
                            entries, "qfe_template_pool_gradients");
        if (rc) return rc;
        ops[o].e1 = (uint32_t)entries.size();
    }
    Single S;
    int rc = single_psi_sigma(t, params, inputs, S);
    if (rc) return rc;
    Packer pk(0);
    const size_t i_l = pk.add(lp.pool.data(), lp.pool.size() * sizeof(int2));
    const size_t i_e = pk.add(entries.data(), entries.size() * sizeof(SecEntry));
    const size_t i_o = pk.add(ops.data(), ops.size() * sizeof(PoolOp));
    const size_t o_out = pk.total;
    const size_t total = o_out + align256(nops * 8 + 8);
    // The tables of the call go through the context's staging and scratch; above
    // kPoolKeep they get memory of their own, given back at the end.
    void* dev = nullptr;
    const bool keep = total <= kPoolKeep;
    std::vector<char> img;
    if (keep) {
        rc = scratch_reserve(total, &dev);
        if (rc) return rc;
        void* host = nullptr;
        rc = staging_begin(pk.total, &host);
        if (rc) return rc;
        pk.fill(static_cast<char*>(host));
        rc = staging_commit(dev, pk.total);
        if (rc) return rc;
    } else {
        QFE_HIP(device_malloc(&dev, total));
        img.resize(pk.total);
        pk.fill(img.data());
        const hipError_t e = hipMemcpy(dev, img.data(), pk.total, hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            (void)hipFree(dev);
            return hip_fail(e, "qfe_template_pool_gradients: upload");
        }
    }
    char* base = (char*)dev;
    // One workgroup per operator and all of them in one launch: an operator needs
    // no memory of its own, so `batch` bounds nothing here (1638 operators at 14
    // qubits in launches of 64 left three CUs of four idle).
    hipError_t e = hipSuccess;
    constexpr uint64_t kGridMax = 1u << 30;
    for (uint64_t b0 = 0; b0 < nops && e == hipSuccess; b0 += kGridMax) {
        const uint64_t b1 = std::min(nops, b0 + kGridMax);
        with_scalar(t, [&](auto z) {
            using A = decltype(z);
            hipLaunchKernelGGL(k_sec_pool<A>, dim3((unsigned)(b1 - b0)), dim3(256), 0, ctx().stream, t->dt,
                               (const SecEntry*)(base + pk.pieces[i_e].off), (const int2*)(base + pk.pieces[i_l].off),
                               (const PoolOp*)(base + pk.pieces[i_o].off) + b0, (const A*)(S.work + t->off_sig),
                               (const A*)(S.work + t->off_psi), (double*)(base + o_out) + b0);
        });
        e = hipGetLastError();
    }
    rc = e != hipSuccess ? hip_fail(e, "qfe_template_pool_gradients: launch")
                         : nops ? fetch_doubles((const double*)(base + o_out), nops, grads) : QFE_OK;
    if (!keep) {
        (void)hipStreamSynchronize(ctx().stream);
        (void)hipFree(dev);
    }
    return rc;
}

int qfe_batch_create(uint64_t hbm_budget_bytes, int max_active, qfe_batch* out) {
    if (!out || max_active < 1 || hbm_budget_bytes == 0) return fail(QFE_ERR_ARG, "qfe_batch_create: invalid argument");
    int rc = ensure_init();
    if (rc) return rc;
    qfe_batch b = new qfe_batch_s();
    b->budget = hbm_budget_bytes;
    b->max_active = max_active;
    b->lanes.resize(kLanes);
    for (int i = 0; i < kLanes; ++i) {
        Lane& L = b->lanes[i];
        L.tier = i / kLanesPerTier;
        rc = lane_stream(i, &L.stream);
        if (rc) {
            qfe_batch_destroy(b);
            return rc;
        }
        const hipError_t e = hipEventCreateWithFlags(&L.done, hipEventDisableTiming);
        if (e != hipSuccess) {
            qfe_batch_destroy(b);
            return hip_fail(e, "qfe_batch_create");
        }
    }
    *out = b;
    return QFE_OK;
}

int qfe_batch_destroy(qfe_batch b) {
    if (!b) return QFE_OK;
    for (auto& L : b->lanes) {
        // the lane streams are shared by every engine: wait for this engine's own last launch only
        if (L.busy && L.done) (void)hipEventSynchronize(L.done);
        if (L.dev) (void)hipFree(L.dev);
        if (L.up) (void)hipHostFree(L.up);
        if (L.out) (void)hipHostFree(L.out);
        if (L.done) (void)hipEventDestroy(L.done);
    }
    delete b;
    return QFE_OK;
}

int qfe_batch_submit(qfe_batch b, qfe_template t, const double* params, const double* inputs, uint64_t* request_id) {
    if (!b || !t || !request_id) return fail(QFE_ERR_ARG, "qfe_batch_submit: invalid argument");
    if ((t->nparam && !params) || (t->ninputs && !inputs)) return fail(QFE_ERR_ARG, "qfe_batch_submit: null parameters");
    if (t->request_bytes > b->budget / kLanes)
        return fail(QFE_ERR_ARG, "qfe_batch_submit: one request exceeds the per-launch share of the HBM budget");
    b->queue[t->tier].push_back(make_request(b, t, params, inputs));
    *request_id = b->queue[t->tier].back().id;
    return QFE_OK;
}

int qfe_batch_submit_gradient(qfe_batch b, qfe_template t, const double* params, const double* inputs,
                              uint64_t* request_id) {
    if (!b || !t || !request_id) return fail(QFE_ERR_ARG, "qfe_batch_submit_gradient: invalid argument");
    if ((t->nparam && !params) || (t->ninputs && !inputs))
        return fail(QFE_ERR_ARG, "qfe_batch_submit_gradient: null parameters");
    if (t->grad_least_bytes > b->budget / kLanes)
        return fail(QFE_ERR_ARG, "qfe_batch_submit_gradient: one request exceeds the per-launch share of the HBM budget");
    b->gqueue[t->tier].push_back(make_request(b, t, params, inputs));
    *request_id = b->gqueue[t->tier].back().id;
    return QFE_OK;
}

int qfe_batch_take_gradient(qfe_batch b, uint64_t request_id, double* grad, uint64_t nparam) {
    if (!b || (nparam && !grad)) return fail(QFE_ERR_ARG, "qfe_batch_take_gradient: invalid argument");
    auto it = b->grads.find(request_id);
    if (it == b->grads.end())
        return fail(QFE_ERR_ARG, "qfe_batch_take_gradient: no completed gradient request with this id");
    if (it->second.size() != nparam) return fail(QFE_ERR_ARG, "qfe_batch_take_gradient: wrong gradient length");
    std::copy(it->second.begin(), it->second.end(), grad);
    b->grads.erase(it);
    return QFE_OK;
}

int qfe_batch_poll(qfe_batch b, uint64_t* done_ids, double* done_energies, uint64_t cap, uint64_t* ndone) {
    if (!b || !ndone || (cap && (!done_ids || !done_energies))) return fail(QFE_ERR_ARG, "qfe_batch_poll: invalid argument");
    int rc = collect(b, false);
    if (!rc) rc = fill_lanes(b);
    if (rc) return rc;
    return hand_out(b, done_ids, done_energies, cap, ndone);
}

int qfe_batch_step(qfe_batch b, uint64_t* done_ids, double* done_energies, uint64_t cap, uint64_t* ndone) {
    if (!b || !ndone || (cap && (!done_ids || !done_energies))) return fail(QFE_ERR_ARG, "qfe_batch_step: invalid argument");
    int rc = collect(b, false);
    if (!rc) rc = fill_lanes(b);
    if (!rc && b->done.empty() && any_busy(b)) {
        rc = collect(b, true);
        if (!rc) rc = fill_lanes(b);
    }
    if (rc) return rc;
    return hand_out(b, done_ids, done_energies, cap, ndone);
}

int qfe_batch_pending(qfe_batch b, uint64_t* queued, uint64_t* active) {
    if (!b) return fail(QFE_ERR_ARG, "qfe_batch_pending: invalid handle");
    if (queued) {
        *queued = 0;
        for (int i = 0; i < 3; ++i) *queued += b->queue[i].size() + b->gqueue[i].size();
    }
    if (active) *active = b->active + b->done.size();
    return QFE_OK;
}

}  // extern "C"
