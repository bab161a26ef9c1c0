// Gate circuits on small states as rounds of register orbits.
//
// X, CNOT and SWAP gates move no amplitude: the host keeps the affine frame
// they make, p = stored index of logical index l, with col[q] the flip of
// logical qubit q in stored indexes and row[q] the functional that reads it
// (row_a . col_b = delta_ab over GF(2)).  Every other gate becomes, in stored
// coordinates, a rotation R on pairs (p, p ^ x) whose role bit is the parity
// of p & f, and phases D that depend on parities of p: a one-qubit matrix is
// diag * rotation * diag, and all of a qubit's matrices between two-qubit
// gates are multiplied first.  A phase whose parities are constant on an orbit
// is one complex factor per thread, so half of a circuit's gates cost a few
// instructions per 16 amplitudes.
//
// A tile is a coset of a space of stored indexes, 2^k amplitudes in LDS.  One
// round is one trip of the tile through registers: up to four rotations with
// flips b_k and functionals r_k, r_j . b_k = delta_jk, so a thread that owns an
// orbit {j ^ span b} applies them at compile-time element pairs, and one
// barrier.  Pass by pass the tiles follow the gates that are ready; the last
// pass stores every amplitude at its logical index.
//
// A round is bound by its chain: the tile's trip through LDS (0.75 us of the
// 1.7 us at 12-bit tiles), the phase tables and the rotations (0.5 us each, FP64
// at one wave per SIMD).  500 random gates on 12 qubits are 28 rounds in one
// launch of one workgroup, 55 us (15 launches of gate-by-gate 8-qubit tiles on
// 16 workgroups: 374 us); 800 on 17 qubits six launches of 20 us (27 of 30 us).
// On states beyond 22 qubits every tile pass is planned on its own and works in
// place (a move's target lies in the tile, so its frame stays in the coset), with
// 11-bit tiles, three flips a round and 8 amplitudes per thread: four waves per
// SIMD hide the rounds' chain behind the other tiles' loads.  Brickwork of 4 layers at 29 qubits: four passes of 7.1 ms
// (nine of 4.6 ms gate by gate; a bare read and write takes 3.4 ms).
// Tiles of 11 or 13 bits (2^(k - 4) threads) were level or slower from 15 qubits
// on: 13 bits halve the workgroups, 11 bits add passes.  64-byte runs against 128:
// 15-20 qubits 2-10 % faster, since a pass has one more free flip.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "qfe_device.h"
#include "qfe_internal.h"

namespace qfe {

namespace {

constexpr int kRoundDims = 4;                        // flips per round: 16 amplitudes per thread
constexpr int kLargeDims = kLargeRoundTile - 8;      // on large states, where waves matter more: 8 amplitudes
constexpr int kRoundLow = 2;                         // lowest index bits in every tile: runs of 64 bytes
constexpr int kOrbitBits = kRoundTileMax - kRoundDims;  // a full tile has 2^8 orbits of 16,
constexpr int kRoundTPB = 1 << kOrbitBits;              // one per thread
constexpr uint32_t kChunkWords = 2 * kRoundTPB;      // 8 KiB of the program staged in LDS at a time
constexpr uint32_t kRoundWords = 6;                  // 16-byte words of a round: header, roles, (cos, sin) of four axes
constexpr uint32_t kPhaseWords = 17, kRotWords = 2;  // of a phase table and of a further rotation
constexpr int kPhaseBits = 4;                        // parities of one phase table (16 factors)
constexpr int kPhasesMax = 16, kRotsMax = 16;        // gates per round: 6 + 16 * 17 + 16 * 2 words fit a chunk

__device__ __forceinline__ uint32_t parity32(uint32_t v) { return (uint32_t)__popc(v) & 1u; }
__device__ __forceinline__ uint32_t sgpr(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// Rotation (c, s) along axis AX of 2^G elements.
template <int G, int AX>
__device__ __forceinline__ void rotate(double2 (&a)[1 << G], double c, double s) {
#pragma unroll
    for (int i = 0; i < (1 << G); ++i) {
        if (i & (1 << AX)) continue;
        const double2 x = a[i], y = a[i | (1 << AX)];
        a[i] = make_double2(fma(-s, y.x, c * x.x), fma(-s, y.y, c * x.y));
        a[i | (1 << AX)] = make_double2(fma(s, x.x, c * y.x), fma(s, x.y, c * y.y));
    }
}

// Factor of a phase table at buf[w] for the thread's parities.
__device__ __forceinline__ double2 phase_of(const uint4* buf, uint32_t w, uint32_t J) {
    const uint4 f = buf[w];
    const uint32_t idx = parity32(f.x & J) | (parity32(f.y & J) << 1) | (parity32(f.z & J) << 2) | (parity32(f.w & J) << 3);
    return reinterpret_cast<const double2*>(buf + w + 1)[idx];
}

// One round of G flips whose record starts at buf[at] (its header is h).  The
// first unconditional rotation of every axis has a place of its own, so its
// data is read ahead of the tile and its axis is known at compile time; the
// others follow in a list.
template <int G>
__device__ __forceinline__ void round_body(double2* tile, const uint4* buf, uint32_t at, uint4 h, uint32_t k, uint32_t number) {
    const uint32_t norb = (1u << k) >> G;
    if (threadIdx.x >= norb) return;
    const uint32_t np = (h.x >> 8) & 0xFFu, nr = (h.x >> 16) & 0xFFu, first = h.x >> 24;
    const uint4 role = buf[at + 1];
    double2 cs[4];
#pragma unroll
    for (int d = 0; d < G; ++d) cs[d] = reinterpret_cast<const double2*>(buf)[at + 2 + d];
    uint32_t j = threadIdx.x;
#pragma unroll
    for (int d = 0; d < G; ++d) j = ins0_32(j, (h.y >> (8 * d)) & 0xFFu);
    const uint32_t J = j | (number << k);
    const uint32_t b[4] = {h.z & 0xFFFFu, h.z >> 16, h.w & 0xFFFFu, h.w >> 16};
    uint32_t q[1 << G];
    double2 a[1 << G];
#pragma unroll
    for (int i = 0; i < (1 << G); ++i) {
        uint32_t o = 0;
#pragma unroll
        for (int d = 0; d < G; ++d)
            if (i & (1 << d)) o ^= b[d];
        q[i] = j ^ o;
        a[i] = tile[q[i]];
    }
    uint32_t w = at + kRoundWords;
    double2 ph = make_double2(1.0, 0.0);
    if (np) {
        ph = phase_of(buf, w, J);
        w += kPhaseWords;
        uint32_t p = 1;
        for (; p + 2 <= np; p += 2, w += 2 * kPhaseWords) {
            const double2 u = phase_of(buf, w, J), v = phase_of(buf, w + kPhaseWords, J);
            ph = cmul(ph, cmul(u, v));
        }
        if (p < np) {
            ph = cmul(ph, phase_of(buf, w, J));
            w += kPhaseWords;
        }
    }
    const uint32_t rf[4] = {role.x, role.y, role.z, role.w};
    auto signed_sin = [&](int d) { return parity32(rf[d] & J) ? -cs[d].y : cs[d].y; };
    if constexpr (G > 0)
        if (first & 1u) rotate<G, 0>(a, cs[0].x, signed_sin(0));
    if constexpr (G > 1)
        if (first & 2u) rotate<G, 1>(a, cs[1].x, signed_sin(1));
    if constexpr (G > 2)
        if (first & 4u) rotate<G, 2>(a, cs[2].x, signed_sin(2));
    if constexpr (G > 3)
        if (first & 8u) rotate<G, 3>(a, cs[3].x, signed_sin(3));
    for (uint32_t r = 0; r < nr; ++r, w += kRotWords) {
        const uint4 f = buf[w];
        const double2 x = reinterpret_cast<const double2*>(buf)[w + 1];
        double c = x.x, sn = parity32(f.x & J) ? -x.y : x.y;
        const uint32_t mode = sgpr(f.z);
        if (mode & 0x100u) {  // under a condition
            const bool on = parity32(f.y & J) == ((mode >> 9) & 1u);
            c = on ? c : 1.0;
            sn = on ? sn : 0.0;
        }
        switch (mode & 3u) {
            case 0:
                if constexpr (G > 0) rotate<G, 0>(a, c, sn);
                break;
            case 1:
                if constexpr (G > 1) rotate<G, 1>(a, c, sn);
                break;
            case 2:
                if constexpr (G > 2) rotate<G, 2>(a, c, sn);
                break;
            default:
                if constexpr (G > 3) rotate<G, 3>(a, c, sn);
                break;
        }
    }
    if (np) {
#pragma unroll
        for (int i = 0; i < (1 << G); ++i) a[i] = cmul(ph, a[i]);
    }
#pragma unroll
    for (int i = 0; i < (1 << G); ++i) tile[q[i]] = a[i];
}

// DIMS: most flips of a round (registers); NT: non-temporal accesses.
template <int DIMS, bool NT>
__global__ __launch_bounds__(kRoundTPB) __attribute__((amdgpu_waves_per_eu(DIMS > 3 ? 2 : 4))) void k_rounds(const double2* src, double2* dst, const RoundsPass P,
                                                      const uint4* __restrict__ prog) {
    extern __shared__ double2 tile[];
    const uint32_t T = 1u << P.k, tid = threadIdx.x, number = (uint32_t)xcd_block();
    uint4* buf = reinterpret_cast<uint4*>(tile + T);
    uint32_t sb = 0, wb = P.w0;
#pragma unroll
    for (int u = 0; u < 32 - kLargeRoundTile; ++u) {
        sb ^= ((number >> u) & 1u) ? P.sq[u] : 0u;
        wb ^= ((number >> u) & 1u) ? P.wq[u] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kOrbitBits; ++i) {
        sb ^= ((tid >> i) & 1u) ? P.sv[i] : 0u;
        wb ^= ((tid >> i) & 1u) ? P.wv[i] : 0u;
    }
    auto upper = [](uint32_t r, const uint32_t (&v)[kRoundTileMax]) {  // tile bits above a thread's number
        uint32_t x = 0;
#pragma unroll
        for (int i = kOrbitBits; i < kRoundTileMax; ++i) x ^= ((r >> (i - kOrbitBits)) & 1u) ? v[i] : 0u;
        return x;
    };
    static_assert(kChunkWords == 2 * kRoundTPB, "two words per thread");
    uint4 next0 = make_uint4(0, 0, 0, 0), next1 = next0;
    if (P.chunks) {
        next0 = prog[tid];
        next1 = prog[tid + kRoundTPB];
    }
    const uint32_t rows = (T + kRoundTPB - 1) / kRoundTPB;
#pragma unroll 8
    for (uint32_t r = 0; r < rows; ++r)
        if (tid < T) tile[tid + r * kRoundTPB] = ld_s<NT>(src + (sb ^ upper(r, P.sv)));
    for (uint32_t c = 0; c < P.chunks; ++c) {
        // the rounds of the chunk before have ended (their last barrier)
        buf[tid] = next0;
        buf[tid + kRoundTPB] = next1;
        if (c + 1 < P.chunks) {
            next0 = prog[(c + 1) * kChunkWords + tid];
            next1 = prog[(c + 1) * kChunkWords + tid + kRoundTPB];
        }
        __syncthreads();
        const uint32_t rounds = sgpr(buf[0].x);
        uint32_t at = 1;
        uint4 h = buf[at];
        for (uint32_t r = 0; r < rounds; ++r) {
            h = make_uint4(sgpr(h.x), sgpr(h.y), sgpr(h.z), sgpr(h.w));
            switch (h.x & 0xFFu) {
                case 0: round_body<0>(tile, buf, at, h, P.k, number); break;
                case 1: round_body<1>(tile, buf, at, h, P.k, number); break;
                case 2: round_body<2>(tile, buf, at, h, P.k, number); break;
                case 3: round_body<3>(tile, buf, at, h, P.k, number); break;
                default:
                    if constexpr (DIMS > 3) round_body<4>(tile, buf, at, h, P.k, number);
                    break;
            }
            at += kRoundWords + ((h.x >> 8) & 0xFFu) * kPhaseWords + ((h.x >> 16) & 0xFFu) * kRotWords;
            h = buf[min(at, kChunkWords - 1u)];  // the next header, if there is one
            __syncthreads();
        }
    }
    __syncthreads();
#pragma unroll 8
    for (uint32_t r = 0; r < rows; ++r)
        if (tid < T) st_s<NT>(dst + (wb ^ upper(r, P.wv)), tile[tid + r * kRoundTPB]);
}

// ---- host: gates to rotations and phases in stored coordinates ------------------------

// Products of gates and of phases are formed in extended precision and rounded
// once, as the (cos, sin) and the table entries of the program: in double, the
// products' own roundings made the amplitudes' error 1.2 to 2 times that of the
// gates applied one by one.
struct Z {
    long double x, y;
};
constexpr Z kOne = {1.0L, 0.0L}, kZero = {0.0L, 0.0L};
Z wide(double2 a) { return {a.x, a.y}; }
double2 narrow(Z a) { return make_double2((double)a.x, (double)a.y); }
inline Z zmul(Z a, Z b) {
    if (a.y == 0.0L) return {a.x * b.x, a.x * b.y};  // real factors are common
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
Z zadd(Z a, Z b) { return {a.x + b.x, a.y + b.y}; }
Z zconj(Z a) { return {a.x, -a.y}; }
Z zneg(Z a) { return {-a.x, -a.y}; }
long double zabs(Z a) { return sqrtl(a.x * a.x + a.y * a.y); }
bool zis(Z a, double re) { return a.x == re && a.y == 0.0L; }

struct RoundOp {
    uint32_t x;       // rotation: flip; 0: phase
    uint32_t f0, f1;  // rotation: role and condition (0: none); phase: its parities (0: none)
    bool want;        // rotation: value of the condition's parity
    double c, s;
    uint32_t tab;     // phase: first of its four factors, by parity of f0 (bit 0) and f1 (bit 1)
};

// m = diag(l) [[c, -s], [s, c]] diag(1, r); false when m is not unitary to
// 1e-15 (no such form then).
bool split_rotation(const Z m[4], Z l[2], double& c, double& s, Z& r) {
    long double n[4];
    for (int i = 0; i < 4; ++i) n[i] = zabs(m[i]);
    auto unit = [](Z v, long double a) { return Z{v.x / a, v.y / a}; };
    l[0] = n[0] > 0.0L ? unit(m[0], n[0]) : kOne;
    l[1] = n[2] > 0.0L ? unit(m[2], n[2]) : kOne;
    if (!(n[0] > 0.0L)) r = n[1] > 0.0L ? unit(zneg(m[1]), n[1]) : kOne;
    else if (!(n[2] > 0.0L)) r = n[3] > 0.0L ? unit(zmul(m[3], zconj(l[0])), n[3]) : kOne;
    else if (n[1] >= n[3]) r = unit(zmul(zneg(m[1]), zconj(l[0])), n[1]);
    else r = unit(zmul(m[3], zconj(l[1])), n[3]);
    if (!(n[2] > 0.0L)) l[1] = l[0];
    c = (double)n[0];
    s = (double)n[2];
    const Z a1 = zmul(l[0], r), a3 = zmul(l[1], r);
    const long double e[8] = {l[0].x * n[0] - m[0].x, l[0].y * n[0] - m[0].y, -a1.x * n[2] - m[1].x, -a1.y * n[2] - m[1].y,
                              l[1].x * n[2] - m[2].x, l[1].y * n[2] - m[2].y, a3.x * n[0] - m[3].x, a3.y * n[0] - m[3].y};
    for (long double v : e)
        if (!(fabsl(v) <= 1e-15L)) return false;
    return true;
}

// Whether an op is a gate that the lowering below takes (a matrix that turns out
// not to be unitary aside): general two-qubit matrices, exponentials and gates
// under several conditions are not.
bool has_form(const DevOp& o) {
    if (o.kind == K_U2) {
        // a swap, or a gate under "qubit c reads 0" (rows and columns 2c + t)
        for (int r = 0; r < 4 && !o.hb; ++r)
            for (int c = 0; c < 4; ++c)
                if ((r > 1 || c > 1) && !zis(wide(o.m[4 * r + c]), r == c ? 1.0 : 0.0)) return false;
        return true;
    }
    return (o.kind == K_U1 || o.kind == K_DIAG1) && __builtin_popcountll(o.cmask) <= 1;
}

struct FrameLowering {
    int n;
    uint32_t col[32], row[32];
    uint32_t neg = 0;  // bit q: logical qubit q reads inverted
    Z acc[32][4];
    uint8_t kind[32];   // of acc: 0 identity, 1 diagonal, 2 antidiagonal, 3 dense
    uint8_t chain[32];  // gates multiplied since the last split for length
    std::vector<RoundOp> out;
    std::vector<Z> tabs;

    explicit FrameLowering(int nq) : n(nq) {
        for (int q = 0; q < n; ++q) {
            col[q] = row[q] = 1u << q;
            kind[q] = chain[q] = 0;
        }
    }
    void classify(int q) {
        const Z* m = acc[q];
        const bool off = !(zis(m[1], 0.0) && zis(m[2], 0.0)), dia = !(zis(m[0], 0.0) && zis(m[3], 0.0));
        kind[q] = off ? (dia ? 3 : 2) : (zis(m[0], 1.0) && zis(m[3], 1.0) ? 0 : 1);
    }
    void set_diag(int q, Z a, Z b) {
        acc[q][0] = a;
        acc[q][1] = acc[q][2] = kZero;
        acc[q][3] = b;
        classify(q);
    }
    void multiply(int q, const Z m[4]) {
        Z* a = acc[q];
        if (!kind[q]) {
            for (int i = 0; i < 4; ++i) a[i] = m[i];
        } else if (zis(m[1], 0.0) && zis(m[2], 0.0)) {
            for (int i = 0; i < 4; ++i) {
                if (kind[q] == 1 && (i == 1 || i == 2)) continue;
                const Z f = m[i < 2 ? 0 : 3];
                if (!zis(f, 1.0)) a[i] = zmul(f, a[i]);
            }
        } else if (kind[q] == 1) {
            const Z d[2] = {a[0], a[3]};
            const bool same[2] = {zis(d[0], 1.0), zis(d[1], 1.0)};
            for (int i = 0; i < 4; ++i) a[i] = same[i & 1] ? m[i] : zmul(m[i], d[i & 1]);
        } else {
            Z r[4];
            for (int i = 0; i < 4; ++i) r[i] = zadd(zmul(m[i & 2], a[i & 1]), zmul(m[(i & 2) + 1], a[2 + (i & 1)]));
            for (int i = 0; i < 4; ++i) a[i] = r[i];
        }
        classify(q);
    }
    // diag(a, b) on qubit t, where qubit c (if any) reads cv
    void phase(int t, int c, bool cv, Z a, Z b) {
        if (zis(a, 1.0) && zis(b, 1.0)) return;
        RoundOp o{};
        const bool nt = (neg >> t) & 1u;
        o.f0 = row[t];
        o.f1 = c >= 0 ? row[c] : 0u;
        o.tab = (uint32_t)tabs.size();
        for (int i = 0; i < 4; ++i) {
            const bool on = c < 0 || (((i >> 1) & 1) != 0) == (cv != (((neg >> c) & 1u) != 0));
            tabs.push_back(on ? ((((i & 1) != 0) != nt) ? b : a) : kOne);
        }
        out.push_back(o);
    }
    void rotation(int t, int c, bool cv, double cs, double sn) {
        RoundOp o{};
        o.x = col[t];
        o.f0 = row[t];
        o.f1 = c >= 0 ? row[c] : 0u;
        o.want = c >= 0 && (cv != (((neg >> c) & 1u) != 0));
        o.c = cs;
        o.s = ((neg >> t) & 1u) ? -sn : sn;
        out.push_back(o);
    }
    void cnot(int t, int c, bool cv) {
        row[t] ^= row[c];
        col[c] ^= col[t];
        neg ^= (((neg >> c) ^ (cv ? 0u : 1u)) & 1u) << t;
    }
    // leave qubit q with a diagonal (or no) matrix to come
    bool flush_dense(int q) {
        if (kind[q] == 2) {
            neg ^= 1u << q;
            set_diag(q, acc[q][1], acc[q][2]);
        } else if (kind[q] == 3) {
            Z l[2], r;
            double c, s;
            if (!split_rotation(acc[q], l, c, s, r)) return false;
            phase(q, -1, false, kOne, r);
            rotation(q, -1, false, c, s);
            set_diag(q, l[0], l[1]);
        }
        return true;
    }
    bool flush(int q) {
        if (!flush_dense(q)) return false;
        if (kind[q]) phase(q, -1, false, acc[q][0], acc[q][3]);
        kind[q] = 0;
        return true;
    }
    // o has a form
    bool add(const DevOp& o) {
        const int t = (int)o.t;
        if (o.kind == K_U2 && !o.hb) {
            const Z m[4] = {wide(o.m[0]), wide(o.m[1]), wide(o.m[4]), wide(o.m[5])};
            return conditioned(t, (int)o.c, false, m);
        }
        if (o.kind == K_U2) {
            const int c = (int)o.c;
            std::swap(row[t], row[c]);
            std::swap(col[t], col[c]);
            std::swap(kind[t], kind[c]);
            std::swap(chain[t], chain[c]);
            for (int i = 0; i < 4; ++i) std::swap(acc[t][i], acc[c][i]);
            const uint32_t d = ((neg >> t) ^ (neg >> c)) & 1u;
            neg ^= (d << t) | (d << c);
            return true;
        }
        const bool diag = o.kind == K_DIAG1;
        const Z m[4] = {wide(o.m[0]), diag ? kZero : wide(o.m[1]), diag ? kZero : wide(o.m[2]), wide(o.m[diag ? 1 : 3])};
        if (!o.cmask) {
            // a long product drifts from unitary by its roundings: split it off
            // well before split_rotation's bound
            if (++chain[t] > 16) {
                if (!flush(t)) return false;
                chain[t] = 1;
            }
            multiply(t, m);
            return true;
        }
        return conditioned(t, __builtin_ctzll(o.cmask), o.cval != 0, m);
    }
    // m on qubit t where qubit c reads cv
    bool conditioned(int t, int c, bool cv, const Z m[4]) {
        if (!flush_dense(c)) return false;
        if (zis(m[1], 0.0) && zis(m[2], 0.0)) {
            if (!flush_dense(t)) return false;
            phase(t, c, cv, m[0], m[3]);
            return true;
        }
        if (!flush(t)) return false;
        if (zis(m[0], 0.0) && zis(m[3], 0.0)) {
            cnot(t, c, cv);
            phase(t, c, cv, m[1], m[2]);
            return true;
        }
        Z l[2], r;
        double cs, sn;
        if (!split_rotation(m, l, cs, sn, r)) return false;
        phase(t, c, cv, kOne, r);
        rotation(t, c, cv, cs, sn);
        phase(t, c, cv, l[0], l[1]);
        return true;
    }
};

// ---- host: rounds and passes -----------------------------------------------------------

inline uint32_t par(uint32_t v) { return (uint32_t)__builtin_parity(v); }

struct Round {
    uint32_t rots[kRotsMax], phases[kPhasesMax];  // ops
    uint8_t axis[kRotsMax];                       // of rots
    int nrots = 0, nphases = 0;
    uint32_t b[kRoundDims], f[kRoundDims];
    int g = 0;
    uint32_t fn[kRoundTileMax + 2];  // basis of every functional in use
    int nfn = 0;
};

struct RoundPlan {
    std::vector<RoundsPass> passes;
    std::vector<uint4> words;
    std::vector<uint32_t> first;  // chunk of a pass
};

class RoundPlanner {
  public:
    RoundPlanner(const FrameLowering& fl, int n, int k, int low, int dims)
        : ops_(fl.out), tabs_(fl.tabs), n_(n), k_(std::min(n, k)), low_(low), dims_(dims) {
        for (auto& w : wx_) w = 0;
        for (auto& w : conf_) w = 0;
        for (auto& w : wf_) w = 0;
        for (auto& w : wg_) w = 0;
        fill();
    }


    void run(RoundPlan& plan) {
        while (pending_) {
            basis_.clear();
            for (int q = 0; q < (n_ > k_ ? std::min(low_, k_) : k_); ++q) basis_.push_back(1u << q);
            collect();
            emit(plan);
        }
    }
    // one pass over the given index bits; false when it does not take every op
    bool run_on(RoundPlan& plan, uint32_t bits) {
        for (uint32_t m = bits; m; m &= m - 1) basis_.push_back(m & (0u - m));
        collect();
        if (pending_) return false;
        emit(plan);
        return true;
    }
    // a pass without rounds
    void empty(RoundPlan& plan) {
        basis_.clear();
        rounds_.clear();
        emit(plan);
    }

  private:
    void collect() {
        rounds_.clear();
        out_ = 0;
        for (;;) {
            Round r;
            if (!form(r)) break;
            rounds_.push_back(r);
        }
    }
    // Slot s of the window holds op slot_[s]; a word per index bit over the
    // slots makes one op's parities against all of them a few XORs.
    void fill() {
        while (next_ < ops_.size()) {
            const uint32_t s = next_ & 63u;
            if ((pending_ >> s) & 1ull) break;
            const RoundOp& o = ops_[next_];
            uint64_t c = along(wf_, o.x) | along(wg_, o.x) | along(wx_, o.f0) | along(wx_, o.f1);
            const uint64_t bit = 1ull << s;
            for (uint64_t& w : conf_) w &= ~bit;  // the slot's last op is done
            conf_[s] = c & pending_;
            const RoundOp none{}, &old = next_ < 64 ? none : ops_[slot_[s]];
            toggle(wx_, o.x ^ old.x, bit);
            toggle(wf_, o.f0 ^ old.f0, bit);
            toggle(wg_, o.f1 ^ old.f1, bit);
            slot_[s] = (uint32_t)next_;
            out_ &= ~bit;
            pending_ |= bit;
            ++next_;
        }
    }
    static void toggle(uint64_t* w, uint32_t mask, uint64_t bit) {
        for (; mask; mask &= mask - 1) w[__builtin_ctz(mask)] ^= bit;
    }
    static uint64_t along(const uint64_t* w, uint32_t mask) {
        uint64_t r = 0;
        for (; mask; mask &= mask - 1) r ^= w[__builtin_ctz(mask)];
        return r;
    }
    uint32_t reduce(uint32_t x) const {
        for (uint32_t v : basis_)
            if ((x >> (31 - __builtin_clz(v))) & 1u) x ^= v;
        return x;
    }
    void extend(uint32_t r) {  // r reduced, not 0
        const int p = 31 - __builtin_clz(r);
        for (uint32_t& v : basis_)
            if ((v >> p) & 1u) v ^= r;
        basis_.push_back(r);
    }
    // The next round from the ops that are ready, oldest first.
    bool form(Round& r) {
        uint64_t phased = 0;  // phases of this round: still before any rotation they do not commute with
        // oldest first, then the ops that came into the window meanwhile (an op
        // that could not be taken does not become takable by a later one)
        uint64_t look = pending_ & ~out_;
        while (look) {
            const uint32_t start = next_ & 63u;
            const size_t before = next_;
            for (int half = 0; half < 2; ++half) {
                uint64_t todo = look & (half ? ((1ull << start) - 1ull) : ~((1ull << start) - 1ull));
                for (; todo; todo &= todo - 1) {
                    const uint32_t s = (uint32_t)__builtin_ctzll(todo);
                    if (!take(r, s)) continue;
                    if (ops_[slot_[s]].x) pending_ &= ~(1ull << s);
                    else phased |= 1ull << s;
                }
            }
            fill();
            look = 0;
            for (size_t i = before; i < next_; ++i) look |= 1ull << (i & 63u);
        }
        pending_ &= ~phased;
        fill();
        return r.nrots || r.nphases;
    }
    // Take functionals u and v into a round of g flips: it must stay possible
    // to pad the flips to k - kOrbitBits of them, orthogonal to every functional.
    bool room(Round& r, uint32_t u, uint32_t v, int g) const {
        if (k_ <= kOrbitBits) return true;
        const int most = k_ - std::max(0, k_ - kOrbitBits - g), had = r.nfn;
        for (uint32_t f : {u, v}) {
            for (int i = 0; i < r.nfn && f; ++i) f = std::min(f, f ^ r.fn[i]);
            if (f) r.fn[r.nfn++] = f;
        }
        if (r.nfn <= most) return true;
        r.nfn = had;
        return false;
    }
    bool take(Round& r, uint32_t s) {
        const RoundOp& o = ops_[slot_[s]];
        if (!o.x) {
            if (conf_[s] & pending_) return false;
            if (r.nphases >= kPhasesMax) return false;
            for (int d = 0; d < r.g; ++d)
                if (par(r.b[d] & o.f0) | par(r.b[d] & o.f1)) return false;
            if (!room(r, o.f0, o.f1, r.g)) return false;
            r.phases[r.nphases++] = slot_[s];
            return true;
        }
        if (conf_[s] & pending_) return false;  // phases of this round count as pending: they come first
        if (r.nrots >= kRotsMax) return false;
        for (int d = 0; d < r.g; ++d)
            if (r.b[d] == o.x && r.f[d] == o.f0) {
                for (int e = 0; e < r.g; ++e)
                    if (par(r.b[e] & o.f1)) return false;
                if (!room(r, o.f1, 0, r.g)) return false;
                r.axis[r.nrots] = (uint8_t)d;
                r.rots[r.nrots++] = slot_[s];
                return true;
            }
        if (r.g == dims_) return false;
        if (par(o.x & o.f1)) return false;
        for (int d = 0; d < r.g; ++d)
            if (par(r.b[d] & o.f0) | par(o.x & r.f[d]) | par(r.b[d] & o.f1)) return false;
        for (int i = 0; i < r.nrots; ++i)
            if (par(o.x & ops_[r.rots[i]].f1)) return false;
        for (int i = 0; i < r.nphases; ++i)
            if (par(o.x & ops_[r.phases[i]].f0) | par(o.x & ops_[r.phases[i]].f1)) return false;
        const uint32_t red = n_ > k_ ? reduce(o.x) : 0u;
        if (red && (int)basis_.size() >= k_) {
            out_ |= 1ull << s;  // not in this pass
            return false;
        }
        if (!room(r, o.f0, o.f1, r.g + 1)) return false;
        if (red) extend(red);
        r.b[r.g] = o.x;
        r.f[r.g] = o.f0;
        r.axis[r.nrots] = (uint8_t)r.g++;
        r.rots[r.nrots++] = slot_[s];
        return true;
    }

    // The pass of the collected rounds: tile bits, program words.
    void emit(RoundPlan& plan) {
        for (int q = 0; q < n_ && (int)basis_.size() < k_; ++q) {
            const uint32_t red = reduce(1u << q);
            if (red) extend(red);
        }
        std::sort(basis_.begin(), basis_.end());  // ascending pivots
        RoundsPass p{};
        p.k = (uint32_t)k_;
        uint32_t pivots = 0;
        for (int i = 0; i < k_; ++i) {
            p.sv[i] = p.wv[i] = basis_[i];
            pivots |= 1u << (31 - __builtin_clz(basis_[i]));
        }
        int u = 0;
        for (int q = 0; q < n_; ++q)
            if (!((pivots >> q) & 1u)) {
                p.sq[u] = p.wq[u] = 1u << q;
                ++u;
            }
        // functional -> tile bits, then bits of the tile's number (linear: one
        // word per index bit); flip -> tile bits
        uint32_t reads[32];
        for (int q = 0; q < n_; ++q) {
            reads[q] = 0;
            for (int i = 0; i < k_; ++i) reads[q] |= ((p.sv[i] >> q) & 1u) << i;
            for (int i = 0; i < u; ++i) reads[q] |= ((p.sq[i] >> q) & 1u) << (k_ + i);
        }
        auto functional = [&](uint32_t f) {
            uint32_t r = 0;
            for (; f; f &= f - 1) r ^= reads[__builtin_ctz(f)];
            return r;
        };
        auto flip = [&](uint32_t x) {
            uint32_t r = 0;
            for (int i = 0; i < k_; ++i) r |= ((x >> (31 - __builtin_clz(p.sv[i]))) & 1u) << i;
            return r;
        };
        plan.first.push_back((uint32_t)(plan.words.size() / kChunkWords));
        size_t start = 0, used = kChunkWords;  // of the open chunk
        for (const Round& r : rounds_) {
            const size_t at0 = scratch_.size();
            scratch_.resize(at0 + kRoundWords, make_uint4(0, 0, 0, 0));
            // the first rotation of an axis, if unconditional, into the axis' own place
            uint32_t role[kRoundDims] = {0, 0, 0, 0}, own = 0, seen = 0;
            auto pack = [](double c, double sn) {
                uint4 w;
                const double cs[2] = {c, sn};
                std::memcpy(&w, cs, 16);
                return w;
            };
            const uint32_t np = pack_phases(r, functional);
            uint32_t nr = 0;
            for (int i = 0; i < r.nrots; ++i) {
                const RoundOp& o = ops_[r.rots[i]];
                const uint32_t bit = 1u << r.axis[i];
                const bool lead = !o.f1 && !(seen & bit);
                seen |= bit;
                if (lead) {
                    own |= bit;
                    role[r.axis[i]] = functional(o.f0);
                    scratch_[at0 + 2 + r.axis[i]] = pack(o.c, o.s);
                    continue;
                }
                scratch_.push_back(make_uint4(functional(o.f0), functional(o.f1), r.axis[i] | (o.f1 ? 0x100u : 0u) | (o.want ? 0x200u : 0u), 0));
                scratch_.push_back(pack(o.c, o.s));
                ++nr;
            }
            scratch_[at0 + 1] = make_uint4(role[0], role[1], role[2], role[3]);
            uint32_t b[kRoundDims] = {0, 0, 0, 0}, e[kRoundDims], piv[kRoundDims];
            int g = r.g;
            for (int d = 0; d < g; ++d) b[d] = flip(r.b[d]);
            if (g < k_ - kOrbitBits) pad(r, functional, b, g);
            for (int d = 0; d < g; ++d) {
                // pivots as high as they get: consecutive threads own consecutive amplitudes
                uint32_t v = b[d];
                for (int c = 0; c < d; ++c)
                    if ((v >> piv[c]) & 1u) v ^= e[c];
                piv[d] = (uint32_t)(31 - __builtin_clz(v));
                for (int c = 0; c < d; ++c)
                    if ((e[c] >> piv[d]) & 1u) e[c] ^= v;
                e[d] = v;
            }
            std::sort(piv, piv + g);
            uint32_t pv = 0;
            for (int d = 0; d < g; ++d) pv |= piv[d] << (8 * d);
            scratch_[at0] = make_uint4((uint32_t)g | (np << 8) | (nr << 16) | (own << 24), pv, b[0] | (b[1] << 16), b[2] | (b[3] << 16));
            const size_t size = scratch_.size() - at0;
            if (used + size > kChunkWords) {
                start = plan.words.size();
                plan.words.resize(start + kChunkWords, make_uint4(0, 0, 0, 0));
                used = 1;
                p.chunks++;
            }
            std::copy(scratch_.begin() + (long)at0, scratch_.end(), plan.words.begin() + (long)(start + used));
            plan.words[start].x++;
            used += size;
            scratch_.clear();
        }
        plan.passes.push_back(p);
    }
    // Flips that nothing in the round reads, up to k - kOrbitBits in all.
    template <typename F>
    void pad(const Round& r, F functional, uint32_t (&b)[kRoundDims], int& g) const {
        std::vector<uint32_t> e;  // reduced echelon form of the functionals on the tile
        std::vector<int> pv;
        uint32_t pivots = 0;
        for (int u = 0; u < r.nfn; ++u) {
            uint32_t v = functional(r.fn[u]) & ((1u << k_) - 1u);
            for (size_t i = 0; i < e.size(); ++i)
                if ((v >> pv[i]) & 1u) v ^= e[i];
            if (!v) continue;
            const int p = __builtin_ctz(v);
            for (uint32_t& w : e)
                if ((w >> p) & 1u) w ^= v;
            e.push_back(v);
            pv.push_back(p);
            pivots |= 1u << p;
        }
        for (int c = k_; c-- > 0 && g < k_ - kOrbitBits;) {
            if ((pivots >> c) & 1u) continue;
            uint32_t v = 1u << c;
            for (size_t i = 0; i < e.size(); ++i)
                if ((e[i] >> c) & 1u) v |= 1u << pv[i];
            b[g++] = v;
        }
    }
    // The phases of a round as products over up to four parities; returns the
    // number of tables.
    template <typename F>
    uint32_t pack_phases(const Round& r, F functional) {
        struct Rec {
            uint32_t f[kPhaseBits];
            int n;
            Z t[1 << kPhaseBits];
        };
        Rec rec[kPhasesMax];
        uint32_t count = 0;
        for (int x = 0; x < r.nphases; ++x) {
            const RoundOp& o = ops_[r.phases[x]];
            const uint32_t fs[2] = {o.f0, o.f1};
            int at[2] = {-1, -1};  // places of f0 and f1 in the table
            for (uint32_t c = 0; c <= count; ++c) {
                Rec& t = rec[c];
                if (c == count) {
                    t.n = 0;
                    t.t[0] = kOne;
                }
                int n = t.n;
                for (int k = 0; k < 2; ++k) {
                    at[k] = -1;
                    if (!fs[k]) continue;
                    for (int i = 0; i < t.n; ++i)
                        if (t.f[i] == fs[k]) at[k] = i;
                    if (at[k] < 0) at[k] = n++;
                }
                if (n > kPhaseBits) continue;
                for (int k = 0; k < 2; ++k)
                    if (at[k] >= t.n) t.f[at[k]] = fs[k];
                for (; t.n < n; ++t.n)
                    for (int i = 0; i < (1 << t.n); ++i) t.t[i | (1 << t.n)] = t.t[i];
                bool one[4];
                for (int j = 0; j < 4; ++j) one[j] = zis(tabs_[o.tab + (uint32_t)j], 1.0);
                for (int i = 0; i < (1 << n); ++i) {
                    const int j = ((i >> at[0]) & 1) | (at[1] >= 0 ? ((i >> at[1]) & 1) << 1 : 0);
                    if (!one[j]) t.t[i] = zmul(t.t[i], tabs_[o.tab + (uint32_t)j]);
                }
                if (c == count) ++count;
                break;
            }
        }
        for (uint32_t c = 0; c < count; ++c) {
            uint32_t f[kPhaseBits] = {0, 0, 0, 0};
            for (int i = 0; i < rec[c].n; ++i) f[i] = functional(rec[c].f[i]);
            scratch_.push_back(make_uint4(f[0], f[1], f[2], f[3]));
            const size_t w = scratch_.size();
            scratch_.resize(w + (1u << kPhaseBits), make_uint4(0, 0, 0, 0));  // unused parities read 0
            for (int i = 0; i < (1 << rec[c].n); ++i) {
                const double2 v = narrow(rec[c].t[i]);
                std::memcpy(&scratch_[w + (size_t)i], &v, sizeof(v));
            }
        }
        return count;
    }

    const std::vector<RoundOp>& ops_;
    const std::vector<Z>& tabs_;
    int n_, k_, low_, dims_;
    size_t next_ = 0;
    uint64_t pending_ = 0, out_ = 0, conf_[64];
    uint32_t slot_[64];
    uint64_t wx_[32], wf_[32], wg_[32];
    std::vector<uint32_t> basis_;
    std::vector<Round> rounds_;
    std::vector<uint4> scratch_;
};

// Let the pass store every amplitude at its logical index.
void to_logical(const FrameLowering& fl, RoundsPass& p) {
    auto logical = [&](uint32_t v) {
        uint32_t l = 0;
        for (int q = 0; q < fl.n; ++q) l |= par(fl.row[q] & v) << q;
        return l;
    };
    for (uint32_t& v : p.wv) v = logical(v);
    for (uint32_t& v : p.wq) v = logical(v);
    p.w0 = fl.neg;
}

// Passes and program of an op list; false when an op has no such form.  The
// stored index that the last pass leaves differs from the logical one unless
// `plain`.
bool plan_rounds(const std::vector<HostOp>& ops, int n, RoundPlan& plan, bool& plain) {
    // first of all: a list with one op that has no form is lowered for nothing
    for (const HostOp& h : ops)
        if (!has_form(h.op)) return false;
    FrameLowering fl(n);
    fl.out.reserve(ops.size());
    for (const HostOp& h : ops)
        if (!fl.add(h.op)) return false;
    for (int q = 0; q < n; ++q)
        if (!fl.flush(q)) return false;
    plain = fl.neg == 0;
    for (int q = 0; q < n; ++q) plain = plain && fl.col[q] == 1u << q;
    RoundPlanner pl(fl, n, kRoundTileMax, kRoundLow, kRoundDims);
    pl.run(plan);
    if (plain) return true;
    // one tile moves its amplitudes by itself; more need a second buffer, so
    // the first pass stores there and the last pass comes back
    const size_t least = n > kRoundTileMax ? 2 : 1;
    while (plan.passes.size() < least) pl.empty(plan);
    to_logical(fl, plan.passes.back());
    return true;
}

template <int DIMS, bool NT>
int launch_rounds(qfe_state_s* st, const double2* src, double2* dst, const RoundsPass& p, const uint4* prog) {
    Context& cx = ctx();
    constexpr int tile = kOrbitBits + DIMS;
    static const hipError_t big = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_rounds<DIMS, NT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                      (sizeof(double2) << tile) + kChunkWords * sizeof(uint4));
    QFE_HIP(big);
    hipLaunchKernelGGL((k_rounds<DIMS, NT>), dim3(1u << (st->n - (int)p.k)), dim3(kRoundTPB),
                       (sizeof(double2) << p.k) + kChunkWords * sizeof(uint4), cx.stream, src, dst, p, prog);
    QFE_HIP(hipGetLastError());
    cx.counters.fused++;
    cx.counters.tile++;
    cx.counters.nt += NT ? 1 : 0;
    cx.counters.bytes += 32.0 * (double)st->N;
    return QFE_OK;
}

}  // namespace

bool plan_tile_rounds(const std::vector<HostOp>& ops, const std::vector<int>& take, int n, uint32_t bits, RoundsPass& p,
                      std::vector<uint4>& words) {
    FrameLowering fl(n);
    for (int i : take)
        if (!has_form(ops[i].op) || !fl.add(ops[i].op)) return false;
    for (int q = 0; q < n; ++q)
        if (!fl.flush(q)) return false;
    RoundPlan plan;
    RoundPlanner pl(fl, n, __builtin_popcount(bits), 0, kLargeDims);
    if (!pl.run_on(plan, bits)) return false;
    p = plan.passes[0];
    to_logical(fl, p);
    words.insert(words.end(), plan.words.begin(), plan.words.end());
    return true;
}

int launch_tile_rounds(qfe_state_s* st, const RoundsPass& p, const uint4* words) {
    return use_nt(st->n, (uint32_t)p.low) ? launch_rounds<kLargeDims, true>(st, st->d, st->d, p, words)
                                          : launch_rounds<kLargeDims, false>(st, st->d, st->d, p, words);
}

int run_rounds(qfe_state_s* st, const std::vector<HostOp>& ops, bool& taken) {
    taken = false;
    Context& cx = ctx();
    RoundPlan plan;
    bool plain = false;
    if (!plan_rounds(ops, st->n, plan, plain)) return QFE_OK;
    taken = true;
    if (plan.passes.empty()) return QFE_OK;
    int rc = QFE_OK;
    const uint4* prog = nullptr;
    if (!plan.words.empty()) {
        const size_t bytes = plan.words.size() * sizeof(uint4);
        void *dev = nullptr, *host = nullptr;
        rc = scratch_reserve(bytes, &dev);
        if (rc) return rc;
        rc = staging_begin(bytes, &host);
        if (rc) return rc;
        std::memcpy(host, plan.words.data(), bytes);
        rc = staging_commit(dev, bytes);
        if (rc) return rc;
        prog = static_cast<const uint4*>(dev);
    }
    double2* other = st->d;
    if (!plain && st->n > kRoundTileMax) {
        other = static_cast<double2*>(slice_memory(sizeof(double2) << st->n));
        if (!other) {
            taken = false;
            return QFE_OK;
        }
    }
    for (size_t i = 0; i < plan.passes.size(); ++i) {
        const RoundsPass& p = plan.passes[i];
        const double2* src = i == 0 ? st->d : other;
        double2* dst = i + 1 == plan.passes.size() ? st->d : other;
        rc = launch_rounds<kRoundDims, false>(st, src, dst, p, p.chunks ? prog + (size_t)plan.first[i] * kChunkWords : nullptr);
        if (rc) return rc;
    }
    return QFE_OK;
}

}  // namespace qfe
