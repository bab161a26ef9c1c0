// Compiled UCC programs: energy, adjoint gradient and pool gradients with the
// ansatz and the Hamiltonian resident in HBM.
//
// The reference rebuilds the ansatz circuit (JW of every pool operator,
// trotterize, gate objects) on every energy_feval (algorithm.py:458-474,
// ansatz.py:25-82) and evaluates the gradient with deep copies and Python
// list conversions (uccvqeabc.py:122-251).  A program is compiled once; the
// amplitudes are the only per-call input.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "qfe_device.h"
#include "qfe_internal.h"

namespace qfe {

// A grouped Pauli table resident in HBM.
struct DevTable {
    PauliGroup* g = nullptr;
    uint64_t* z = nullptr;
    double2* c = nullptr;
    uint32_t ngroups = 0;
};

static int table_upload(const std::vector<PauliGroup>& groups, const std::vector<uint64_t>& zs,
                        const std::vector<double2>& cs, DevTable& t) {
    t.ngroups = (uint32_t)groups.size();
    if (groups.empty()) return QFE_OK;
    QFE_HIP(device_malloc(&t.g, groups.size() * sizeof(PauliGroup)));
    QFE_HIP(device_malloc(&t.z, zs.size() * sizeof(uint64_t)));
    QFE_HIP(device_malloc(&t.c, cs.size() * sizeof(double2)));
    QFE_HIP(hipMemcpy(t.g, groups.data(), groups.size() * sizeof(PauliGroup), hipMemcpyHostToDevice));
    QFE_HIP(hipMemcpy(t.z, zs.data(), zs.size() * sizeof(uint64_t), hipMemcpyHostToDevice));
    QFE_HIP(hipMemcpy(t.c, cs.data(), cs.size() * sizeof(double2), hipMemcpyHostToDevice));
    return QFE_OK;
}

static void table_free(DevTable& t) {
    if (t.g) (void)hipFree(t.g);
    if (t.z) (void)hipFree(t.z);
    if (t.c) (void)hipFree(t.c);
    t = DevTable{};
}

// Concatenate the groupings of several operators; ranges[k]..ranges[k+1] are
// the groups of operator k.
static void group_many(const qfe_pauli* terms, const uint64_t* offsets, uint64_t nops, std::vector<PauliGroup>& groups,
                       std::vector<uint64_t>& zs, std::vector<double2>& cs, std::vector<uint32_t>& ranges) {
    groups.clear();
    zs.clear();
    cs.clear();
    ranges.assign(1, 0);
    std::vector<PauliGroup> g1;
    std::vector<uint64_t> z1;
    std::vector<double2> c1;
    for (uint64_t k = 0; k < nops; ++k) {
        group_terms(terms + offsets[k], offsets[k + 1] - offsets[k], g1, z1, c1);
        const uint32_t shift = (uint32_t)zs.size();
        for (PauliGroup g : g1) {
            g.first += shift;
            groups.push_back(g);
        }
        zs.insert(zs.end(), z1.begin(), z1.end());
        cs.insert(cs.end(), c1.begin(), c1.end());
        ranges.push_back((uint32_t)groups.size());
    }
}

// ---- captured energy sequence --------------------------------------------------------------
// The ansatz is planned once with device-side angles: every exponential's
// (cos, sin) lives in a descriptor image in HBM and a kernel rewrites them
// from the amplitudes before the passes run.  Parameter upload, that kernel,
// the reference state, the exponential passes, the expectation value and the
// result download are captured once as a hipGraph; each energy call then
// writes the amplitudes into pinned memory and replays the graph.
struct DevAngle {
    uint64_t off;  // byte offset of the (cos, sin) pair in the descriptor image
    uint32_t param;
    uint32_t pad;
    double scale;  // generator scale
    double cim;    // Im(coefficient) of the Pauli term
};

__global__ __launch_bounds__(256) void k_program_angles(const double* __restrict__ params,
                                                        const DevAngle* __restrict__ a, uint32_t n,
                                                        char* __restrict__ image) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const DevAngle d = a[i];
    double sn, c;
    sincos((params[d.param] * d.scale) * d.cim, &sn, &c);
    double* dst = reinterpret_cast<double*>(image + d.off);  // 8-byte aligned in every descriptor kind
    dst[0] = c;
    dst[1] = sn;
}

struct ProgramGraph {
    OpPlan* plan = nullptr;
    char* image = nullptr;
    DevAngle* angles = nullptr;
    uint32_t nangles = 0;
    double* dparams = nullptr;
    double* hparams = nullptr;  // pinned; read by the graph's first node
    double2* partial = nullptr;
    double2* gout = nullptr;
    double2* hout = nullptr;  // pinned; written by the graph's last node
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

static void graph_free(ProgramGraph* g) {
    if (!g) return;
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    if (g->image) (void)hipFree(g->image);
    if (g->angles) (void)hipFree(g->angles);
    if (g->dparams) (void)hipFree(g->dparams);
    if (g->partial) (void)hipFree(g->partial);
    if (g->gout) (void)hipFree(g->gout);
    if (g->hparams) (void)hipHostFree(g->hparams);
    if (g->hout) (void)hipHostFree(g->hout);
    plan_free(g->plan);
    delete g;
}

// ---- generator tiles ----------------------------------------------------------------
// A run of generator terms with one X mask x and commuting strings is the
// exponential of K = sum_t kappa_t P_t, which maps j to j ^ x with weight
// alpha(j) = sum_t kappa_t (-1)^{j.z_t}, alpha(j ^ x) = -conj(alpha(j)): on
// every pair exp(theta K) = cos(theta w) + sin(theta w) / w K, w = |alpha|.
// When |alpha| takes one non-zero value (every fermionic or qubit excitation),
// a run is a rotation of the pairs that have it, instead of one exponential
// per term.  Consecutive generators whose masks span at most kProgDims
// dimensions over GF(2) form a pass: a workgroup takes one coset of the span
// in LDS (psi, or psi and sigma) through all of them.  The reverse sweep also
// adds up each generator's Re<sigma|K|psi>.  It used to take five kernels and
// two copies per generator (14-qubit UCCSD gradient: 204 generators, 9.2 ms).
// Tile width, in dimensions: wider tiles take fewer passes with longer chains
// (UCCSD gradients at 14 / 16 / 20 / 24 qubits in us: 549 / 1059 / 11388 /
// 199353 with 8, 521 / 1017 / 9789 / 194284 with 9, 642 / 1168 / 9698 / 194497
// with 10; one exponential at a time 12567 / 21971 / 78345 / 645992).
constexpr int kProgDims = 9;
constexpr int kProgLow = 3;          // the lowest qubits are always in the span: whole 128-byte lines
constexpr int kProgThreads = 256;
constexpr uint32_t kProgTerms = 512;  // terms of a pass

struct ProgTerm {
    uint64_t z;
    double2 kappa;
};
struct ProgRun {  // v: flip in tile coordinates, hb: its top bit
    uint32_t v, hb, t0, nt, run, flags;
    double w2;  // |alpha|^2 of the pairs that rotate
};
constexpr uint32_t kRunGenEnd = 1;  // last run of a generator (in pass order)
constexpr uint32_t kRunOnlyOv = 2;  // overlap without rotation
constexpr uint32_t kRunOnlyRot = 4;

struct ProgPass {
    uint64_t basis[kProgDims];
    uint32_t piv[kProgDims];
    uint32_t dims, run0, nrun, term0, nterm, part;
};

// MODE 0: the pass's runs on x; MODE 1: their inverses, last first, on x;
// MODE 2: reverse sweep on x = psi and y = sigma (first: adds Re<psi|sigma>).
template <int MODE>
__global__ __launch_bounds__(kProgThreads) void k_program_tile(double2* __restrict__ gx, double2* __restrict__ gy,
                                                               const ProgPass* __restrict__ passes, uint32_t pass,
                                                               const ProgRun* __restrict__ runs,
                                                               const ProgTerm* __restrict__ terms,
                                                               const double2* __restrict__ cs, double* __restrict__ partial,
                                                               uint32_t first) {
    extern __shared__ double2 prog_lds[];
    __shared__ uint64_t lo[32], hi[32];
    __shared__ double2 kap[kProgTerms];
    __shared__ uint32_t zloc[kProgTerms];
    __shared__ double red[2][kProgThreads / kWave];  // wave sums of the last two outputs
    const ProgPass& P = passes[pass];
    const uint32_t d = P.dims, n = 1u << d, tid = threadIdx.x;
    double2 *X = prog_lds, *Y = prog_lds + n;
    uint64_t j = blockIdx.x;
    for (uint32_t k = 0; k < d; ++k) j = ins0(j, P.piv[k]);
    if (tid < 64) {
        uint64_t c = 0;
        for (uint32_t k = 0; k < 5; ++k) {
            const uint32_t b = tid < 32 ? k : k + 5;
            if (((tid & 31u) >> k) & 1u && b < d) c ^= P.basis[b];
        }
        (tid < 32 ? lo : hi)[tid & 31u] = c;
    }
    for (uint32_t t = tid; t < P.nterm; t += kProgThreads) {
        const ProgTerm T = terms[P.term0 + t];
        uint32_t m = 0;
        for (uint32_t k = 0; k < d; ++k) m |= (uint32_t)(__popcll(P.basis[k] & T.z) & 1) << k;
        zloc[t] = m;
        kap[t] = __popcll(j & T.z) & 1 ? make_double2(-T.kappa.x, -T.kappa.y) : T.kappa;
    }
    __syncthreads();
    double acc = 0.0;
    for (uint32_t i = tid; i < n; i += kProgThreads) {
        const uint64_t g = j ^ lo[i & 31u] ^ hi[i >> 5];
        X[i] = gx[g];
        if (MODE == 2) {
            Y[i] = gy[g];
            if (first) acc += X[i].x * Y[i].x + X[i].y * Y[i].y;
        }
    }
    // an output is its waves' sums, added up and stored after the next barrier
    uint32_t nout = 0;
    bool pending = false;
    auto flush = [&]() {
        const double v = wave_sum_last(acc);
        if ((tid & (kWave - 1)) == kWave - 1) red[nout & 1u][tid / kWave] = v;
        acc = 0.0;
        pending = true;
    };
    auto store = [&]() {
        if (!pending) return;
        if (tid == 0) {
            double v = 0.0;
            for (int w = 0; w < kProgThreads / kWave; ++w) v += red[nout & 1u][w];
            partial[P.part + nout * gridDim.x + blockIdx.x] = v;
        }
        ++nout;
        pending = false;
    };
    if (MODE == 2 && first) flush();
    __syncthreads();
    if (MODE == 2) store();
    for (uint32_t q = 0; q < P.nrun; ++q) {
        const ProgRun R = runs[P.run0 + (MODE == 1 ? P.nrun - 1 - q : q)];
        const double2 rot = cs[R.run];  // cos(theta w), sin(theta w) / w
        const double c = rot.x, s = MODE == 0 ? rot.y : -rot.y;
        const bool ov = MODE == 2 && !(R.flags & kRunOnlyRot), turn = MODE != 2 || !(R.flags & kRunOnlyOv);
        for (uint32_t p = tid; p < n / 2; p += kProgThreads) {
            const uint32_t ia = ins0_32(p, R.hb), ib = ia ^ R.v;
            double2 al = make_double2(0.0, 0.0);  // alpha on the pair's first index
#pragma unroll 8
            for (uint32_t t = R.t0; t < R.t0 + R.nt; ++t) {
                const int neg = (int)((uint32_t)__popc(ia & zloc[t]) << 31);
                const double2 k = kap[t];
                al.x += __hiloint2double(__double2hiint(k.x) ^ neg, __double2loint(k.x));
                al.y += __hiloint2double(__double2hiint(k.y) ^ neg, __double2loint(k.y));
            }
            // |alpha|^2 is w^2 or zero: the pair rotates or stays
            if (2.0 * (al.x * al.x + al.y * al.y) < R.w2) continue;
            const double2 be = make_double2(-al.x, al.y);  // alpha on the second
            const double2 a = X[ia], b = X[ib];
            const double2 ka = cmul(be, b), kb = cmul(al, a);  // K x
            if (MODE == 2) {
                const double2 ya = Y[ia], yb = Y[ib];
                if (ov) acc += (ya.x * ka.x + ya.y * ka.y) + (yb.x * kb.x + yb.y * kb.y);
                if (turn) {
                    const double2 la = cmul(be, yb), lb = cmul(al, ya);
                    Y[ia] = make_double2(c * ya.x + s * la.x, c * ya.y + s * la.y);
                    Y[ib] = make_double2(c * yb.x + s * lb.x, c * yb.y + s * lb.y);
                }
            }
            if (turn) {
                X[ia] = make_double2(c * a.x + s * ka.x, c * a.y + s * ka.y);
                X[ib] = make_double2(c * b.x + s * kb.x, c * b.y + s * kb.y);
            }
        }
        if (MODE == 2 && (R.flags & kRunGenEnd)) flush();
        __syncthreads();
        if (MODE == 2) store();
    }
    for (uint32_t i = tid; i < n; i += kProgThreads) {
        const uint64_t g = j ^ lo[i & 31u] ^ hi[i >> 5];
        gx[g] = X[i];
        if (MODE == 2) gy[g] = Y[i];
    }
}

// out[k] = sum of partial[range k], one wave each, in a fixed order.
__global__ __launch_bounds__(256) void k_program_sum(const double* __restrict__ partial, const uint2* __restrict__ ranges,
                                                     uint32_t count, double* __restrict__ out) {
    const uint32_t k = blockIdx.x * (256 / kWave) + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (k >= count) return;
    double acc = 0.0;
    for (uint32_t i = lane; i < ranges[k].y; i += kWave) acc += partial[ranges[k].x + i];
    const double v = wave_sum_last(acc);
    if (lane == kWave - 1) out[k] = v;
}

// Host side: runs, passes and the tables of both directions.
struct ProgTiles {
    bool ok = false;
    struct Run {
        uint64_t x;
        uint32_t gen, t0, nt;
        double w;  // |alpha| where it is not zero
    };
    std::vector<Run> runs;
    std::vector<ProgPass> fwd, rev;
    std::vector<ProgRun> fruns, rruns;
    std::vector<ProgTerm> terms;
    std::vector<uint2> ranges;  // partial sums: the energy, then generator k
    uint32_t parts = 0, dims = 0;
    void* dev = nullptr;  // tables, (cos, sin / w) of every run, results
    double* part = nullptr;  // partial sums, from the first gradient on
    size_t o_fwd = 0, o_rev = 0, o_fruns = 0, o_rruns = 0, o_terms = 0, o_ranges = 0, o_cs = 0, o_out = 0;

    // |alpha| over the patterns of the bits it depends on; false unless all of
    // them are one value or zero, to the rounding of their sums: a rotation by
    // the mean is then as close to the string's exponentials as these are.
    static bool weight(const std::vector<qfe_pauli>& t, uint64_t b, uint64_t e, double& w) {
        uint64_t m = 0;
        double total = 0.0;
        for (uint64_t k = b; k < e; ++k) {
            m |= t[k].z ^ t[b].z;
            total += std::fabs(t[k].coeff.im);
        }
        if (__builtin_popcountll(m) > 12) return false;
        w = 0.0;
        const double tol = 4.0 * 0x1p-52 * total;
        std::vector<double> seen;
        for (uint64_t p = m;; p = (p - 1) & m) {
            double re = 0.0, im = 0.0;
            for (uint64_t k = b; k < e; ++k) {
                const double sg = __builtin_popcountll(p & (t[k].z ^ t[b].z)) & 1 ? -t[k].coeff.im : t[k].coeff.im;
                re -= sg * t[k].phase.im;  // kappa = i Im(coeff) phase
                im += sg * t[k].phase.re;
            }
            const double v = std::hypot(re, im);
            if (v > tol) seen.push_back(v);
            if (!p) break;
        }
        if (seen.empty()) return false;
        for (double v : seen) w += v / (double)seen.size();
        for (double v : seen)
            if (std::fabs(v - w) > tol) return false;
        return true;
    }

    // Reduced basis of a span, every pivot (highest bit) in one vector only.
    struct Basis {
        std::vector<uint64_t> b;
        bool add(uint64_t x, int most) {
            for (uint64_t v : b)
                if ((x >> (63 - __builtin_clzll(v))) & 1ull) x ^= v;
            if (!x) return true;
            if ((int)b.size() >= most) return false;
            const int p = 63 - __builtin_clzll(x);
            for (uint64_t& v : b)
                if ((v >> p) & 1ull) v ^= x;
            b.push_back(x);
            return true;
        }
    };

    void build(int n, const std::vector<qfe_pauli>& t, const std::vector<uint64_t>& gen_off) {
        const uint64_t ngen = gen_off.size() - 1;
        dims = (uint32_t)std::min(n, kProgDims);
        std::vector<uint32_t> gen_run{0};
        for (uint64_t k = 0; k < ngen; ++k) {
            for (uint64_t b = gen_off[k]; b < gen_off[k + 1];) {
                uint64_t e = b + 1;
                while (e < gen_off[k + 1] && t[e].x == t[b].x && !(__builtin_popcountll(t[b].x & (t[e].z ^ t[b].z)) & 1)) ++e;
                Run r{t[b].x, (uint32_t)k, (uint32_t)b, (uint32_t)(e - b), 0.0};
                if (!r.x || r.nt > kProgTerms || !weight(t, b, e, r.w)) return;
                runs.push_back(r);
                b = e;
            }
            gen_run.push_back((uint32_t)runs.size());
        }
        for (const qfe_pauli& q : t)
            terms.push_back(ProgTerm{q.z, make_double2(-q.coeff.im * q.phase.im, q.coeff.im * q.phase.re)});
        struct Seg {
            uint64_t g0, g1;
        };
        std::vector<Seg> segs;
        std::vector<Basis> bases;
        for (uint64_t g = 0; g < ngen;) {
            Basis cur;
            for (int q = 0; q < std::min(kProgLow, (int)dims); ++q) cur.add(1ull << q, (int)dims);
            uint64_t g1 = g;
            while (g1 < ngen && gen_off[g1 + 1] - gen_off[g] <= kProgTerms) {
                Basis trial = cur;
                bool fits = true;
                for (uint32_t r = gen_run[g1]; fits && r < gen_run[g1 + 1]; ++r) fits = trial.add(runs[r].x, (int)dims);
                if (!fits) break;
                cur = trial;
                ++g1;
            }
            if (g1 == g) return;  // one generator spans more than a tile
            for (int q = 0; (int)cur.b.size() < (int)dims; ++q) cur.add(1ull << q, (int)dims);
            std::sort(cur.b.begin(), cur.b.end());
            segs.push_back({g, g1});
            bases.push_back(cur);
            g = g1;
        }
        if ((ngen + 1) << (n - (int)dims) > (1ull << 25)) return;  // partial sums: at most 256 MiB
        const uint32_t per = 1u << (n - (int)dims);
        ranges.assign(ngen + 1, make_uint2(0, 0));
        auto add = [&](size_t sg, bool reverse) {
            ProgPass P{};
            for (uint32_t k = 0; k < dims; ++k) {
                P.basis[k] = bases[sg].b[k];
                P.piv[k] = (uint32_t)(63 - __builtin_clzll(bases[sg].b[k]));
            }
            P.dims = dims;
            P.term0 = (uint32_t)gen_off[segs[sg].g0];
            P.nterm = (uint32_t)gen_off[segs[sg].g1] - P.term0;
            P.part = parts;
            std::vector<ProgRun>& out = reverse ? rruns : fruns;
            P.run0 = (uint32_t)out.size();
            auto push = [&](uint32_t r, uint32_t flags) {
                uint32_t v = 0;
                for (uint32_t k = 0; k < dims; ++k) v |= (uint32_t)((runs[r].x >> P.piv[k]) & 1ull) << k;
                out.push_back(ProgRun{v, (uint32_t)(31 - __builtin_clz(v)), runs[r].t0 - P.term0, runs[r].nt, r, flags,
                                      runs[r].w * runs[r].w});
            };
            if (!reverse) {
                for (uint32_t r = gen_run[segs[sg].g0]; r < gen_run[segs[sg].g1]; ++r) push(r, 0);
            } else {
                if (rev.empty()) {
                    ranges[0] = make_uint2(parts, per);
                    parts += per;
                }
                for (uint64_t k = segs[sg].g1; k-- > segs[sg].g0;) {
                    const uint32_t r0 = gen_run[k], r1 = gen_run[k + 1];
                    if (r0 == r1) continue;
                    ranges[k + 1] = make_uint2(parts, per);
                    parts += per;
                    if (r1 == r0 + 1) {
                        push(r0, kRunGenEnd);
                        continue;
                    }
                    for (uint32_t r = r0; r < r1; ++r) push(r, kRunOnlyOv | (r + 1 == r1 ? kRunGenEnd : 0u));
                    for (uint32_t r = r1; r-- > r0;) push(r, kRunOnlyRot);
                }
            }
            P.nrun = (uint32_t)out.size() - P.run0;
            (reverse ? rev : fwd).push_back(P);
        };
        for (size_t i = 0; i < segs.size(); ++i) add(i, false);
        for (size_t i = segs.size(); i-- > 0;) add(i, true);
        ok = !segs.empty();
    }

    // Tables on the device; dev stays null when memory is short, and the caller
    // goes one exponential at a time.
    int upload() {
        if (!ok || dev) return QFE_OK;
        size_t at = 0;
        auto place = [&](size_t bytes) {
            const size_t o = at;
            at += (bytes + 255) & ~(size_t)255;
            return o;
        };
        o_fwd = place(fwd.size() * sizeof(ProgPass));
        o_rev = place(rev.size() * sizeof(ProgPass));
        o_fruns = place(fruns.size() * sizeof(ProgRun));
        o_rruns = place(rruns.size() * sizeof(ProgRun));
        o_terms = place(terms.size() * sizeof(ProgTerm));
        o_ranges = place(ranges.size() * sizeof(uint2));
        const size_t tables = at;
        o_cs = place(runs.size() * sizeof(double2));
        o_out = place(ranges.size() * sizeof(double));
        std::vector<char> img(tables);
        auto put = [&](size_t o, const void* src, size_t bytes) { std::memcpy(img.data() + o, src, bytes); };
        put(o_fwd, fwd.data(), fwd.size() * sizeof(ProgPass));
        put(o_rev, rev.data(), rev.size() * sizeof(ProgPass));
        put(o_fruns, fruns.data(), fruns.size() * sizeof(ProgRun));
        put(o_rruns, rruns.data(), rruns.size() * sizeof(ProgRun));
        put(o_terms, terms.data(), terms.size() * sizeof(ProgTerm));
        put(o_ranges, ranges.data(), ranges.size() * sizeof(uint2));
        if (!try_malloc(&dev, at)) return QFE_OK;
        const hipError_t e = hipMemcpy(dev, img.data(), tables, hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            release();
            return hip_fail(e, "qfe_program: table upload");
        }
        return QFE_OK;
    }
    template <typename T>
    static bool try_malloc(T** p, size_t bytes) {
        if (device_malloc(p, bytes) == hipSuccess) return true;
        (void)hipGetLastError();  // no error of the call
        *p = nullptr;
        return false;
    }
    // Whether a reverse sweep can take the tiles.
    bool sums() { return dev && (part || try_malloc(&part, (size_t)parts * sizeof(double))); }
    void release() {
        if (dev) (void)hipFree(dev);
        if (part) (void)hipFree(part);
        dev = nullptr;
        part = nullptr;
    }
    template <typename T>
    T* at(size_t o) const {
        return reinterpret_cast<T*>(static_cast<char*>(dev) + o);
    }

    // (cos, sin / w) of every run for these amplitudes.
    int angles(const double* params, const std::vector<int32_t>& gparam, const std::vector<double>& gscale) {
        int rc = upload();
        if (rc || !dev) return rc;
        void* host = nullptr;
        rc = staging_begin(runs.size() * sizeof(double2), &host);
        if (rc) return rc;
        double2* h = static_cast<double2*>(host);
        for (size_t r = 0; r < runs.size(); ++r) {
            const double a = params[gparam[runs[r].gen]] * gscale[runs[r].gen] * runs[r].w;
            h[r] = make_double2(std::cos(a), std::sin(a) / runs[r].w);
        }
        return staging_commit(at<char>(o_cs), runs.size() * sizeof(double2));
    }

    template <int MODE>
    int launch(int n, double2* x, double2* y) {
        Context& cx = ctx();
        const auto& ps = MODE == 2 ? rev : fwd;
        const size_t lds = ((size_t)sizeof(double2) << dims) * (MODE == 2 ? 2 : 1);
        for (size_t i = 0; i < ps.size(); ++i) {
            const uint32_t pass = (uint32_t)(MODE == 1 ? ps.size() - 1 - i : i);
            hipLaunchKernelGGL(k_program_tile<MODE>, dim3((unsigned)(1ull << (n - (int)dims))), dim3(kProgThreads), lds, cx.stream,
                               x, y, at<const ProgPass>(MODE == 2 ? o_rev : o_fwd), pass,
                               at<const ProgRun>(MODE == 2 ? o_rruns : o_fruns), at<const ProgTerm>(o_terms),
                               at<const double2>(o_cs), part, (uint32_t)(MODE == 2 && i == 0));
            QFE_HIP(hipGetLastError());
            cx.counters.fused++;
            cx.counters.tile++;
            cx.counters.bytes += (MODE == 2 ? 64.0 : 32.0) * (double)(1ull << n);
        }
        return QFE_OK;
    }
};

}  // namespace qfe

struct qfe_program_s {
    int n = 0;
    uint64_t ref = 0;
    std::vector<qfe_pauli> gen_terms;
    std::vector<uint64_t> gen_off;
    std::vector<int32_t> gparam;
    std::vector<double> gscale;
    uint64_t nparam = 0;
    std::vector<qfe_pauli> ham_terms;
    qfe::DevTable ham;      // Hamiltonian grouped by X mask
    std::vector<qfe::PauliGroup> hgroups;  // the same on the host, for the expectation passes
    std::vector<uint64_t> hz;
    std::vector<double2> hc;
    qfe::DevTable gens;     // every generator grouped by X mask
    std::vector<uint32_t> gen_ranges;
    double2* partial = nullptr;  // reduction partials (reused launch to launch)
    size_t partial_cap = 0;
    double2* gout = nullptr;     // per-group results (generators, then Hamiltonian)
    size_t gout_cap = 0;
    qfe_state psi = nullptr;
    qfe_state sig = nullptr;
    qfe::ProgTiles tiles;
    qfe::ProgramGraph* graph = nullptr;  // captured energy sequence (first graph energy call)
};

namespace qfe {

static int ensure_partial(qfe_program p, size_t entries) {
    if (p->partial_cap >= entries) return QFE_OK;
    if (p->partial) {
        QFE_HIP(hipStreamSynchronize(ctx().stream));
        QFE_HIP(hipFree(p->partial));
        p->partial = nullptr;
    }
    QFE_HIP(device_malloc(&p->partial, entries * sizeof(double2)));
    p->partial_cap = entries;
    return QFE_OK;
}

static int ensure_gout(qfe_program p, size_t entries) {
    if (p->gout_cap >= entries) return QFE_OK;
    if (p->gout) {
        QFE_HIP(hipStreamSynchronize(ctx().stream));
        QFE_HIP(hipFree(p->gout));
        p->gout = nullptr;
    }
    QFE_HIP(device_malloc(&p->gout, entries * sizeof(double2)));
    p->gout_cap = entries;
    return QFE_OK;
}

static int ensure_states(qfe_program p, bool need_sigma) {
    int rc = QFE_OK;
    if (!p->psi) rc = qfe_state_create(p->n, &p->psi);
    if (rc) return rc;
    if (need_sigma && !p->sig) rc = qfe_state_create(p->n, &p->sig);
    return rc;
}

// Lower generator k (forward: sign = +1; inverse: sign = -1, terms reversed).
static int lower_generator(qfe_program p, uint64_t k, const double* params, double sign, std::vector<HostOp>& ops) {
    const double theta = params[p->gparam[k]] * p->gscale[k] * sign;
    const uint64_t b = p->gen_off[k], e = p->gen_off[k + 1];
    for (uint64_t i = 0; i < e - b; ++i) {
        const qfe_pauli& t = p->gen_terms[sign > 0 ? b + i : e - 1 - i];
        // exp(theta * coeff * P) with coeff purely imaginary = exp(i * theta * Im(coeff) * P)
        int rc = lower_pexp(t, theta * t.coeff.im, p->n, ops);
        if (rc) return rc;
    }
    return QFE_OK;
}

static int prepare(qfe_program p, const double* params, qfe_state out) {
    int rc = launch_basis(out->d, out->N, p->ref, ctx().stream);
    if (rc) return rc;
    if (p->tiles.ok) {
        rc = p->tiles.angles(params, p->gparam, p->gscale);
        if (rc) return rc;
        if (p->tiles.dev) return p->tiles.launch<0>(p->n, out->d, nullptr);
    }
    std::vector<HostOp> ops;
    ops.reserve(p->gen_terms.size());
    for (uint64_t k = 0; k + 1 < p->gen_off.size(); ++k) {
        rc = lower_generator(p, k, params, +1.0, ops);
        if (rc) return rc;
    }
    return run_ops(out, ops);
}

static int fetch(const double2* dev, size_t count, std::vector<double2>& host) {
    host.resize(count);
    if (!count) return QFE_OK;
    void* pin = nullptr;
    int rc = pinned_reserve(count * sizeof(double2), &pin);
    if (rc) return rc;
    QFE_HIP(hipMemcpyAsync(pin, dev, count * sizeof(double2), hipMemcpyDeviceToHost, ctx().stream));
    QFE_HIP(hipStreamSynchronize(ctx().stream));
    std::memcpy(host.data(), pin, count * sizeof(double2));
    return QFE_OK;
}

static int energy_of(qfe_program p, qfe_state s, double* energy) {
    if (takes_orbits(p->n, true)) {
        std::vector<double2> per(p->hgroups.size());
        int rc = expval_groups(s->d, s->d, p->n, p->hgroups, p->hz, p->hc, per.data());
        if (rc) return rc;
        *energy = 0.0;
        for (const double2& v : per) *energy += v.x;
        return QFE_OK;
    }
    const uint32_t nch = expval_chunks(p->n, p->ham.ngroups);
    int rc = ensure_partial(p, (size_t)p->ham.ngroups * nch);
    if (rc) return rc;
    rc = ensure_gout(p, p->ham.ngroups);
    if (rc) return rc;
    rc = launch_expval_async(s->d, s->d, p->n, p->ham.g, p->ham.ngroups, p->ham.z, p->ham.c, p->partial, nch, p->gout);
    if (rc) return rc;
    std::vector<double2> per;
    rc = fetch(p->gout, p->ham.ngroups, per);
    if (rc) return rc;
    double e = 0.0;
    for (const double2& v : per) e += v.x;
    *energy = e;
    return QFE_OK;
}

// Plan the ansatz with device-side angles and capture the energy sequence.
static int graph_build(qfe_program p) {
    int rc = ensure_states(p, false);
    if (rc) return rc;
    // every term with a nonzero coefficient becomes an op, whatever the amplitudes
    std::vector<HostOp> ops;
    std::vector<DevAngle> table;
    for (uint64_t k = 0; k + 1 < p->gen_off.size(); ++k) {
        if (p->gscale[k] == 0.0) continue;
        for (uint64_t i = p->gen_off[k]; i < p->gen_off[k + 1]; ++i) {
            const qfe_pauli& t = p->gen_terms[i];
            if (t.coeff.im == 0.0) continue;
            rc = lower_pexp(t, 1.0, p->n, ops);
            if (rc) return rc;
            ops.back().src = (int32_t)table.size();
            table.push_back(DevAngle{0, (uint32_t)p->gparam[k], 0, p->gscale[k], t.coeff.im});
        }
    }
    ProgramGraph* g = new ProgramGraph();
    std::vector<char> image;
    std::vector<AngleRef> refs;
    rc = plan_build(ops, p->n, true, &g->plan, image, refs);
    if (rc) {
        graph_free(g);
        return rc;
    }
    std::vector<DevAngle> angles;
    angles.reserve(refs.size());
    for (const AngleRef& r : refs) {
        DevAngle a = table[r.src];
        a.off = r.off;
        angles.push_back(a);
    }
    g->nangles = (uint32_t)angles.size();
    const uint32_t nhg = p->ham.ngroups;
    const uint32_t nch = expval_chunks(p->n, nhg);
    auto alloc = [&]() -> int {
        if (!image.empty()) QFE_HIP(device_malloc(&g->image, image.size()));
        if (!angles.empty()) QFE_HIP(device_malloc(&g->angles, angles.size() * sizeof(DevAngle)));
        QFE_HIP(device_malloc(&g->dparams, (p->nparam + 1) * sizeof(double)));
        QFE_HIP(device_malloc(&g->partial, ((size_t)nhg * nch + 1) * sizeof(double2)));
        QFE_HIP(device_malloc(&g->gout, ((size_t)nhg + 1) * sizeof(double2)));
        QFE_HIP(hipHostMalloc(reinterpret_cast<void**>(&g->hparams), (p->nparam + 1) * sizeof(double), hipHostMallocDefault));
        QFE_HIP(hipHostMalloc(reinterpret_cast<void**>(&g->hout), ((size_t)nhg + 1) * sizeof(double2), hipHostMallocDefault));
        if (!image.empty()) QFE_HIP(hipMemcpy(g->image, image.data(), image.size(), hipMemcpyHostToDevice));
        if (!angles.empty())
            QFE_HIP(hipMemcpy(g->angles, angles.data(), angles.size() * sizeof(DevAngle), hipMemcpyHostToDevice));
        return QFE_OK;
    };
    rc = alloc();
    if (rc) {
        graph_free(g);
        return rc;
    }
    hipStream_t st = ctx().stream;
    QFE_HIP(hipStreamSynchronize(st));
    hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed);
    if (e != hipSuccess) {
        graph_free(g);
        return hip_fail(e, "qfe_program_energy_graph: begin capture");
    }
    // launches below only record; the capture is always ended before returning
    auto record = [&]() -> int {
        if (p->nparam)
            QFE_HIP(hipMemcpyAsync(g->dparams, g->hparams, p->nparam * sizeof(double), hipMemcpyHostToDevice, st));
        if (g->nangles) {
            hipLaunchKernelGGL(k_program_angles, dim3((g->nangles + 255) / 256), dim3(256), 0, st, g->dparams, g->angles,
                               g->nangles, g->image);
            QFE_HIP(hipGetLastError());
        }
        int r = launch_basis(p->psi->d, p->psi->N, p->ref, st);
        if (!r) r = plan_launch(g->plan, p->psi, g->image);
        if (!r) r = launch_expval_async(p->psi->d, p->psi->d, p->n, p->ham.g, nhg, p->ham.z, p->ham.c, g->partial, nch, g->gout);
        if (r) return r;
        if (nhg) QFE_HIP(hipMemcpyAsync(g->hout, g->gout, nhg * sizeof(double2), hipMemcpyDeviceToHost, st));
        return QFE_OK;
    };
    rc = record();
    e = hipStreamEndCapture(st, &g->graph);
    if (!rc && e != hipSuccess) rc = hip_fail(e, "qfe_program_energy_graph: end capture");
    if (!rc) {
        e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
        if (e != hipSuccess) rc = hip_fail(e, "qfe_program_energy_graph: instantiate");
    }
    if (rc) {
        graph_free(g);
        return rc;
    }
    p->graph = g;
    return QFE_OK;
}

static int graph_energy(qfe_program p, const double* params, double* energy) {
    ProgramGraph* g = p->graph;
    hipStream_t st = ctx().stream;
    // the previous replay has finished (every call synchronizes), so the pinned buffers are free
    if (p->nparam) std::memcpy(g->hparams, params, p->nparam * sizeof(double));
    QFE_HIP(hipGraphLaunch(g->exec, st));
    QFE_HIP(hipStreamSynchronize(st));
    double e = 0.0;
    for (uint32_t i = 0; i < p->ham.ngroups; ++i) e += g->hout[i].x;
    *energy = e;
    return QFE_OK;
}

int program_nqubit(qfe_program p) { return p->n; }
uint64_t program_nparam(qfe_program p) { return p->nparam; }
ProgramView program_view(qfe_program p) {
    return ProgramView{p->n, p->ref, p->nparam, &p->gen_terms, &p->gen_off, &p->gparam, &p->gscale, &p->ham_terms};
}

}  // namespace qfe

using namespace qfe;

extern "C" {

int qfe_program_create(int nqubit, uint64_t ref_index, const qfe_pauli* gen_terms, const uint64_t* gen_offsets,
                       uint64_t ngen, const int32_t* gen_param, const double* gen_scale, uint64_t nparam,
                       const qfe_pauli* ham_terms, uint64_t nham, qfe_program* out) {
    if (!out) return fail(QFE_ERR_ARG, "qfe_program_create: null output");
    *out = nullptr;
    if (nqubit < 1 || nqubit > 36) return fail(QFE_ERR_ARG, "qfe_program_create: nqubit must be in [1, 36]");
    if (ref_index >> nqubit) return fail(QFE_ERR_ARG, "qfe_program_create: reference index out of range");
    if (ngen && (!gen_terms || !gen_offsets || !gen_param || !gen_scale))
        return fail(QFE_ERR_ARG, "qfe_program_create: null generator arrays");
    if (nham && !ham_terms) return fail(QFE_ERR_ARG, "qfe_program_create: null Hamiltonian");
    const uint64_t lim = (1ull << nqubit) - 1ull;
    if (ngen && gen_offsets[0] != 0) return fail(QFE_ERR_ARG, "qfe_program_create: gen_offsets[0] must be 0");
    for (uint64_t k = 0; k < ngen; ++k) {
        if (gen_offsets[k + 1] < gen_offsets[k]) return fail(QFE_ERR_ARG, "qfe_program_create: offsets must be non-decreasing");
        if (gen_param[k] < 0 || (uint64_t)gen_param[k] >= nparam)
            return fail(QFE_ERR_ARG, "qfe_program_create: generator parameter index out of range");
    }
    const uint64_t nterms = ngen ? gen_offsets[ngen] : 0;
    for (uint64_t i = 0; i < nterms; ++i) {
        const qfe_pauli& t = gen_terms[i];
        if ((t.x | t.z) & ~lim) return fail(QFE_ERR_ARG, "qfe_program_create: generator term acts outside the register");
        if (std::fabs(t.coeff.re) > 1.0e-14)
            return fail(QFE_ERR_ARG, "qfe_program_create: generator coefficients must be purely imaginary");
    }
    for (uint64_t i = 0; i < nham; ++i)
        if ((ham_terms[i].x | ham_terms[i].z) & ~lim) return fail(QFE_ERR_ARG, "qfe_program_create: Hamiltonian term acts outside the register");
    int rc = ensure_init();
    if (rc) return rc;
    qfe_program p = new qfe_program_s();
    p->n = nqubit;
    p->ref = ref_index;
    p->gen_terms.assign(gen_terms, gen_terms + nterms);
    p->gen_off.assign(gen_offsets, gen_offsets + (ngen ? ngen + 1 : 1));
    if (!ngen) p->gen_off[0] = 0;
    p->gparam.assign(gen_param, gen_param + ngen);
    p->gscale.assign(gen_scale, gen_scale + ngen);
    p->nparam = nparam;
    p->ham_terms.assign(ham_terms, ham_terms + nham);
    std::vector<PauliGroup> g;
    std::vector<uint64_t> z;
    std::vector<double2> c;
    group_terms(ham_terms, nham, g, z, c);
    rc = table_upload(g, z, c, p->ham);
    p->hgroups = g;
    p->hz = z;
    p->hc = c;
    if (!rc && ngen) {
        group_many(gen_terms, gen_offsets, ngen, g, z, c, p->gen_ranges);
        rc = table_upload(g, z, c, p->gens);
    }
    if (rc) {
        qfe_program_destroy(p);
        return rc;
    }
    // strings that are not Hermitian keep the lowering, which reports them
    bool hermitian = true;
    for (const qfe_pauli& t : p->gen_terms) hermitian = hermitian && !pexp_refusal(t);
    if (ngen && hermitian) p->tiles.build(p->n, p->gen_terms, p->gen_off);
    *out = p;
    return QFE_OK;
}

int qfe_program_destroy(qfe_program p) {
    if (!p) return QFE_OK;
    (void)hipStreamSynchronize(ctx().stream);
    table_free(p->ham);
    table_free(p->gens);
    p->tiles.release();
    if (p->partial) (void)hipFree(p->partial);
    if (p->gout) (void)hipFree(p->gout);
    graph_free(p->graph);
    qfe_state_destroy(p->psi);
    qfe_state_destroy(p->sig);
    delete p;
    return QFE_OK;
}

int qfe_program_prepare(qfe_program p, const double* params, qfe_state out) {
    if (!p || !out || !out->d || (p->nparam && !params)) return fail(QFE_ERR_ARG, "qfe_program_prepare: invalid argument");
    if (out->n != p->n) return fail(QFE_ERR_ARG, "qfe_program_prepare: state has the wrong number of qubits");
    return prepare(p, params, out);
}

int qfe_program_energy(qfe_program p, const double* params, double* energy) {
    if (!p || !energy || (p->nparam && !params)) return fail(QFE_ERR_ARG, "qfe_program_energy: invalid argument");
    int rc = ensure_states(p, false);
    if (rc) return rc;
    rc = prepare(p, params, p->psi);
    if (rc) return rc;
    return energy_of(p, p->psi, energy);
}

int qfe_program_energy_graph(qfe_program p, const double* params, double* energy) {
    if (!p || !energy || (p->nparam && !params)) return fail(QFE_ERR_ARG, "qfe_program_energy_graph: invalid argument");
    if (!p->graph) {
        int rc = graph_build(p);
        if (rc) return rc;
    }
    return graph_energy(p, params, energy);
}

int qfe_program_gradient(qfe_program p, const double* params, double* grad, double* energy) {
    if (!p || !grad || (p->nparam && !params)) return fail(QFE_ERR_ARG, "qfe_program_gradient: invalid argument");
    int rc = ensure_states(p, true);
    if (rc) return rc;
    rc = prepare(p, params, p->psi);
    if (rc) return rc;
    const uint64_t ngen = p->gen_off.size() - 1;
    const uint32_t ngg = p->gens.ngroups;
    const uint32_t nhg = p->ham.ngroups;
    // sigma = H psi
    rc = launch_apply_sum_async(p->psi->d, p->sig->d, p->n, p->ham.g, nhg, p->ham.z, p->ham.c);
    if (rc) return rc;
    if (p->tiles.sums()) {
        ProgTiles& T = p->tiles;
        rc = T.launch<2>(p->n, p->psi->d, p->sig->d);
        if (rc) return rc;
        hipLaunchKernelGGL(k_program_sum, dim3((unsigned)(ngen / 4 + 1)), dim3(256), 0, ctx().stream, T.part,
                           T.at<const uint2>(T.o_ranges), (uint32_t)(ngen + 1), T.at<double>(T.o_out));
        QFE_HIP(hipGetLastError());
        void* pin = nullptr;
        rc = pinned_reserve((ngen + 1) * sizeof(double), &pin);
        if (rc) return rc;
        QFE_HIP(hipMemcpyAsync(pin, T.at<double>(T.o_out), (ngen + 1) * sizeof(double), hipMemcpyDeviceToHost, ctx().stream));
        QFE_HIP(hipStreamSynchronize(ctx().stream));
        const double* r = static_cast<const double*>(pin);
        for (uint64_t i = 0; i < p->nparam; ++i) grad[i] = 0.0;
        for (uint64_t k = 0; k < ngen; ++k) grad[p->gparam[k]] += 2.0 * p->gscale[k] * r[k + 1];
        if (energy) *energy = r[0];
        return QFE_OK;
    }
    uint32_t maxg = nhg;
    for (uint64_t k = 0; k < ngen; ++k) maxg = std::max(maxg, p->gen_ranges[k + 1] - p->gen_ranges[k]);
    const uint32_t nch = expval_chunks(p->n, maxg);
    rc = ensure_partial(p, (size_t)maxg * nch);
    if (rc) return rc;
    rc = ensure_gout(p, (size_t)ngg + nhg);
    if (rc) return rc;
    if (energy) {
        rc = launch_expval_async(p->psi->d, p->psi->d, p->n, p->ham.g, nhg, p->ham.z, p->ham.c, p->partial, nch,
                                 p->gout + ngg);
        if (rc) return rc;
    }
    // reverse sweep: <sigma_k| A_k |psi_k>, then un-apply generator k on both
    for (uint64_t kk = ngen; kk-- > 0;) {
        const uint32_t g0 = p->gen_ranges[kk], g1 = p->gen_ranges[kk + 1];
        rc = launch_expval_async(p->sig->d, p->psi->d, p->n, p->gens.g + g0, g1 - g0, p->gens.z, p->gens.c, p->partial,
                                 nch, p->gout + g0);
        if (rc) return rc;
        if (kk == 0) break;
        std::vector<HostOp> ops;
        rc = lower_generator(p, kk, params, -1.0, ops);
        if (rc) return rc;
        std::vector<HostOp> ops2 = ops;
        rc = run_ops(p->psi, ops);
        if (rc) return rc;
        rc = run_ops(p->sig, ops2);
        if (rc) return rc;
    }
    std::vector<double2> per;
    rc = fetch(p->gout, (size_t)ngg + nhg, per);
    if (rc) return rc;
    for (uint64_t i = 0; i < p->nparam; ++i) grad[i] = 0.0;
    for (uint64_t k = 0; k < ngen; ++k) {
        double acc = 0.0;
        for (uint32_t g = p->gen_ranges[k]; g < p->gen_ranges[k + 1]; ++g) acc += per[g].x;
        grad[p->gparam[k]] += 2.0 * p->gscale[k] * acc;
    }
    if (energy) {
        double e = 0.0;
        for (uint32_t g = 0; g < nhg; ++g) e += per[ngg + g].x;
        *energy = e;
    }
    return QFE_OK;
}

int qfe_program_residuals(qfe_program p, const double* params, const uint64_t* idx, uint64_t count, qfe_c64* out) {
    if (!p || (count && (!idx || !out)) || (p->nparam && !params))
        return fail(QFE_ERR_ARG, "qfe_program_residuals: invalid argument");
    for (uint64_t i = 0; i < count; ++i)
        if (idx[i] >> p->n) return fail(QFE_ERR_ARG, "qfe_program_residuals: basis index out of range");
    int rc = ensure_states(p, true);
    if (rc) return rc;
    rc = prepare(p, params, p->psi);
    if (rc) return rc;
    // sigma = H U|ref>, then U^dag: generators last to first, terms reversed
    rc = launch_apply_sum_async(p->psi->d, p->sig->d, p->n, p->ham.g, p->ham.ngroups, p->ham.z, p->ham.c);
    if (rc) return rc;
    if (p->tiles.dev) {
        rc = p->tiles.launch<1>(p->n, p->sig->d, nullptr);
    } else {
        std::vector<HostOp> ops;
        for (uint64_t kk = p->gen_off.size() - 1; kk-- > 0;) {
            rc = lower_generator(p, kk, params, -1.0, ops);
            if (rc) return rc;
        }
        rc = run_ops(p->sig, ops);
    }
    if (rc) return rc;
    for (uint64_t i = 0; i < count; ++i) {
        rc = qfe_state_get_amp(p->sig, idx[i], &out[i]);
        if (rc) return rc;
    }
    return QFE_OK;
}

int qfe_program_pool_gradients(qfe_program p, const double* params, const qfe_pauli* pool_terms,
                               const uint64_t* op_offsets, uint64_t nops, uint64_t batch, double* grads) {
    if (!p || (nops && (!pool_terms || !op_offsets || !grads)) || (p->nparam && !params))
        return fail(QFE_ERR_ARG, "qfe_program_pool_gradients: invalid argument");
    if (nops == 0) return QFE_OK;
    if (batch == 0) batch = 64;
    const uint64_t lim = (1ull << p->n) - 1ull;
    for (uint64_t i = 0; i < op_offsets[nops]; ++i)
        if ((pool_terms[i].x | pool_terms[i].z) & ~lim) return fail(QFE_ERR_ARG, "qfe_program_pool_gradients: term outside the register");
    int rc = ensure_states(p, true);
    if (rc) return rc;
    rc = prepare(p, params, p->psi);
    if (rc) return rc;
    rc = launch_apply_sum_async(p->psi->d, p->sig->d, p->n, p->ham.g, p->ham.ngroups, p->ham.z, p->ham.c);
    if (rc) return rc;
    std::vector<PauliGroup> g;
    std::vector<uint64_t> z;
    std::vector<double2> c;
    std::vector<uint32_t> ranges;
    group_many(pool_terms, op_offsets, nops, g, z, c, ranges);
    DevTable t;
    rc = table_upload(g, z, c, t);
    if (rc) {
        table_free(t);
        return rc;
    }
    rc = ensure_gout(p, g.size());
    // batches of `batch` operators per launch
    for (uint64_t b0 = 0; !rc && b0 < nops; b0 += batch) {
        const uint64_t b1 = std::min(nops, b0 + batch);
        const uint32_t g0 = ranges[b0], g1 = ranges[b1];
        if (g1 == g0) continue;
        const uint32_t nch = expval_chunks(p->n, g1 - g0);
        rc = ensure_partial(p, (size_t)(g1 - g0) * nch);
        if (!rc)
            rc = launch_expval_async(p->sig->d, p->psi->d, p->n, t.g + g0, g1 - g0, t.z, t.c, p->partial, nch,
                                     p->gout + g0);
    }
    std::vector<double2> per;
    if (!rc) rc = fetch(p->gout, g.size(), per);
    if (!rc) {
        for (uint64_t k = 0; k < nops; ++k) {
            double acc = 0.0;
            for (uint32_t gi = ranges[k]; gi < ranges[k + 1]; ++gi) acc += per[gi].x;
            grads[k] = 2.0 * acc;
        }
    }
    (void)hipStreamSynchronize(ctx().stream);
    table_free(t);
    return rc;
}

}  // extern "C"
