// nbx_ref64.hip -- FP64 kernels that reproduce the reference's arithmetic bit for bit.
//
// Built with -ffp-contract=off: every a*b+c rounds twice, as Julia does without
// @fastmath/@muladd.  Every per-target sum takes the source atoms in ascending index
// order (the reference's `for j in indxs`): a target has a wavefront whose lanes compute
// the pair terms of 64 sources at once before the terms are added in j order (gravity of
// many bodies: one thread per target, sources staged through LDS tiles).  Neither changes
// the order or the rounding of the sums.  Device state is SoA: x[k * n + i].
#include <algorithm>
#include <mutex>

#include "nbx_internal.h"

#define REF_TILE 256

// ---------------------------------------------------------------------------
// Layout / fill helpers
// ---------------------------------------------------------------------------

__global__ void k_fill(double* __restrict__ p, int64_t count, double value) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < count) p[t] = value;
}

__global__ void k_aos_to_soa(const double* __restrict__ aos, double* __restrict__ soa,
                             int64_t n) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 3 * n) {
        int64_t i = t / 3, k = t - 3 * i;
        soa[k * n + i] = aos[t];
    }
}

__global__ void k_soa_to_aos(const double* __restrict__ soa, double* __restrict__ aos,
                             int64_t n) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 3 * n) {
        int64_t i = t / 3, k = t - 3 * i;
        aos[t] = soa[k * n + i];
    }
}

// one saved frame: positions and velocities to the caller's layout
__global__ void k_save_frame(const double* __restrict__ x, const double* __restrict__ v,
                             double* __restrict__ uf, double* __restrict__ vf, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * n) return;
    const int64_t i = t / 3, k = t - 3 * i;
    uf[t] = x[k * n + i];
    vf[t] = v[k * n + i];
}

void ref64_save_frame(hipStream_t s, const double* x, const double* v, double* uf, double* vf,
                      int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_save_frame, dim3(nbx_blocks(3 * n, 256)), dim3(256), 0, s, x, v, uf, vf, n);
}

void ref64_fill(hipStream_t s, double* p, int64_t count, double value) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_fill, dim3(nbx_blocks(count, 256)), dim3(256), 0, s, p, count, value);
}
void ref64_aos_to_soa(hipStream_t s, const double* aos, double* soa, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_aos_to_soa, dim3(nbx_blocks(3 * n, 256)), dim3(256), 0, s, aos, soa, n);
}
void ref64_soa_to_aos(hipStream_t s, const double* soa, double* aos, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_soa_to_aos, dim3(nbx_blocks(3 * n, 256)), dim3(256), 0, s, soa, aos, n);
}

// ---------------------------------------------------------------------------
// Pair terms in the reference's order: Lennard-Jones (src/basic_potentials.jl:240-272),
// truncated Coulomb (:274-304) and reaction field, gravity (:306-331)
// ---------------------------------------------------------------------------

// Wavefront per target.  Its 64 lanes evaluate the pair terms factor * r_ij of up to 64
// sources at once; the terms of the pairs in range go to LDS in ascending j, and lanes 0..2
// add them to the x, y, z sums one after another, so every sum sees the reference's terms in
// the reference's order: the result is bit for bit a loop over j.  A pair out of range is
// left out: its term would be +0.0, which leaves a sum unchanged (the sums start at +0.0 and
// never become -0.0 under round-to-nearest).
//
// FILTER (cubic box, finite cutoff): sources first pass an FP32 distance test on box
// fractions, widened by 2e-6 of the box (the fractions are within 1e-7), and only the
// survivors are gathered, 64 at a time, for the FP64 evaluation.  With 55 of 4,000 sources in
// range the FP64 work per target is one or two passes instead of 63, and the ordered adds
// are 55 instead of 4,032.  us per evaluation, against adding all 64 lanes' terms of every
// chunk through v_readlane: n = 864 36.6 -> 7.9 (the fused step included), n = 4,000
// 341 -> 22; water's Coulomb and Lennard-Jones terms (1,029 atoms, cutoff 0.45 L) 71 -> 13.6.
// A few targets per SIMD make it a latency chain: one wavefront's fractions, gathers, pair
// terms and about 13 cycles per ordered add; up to REF_SPLIT_TARGETS targets share it among
// four wavefronts each (ref_block_sum; n = 864 7.7 -> 6.5).
#define REF_WAVES 4   // targets (wavefronts) per block
// Targets that get a block of four wavefronts each (filtered sums): as many as run at once,
// six blocks (27 KB of LDS each) on each of 256 CUs.  us per step with one / four
// wavefronts: Lennard-Jones n = 256 5.4 / 5.2, 500 6.3 / 5.5, 864 7.7 / 6.3, 1,372 9.7 / 9.5,
// 2,048 11.2 / 13.1, 4,000 20 / 33; water (4/3 targets an atom) 375 atoms 13.1 / 10.9, 1,029
// 17.9 / 17.1, 1,536 19.4 / 19.2, 2,187 24.1 / 28.2.
#define REF_SPLIT_BLOCKS 6
#define REF_SPLIT_TARGETS (256 * REF_SPLIT_BLOCKS)
enum { REF_LJ = 0, REF_COULOMB = 1, REF_RF = 2, REF_GRAV = 3 };

struct ref_law {
    double s2, R2;     // sigma^2, cutoff^2
    double c;          // Lennard-Jones eps, Coulomb k, gravity G
    double krf2;       // 2 k_rf
    float lim;         // FILTER: squared cutoff in box fractions, widened
    int jstride, water;
    int64_t nj;
};

struct ref_atoms {
    const double* x;       // SoA
    const float4* frac;    // box fractions (FILTER)
    const double* ms;
    const double* qs;
    int64_t n;
};

__device__ __forceinline__ bool ref_excluded(int64_t i, int64_t j, int water) {
    return water ? (i / 3) == (j / 3) : i == j;   // src/nbody_to_ode.jl:326, :346-348
}

// box fraction of a coordinate for the filter; NaN (passes every test) where x / L is too
// large for the margin to hold
__device__ __forceinline__ float ref_frac(double x, double invL) {
    const double t = x * invL;
    return fabs(t) < 1048576.0 ? (float)(t - floor(t)) : __builtin_nanf("");
}

// factor * r_ij of one pair; false when it is out of range
template <int KIND>
__device__ __forceinline__ bool ref_pair_term(const ref_law& law, double xi, double yi, double zi,
                                              double xj, double yj, double zj, double wj,
                                              const nbx_bcv& bc, double* t) {
    if (KIND == REF_GRAV) {
        const double rx = xi - xj, ry = yi - yj, rz = zi - zj;
        const double ss = rx * rx + ry * ry;
        const double nr = sqrt(ss + rz * rz);
        const double factor = -law.c * wj / (nr * nr * nr);
        t[0] = factor * rx;
        t[1] = factor * ry;
        t[2] = factor * rz;
        return true;
    }
    double rx, ry, rz, r2;
    nbx_displacement(xi, yi, zi, xj, yj, zj, bc, rx, ry, rz, r2);
    if (!(r2 < law.R2)) return false;
    double factor;
    if (KIND == REF_LJ) {
        const double qq = law.s2 / r2;
        const double s6 = qq * qq * qq;
        const double s12 = s6 * s6;
        factor = (2.0 * s12 - s6) / r2;
    } else {
        const double r = sqrt(r2);
        if (KIND == REF_RF) factor = wj * (1.0 / (r * r2) - law.krf2);
        else factor = wj / (r * r2);
    }
    t[0] = factor * rx;
    t[1] = factor * ry;
    t[2] = factor * rz;
    return true;
}

// component c of cnt terms added to f one after another
__device__ __forceinline__ double ref_add_terms(double f, const double* term, int cnt, int c) {
    int q = 0;
    for (; q + 16 <= cnt; q += 16) {
        double u[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) u[k] = term[3 * (q + k) + c];
#pragma unroll
        for (int k = 0; k < 16; ++k) f += u[k];
    }
    for (; q + 4 <= cnt; q += 4) {
        double u[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) u[k] = term[3 * (q + k) + c];
#pragma unroll
        for (int k = 0; k < 4; ++k) f += u[k];
    }
    for (; q < cnt; ++q) f += term[3 * q + c];
    return f;
}

// the whole wavefront's sum over the sources of target i: component min(lane, 2) in each lane
template <int KIND, bool FILTER>
__device__ __forceinline__ double ref_wave_sum(const ref_atoms& A, const ref_law& law,
                                               const nbx_bcv& bc, int64_t i, int* cand,
                                               double* term) {
    const int lane = threadIdx.x & 63;
    const int c = lane < 2 ? lane : 2;
    const int64_t n = A.n;
    const double xi = A.x[i], yi = A.x[n + i], zi = A.x[2 * n + i];
    const double* const w = KIND == REF_GRAV ? A.ms : (KIND == REF_LJ ? nullptr : A.qs);
    double f = 0.0;
    // the terms of up to 64 sources, one per lane (in ascending j), added in order
    const auto add = [&](bool ok, double xj, double yj, double zj, double wj) {
        double t[3] = {0.0, 0.0, 0.0};
        const bool hit = ok && ref_pair_term<KIND>(law, xi, yi, zi, xj, yj, zj, wj, bc, t);
        const unsigned long long mask = __ballot(hit);
        if (mask == 0ull) return;
        const int at = (int)__builtin_amdgcn_mbcnt_hi(
            (unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
        if (hit) {
            term[3 * at] = t[0];
            term[3 * at + 1] = t[1];
            term[3 * at + 2] = t[2];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        f = ref_add_terms(f, term, __popcll(mask), c);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    if constexpr (FILTER) {
        const float4 fi = A.frac[i];
        int pending = 0;   // uniform
        const auto eval = [&](int cnt) {
            const bool ok = lane < cnt;
            const int64_t j = ok ? cand[lane] : i;
            add(ok, A.x[j], A.x[n + j], A.x[2 * n + j], w != nullptr ? w[j] : 0.0);
        };
        constexpr int U = 4;   // chunks of 64 whose fractions are in flight together
        for (int64_t base = 0; base < law.nj; base += 64 * U) {
            float4 fj[U];
#pragma unroll
            for (int q = 0; q < U; ++q) {
                const int64_t jj = base + 64 * q + lane;
                fj[q] = A.frac[jj < law.nj ? jj * law.jstride : i];
            }
#pragma unroll
            for (int q = 0; q < U; ++q) {
                const int64_t jj = base + 64 * q + lane, j = jj * law.jstride;
                float dx = fi.x - fj[q].x, dy = fi.y - fj[q].y, dz = fi.z - fj[q].z;
                dx -= rintf(dx);
                dy -= rintf(dy);
                dz -= rintf(dz);
                const bool near = jj < law.nj && !ref_excluded(i, j, law.water) &&
                                  !(dx * dx + dy * dy + dz * dz >= law.lim);
                const unsigned long long mask = __ballot(near);
                if (mask == 0ull) continue;
                const int at = pending + (int)__builtin_amdgcn_mbcnt_hi(
                    (unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
                if (near) cand[at] = (int)j;
                pending += __popcll(mask);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (pending >= 64) {
                    eval(64);
                    pending -= 64;
                    const int rest = cand[64 + lane];   // moved down (past the count: unused)
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    cand[lane] = rest;
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
            }
        }
        if (pending > 0) eval(pending);
    } else {
        // every source: the next chunk's atoms are loaded while this one is added
        const auto load = [&](int64_t jj, double* p) {
            const int64_t j = jj < law.nj ? jj * law.jstride : i;
            p[0] = A.x[j]; p[1] = A.x[n + j]; p[2] = A.x[2 * n + j];
            p[3] = w != nullptr ? w[j] : 0.0;
        };
        double nx[4];
        load(lane, nx);
        for (int64_t base = 0; base < law.nj; base += 64) {
            const double px = nx[0], py = nx[1], pz = nx[2], pw = nx[3];
            if (base + 64 < law.nj) load(base + 64 + lane, nx);
            const int64_t jj = base + lane;
            add(jj < law.nj && !ref_excluded(i, jj * law.jstride, law.water), px, py, pz, pw);
        }
    }
    return f;
}

// The filtered sum of one target by a block of four wavefronts: in a round of at most 1,024
// sources each takes up to 256 consecutive ones, filters them and leaves its terms in LDS in
// ascending j; the first wavefront then adds the four runs of terms in order, so the sum is
// that of ref_wave_sum bit for bit.  With few targets the sum is a latency chain, and a
// wavefront alone spends most of it in the filter (n = 864, us: filter 3.3, terms and adds
// 1.5, end of the step 0.6).  The result is valid in wavefront 0.
struct ref_block_lds {
    uint16_t cand[4][256];
    double term[4][3 * 256];
    int count[4];
};

template <int KIND>
__device__ __forceinline__ double ref_block_sum(const ref_atoms& A, const ref_law& law,
                                                const nbx_bcv& bc, int64_t i, ref_block_lds& S) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane < 2 ? lane : 2;
    const int64_t n = A.n;
    const double xi = A.x[i], yi = A.x[n + i], zi = A.x[2 * n + i];
    const float4 fi = A.frac[i];
    const double* const w = KIND == REF_LJ ? nullptr : A.qs;
    const int64_t chunks = (law.nj + 63) >> 6;
    // rounds of equal size, at most four chunks per wavefront
    const int64_t rounds = (chunks + 15) >> 4;
    const int u = (int)((chunks + 4 * rounds - 1) / (4 * rounds));
    double f = 0.0;
    for (int64_t first = 0; first < chunks;) {   // the same for the whole block
        const int64_t base = 64 * (first + wave * u);
        float4 fj[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t jj = base + 64 * q + lane;
            fj[q] = A.frac[q < u && jj < law.nj ? jj * law.jstride : i];
        }
        int pending = 0;   // uniform over the wavefront
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t jj = base + 64 * q + lane;
            float dx = fi.x - fj[q].x, dy = fi.y - fj[q].y, dz = fi.z - fj[q].z;
            dx -= rintf(dx);
            dy -= rintf(dy);
            dz -= rintf(dz);
            const bool near = q < u && jj < law.nj && !ref_excluded(i, jj * law.jstride, law.water) &&
                              !(dx * dx + dy * dy + dz * dz >= law.lim);
            const unsigned long long mask = __ballot(near);
            const int at = pending + (int)__builtin_amdgcn_mbcnt_hi(
                (unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
            if (near) S.cand[wave][at] = (uint16_t)(64 * q + lane);
            pending += __popcll(mask);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        int got = 0;
        for (int p = 0; p < pending; p += 64) {
            const bool ok = p + lane < pending;
            const int64_t j = ok ? (base + S.cand[wave][p + lane]) * law.jstride : i;
            double t[3] = {0.0, 0.0, 0.0};
            const bool hit = ok && ref_pair_term<KIND>(law, xi, yi, zi, A.x[j], A.x[n + j],
                                                       A.x[2 * n + j], w != nullptr ? w[j] : 0.0,
                                                       bc, t);
            const unsigned long long mask = __ballot(hit);
            const int at = got + (int)__builtin_amdgcn_mbcnt_hi(
                (unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
            if (hit) {
#pragma unroll
                for (int k = 0; k < 3; ++k) S.term[wave][3 * at + k] = t[k];
            }
            got += __popcll(mask);
        }
        if (lane == 0) S.count[wave] = got;
        first += 4 * u;
        __syncthreads();
        if (wave == 0)
            for (int v = 0; v < 4; ++v) f = ref_add_terms(f, S.term[v], S.count[v], c);
        if (first < chunks) __syncthreads();   // read before the next round writes
    }
    return f;
}

// the closure's contribution to atom i from the sum: dv += coeff * f
template <int KIND>
__device__ __forceinline__ double ref_contribution(const ref_atoms& A, const ref_law& law,
                                                   int64_t i, double f) {
    if (KIND == REF_LJ) return 24.0 * law.c / A.ms[i] * f;
    if (KIND == REF_GRAV) return f;
    return law.c * A.qs[i] / A.ms[i] * f;
}

// End of step `step` for component c of atom i, with the acceleration a of its potentials:
// thermostat force, kick, Langevin B and Andersen; then (drift) the start of step + 1:
// Langevin A, positions into the other buffer, half-kicked velocity, box fraction.  The
// expressions of k_ref_berendsen, k_ref_kick, k_ref_langevin_half, k_ref_andersen and
// k_ref_drift; counter: the atom whose number decides an Andersen collision (the molecule's
// O for water), m_andersen its mass.
__device__ __forceinline__ void ref_end_step(const ref64_step& st, int64_t n, int64_t i, int c,
                                             double a, double mi, int64_t counter,
                                             double m_andersen) {
    const int64_t k = c * n + i;
    const double h = st.vh[k];
    if (st.therm == NBX_THERM_BERENDSEN) {
        const double T = st.d_T[0];
        if (1.0 / T == __builtin_inf()) a += st.gamma * h;
        else {
            const double cb = st.gamma * (st.T / T - 1.0);
            a += cb * h;
        }
    }
    st.a[k] = a;
    double v = h + st.dt * (0.5 * a);
    double g[3], sig = 0.0;
    if (st.therm == NBX_THERM_LANGEVIN) {
        sig = st.c2 * sqrt(st.kb * st.T / mi);
        nbx_rng_normals3(st.seed, i, st.step, NBX_RNG_LANGEVIN_B, g);
        v = st.c1 * v + sig * (c == 0 ? g[0] : (c == 1 ? g[1] : g[2]));
    } else if (st.therm == NBX_THERM_ANDERSEN &&
               nbx_rng_uniform(st.seed, counter, st.step, NBX_RNG_ANDERSEN) < st.prob) {
        const double vdev = sqrt(st.kb * st.T / m_andersen);
        nbx_rng_normals3(st.seed, i, st.step, NBX_RNG_ANDERSEN, g);
        v = vdev * (c == 0 ? g[0] : (c == 1 ? g[1] : g[2]));
    }
    st.v[k] = v;
    if (!st.drift) return;
    if (st.therm == NBX_THERM_LANGEVIN) {
        nbx_rng_normals3(st.seed, i, st.step + 1, NBX_RNG_LANGEVIN_A, g);
        v = st.c1 * v + sig * (c == 0 ? g[0] : (c == 1 ? g[1] : g[2]));
    }
    const double half = 0.5, dtsq = st.dt * st.dt;
    const double px = st.x_in[k] + st.dt * v + dtsq * (half * a);
    st.x_out[k] = px;
    st.vh[k] = v + st.dt * (half * a);
    if (st.frac_out != nullptr)
        reinterpret_cast<float*>(st.frac_out + i)[c] = ref_frac(px, st.invL);
}

// targets i = ib, ib + istride, ...: dv += contribution, or (STEP) the acceleration a_in
// (nullptr: 0) + contribution and the end of the step
template <int KIND, bool FILTER, bool STEP>
__global__ void __launch_bounds__(64 * REF_WAVES)
k_ref_pairs(ref_atoms A, ref_law law, nbx_bcv bc, int64_t ib, int64_t cnt, int istride,
            double* __restrict__ dv, ref64_step st) {
    __shared__ int cand[REF_WAVES][128];
    __shared__ double term[REF_WAVES][192];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * REF_WAVES + wave;
    if (t >= cnt) return;   // the whole wavefront
    const int64_t i = ib + t * istride;
    const double f = ref_wave_sum<KIND, FILTER>(A, law, bc, i, cand[wave], term[wave]);
    if (lane >= 3) return;
    const double add = ref_contribution<KIND>(A, law, i, f);
    const int64_t k = lane * A.n + i;
    if constexpr (STEP) {
        ref_end_step(st, A.n, i, lane, (st.a_in != nullptr ? st.a_in[k] : 0.0) + add, A.ms[i], i,
                     A.ms[0]);
    } else {
        dv[k] += add;
    }
}

// a block per target: few targets (REF_SPLIT_TARGETS)
template <int KIND, bool STEP>
__global__ void __launch_bounds__(256, REF_SPLIT_BLOCKS)
k_ref_pairs_split(ref_atoms A, ref_law law, nbx_bcv bc, int64_t ib, int istride,
                  double* __restrict__ dv, ref64_step st) {
    __shared__ ref_block_lds S;
    const int64_t i = ib + (int64_t)blockIdx.x * istride;
    const double f = ref_block_sum<KIND>(A, law, bc, i, S);
    if (threadIdx.x >= 3) return;
    const int c = threadIdx.x;
    const double add = ref_contribution<KIND>(A, law, i, f);
    const int64_t k = c * A.n + i;
    if constexpr (STEP) {
        ref_end_step(st, A.n, i, c, (st.a_in != nullptr ? st.a_in[k] : 0.0) + add, A.ms[i], i,
                     A.ms[0]);
    } else {
        dv[k] += add;
    }
}

static double rf_krf(double R, double eps_rf) {
    if (__builtin_isinf(eps_rf)) return 1.0 / (2.0 * R * R * R);
    return (eps_rf - 1.0) / ((2.0 * eps_rf + 1.0) * (R * R * R));
}

static ref_law make_law(const ref64_term& t, const nbx_bcv& bc) {
    ref_law law{};
    law.jstride = t.jstride;
    law.nj = t.nj;
    law.water = t.water;
    if (t.kind == NBX_TERM_LJ) {
        law.c = t.p[0];
        law.s2 = t.p[1] * t.p[1];
        law.R2 = t.p[2] * t.p[2];
    } else if (t.kind == NBX_TERM_GRAV) {
        law.c = t.p[0];
    } else {
        law.c = t.p[0];
        law.R2 = t.p[1] * t.p[1];
        if (t.kind == NBX_TERM_RF) law.krf2 = 2.0 * rf_krf(t.p[1], t.p[2]);
    }
    if (t.filter) {
        const double R = (t.kind == NBX_TERM_LJ ? t.p[2] : t.p[1]) / bc.b[0] + 2e-6;
        law.lim = (float)(R * R * (1.0 + 1e-6));
    }
    return law;
}

bool ref64_filters(const ref64_term& t, const nbx_bcv& bc) {
    if (bc.kind != NBX_BC_CUBIC || t.kind == NBX_TERM_GRAV) return false;
    const double R = t.kind == NBX_TERM_LJ ? t.p[2] : t.p[1];
    // from half the box on nearly every source passes: the test would only add work
    return R < 0.5 * bc.b[0];
}

template <int KIND, bool STEP>
static void launch_pairs(hipStream_t s, const ref64_term& t, const ref_atoms& A,
                         const nbx_bcv& bc, int64_t ib, int64_t ie, double* dv,
                         const ref64_step& st) {
    const ref_law law = make_law(t, bc);
    const int64_t cnt = (ie - ib + t.istride - 1) / t.istride;
    const dim3 grid(nbx_blocks(cnt, REF_WAVES)), block(64 * REF_WAVES);
    if constexpr (KIND != REF_GRAV) {
        if (t.filter && cnt <= REF_SPLIT_TARGETS) {
            hipLaunchKernelGGL((k_ref_pairs_split<KIND, STEP>), dim3((unsigned)cnt), dim3(256), 0, s,
                               A, law, bc, ib, t.istride, dv, st);
            return;
        }
        if (t.filter) {
            hipLaunchKernelGGL((k_ref_pairs<KIND, true, STEP>), grid, block, 0, s, A, law, bc, ib,
                               cnt, t.istride, dv, st);
            return;
        }
    }
    hipLaunchKernelGGL((k_ref_pairs<KIND, false, STEP>), grid, block, 0, s, A, law, bc, ib, cnt,
                       t.istride, dv, st);
}

void ref64_pairs(hipStream_t s, const ref64_term& t, const double* x, const float4* frac,
                 const double* ms, const double* qs, int64_t n, int64_t ib, int64_t ie,
                 const nbx_bcv& bc, double* dv, const ref64_step* step) {
    if (ie <= ib) return;
    const ref_atoms A{x, frac, ms, qs, n};
    const ref64_step st = step ? *step : ref64_step{};
#define REF_GO(KIND)                                                            \
    do {                                                                        \
        if (step) launch_pairs<KIND, true>(s, t, A, bc, ib, ie, dv, st);        \
        else launch_pairs<KIND, false>(s, t, A, bc, ib, ie, dv, st);            \
    } while (0)
    switch (t.kind) {
    case NBX_TERM_LJ: REF_GO(REF_LJ); break;
    case NBX_TERM_ELEC: REF_GO(REF_COULOMB); break;
    case NBX_TERM_RF: REF_GO(REF_RF); break;
    case NBX_TERM_GRAV: REF_GO(REF_GRAV); break;
    default: break;
    }
#undef REF_GO
}

__global__ void k_ref_fractions(const double* __restrict__ x, int64_t n, double invL,
                                float4* __restrict__ frac) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    frac[i] = make_float4(ref_frac(x[i], invL), ref_frac(x[n + i], invL),
                          ref_frac(x[2 * n + i], invL), 0.0f);
}

void ref64_fractions(hipStream_t s, const double* x, int64_t n, double L, float4* frac) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_ref_fractions, dim3(nbx_blocks(n, 256)), dim3(256), 0, s, x, n, 1.0 / L,
                       frac);
}

// ---------------------------------------------------------------------------
// Gravity of many bodies: src/basic_potentials.jl:306-331 (no boundary conditions, no
// cutoff).  One thread per target walks the sources: a third of the instructions of a
// wavefront per target, once there are targets enough to fill the chip (NBX_REF_GRAV_WAVES).
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(REF_TILE)
k_ref_grav(const double* __restrict__ x, double* __restrict__ dv, const double* __restrict__ ms,
           int64_t n, int64_t ib, int64_t ie, double G) {
    __shared__ double sx[REF_TILE], sy[REF_TILE], sz[REF_TILE], sm[REF_TILE];
    const int64_t i = ib + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = i < ie;
    double xi = 0.0, yi = 0.0, zi = 0.0;
    if (active) { xi = x[i]; yi = x[n + i]; zi = x[2 * n + i]; }
    double a1 = 0.0, a2 = 0.0, a3 = 0.0;
    for (int64_t base = 0; base < n; base += REF_TILE) {
        const int64_t j = base + threadIdx.x;
        if (j < n) {
            sx[threadIdx.x] = x[j]; sy[threadIdx.x] = x[n + j];
            sz[threadIdx.x] = x[2 * n + j]; sm[threadIdx.x] = ms[j];
        }
        __syncthreads();
        const int lim = (int)((n - base) < REF_TILE ? (n - base) : REF_TILE);
        if (active) {
            for (int q = 0; q < lim; ++q) {
                if (base + q == i) continue;
                double rx = xi - sx[q], ry = yi - sy[q], rz = zi - sz[q];
                double ss = rx * rx + ry * ry;
                double nr = sqrt(ss + rz * rz);
                double factor = -G * sm[q] / (nr * nr * nr);
                a1 += factor * rx;
                a2 += factor * ry;
                a3 += factor * rz;
            }
        }
        __syncthreads();
    }
    if (active) {
        dv[i] += a1;
        dv[n + i] += a2;
        dv[2 * n + i] += a3;
    }
}

void ref64_grav(hipStream_t s, const double* x, double* dv, const double* ms, int64_t n,
                int64_t ib, int64_t ie, double G) {
    if (ie <= ib) return;
    hipLaunchKernelGGL(k_ref_grav, dim3(nbx_blocks(ie - ib, REF_TILE)), dim3(REF_TILE), 0, s,
                       x, dv, ms, n, ib, ie, G);
}

// sqrt((x^2 + y^2) + z^2)
__device__ __forceinline__ double ref_norm3(double x, double y, double z) {
    double s = x * x + y * y;
    return sqrt(s + z * z);
}

// ---------------------------------------------------------------------------
// Magnetic dipoles: src/basic_potentials.jl:333-365 (no boundary conditions, as the
// reference).  Per source j, in the reference's expression order:
//   rij4 = dot(rij, rij)^2, r = rij / norm(rij), mir = mi.r, mij = mj.r,
//   c_k = (((mi_k mij + mj_k mir) + r_k (mi.mj)) - ((5 r_k) mir) mij) / rij4
// then dv += (3 mu_4pi / m_i) * sum_j c.  mm: moments SoA (component k at k*n + j).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ref_mag_term(double rx, double ry, double rz, const double* mi,
                                             const double* mj, double* t) {
    const double d = (rx * rx + ry * ry) + rz * rz;
    const double rij4 = d * d;
    const double nr = ref_norm3(rx, ry, rz);
    const double r1 = rx / nr, r2 = ry / nr, r3 = rz / nr;
    const double mir = (mi[0] * r1 + mi[1] * r2) + mi[2] * r3;
    const double mij = (mj[0] * r1 + mj[1] * r2) + mj[2] * r3;
    const double dmm = (mi[0] * mj[0] + mi[1] * mj[1]) + mi[2] * mj[2];
    t[0] = (((mi[0] * mij + mj[0] * mir) + r1 * dmm) - ((5.0 * r1) * mir) * mij) / rij4;
    t[1] = (((mi[1] * mij + mj[1] * mir) + r2 * dmm) - ((5.0 * r2) * mir) * mij) / rij4;
    t[2] = (((mi[2] * mij + mj[2] * mir) + r3 * dmm) - ((5.0 * r3) * mir) * mij) / rij4;
}

__global__ void __launch_bounds__(REF_TILE)
k_ref_mag(const double* __restrict__ x, double* __restrict__ dv, const double* __restrict__ ms,
          const double* __restrict__ mm, int64_t n, int64_t ib, int64_t ie, double mu_4pi) {
    __shared__ double sx[REF_TILE], sy[REF_TILE], sz[REF_TILE];
    __shared__ double smx[REF_TILE], smy[REF_TILE], smz[REF_TILE];
    const int64_t i = ib + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = i < ie;
    double xi = 0.0, yi = 0.0, zi = 0.0, mix = 0.0, miy = 0.0, miz = 0.0;
    if (active) {
        xi = x[i]; yi = x[n + i]; zi = x[2 * n + i];
        mix = mm[i]; miy = mm[n + i]; miz = mm[2 * n + i];
    }
    double f1 = 0.0, f2 = 0.0, f3 = 0.0;
    for (int64_t base = 0; base < n; base += REF_TILE) {
        const int64_t j = base + threadIdx.x;
        if (j < n) {
            sx[threadIdx.x] = x[j]; sy[threadIdx.x] = x[n + j]; sz[threadIdx.x] = x[2 * n + j];
            smx[threadIdx.x] = mm[j]; smy[threadIdx.x] = mm[n + j]; smz[threadIdx.x] = mm[2 * n + j];
        }
        __syncthreads();
        const int lim = (int)((n - base) < REF_TILE ? (n - base) : REF_TILE);
        if (active) {
            for (int q = 0; q < lim; ++q) {
                if (base + q == i) continue;
                const double mi[3] = {mix, miy, miz}, mj[3] = {smx[q], smy[q], smz[q]};
                double t[3];
                ref_mag_term(xi - sx[q], yi - sy[q], zi - sz[q], mi, mj, t);
                f1 += t[0];
                f2 += t[1];
                f3 += t[2];
            }
        }
        __syncthreads();
    }
    if (active) {
        const double coeff = 3.0 * mu_4pi / ms[i];
        dv[i] += coeff * f1;
        dv[n + i] += coeff * f2;
        dv[2 * n + i] += coeff * f3;
    }
}

void ref64_mag(hipStream_t s, const double* x, double* dv, const double* ms, const double* mm,
               int64_t n, int64_t ib, int64_t ie, double mu_4pi) {
    if (ie <= ib) return;
    hipLaunchKernelGGL(k_ref_mag, dim3(nbx_blocks(ie - ib, REF_TILE)), dim3(REF_TILE), 0, s, x,
                       dv, ms, mm, n, ib, ie, mu_4pi);
}

// ---------------------------------------------------------------------------
// Few bodies: a whole run of velocity-Verlet steps in one workgroup
// ---------------------------------------------------------------------------

// With a few bodies a step is a handful of dependent FP64 operations, and launches are all
// its cost (8 bodies: a force kernel and a frame kernel per step, 7.0 us; here 0.7).  The
// state lives in LDS.  Per potential, every ordered pair's term is evaluated by a thread of
// its own (phase A), then a thread per body and component adds its row in ascending j
// (phase B) -- the sums of k_ref_pairs, bit for bit; a pair out of range or the body itself
// contributes the +0.0 that leaves a sum unchanged.  Then the same thread kicks, writes the
// frame if one is due, and drifts.  A latency chain of about 1,600 cycles and two barriers
// per step, most of it the square root, the division and the ordered adds.
struct ref_small_laws {
    ref_law law[8];
    int kind[8];
    int count;
};

template <int KIND>
__device__ __forceinline__ void ref_small_term(const ref_law& law, const double* x, const double* w,
                                               const nbx_bcv& bc, int i, int j, double* t) {
    t[0] = t[1] = t[2] = 0.0;
    if (i != j)
        (void)ref_pair_term<KIND>(law, x[3 * i], x[3 * i + 1], x[3 * i + 2], x[3 * j],
                                  x[3 * j + 1], x[3 * j + 2], w[j], bc, t);
}

__global__ void __launch_bounds__(1024)
k_ref_small(int n, double* __restrict__ gx, double* __restrict__ gv, double* __restrict__ ga,
            const double* __restrict__ gms, const double* __restrict__ gqs,
            const double* __restrict__ gmm, ref_small_laws laws, nbx_bcv bc, double dt, int64_t step0,
            int64_t nsteps, int64_t save_every, double* __restrict__ uf, double* __restrict__ vf) {
    constexpr int N = NBX_REF_SMALL;
    __shared__ double term[3 * N * (N + 1)];
    __shared__ double x[3 * N], mm[3 * N], ms[N], qs[N];
    const int tid = threadIdx.x;
    const int ld = n | 1;          // odd: the rows of phase B start in different banks
    const int n3 = 3 * n;
    if (tid < n) {
        ms[tid] = gms[tid];
        qs[tid] = gqs[tid];
    }
    // thread t < 3 n: component c of body b
    const int b = tid / 3, c = tid - 3 * b;
    const bool own = tid < n3;
    double px = 0.0, v = 0.0, a = 0.0, vh = 0.0;
    const double half = 0.5, dtsq = dt * dt;
    if (own) {
        px = gx[c * n + b];
        v = gv[c * n + b];
        a = ga[c * n + b];
        if (gmm != nullptr) mm[tid] = gmm[c * n + b];
    }
    // the thread's pairs of phase A, and the frame that is due next
    constexpr int PAIRS = (N * N + 1023) / 1024;
    int pi[PAIRS], pj[PAIRS];
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
        const int p = tid + q * (int)blockDim.x;
        pi[q] = p < n * n ? p / n : -1;
        pj[q] = p - pi[q] * n;
    }
    int64_t due = save_every > 0 ? save_every - step0 % save_every : nsteps + 1;
    double* fu = uf + tid;
    double* fv = vf + tid;
    __syncthreads();
    for (int64_t s = 1; s <= nsteps; ++s) {
        if (own) {   // drift
            px = px + dt * v + dtsq * (half * a);
            vh = v + dt * (half * a);
            x[tid] = px;
            a = 0.0;
        }
        __syncthreads();
        for (int q = 0; q < laws.count; ++q) {
            const ref_law& law = laws.law[q];
            const int kind = laws.kind[q];
#pragma unroll
            for (int r = 0; r < PAIRS; ++r) {
                const int i = pi[r], j = pj[r];
                if (i < 0) break;
                double t[3];
                if (kind == NBX_TERM_LJ) ref_small_term<REF_LJ>(law, x, ms, bc, i, j, t);
                else if (kind == NBX_TERM_ELEC) ref_small_term<REF_COULOMB>(law, x, qs, bc, i, j, t);
                else if (kind == NBX_TERM_RF) ref_small_term<REF_RF>(law, x, qs, bc, i, j, t);
                else if (kind == NBX_TERM_GRAV) ref_small_term<REF_GRAV>(law, x, ms, bc, i, j, t);
                else if (i == j) t[0] = t[1] = t[2] = 0.0;
                else ref_mag_term(x[3 * i] - x[3 * j], x[3 * i + 1] - x[3 * j + 1],
                                  x[3 * i + 2] - x[3 * j + 2], mm + 3 * i, mm + 3 * j, t);
#pragma unroll
                for (int k = 0; k < 3; ++k) term[(3 * i + k) * ld + j] = t[k];
            }
            __syncthreads();
            if (own) {
                const double* row = term + tid * ld;
                double f = 0.0;
                int j = 0;
                for (; j + 8 <= n; j += 8) {
                    double u[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) u[k] = row[j + k];
#pragma unroll
                    for (int k = 0; k < 8; ++k) f += u[k];
                }
                for (; j < n; ++j) f += row[j];
                double add = f;
                if (kind == NBX_TERM_LJ) add = 24.0 * law.c / ms[b] * f;
                else if (kind == NBX_TERM_MAG) add = 3.0 * law.c / ms[b] * f;
                else if (kind != NBX_TERM_GRAV) add = law.c * qs[b] / ms[b] * f;
                a += add;
            }
            if (q + 1 < laws.count) __syncthreads();   // the rows are read before the next terms
        }
        if (own) {   // kick; the barrier after the next drift separates it from the terms
            v = vh + dt * (0.5 * a);
            if (s == due) {
                *fu = px;
                *fv = v;
                fu += n3;
                fv += n3;
                due += save_every;
            }
        }
    }
    if (own) {
        gx[c * n + b] = px;
        gv[c * n + b] = v;
        ga[c * n + b] = a;
    }
}

void ref64_small_run(hipStream_t s, int n, double* x, double* v, double* a, const double* ms,
                     const double* qs, const double* mm, const ref64_term* terms, int count,
                     const nbx_bcv& bc, double dt, int64_t step0, int64_t nsteps, int64_t save_every,
                     double* uf, double* vf) {
    ref_small_laws laws{};
    laws.count = count;
    for (int q = 0; q < count; ++q) {
        ref64_term t = terms[q];
        t.filter = false;
        laws.kind[q] = t.kind;
        if (t.kind == NBX_TERM_MAG) laws.law[q].c = t.p[0];
        else laws.law[q] = make_law(t, bc);
    }
    const int want = std::max(n * n, 3 * n);
    const int threads = std::min(1024, (want + 63) / 64 * 64);
    hipLaunchKernelGGL(k_ref_small, dim3(1), dim3(threads), 0, s, n, x, v, a, ms, qs, mm, laws, bc, dt,
                       step0, nsteps, save_every, uf, vf);
}

// ---------------------------------------------------------------------------
// SPC/Fw bonded terms: src/basic_potentials.jl:367-433
// ---------------------------------------------------------------------------

// bond force / mass-free sum of atom i (src/nbody_to_ode.jl:274-284)
__device__ __forceinline__ void ref_bond_force(const double* __restrict__ x, int64_t n, int64_t i,
                                               double rOH, double kbond, double* f) {
    const int64_t o = 3 * (i / 3);
    int64_t nb[2];
    int nn;
    if (i == o) { nb[0] = o + 1; nb[1] = o + 2; nn = 2; }
    else { nb[0] = o; nb[1] = o; nn = 1; }
    double f1 = 0.0, f2 = 0.0, f3 = 0.0;
    const double xi = x[i], yi = x[n + i], zi = x[2 * n + i];
    for (int t = 0; t < nn; ++t) {
        const int64_t j = nb[t];
        double rx = xi - x[j], ry = yi - x[n + j], rz = zi - x[2 * n + j];
        double r = ref_norm3(rx, ry, rz);
        double d = r - rOH;
        double factor = -d * kbond / r;
        f1 += factor * rx;
        f2 += factor * ry;
        f3 += factor * rz;
    }
    f[0] = f1; f[1] = f2; f[2] = f3;
}

__global__ void k_ref_bond(const double* __restrict__ x, double* __restrict__ dv,
                           const double* __restrict__ ms, int64_t n, int64_t ib, int64_t ie,
                           double rOH, double kbond) {
    const int64_t i = ib + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ie) return;
    double f[3];
    ref_bond_force(x, n, i, rOH, kbond, f);
    double coeff = 1.0 / ms[i];
    dv[i] += coeff * f[0];
    dv[n + i] += coeff * f[1];
    dv[2 * n + i] += coeff * f[2];
}

void ref64_bond(hipStream_t s, const double* x, double* dv, const double* ms, int64_t n,
                int64_t ib, int64_t ie, double rOH, double kbond) {
    if (ie <= ib) return;
    hipLaunchKernelGGL(k_ref_bond, dim3(nbx_blocks(ie - ib, 256)), dim3(256), 0, s, x, dv, ms,
                       n, ib, ie, rOH, kbond);
}

__device__ __forceinline__ void ref_cross(double a0, double a1, double a2, double b0, double b1,
                                          double b2, double& c0, double& c1, double& c2) {
    c0 = a1 * b2 - a2 * b1;
    c1 = a2 * b0 - a0 * b2;
    c2 = a0 * b1 - a1 * b0;
}

// valence_angle_potential_acceleration!(dv, rs, a=H1, b=O, c=H2, ...) of molecule m: the
// forces on H1 (fa) and H2 (fc); O takes -(fa + fc)
__device__ __forceinline__ void ref_angle_force(const double* __restrict__ x, int64_t n, int64_t m,
                                                double aHOH, double ka, double* fa, double* fc) {
    const int64_t a = 3 * m + 1, b = 3 * m, c = 3 * m + 2;
    double ra[3] = {x[a], x[n + a], x[2 * n + a]};
    double rb[3] = {x[b], x[n + b], x[2 * n + b]};
    double rc[3] = {x[c], x[n + c], x[2 * n + c]};
    double rba[3], rbc[3], rcb[3];
    for (int k = 0; k < 3; ++k) {
        rba[k] = ra[k] - rb[k];
        rbc[k] = rc[k] - rb[k];
        rcb[k] = rb[k] - rc[k];
    }
    double X[3], ta[3], tc[3];
    ref_cross(rba[0], rba[1], rba[2], rbc[0], rbc[1], rbc[2], X[0], X[1], X[2]);
    ref_cross(rba[0], rba[1], rba[2], X[0], X[1], X[2], ta[0], ta[1], ta[2]);
    ref_cross(rcb[0], rcb[1], rcb[2], X[0], X[1], X[2], tc[0], tc[1], tc[2]);
    double ia = 1.0 / ref_norm3(ta[0], ta[1], ta[2]);
    double ic = 1.0 / ref_norm3(tc[0], tc[1], tc[2]);
    double nba = ref_norm3(rba[0], rba[1], rba[2]);
    double nbc = ref_norm3(rbc[0], rbc[1], rbc[2]);
    double dt = rba[0] * rbc[0] + rba[1] * rbc[1];
    dt = dt + rba[2] * rbc[2];
    double cosine = dt / (nba * nbc);
    if (cosine > 1.0) cosine = 1.0;
    else if (cosine < -1.0) cosine = -1.0;
    double ang = acos(cosine);
    double force = -ka * (ang - aHOH);
    for (int k = 0; k < 3; ++k) {
        double pa = ia * ta[k], pc = ic * tc[k];
        fa[k] = pa * force / nba;
        fc[k] = pc * force / nbc;
    }
}

__global__ void k_ref_angle(const double* __restrict__ x, double* __restrict__ dv,
                            const double* __restrict__ ms, int64_t n, int64_t mb, int64_t me,
                            double aHOH, double ka) {
    const int64_t m = mb + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= me) return;
    const int64_t a = 3 * m + 1, b = 3 * m, c = 3 * m + 2;
    double fa[3], fc[3];
    ref_angle_force(x, n, m, aHOH, ka, fa, fc);
    for (int k = 0; k < 3; ++k) {
        double fb = -(fa[k] + fc[k]);
        dv[k * n + a] += fa[k] / ms[a];
        dv[k * n + b] += fb / ms[b];
        dv[k * n + c] += fc[k] / ms[c];
    }
}

// Water, one step's right-hand side and end in two launches: the electrostatic sums of all
// atoms into elec and the Lennard-Jones sums of the O atoms into lj (one launch, a wavefront
// per sum), then per atom the reference's closure order -- electrostatic, bond, LJ (O), then
// the molecule's angle -- and the end of the step.
template <int KIND, bool FILTER>
__global__ void __launch_bounds__(64 * REF_WAVES)
k_ref_water_pairs(ref_atoms A, ref_law el, ref_law lj, nbx_bcv bc, double* __restrict__ elec,
                  double* __restrict__ ljv) {
    __shared__ int cand[REF_WAVES][128];
    __shared__ double term[REF_WAVES][192];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * REF_WAVES + wave;
    const int64_t n = A.n;
    if (t < n) {
        const double f = ref_wave_sum<KIND, FILTER>(A, el, bc, t, cand[wave], term[wave]);
        if (lane < 3) elec[lane * n + t] = ref_contribution<KIND>(A, el, t, f);
    } else if (t < n + n / 3) {
        const int64_t i = 3 * (t - n);
        const double f = ref_wave_sum<REF_LJ, FILTER>(A, lj, bc, i, cand[wave], term[wave]);
        if (lane < 3) ljv[lane * n + i] = ref_contribution<REF_LJ>(A, lj, i, f);
    }
}

template <int KIND>
__global__ void __launch_bounds__(256, REF_SPLIT_BLOCKS)
k_ref_water_pairs_split(ref_atoms A, ref_law el, ref_law lj, nbx_bcv bc, double* __restrict__ elec,
                        double* __restrict__ ljv) {
    __shared__ ref_block_lds S;
    const int64_t n = A.n, t = blockIdx.x;
    const int c = threadIdx.x;
    if (t < n) {
        const double f = ref_block_sum<KIND>(A, el, bc, t, S);
        if (c < 3) elec[c * n + t] = ref_contribution<KIND>(A, el, t, f);
    } else {
        const int64_t i = 3 * (t - n);
        const double f = ref_block_sum<REF_LJ>(A, lj, bc, i, S);
        if (c < 3) ljv[c * n + i] = ref_contribution<REF_LJ>(A, lj, i, f);
    }
}

// one thread per component of an atom (thread t: atom t / 3, component t % 3)
__global__ void __launch_bounds__(192)
k_ref_water_step(const double* __restrict__ ms, int64_t n, const double* __restrict__ elec,
                 const double* __restrict__ ljv, double rOH, double kbond, double aHOH, double ka,
                 ref64_step st) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = t / 3;
    if (i >= n) return;
    const int c = (int)(t - 3 * i);
    const int64_t m = i / 3, o = 3 * m;
    const double* const x = st.x_in;
    double fb[3], fa[3], fc[3];
    ref_bond_force(x, n, i, rOH, kbond, fb);
    ref_angle_force(x, n, m, aHOH, ka, fa, fc);
    const auto pick = [c](const double* f) { return c == 0 ? f[0] : (c == 1 ? f[1] : f[2]); };
    const double mi = ms[i];
    double a = 0.0 + elec[c * n + i];
    const double coeff = 1.0 / mi;
    a += coeff * pick(fb);
    if (i == o) a += ljv[c * n + i];
    const double f1 = pick(fa), f2 = pick(fc);
    if (i == o) a += -(f1 + f2) / mi;
    else if (i == o + 1) a += f1 / mi;
    else a += f2 / mi;
    ref_end_step(st, n, i, c, a, mi, o, mi);
}

void ref64_water_step(hipStream_t s, const ref64_term& el, const ref64_term& lj, const float4* frac,
                      const double* ms, const double* qs, int64_t n, const nbx_bcv& bc,
                      double* elec, double* ljv, double rOH, double kbond, double aHOH, double ka,
                      const ref64_step& st) {
    if (n <= 0) return;
    const ref_atoms A{st.x_in, frac, ms, qs, n};
    const ref_law le = make_law(el, bc), ll = make_law(lj, bc);
    const dim3 grid(nbx_blocks(n + n / 3, REF_WAVES)), block(64 * REF_WAVES);
    const bool rf = el.kind == NBX_TERM_RF;
    // both laws filter, or neither (el.filter == lj.filter)
    if (el.filter && n + n / 3 <= REF_SPLIT_TARGETS) {
        const dim3 each((unsigned)(n + n / 3)), four(256);
        if (rf) hipLaunchKernelGGL((k_ref_water_pairs_split<REF_RF>), each, four, 0, s, A, le, ll, bc, elec, ljv);
        else hipLaunchKernelGGL((k_ref_water_pairs_split<REF_COULOMB>), each, four, 0, s, A, le, ll, bc, elec, ljv);
    } else if (el.filter) {
        if (rf) hipLaunchKernelGGL((k_ref_water_pairs<REF_RF, true>), grid, block, 0, s, A, le, ll, bc, elec, ljv);
        else hipLaunchKernelGGL((k_ref_water_pairs<REF_COULOMB, true>), grid, block, 0, s, A, le, ll, bc, elec, ljv);
    } else {
        if (rf) hipLaunchKernelGGL((k_ref_water_pairs<REF_RF, false>), grid, block, 0, s, A, le, ll, bc, elec, ljv);
        else hipLaunchKernelGGL((k_ref_water_pairs<REF_COULOMB, false>), grid, block, 0, s, A, le, ll, bc, elec, ljv);
    }
    hipLaunchKernelGGL(k_ref_water_step, dim3(nbx_blocks(3 * n, 192)), dim3(192), 0, s, ms, n, elec,
                       ljv, rOH, kbond, aHOH, ka, st);
}

void ref64_angle(hipStream_t s, const double* x, double* dv, const double* ms, int64_t n,
                 int64_t mb, int64_t me, double aHOH, double ka) {
    if (me <= mb) return;
    hipLaunchKernelGGL(k_ref_angle, dim3(nbx_blocks(me - mb, 256)), dim3(256), 0, s, x, dv, ms,
                       n, mb, me, aHOH, ka);
}

// ---------------------------------------------------------------------------
// Temperature and Berendsen: src/thermostats.jl:76-91
// ---------------------------------------------------------------------------

// Sum of term(0) .. term(count - 1) in index order, by one block of 256 threads: the block
// computes 1,024 terms at a time into LDS (the next ones while these are added) and the
// first wavefront adds them one after another, every lane the same sum.  Bound by the
// dependent FP64 adds of a single wavefront, 5.6 ns per term (one thread reading its terms
// from memory took 51 ns; 10,976 terms 560 -> 62 us; batches of 64 terms per LDS wait, and
// reading ahead of the adds, measured the same or slower).  The result is valid in
// wavefront 0.
#define SEQ_CHUNK 1024
template <class Term>
__device__ __forceinline__ double ref_ordered_sum(int64_t count, Term term) {
    __shared__ __attribute__((aligned(16))) double buf[2][SEQ_CHUNK];
    const int tid = threadIdx.x;
    constexpr int PER = SEQ_CHUNK / 256;
    double w[PER];
    const auto fetch = [&](int64_t base) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int64_t i = base + tid + q * 256;
            w[q] = i < count ? term(i) : 0.0;
        }
    };
    double e = 0.0;
    fetch(0);
    int par = 0;
    for (int64_t base = 0; base < count; base += SEQ_CHUNK, par ^= 1) {
#pragma unroll
        for (int q = 0; q < PER; ++q) buf[par][tid + q * 256] = w[q];
        __syncthreads();   // the other buffer is written after the adds of the chunk before it
        if (base + SEQ_CHUNK < count) fetch(base + SEQ_CHUNK);
        if (tid < 64) {
            const int cnt = (int)(count - base < SEQ_CHUNK ? count - base : SEQ_CHUNK);
            const double* p = buf[par];
            int q = 0;
            for (; q + 16 <= cnt; q += 16) {
                double t[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) t[u] = p[q + u];
#pragma unroll
                for (int u = 0; u < 16; ++u) e += t[u];
            }
            for (; q < cnt; ++q) e += p[q];
        }
    }
    return e;
}

// term i of the kinetic energy (half mass) or of md_temperature
__device__ __forceinline__ double ref_mv2(const double* __restrict__ v,
                                          const double* __restrict__ ms, int64_t n, int64_t i,
                                          bool half_mass) {
    const double a = v[i], b = v[n + i], c = v[2 * n + i];
    double s = a * a + b * b;
    s = s + c * c;
    return half_mass ? s * (ms[i] / 2.0) : ms[i] * s;
}

// mode 0: out = sum; 1: out = sum / c; 2: out = c * sum
__device__ __forceinline__ void ref_store_sum(double e, int mode, double c, double* out) {
    if (threadIdx.x == 0) out[0] = mode == 1 ? e / c : (mode == 2 ? c * e : e);
}

__global__ void __launch_bounds__(256)
k_seq_sum(const double* __restrict__ terms, int64_t count, int mode, double c,
          double* __restrict__ out) {
    ref_store_sum(ref_ordered_sum(count, [&](int64_t i) { return terms[i]; }), mode, c, out);
}

__global__ void __launch_bounds__(256)
k_seq_mv2(const double* __restrict__ v, const double* __restrict__ ms, int64_t n, int half_mass,
          int mode, double c, double* __restrict__ out) {
    const bool half = half_mass != 0;
    ref_store_sum(ref_ordered_sum(n, [&](int64_t i) { return ref_mv2(v, ms, n, i, half); }), mode,
                  c, out);
}

void ref64_temperature(hipStream_t s, const double* v, const double* ms, int64_t n,
                       double kb, int64_t Nc, double* d_T) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_seq_mv2, dim3(1), dim3(256), 0, s, v, ms, n, 0, 1,
                       kb * (double)(3 * n - Nc), d_T);
}

__global__ void k_ref_berendsen(double* __restrict__ dv, const double* __restrict__ v,
                                int64_t n3, const double* __restrict__ d_T, double T0,
                                double gamma) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n3) return;
    const double T = d_T[0];
    if (1.0 / T == __builtin_inf()) dv[t] += gamma * v[t];
    else {
        double c = gamma * (T0 / T - 1.0);
        dv[t] += c * v[t];
    }
}

void ref64_berendsen(hipStream_t s, double* dv, const double* v, int64_t n, const double* d_T,
                     double T0, double gamma) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_ref_berendsen, dim3(nbx_blocks(3 * n, 256)), dim3(256), 0, s, dv, v,
                       3 * n, d_T, T0, gamma);
}

// ---------------------------------------------------------------------------
// Velocity Verlet and stochastic thermostats
// ---------------------------------------------------------------------------

// x_out may be x; frac: box fractions of the new positions (nullptr: none)
__global__ void k_ref_drift(const double* x, double* x_out, const double* __restrict__ v,
                            const double* __restrict__ a, double* __restrict__ vh, int64_t n,
                            double dt, float4* frac, double invL) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * n) return;
    const double half = 0.5, dtsq = dt * dt;
    const double px = x[t] + dt * v[t] + dtsq * (half * a[t]);
    x_out[t] = px;
    vh[t] = v[t] + dt * (half * a[t]);
    if (frac != nullptr) {
        const int64_t c = t / n;
        reinterpret_cast<float*>(frac + (t - c * n))[c] = ref_frac(px, invL);
    }
}

__global__ void k_ref_kick(double* __restrict__ v, const double* __restrict__ vh,
                           const double* __restrict__ a, int64_t n3, double dt) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n3) return;
    v[t] = vh[t] + dt * (0.5 * a[t]);
}

void ref64_drift(hipStream_t s, const double* x, double* x_out, const double* v, const double* a,
                 double* vh, int64_t n, double dt, float4* frac, double L) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_ref_drift, dim3(nbx_blocks(3 * n, 256)), dim3(256), 0, s, x, x_out, v, a,
                       vh, n, dt, frac, 1.0 / L);
}

void ref64_kick(hipStream_t s, double* v, const double* vh, const double* a, int64_t n,
                double dt) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_ref_kick, dim3(nbx_blocks(3 * n, 256)), dim3(256), 0, s, v, vh, a,
                       3 * n, dt);
}

__global__ void k_ref_langevin_half(double* __restrict__ v, const double* __restrict__ ms,
                                    int64_t n, double kb, double T, double c1, double c2,
                                    uint64_t seed, int64_t step, uint32_t stream) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double sig = c2 * sqrt(kb * T / ms[i]);
    double g[3];
    nbx_rng_normals3(seed, i, step, stream, g);
    for (int k = 0; k < 3; ++k) v[k * n + i] = c1 * v[k * n + i] + sig * g[k];
}

void ref64_langevin_half(hipStream_t s, double* v, const double* ms, int64_t n, double kb,
                         double T, double gamma, double dt, uint64_t seed, int64_t step,
                         uint32_t stream) {
    if (n <= 0) return;
    const double c1 = exp(-gamma * (0.5 * dt));
    const double c2 = sqrt(1.0 - c1 * c1);
    hipLaunchKernelGGL(k_ref_langevin_half, dim3(nbx_blocks(n, 256)), dim3(256), 0, s, v, ms, n,
                       kb, T, c1, c2, seed, step, stream);
}

// Euler-Maruyama step of the Langevin SDE (src/nbody_to_ode.jl:567-598), one thread per
// atom, from the state (x, v) and a = f(x): x' = x + dt v and
// v' = v + dt (a - gamma v) + sigma (sqrt(dt) xi), sigma = sqrt(2 gamma kb T / m_1)
__global__ void k_ref_em(double* __restrict__ x, double* __restrict__ v,
                         const double* __restrict__ a, int64_t n, double dt, double gamma,
                         double sigma, double sqrt_dt, uint64_t seed, int64_t step) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double g[3];
    nbx_rng_normals3(seed, i, step, NBX_RNG_EM, g);
    for (int k = 0; k < 3; ++k) {
        const double vk = v[k * n + i];
        x[k * n + i] = x[k * n + i] + dt * vk;
        v[k * n + i] = vk + dt * (a[k * n + i] - gamma * vk) + sigma * (sqrt_dt * g[k]);
    }
}

void ref64_em(hipStream_t s, double* x, double* v, const double* a, int64_t n, double dt,
              double gamma, double sigma, uint64_t seed, int64_t step) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_ref_em, dim3(nbx_blocks(n, 256)), dim3(256), 0, s, x, v, a, n, dt, gamma,
                       sigma, sqrt(dt), seed, step);
}

// Andersen collisions (src/nbody_simulation_result.jl:511-540), one thread per body
__global__ void k_ref_andersen(double* __restrict__ v, const double* __restrict__ ms, int64_t n,
                               int water, double kb, double T, double prob, uint64_t seed,
                               int64_t step) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nb = water ? n / 3 : n;
    if (b >= nb) return;
    const int64_t first = water ? 3 * b : b;
    if (!(nbx_rng_uniform(seed, first, step, NBX_RNG_ANDERSEN) < prob)) return;
    const int natoms = water ? 3 : 1;
    for (int t = 0; t < natoms; ++t) {
        const int64_t i = first + t;
        const double m = water ? ms[i] : ms[0];
        const double vdev = sqrt(kb * T / m);
        double g[3];
        nbx_rng_normals3(seed, i, step, NBX_RNG_ANDERSEN, g);
        v[i] = vdev * g[0];
        v[n + i] = vdev * g[1];
        v[2 * n + i] = vdev * g[2];
    }
}

void ref64_andersen(hipStream_t s, double* v, const double* ms, int64_t n, int water,
                    double kb, double T, double prob, uint64_t seed, int64_t step) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_ref_andersen, dim3(nbx_blocks(n, 256)), dim3(256), 0, s, v, ms, n,
                       water, kb, T, prob, seed, step);
}

// ---------------------------------------------------------------------------
// Energies: src/nbody_simulation_result.jl:209-397
// ---------------------------------------------------------------------------

void ref64_kinetic(hipStream_t s, const double* v, const double* ms, int64_t n,
                   double* d_out) {
    if (n <= 0) { ref64_fill(s, d_out, 1, 0.0); return; }
    hipLaunchKernelGGL(k_seq_mv2, dim3(1), dim3(256), 0, s, v, ms, n, 1, 0, 0.0, d_out);
}

// box fractions in units of 2^-32; false where the coordinate is more than 1,024 boxes away (or
// no number), too far for the bound on the difference to the FP64 distance
__device__ __forceinline__ bool box_fixed(double x, double y, double z, double invL, uint32_t* q) {
    const double t[3] = {x * invL, y * invL, z * invL};
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        ok = ok && fabs(t[k]) < 1024.0;
        q[k] = ok ? (uint32_t)(uint64_t)((t[k] - floor(t[k])) * 4294967296.0) : 0u;
    }
    return ok;
}

// Pair energies of the pairs i < j of nj atoms: a wavefront takes 64 x 64 tiles of the upper
// triangle (64 atoms i in its lanes, 64 atoms j from LDS), adds per lane in FP64, and the
// lanes, wavefronts and blocks are added in a fixed order (k_ref_pe_sum).  Bound by FP64
// VALU work; one thread per atom i with the triangle's long and short rows took 5,300 us for
// 10,976 Lennard-Jones atoms, this took 108 with every pair in FP64.
//   LJ (:293-319): 4 (s12 - s6), a pair beyond the cutoff at the cutoff's value; those are
//   counted and their constant is added once per lane.  In a cubic box wider than four cutoffs
//   (FILTER) an FP32 distance of fixed-point box fractions, off by less than 1e-6 and 4e-9 of
//   the box, finds the few pairs that can be in range; they queue in LDS, and 64 at a time are
//   taken in FP64.  The same atoms then take 71 us, 62 of them block 0's ordered sum (leaving
//   out only the atoms j that no lane has in range: 81).  A tile with an atom more than 1,024
//   boxes away takes every pair in FP64.
//   Coulomb (:321-351): q_j / r, beyond the cutoff q_j / R; reaction field: in the cutoff only.
// Block 0 of the launch adds the kinetic energy in index order meanwhile (ke_out).
enum { REF_PE_LJ = 0, REF_PE_COULOMB = 1, REF_PE_RF = 2 };
struct ref_pe_law {
    double s2, R, R2, krf, crf;
    double invL;     // FILTER: 1 / L
    float near2;     // FILTER: above the cutoff's square in the units of the box fractions
    int jstride, water;
};

template <int KIND, bool FILTER>
__global__ void __launch_bounds__(256)
k_ref_pair_pe(const double* __restrict__ x, const double* __restrict__ qs, int64_t n, int64_t nj,
              ref_pe_law law, nbx_bcv bc, double* __restrict__ part,
              const double* __restrict__ v, const double* __restrict__ ms,
              double* __restrict__ ke_out) {
    if (blockIdx.x == 0) {
        if (ke_out != nullptr)
            ref_store_sum(ref_ordered_sum(n, [&](int64_t i) { return ref_mv2(v, ms, n, i, true); }),
                          0, 0.0, ke_out);
        return;
    }
    __shared__ double sj[4][64][4];
    __shared__ uint16_t queue[FILTER ? 4 : 1][128];
    __shared__ double red[4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t T = (nj + 63) >> 6, items = T * (T + 1) / 2;
    double e = 0.0;
    int64_t far = 0;
    for (int64_t it = (int64_t)(blockIdx.x - 1) * 4 + wave; it < items;
         it += (int64_t)(gridDim.x - 1) * 4) {
        // row J of the triangle holds the tiles I = 0..J
        int64_t J = (int64_t)((sqrt(8.0 * (double)it + 1.0) - 1.0) * 0.5);
        while (J * (J + 1) / 2 > it) --J;
        while ((J + 1) * (J + 2) / 2 <= it) ++J;
        const int64_t I = it - J * (J + 1) / 2;
        const int64_t a = (I << 6) + lane, b0 = J << 6;
        const int nb = (int)(nj - b0 < 64 ? nj - b0 : 64);
        double xi = 0.0, yi = 0.0, zi = 0.0, qi = 0.0;
        if (a < nj) {
            const int64_t i = a * law.jstride;
            xi = x[i]; yi = x[n + i]; zi = x[2 * n + i];
            if (KIND != REF_PE_LJ) qi = qs[i];
        }
        if (lane < nb) {
            const int64_t j = (b0 + lane) * law.jstride;
            sj[wave][lane][0] = x[j]; sj[wave][lane][1] = x[n + j]; sj[wave][lane][2] = x[2 * n + j];
            sj[wave][lane][3] = KIND != REF_PE_LJ ? qs[j] : 0.0;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t ui[3] = {0u, 0u, 0u}, uj[3] = {0u, 0u, 0u};
        bool ok = FILTER;
        if (FILTER) {
            if (a < nj) ok = box_fixed(xi, yi, zi, law.invL, ui);
            if (lane < nb)
                ok = box_fixed(sj[wave][lane][0], sj[wave][lane][1], sj[wave][lane][2], law.invL,
                               uj) && ok;
        }
        double ei = 0.0;
        const auto exact = [&](int k) {
            double rx, ry, rz, r2;
            nbx_displacement(xi, yi, zi, sj[wave][k][0], sj[wave][k][1], sj[wave][k][2], bc, rx, ry,
                             rz, r2);
            const bool pair = a < nj && b0 + k > a &&
                              (KIND == REF_PE_LJ || !ref_excluded(a, b0 + k, law.water));
            const bool in = pair && r2 < law.R2;
            if (KIND == REF_PE_LJ) {
                if (in) {
                    const double q = law.s2 / r2;
                    const double s6 = q * q * q;
                    const double s12 = s6 * s6;
                    ei += s12 - s6;
                }
                far += pair && !in;
            } else if (KIND == REF_PE_RF) {
                if (in) ei += sj[wave][k][3] * (1.0 / sqrt(r2) + law.krf * r2 - law.crf);
            } else if (pair) {
                ei += sj[wave][k][3] / (in ? sqrt(r2) : law.R);
            }
        };
        if (FILTER && !__any(!ok)) {   // off the diagonal every lane holds an atom, a < b
            const bool diagonal = I == J;
            int queued = 0, found = 0;
            // the term of a queued pair: a source lane's atom and a staged atom
            const auto term = [&](int slot, bool live) {
                const int w = live ? queue[wave][slot] : 0;
                const double x0 = __shfl(xi, w >> 6, 64), y0 = __shfl(yi, w >> 6, 64),
                             z0 = __shfl(zi, w >> 6, 64);
                const double* const q = sj[wave][w & 63];
                double rx, ry, rz, r2;
                nbx_displacement(x0, y0, z0, q[0], q[1], q[2], bc, rx, ry, rz, r2);
                if (live && r2 < law.R2) {
                    const double q2 = law.s2 / r2;
                    const double s6 = q2 * q2 * q2;
                    const double s12 = s6 * s6;
                    ei += s12 - s6;
                    ++found;
                }
            };
            for (int k = 0; k < nb; ++k) {
                const float dx = (float)(int)(ui[0] - __builtin_amdgcn_readlane(uj[0], k));
                const float dy = (float)(int)(ui[1] - __builtin_amdgcn_readlane(uj[1], k));
                const float dz = (float)(int)(ui[2] - __builtin_amdgcn_readlane(uj[2], k));
                const bool pair = !diagonal || k > lane;
                const bool near = pair && fmaf(dz, dz, fmaf(dy, dy, dx * dx)) < law.near2;
                const unsigned long long mask = __ballot(near);
                if (mask == 0ull) continue;
                const int at = (int)__builtin_amdgcn_mbcnt_hi(
                    (unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, (unsigned)queued));
                if (near) queue[wave][at] = (uint16_t)(lane << 6 | k);
                queued += __popcll(mask);
                if (queued >= 64) {
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    queued -= 64;
                    term(queued + lane, true);   // the newest: the older stay where they are
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
            }
            if (queued > 0) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                term(lane, lane < queued);
            }
            far += (diagonal ? (lane < nb ? nb - 1 - lane : 0) : nb) - found;
        } else {
            for (int k = 0; k < nb; ++k) exact(k);
        }
        e += KIND == REF_PE_LJ ? ei : ei * qi;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (KIND == REF_PE_LJ) {
        const double q = law.s2 / law.R2;
        const double s6 = q * q * q;
        if (far) e += (double)far * (s6 * s6 - s6);   // R = Inf has no far pairs
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off, 64);
    if (lane == 0) red[wave] = e;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x - 1] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ void __launch_bounds__(256)
k_ref_pe_sum(const double* __restrict__ part, int count, double* __restrict__ out) {
    __shared__ double red[256];
    double e = 0.0;
    for (int p = threadIdx.x; p < count; p += 256) e += part[p];
    red[threadIdx.x] = e;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

template <int KIND>
static void pair_pe(hipStream_t s, const double* x, const double* qs, int64_t n, int64_t nj,
                    const ref_pe_law& law, const nbx_bcv& bc, double* d_part, double* d_out,
                    const ref64_ke& ke) {
    const int64_t T = (nj + 63) >> 6;
    // 2,048 blocks of four wavefronts fill the chip (d_part holds 8,192 doubles at least)
    const int blocks = (int)std::min<int64_t>((T * (T + 1) / 2 + 3) / 4, 2048);
    if (law.near2 > 0.0f)
        hipLaunchKernelGGL((k_ref_pair_pe<KIND, KIND == REF_PE_LJ>), dim3(blocks + 1), dim3(256), 0,
                           s, x, qs, n, nj, law, bc, d_part, ke.v, ke.ms, ke.out);
    else
        hipLaunchKernelGGL((k_ref_pair_pe<KIND, false>), dim3(blocks + 1), dim3(256), 0, s, x, qs, n,
                           nj, law, bc, d_part, ke.v, ke.ms, ke.out);
    hipLaunchKernelGGL(k_ref_pe_sum, dim3(1), dim3(256), 0, s, d_part, blocks, d_out);
}

void ref64_lj_pe(hipStream_t s, const double* x, int64_t n, int jstride, int64_t nj,
                 double sigma, double R, const nbx_bcv& bc, double* d_part, double* d_out,
                 const ref64_ke& ke) {
    ref_pe_law law{};
    law.s2 = sigma * sigma;
    law.R2 = R * R;
    law.jstride = jstride;
    if (bc.kind == NBX_BC_CUBIC && R < 0.25 * bc.b[0]) {
        law.invL = 1.0 / bc.b[0];
        const double near = (R * law.invL * (1.0 + 1e-6) + 4e-9) * 4294967296.0;
        law.near2 = (float)(near * near);
    }
    pair_pe<REF_PE_LJ>(s, x, nullptr, n, nj, law, bc, d_part, d_out, ke);
}

void ref64_elec_pe(hipStream_t s, const double* x, const double* qs, int64_t n, int water,
                   double R, int rf, double eps_rf, const nbx_bcv& bc, double* d_part,
                   double* d_out, const ref64_ke& ke) {
    ref_pe_law law{};
    law.R = R;
    law.R2 = R * R;
    law.jstride = 1;
    law.water = water;
    if (rf) {
        law.krf = rf_krf(R, eps_rf);
        law.crf = 1.0 / R + law.krf * (R * R);
        pair_pe<REF_PE_RF>(s, x, qs, n, n, law, bc, d_part, d_out, ke);
    } else {
        pair_pe<REF_PE_COULOMB>(s, x, qs, n, n, law, bc, d_part, d_out, ke);
    }
}

__global__ void k_ref_grav_pe(const double* __restrict__ x, const double* __restrict__ ms,
                              int64_t n, double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double xi = x[i], yi = x[n + i], zi = x[2 * n + i];
    double ei = 0.0;
    for (int64_t j = i + 1; j < n; ++j)
        ei += ms[j] / ref_norm3(xi - x[j], yi - x[n + j], zi - x[2 * n + j]);
    out[i] = ei * ms[i];
}

void ref64_grav_pe(hipStream_t s, const double* x, const double* ms, int64_t n, double G,
                   double* d_tmp, double* d_out) {
    if (n <= 0) { ref64_fill(s, d_out, 1, 0.0); return; }
    hipLaunchKernelGGL(k_ref_grav_pe, dim3(nbx_blocks(n, 128)), dim3(128), 0, s, x, ms, n,
                       d_tmp);
    hipLaunchKernelGGL(k_seq_sum, dim3(1), dim3(256), 0, s, d_tmp, n, 2, -G, d_out);
}

// Bonds (:353-372, each bond seen from both ends, / 4) and angles (:374-397, / 2)
__global__ void k_ref_bonded_terms(const double* __restrict__ x, int64_t n, double rOH,
                                   double kbond, double aHOH, double ka,
                                   double* __restrict__ out) {
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nmol = n / 3;
    if (m >= nmol) return;
    const int64_t o = 3 * m;
    // bond terms in visit order: O->H1, O->H2, H1->O, H2->O
    const int64_t pi[4] = {o, o, o + 1, o + 2};
    const int64_t pj[4] = {o + 1, o + 2, o, o};
    for (int t = 0; t < 4; ++t) {
        double d = ref_norm3(x[pi[t]] - x[pj[t]], x[n + pi[t]] - x[n + pj[t]],
                             x[2 * n + pi[t]] - x[2 * n + pj[t]]) - rOH;
        out[4 * m + t] = d * d * kbond;
    }
    const int64_t a = o + 1, b = o, c = o + 2;
    double rba0 = x[a] - x[b], rba1 = x[n + a] - x[n + b], rba2 = x[2 * n + a] - x[2 * n + b];
    double rbc0 = x[c] - x[b], rbc1 = x[n + c] - x[n + b], rbc2 = x[2 * n + c] - x[2 * n + b];
    double dt = rba0 * rbc0 + rba1 * rbc1;
    dt = dt + rba2 * rbc2;
    double ang = acos(dt / (ref_norm3(rba0, rba1, rba2) * ref_norm3(rbc0, rbc1, rbc2)));
    double d = ang - aHOH;
    out[4 * nmol + m] = ka * (d * d);
}

// block 0: the bonds, block 1: the angles
__global__ void __launch_bounds__(256)
k_ref_bonded_sum(const double* __restrict__ terms, int64_t nmol, double* __restrict__ out2) {
    const int64_t first = blockIdx.x ? 4 * nmol : 0;
    ref_store_sum(ref_ordered_sum(blockIdx.x ? nmol : 4 * nmol,
                                  [&](int64_t t) { return terms[first + t]; }),
                  1, blockIdx.x ? 2.0 : 4.0, out2 + blockIdx.x);
}

void ref64_bonded_pe(hipStream_t s, const double* x, int64_t n, double rOH, double kbond,
                     double aHOH, double ka, double* d_tmp, double* d_out2) {
    const int64_t nmol = n / 3;
    if (nmol <= 0) { ref64_fill(s, d_out2, 2, 0.0); return; }
    hipLaunchKernelGGL(k_ref_bonded_terms, dim3(nbx_blocks(nmol, 256)), dim3(256), 0, s, x, n,
                       rOH, kbond, aHOH, ka, d_tmp);
    hipLaunchKernelGGL(k_ref_bonded_sum, dim3(2), dim3(256), 0, s, d_tmp, nmol, d_out2);
}

// ---------------------------------------------------------------------------
// RDF histogram (src/nbody_simulation_result.jl:664-693): frames in AoS (3 x n each)
// ---------------------------------------------------------------------------

// Bound by VALU work.  A wavefront takes 64 atoms a (one per lane) against 64 atoms b, pairs
// b > a; wavefronts stride over the upper triangle of 64 x 64 tiles of all frames, so few
// atoms or frames still spread over the chip.  The bin is estimated in FP32 from fixed-point
// box fractions (the integer wrap-around is the minimum image); only where a lane's estimate
// lies so near the edge of a bin or of the range that FP64 may put it on the other side
// (6e-7 of the distance for the FP32 operations, 2e-9 of the box for the fractions) does the
// wavefront take the FP64 displacement, square root and division: one iteration in 20 with
// 1,000 bins.  Counts go to a histogram in LDS shared by the block (one ds_add_u32 per pair
// in range) and reach memory once per block.  10 frames of 4,000 atoms: 99 us, all pairs in
// FP64 220; device-scope 64-bit atomics per pair from n / 128 blocks took 3,170 a frame.
// Above RDF_LDS_BINS bins (64 KiB of LDS with the staged atoms) the counts go to memory
// directly, and every pair takes FP64 (the estimate is open too often to pay).
#define RDF_LDS_BINS 8000

template <bool LDS>
__global__ void __launch_bounds__(1024)
k_ref_rdf(const double* __restrict__ f, int64_t n, int jstride, int64_t nj, int64_t nframes,
          double L, double dr, int64_t maxbin, unsigned long long* __restrict__ hist) {
    extern __shared__ double rdf_shared[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    double* const sb = rdf_shared + (size_t)wave * 64 * 4;   // this wavefront's atoms b
    unsigned* const cnt = reinterpret_cast<unsigned*>(rdf_shared + (size_t)waves * 64 * 4);
    if (LDS) {
        for (int64_t k = threadIdx.x; k <= maxbin; k += blockDim.x) cnt[k] = 0u;
        __syncthreads();
    }
    const auto flush = [&]() {
        __syncthreads();
        for (int64_t k = threadIdx.x; k <= maxbin; k += blockDim.x) {
            const unsigned c = cnt[k];
            cnt[k] = 0u;
            if (c) atomicAdd(&hist[k], 2ull * c);
        }
        __syncthreads();
    };
    const double radius = 0.5 * L, lim = (0.5 * L) * (0.5 * L), invL = 1.0 / L;
    const float per_bin = (float)((double)maxbin * 0x1p-32), half = 0.5f * (float)maxbin;
    const float open_abs = (float)maxbin * 2e-9f;
    const int64_t T = (nj + 63) >> 6, per_frame = T * (T + 1) / 2, items = per_frame * nframes;
    const int64_t stride = (int64_t)gridDim.x * waves;
    // 2^19 tiles of 2^12 pairs at most between two flushes: a counter stays below 2^32
    const int64_t rounds = (items + stride - 1) / stride;
    const int64_t flush_every = ((int64_t)1 << 19) / waves;
    for (int64_t r = 0; r < rounds; ++r) {
        const int64_t it = (int64_t)blockIdx.x * waves + wave + r * stride;
        if (it < items) {   // the whole wavefront
            const int64_t fr = it / per_frame, q = it - fr * per_frame;
            // row J of the triangle holds the tiles I = 0..J
            int64_t J = (int64_t)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
            while (J * (J + 1) / 2 > q) --J;
            while ((J + 1) * (J + 2) / 2 <= q) ++J;
            const int64_t I = q - J * (J + 1) / 2;
            const double* const x = f + fr * 3 * n;
            const int64_t a = (I << 6) + lane, b0 = J << 6;
            const int nb = (int)(nj - b0 < 64 ? nj - b0 : 64);
            double xi = 0.0, yi = 0.0, zi = 0.0;
            if (a < nj) {
                const double* p = x + 3 * a * jstride;
                xi = p[0]; yi = p[1]; zi = p[2];
            }
            if (lane < nb) {
                const double* p = x + 3 * (b0 + lane) * jstride;
                sb[4 * lane] = p[0]; sb[4 * lane + 1] = p[1]; sb[4 * lane + 2] = p[2];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const auto exact = [&](int k) {   // atom k of the staged against the lane's
                const double rx = nbx_wrap_cubic(xi - sb[4 * k], L, radius);
                const double ry = nbx_wrap_cubic(yi - sb[4 * k + 1], L, radius);
                const double rz = nbx_wrap_cubic(zi - sb[4 * k + 2], L, radius);
                const double s = rx * rx + ry * ry;
                const double r2 = s + rz * rz;
                if (r2 < lim && a < nj && b0 + k > a) {
                    const double fb = ceil(sqrt(r2) / dr);
                    if (fb > 1.0 && fb <= (double)maxbin) {
                        if (LDS) atomicAdd(&cnt[(unsigned)fb], 1u);
                        else atomicAdd(&hist[(int64_t)fb], 2ull);
                    }
                }
            };
            uint32_t qi[3] = {0u, 0u, 0u}, qj[3] = {0u, 0u, 0u};
            bool ok = true;
            if (LDS) {
                if (a < nj) ok = box_fixed(xi, yi, zi, invL, qi);
                if (lane < nb)
                    ok = box_fixed(sb[4 * lane], sb[4 * lane + 1], sb[4 * lane + 2], invL, qj) && ok;
            }
            if (!LDS || __any(!ok)) {
                for (int k = 0; k < nb; ++k) exact(k);
            } else {
                const bool diagonal = I == J;   // off it every lane holds an atom, a < b
                for (int k = 0; k < nb; ++k) {
                    const float dx = (float)(int)(qi[0] - __builtin_amdgcn_readlane(qj[0], k));
                    const float dy = (float)(int)(qi[1] - __builtin_amdgcn_readlane(qj[1], k));
                    const float dz = (float)(int)(qi[2] - __builtin_amdgcn_readlane(qj[2], k));
                    const float g = __builtin_amdgcn_sqrtf(fmaf(dz, dz, fmaf(dy, dy, dx * dx))) * per_bin;
                    const float open = fmaf(g, 6e-7f, open_abs);
                    const bool pair = !diagonal || k > lane;
                    if (__any(pair && (fabsf(g - rintf(g)) <= open || fabsf(g - half) <= open)))
                        exact(k);
                    else if (pair && g < half && g > 1.0f)
                        atomicAdd(&cnt[(unsigned)ceilf(g)], 1u);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        if (LDS && (r + 1) % flush_every == 0) flush();   // uniform over the block
    }
    if (LDS) flush();
}

void ref64_rdf_hist(hipStream_t s, const double* frames_aos, int64_t nframes, int64_t n,
                    int jstride, int64_t nj, double L, int64_t maxbin,
                    unsigned long long* d_hist) {
    if (nj <= 0 || nframes <= 0) return;
    const int64_t T = (nj + 63) >> 6, items = T * (T + 1) / 2 * nframes;
    // single wavefronts while they leave CUs free, then blocks of 16 that share a histogram,
    // at most two per CU
    const int threads = items <= 256 ? 64 : (items <= 4096 ? 256 : 1024);
    const int waves = threads / 64;
    const unsigned blocks = (unsigned)std::min<int64_t>((items + waves - 1) / waves,
                                                        threads == 1024 ? 512 : 1024);
    const size_t stage = sizeof(double) * 4 * 64 * waves;
    const double dr = L / (double)maxbin;
    if (maxbin <= RDF_LDS_BINS)
        hipLaunchKernelGGL(k_ref_rdf<true>, dim3(blocks), dim3(threads),
                           stage + sizeof(unsigned) * (size_t)(maxbin + 1), s, frames_aos, n,
                           jstride, nj, nframes, L, dr, maxbin, d_hist);
    else
        hipLaunchKernelGGL(k_ref_rdf<false>, dim3(blocks), dim3(threads), stage, s, frames_aos, n,
                           jstride, nj, nframes, L, dr, maxbin, d_hist);
}

// Histogram of nbx_rdf_noalloc: library-owned device memory (bins 0..NBX_RDF_NOALLOC_MAXBIN,
// 128 KiB), one copy per GPU, held until the process ends.  Host code never passes the
// array's name to a kernel: it uses the address that hipGetSymbolAddress returned for the
// device (ref64_rdf_scratch).
static __device__ __align__(256) unsigned long long scratch[NBX_RDF_NOALLOC_MAXBIN + 1];

int ref64_rdf_scratch(int device, unsigned long long** out) {
    static std::mutex mu;
    static unsigned long long* ptr[NBX_MAX_DEVICES] = {};
    if (device < 0 || device >= NBX_MAX_DEVICES) return -1;
    std::lock_guard<std::mutex> lock(mu);
    if (!ptr[device]) {
        int cur = -1;
        if (hipGetDevice(&cur) != hipSuccess) return -1;
        if (cur != device && hipSetDevice(device) != hipSuccess) return -1;
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess || !p) return -1;
        ptr[device] = static_cast<unsigned long long*>(p);
    }
    *out = ptr[device];
    return 0;
}

__global__ void k_fill_u64(unsigned long long* __restrict__ p, int64_t count) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < count) p[t] = 0ull;
}

void ref64_zero_u64(hipStream_t s, unsigned long long* p, int64_t count) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_fill_u64, dim3(nbx_blocks(count, 256)), dim3(256), 0, s, p, count);
}

__global__ void k_check_finite(const double* __restrict__ a, const double* __restrict__ b,
                               int64_t count, int* flag) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < count && !(isfinite(a[t]) && isfinite(b[t]))) flag[0] = 1;
}

void ref64_check_finite(hipStream_t s, const double* a, const double* b, int64_t count, int* d_flag) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_check_finite, dim3(nbx_blocks(count, 256)), dim3(256), 0, s, a, b, count,
                       d_flag);
}

__global__ void __launch_bounds__(256)
k_copy_words(ref64_copies c) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int k = 0; k < REF64_COPIES; ++k)
        if (t < c.words[k]) c.dst[k][t] = c.src[k][t];
}

void ref64_copy_words(hipStream_t s, const ref64_copies& c) {
    const int64_t most = *std::max_element(c.words, c.words + REF64_COPIES);
    if (most <= 0) return;
    hipLaunchKernelGGL(k_copy_words, dim3(nbx_blocks(most, 256)), dim3(256), 0, s, c);
}

// ---------------------------------------------------------------------------
// Nose-Hoover thermostat: src/thermostats.jl:116-122.  The reference keeps zeta in the
// position part of an extra coordinate column and writes its rate into the velocity part
// on every right-hand side; here both live in device scalars.
// ---------------------------------------------------------------------------
__global__ void k_ref_nosehoover(double* __restrict__ dv, const double* __restrict__ v, int64_t n,
                                 const double* __restrict__ scal, double* __restrict__ xi_out,
                                 double T0, double tau, int64_t ndf) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const double zeta = scal[NBX_SCAL_ZETA];
    if (i < 3 * n) dv[i] -= zeta * v[i];               // @. dv -= u[zind] * v
    if (i == 0) {
        const double it = 1.0 / tau;                     // inv(p.tau)^2
        const double T = scal[NBX_SCAL_T];
        xi_out[0] = (it * it) * (T / T0 - (double)(ndf + 1) / (double)ndf);
    }
}

void ref64_nosehoover(hipStream_t s, double* dv, const double* v, int64_t n, const double* scal,
                      double* xi_out, double T0, double tau, int64_t ndf) {
    const int64_t cnt = 3 * n > 0 ? 3 * n : 1;
    hipLaunchKernelGGL(k_ref_nosehoover, dim3(nbx_blocks(cnt, 256)), dim3(256), 0, s, dv, v, n,
                       scal, xi_out, T0, tau, ndf);
}

__global__ void k_ref_nh_drift(double* scal, double dt) {
    if (threadIdx.x == 0 && blockIdx.x == 0)
        scal[NBX_SCAL_ZETA] = scal[NBX_SCAL_ZETA] + dt * scal[NBX_SCAL_XI];
}

void ref64_nh_drift(hipStream_t s, double* scal, double dt) {
    hipLaunchKernelGGL(k_ref_nh_drift, dim3(1), dim3(64), 0, s, scal, dt);
}
