// nbx_gravity.hip -- all-pairs gravity (src/basic_potentials.jl:306-331) in mixed
// precision on gfx950.
//
//   a_i = G * sum_j m_j (r_j - r_i) / |r_j - r_i|^3      (= -G m_j r_ij / |r_ij|^3)
//
// pos = float4 (x, y, z, m) per body, written by the drift kernel from the FP64 state.
// Bound by FP32 VALU issue, so every unordered pair is evaluated once: the displacement
// and 1/r^3 (3 sub, 3 FMA, v_rsq_f32 at a quarter of the rate, 2 mul) serve body i and,
// with the opposite sign, body j (3 FMA each): 14 plain instructions and one v_rsq_f32
// per two interactions instead of 22 and two.
//
// The bodies form M tiles of S.  A block holds the S targets of tile I in registers (TPT
// per lane) and meets the tiles I .. I + M/2 of the ring of tiles (offset o = 0 the tile
// itself, one-sided; with M even, offset M/2 only from I < M/2), so each pair of tiles
// meets once.  Sources come 64 at a time through LDS: in step k lane l takes source
// (l + k) % 64, and the source's accumulated acceleration moves through the wavefront one
// lane per step (DPP rotation, 3 moves shared by the lane's TPT pairs), so that after 64
// steps every source has met every lane and its sum is back in its own lane.  (Measured at
// N = 65,536: rotating the positions too, without LDS, 897 us for this kernel against 779;
// sums kept in LDS and updated by ds_add_f32, ten times slower: the unit serialises the
// 64 lanes.)  No atomics: a source's sum over the S targets goes to a partial slot per
// offset, a target's sum over its chunk of sources to a slot per chunk, and k_grav_finish
// adds the slots in a fixed order.
//   WIDE   (n > 32,768): the four wavefronts hold different targets (S = 256 TPT) and
//          share the sources; their source sums are added in FP64 through LDS.  The
//          partial slots cost n^2 / (2 S) words, so large n wants the large tile.
//   narrow (n <= 32,768): the wavefronts hold the same S = 64 TPT targets and take
//          different sources, so that a few thousand bodies still fill the chip.
// Sums: plain FP32 over 64 sources (target side) and over the wavefront's 64 TPT <= 256
// targets (source side), Kahan across a target's source tiles, FP64 above.
//
// Measured, us per step with k_grav_finish, against one-sided tiles that evaluated every
// ordered pair: N = 65,536 equal masses 1,290 -> 802 (1,100 at its best tile shape), unequal
// 881; N = 3,001 unequal 178 -> 14 (12 blocks had 256 CUs to themselves); N = 1,000 9.
// 20 ns of a SIMD per 64 unordered pairs when the chip is full.
//
// The self term is removed by adding 1e-24 to r^2 inside the FMA chain (no extra
// instruction): for j == i the displacement is exactly zero and 1/r^3 = 1e36 is finite,
// so the contribution is exactly zero.  The mass in .w is m / m_max <= 1 (k_grav_finish
// multiplies by G m_max), so m_j / r^3 stays finite for any mass scale; for distinct
// bodies the 1e-24 rounds away unless r^2 < 2^24 * 1e-24 (r < 4e-9 in the caller's
// length unit).  Lanes past the last body hold a massless body at 1.8e19 per axis: r^2
// overflows to infinity, 1/r to zero, and the pair adds exactly zero to both sides.
// When every body has the same mass m (EQM), the tiles sum (r_j - r_i) / |r_j - r_i|^3
// and k_grav_finish multiplies by G m in FP64 (two multiplies fewer per pair).
#include <algorithm>

#include "nbx_mixed.h"

#define GR_THREADS 256
#define GR_TILE 256

// the wavefront's values moved on by one lane
__device__ __forceinline__ float grav_rot(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x134 /* wave_rol:1 */, 0xf,
                                                   0xf, false));
}

__device__ __forceinline__ float4 grav_body(const float4* __restrict__ pos, int i, int n) {
    return i < n ? pos[i] : make_float4(1.8e19f, 1.8e19f, 1.8e19f, 0.0f);
}

// 64 steps of one source tile against the lane's TPT targets: target sums into s, and
// (SYM) the source's own sum into g, which ends in the source's lane.  jt: the tile's
// bodies twice over, so that lane l reads source (l + k) % 64 of step k at a constant
// distance from its own place (no address arithmetic, no rotation of the positions).
// With four targets the loop is not unrolled: the lane's own pairs give independent chains,
// and unrolling only groups the LDS reads and costs registers (24.8 against 20.9 ns of a
// SIMD per 64 pairs); a single target needs the neighbouring steps for that.
template <int TPT, bool EQM, bool SYM>
__device__ __forceinline__ void grav_sweep(const float* xi, const float* yi, const float* zi,
                                           const float* mi, const float4* jt, float* sx,
                                           float* sy, float* sz, float* g) {
    float gx = 0.0f, gy = 0.0f, gz = 0.0f;
    constexpr int unroll = TPT == 1 ? 4 : (TPT == 2 ? 2 : 1);
#pragma unroll unroll
    for (int k = 0; k < 64; ++k) {
        const float4 pj = jt[k];
#pragma unroll
        for (int t = 0; t < TPT; ++t) {
            const float dx = pj.x - xi[t], dy = pj.y - yi[t], dz = pj.z - zi[t];
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, 1e-24f)));
            const float rinv = __builtin_amdgcn_rsqf(r2);
            const float r3 = rinv * rinv * rinv;
            const float si = EQM ? r3 : pj.w * r3;
            sx[t] = fmaf(dx, si, sx[t]);
            sy[t] = fmaf(dy, si, sy[t]);
            sz[t] = fmaf(dz, si, sz[t]);
            if (SYM) {
                const float sj = EQM ? r3 : mi[t] * r3;
                gx = fmaf(dx, sj, gx);
                gy = fmaf(dy, sj, gy);
                gz = fmaf(dz, sj, gz);
            }
        }
        if (SYM) {
            gx = grav_rot(gx);
            gy = grav_rot(gy);
            gz = grav_rot(gz);
        }
    }
    if (SYM) { g[0] = -gx; g[1] = -gy; g[2] = -gz; }
}

// Offsets [o0, o1) of the ring (o0 = 0: with the tile itself), blockIdx.x the target tile,
// blockIdx.y its chunk of them.  part: chunks target slots, then a source slot per offset
// from max(o0, 1) on; a slot is 3 n doubles.
template <int TPT, bool EQM, bool WIDE>
__global__ void __launch_bounds__(GR_THREADS)
k_grav_tiled(const float4* __restrict__ pos, int n, int tiles, int o0, int o1,
             double* __restrict__ part) {
    constexpr int S = (WIDE ? GR_THREADS : 64) * TPT;
    constexpr int JT = S / 64;                        // source tiles of 64 per tile
    constexpr int TS = WIDE ? GR_THREADS : 64;        // distance of a lane's targets
    // the source tile, twice over: WIDE two buffers that the block shares, narrow one per
    // wavefront
    __shared__ float4 jt[WIDE ? 2 : 4][128];
    __shared__ float wsum[WIDE ? 2 : 1][4][3][64];    // WIDE: source sums by wavefront
    __shared__ double tsum[WIDE ? 1 : 4][3][64];      // narrow: target sums by wavefront
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int I = blockIdx.x, chunk = blockIdx.y, chunks = gridDim.y;
    const int ibase = I * S + (WIDE ? tid : lane);
    float xi[TPT], yi[TPT], zi[TPT], mi[TPT];
    nbx_kahan ax[TPT], ay[TPT], az[TPT];
#pragma unroll
    for (int t = 0; t < TPT; ++t) {
        const float4 p = grav_body(pos, ibase + t * TS, n);
        xi[t] = p.x; yi[t] = p.y; zi[t] = p.z; mi[t] = p.w;
        ax[t].init(); ay[t].init(); az[t].init();
    }
    const int half = tiles >> 1;
    // offset M/2 of an even ring belongs to the lower half's blocks
    const int oend = min(o1, half + 1 - ((tiles & 1) == 0 && I >= half ? 1 : 0));
    const int items = oend > o0 ? (oend - o0) * JT : 0;
    const int b0 = (int)((int64_t)items * chunk / chunks);
    const int b1 = (int)((int64_t)items * (chunk + 1) / chunks);
    const int obase = o0 > 0 ? o0 : 1;
    double* const jpart = part + (size_t)chunks * 3 * n;
    constexpr int STEP = WIDE ? 1 : 4;
    const bool loads = !WIDE || wave == 0;   // the wavefront that fetches the source tile
    int item = b0 + (WIDE ? 0 : wave);
    const auto jlane = [&](int it) {
        int J = I + o0 + it / JT;
        J = J >= tiles ? J - tiles : J;
        return J * S + (it % JT) * 64 + lane;
    };
    const auto stage = [&](int buf, float4 p) {
        jt[buf][lane] = p;
        jt[buf][lane + 64] = p;
    };
    if (item < b1 && loads) stage(WIDE ? 0 : wave, grav_body(pos, jlane(item), n));
    if (WIDE) __syncthreads();
    else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // other lanes read the tile
    int par = 0;
    for (; item < b1; item += STEP) {
        float4 nxt = make_float4(0.f, 0.f, 0.f, 0.f);
        const bool more = item + STEP < b1 && loads;
        if (more) nxt = grav_body(pos, jlane(item + STEP), n);
        float sx[TPT], sy[TPT], sz[TPT], g[3];
#pragma unroll
        for (int t = 0; t < TPT; ++t) { sx[t] = 0.f; sy[t] = 0.f; sz[t] = 0.f; }
        const int o = o0 + item / JT;
        const float4* const tile = &jt[WIDE ? par : wave][lane];
        if (o == 0) grav_sweep<TPT, EQM, false>(xi, yi, zi, mi, tile, sx, sy, sz, g);
        else grav_sweep<TPT, EQM, true>(xi, yi, zi, mi, tile, sx, sy, sz, g);
        double* const slot = jpart + (size_t)(o - obase) * 3 * n;
        const int j = jlane(item);
        if constexpr (WIDE) {
            if (o != 0) {
#pragma unroll
                for (int k = 0; k < 3; ++k) wsum[par][wave][k][lane] = g[k];
            }
            if (more) stage(par ^ 1, nxt);
            // one barrier per tile: what this tile read is written again only after the next
            // barrier
            __syncthreads();
            if (o != 0 && wave < 3 && j < n)
                slot[(size_t)wave * n + j] =
                    ((double)wsum[par][0][wave][lane] + (double)wsum[par][1][wave][lane]) +
                    ((double)wsum[par][2][wave][lane] + (double)wsum[par][3][wave][lane]);
            par ^= 1;
        } else {
            if (o != 0 && j < n) {
#pragma unroll
                for (int k = 0; k < 3; ++k) slot[(size_t)k * n + j] = (double)g[k];
            }
            // the wavefront's own tile: its reads above are done (their values are used),
            // its LDS operations stay in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (more) stage(wave, nxt);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
#pragma unroll
        for (int t = 0; t < TPT; ++t) { ax[t].add(sx[t]); ay[t].add(sy[t]); az[t].add(sz[t]); }
    }
    double* const pc = part + (size_t)chunk * 3 * n;
#pragma unroll
    for (int t = 0; t < TPT; ++t) {
        const int i = ibase + t * TS;
        if constexpr (WIDE) {
            if (i < n) {
                pc[i] = ax[t].value();
                pc[n + i] = ay[t].value();
                pc[2 * (size_t)n + i] = az[t].value();
            }
        } else {
            tsum[wave][0][lane] = ax[t].value();
            tsum[wave][1][lane] = ay[t].value();
            tsum[wave][2][lane] = az[t].value();
            __syncthreads();
            if (wave < 3 && i < n)
                pc[(size_t)wave * n + i] = (tsum[0][wave][lane] + tsum[1][wave][lane]) +
                                           (tsum[2][wave][lane] + tsum[3][wave][lane]);
            __syncthreads();
        }
    }
}

// The slots of one launch for the block's 64 bodies: target slots in chunk order, then
// source slots in offset order (an even ring's offset M/2 wrote only the upper half's
// tiles).  Wavefront w adds slots w, w + 4, ... of body i (64 consecutive doubles per load,
// 4 slots in flight), the four sums meet in LDS in wavefront order: a few dozen slots per
// body are a latency chain, and n / 64 blocks of four wavefronts spread it over the chip
// (n = 4,096, 48 slots: 15.2 us per step; 19.9 with one thread per body in n / 256 blocks).
#define GR_BODIES 64
__device__ __forceinline__ void grav_add_slots(const double* __restrict__ part, int i, int n,
                                               const mx_grav_slots& g, double* s) {
    __shared__ double ws[4][3][GR_BODIES];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double a[3] = {0.0, 0.0, 0.0};
    if (i < n) {
        const int half = g.tiles >> 1;
        int oe = g.o1 < half + 1 ? g.o1 : half + 1;
        if ((g.tiles & 1) == 0 && oe == half + 1 && i / g.S < half) oe = half;
        const int ob = g.o0 > 0 ? g.o0 : 1;
        const int cnt = g.chunks + (oe > ob ? oe - ob : 0);
        const size_t step = 3 * (size_t)n;
        int c = wave;
        const double* p = part + (size_t)wave * step + i;
        for (; c + 12 < cnt; c += 16, p += 16 * step) {
            double w[3][4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int k = 0; k < 3; ++k) w[k][q] = p[4 * q * step + (size_t)k * n];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int k = 0; k < 3; ++k) a[k] += w[k][q];
        }
        for (; c < cnt; c += 4, p += 4 * step)
#pragma unroll
            for (int k = 0; k < 3; ++k) a[k] += p[(size_t)k * n];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) ws[wave][k][lane] = a[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k)
        s[k] += (ws[0][k][lane] + ws[1][k][lane]) + (ws[2][k][lane] + ws[3][k][lane]);
}

// the slots of a launch that is not the step's last one, into the running sum
__global__ void __launch_bounds__(256)
k_grav_accumulate(const double* __restrict__ part, int n, mx_grav_slots g, double* __restrict__ run,
                  int first) {
    const int i = blockIdx.x * GR_BODIES + (threadIdx.x & 63);
    double s[3] = {0.0, 0.0, 0.0};
    if (!first && i < n) { s[0] = run[i]; s[1] = run[n + i]; s[2] = run[2 * (size_t)n + i]; }
    grav_add_slots(part, i, n, g, s);
    if (threadIdx.x < GR_BODIES && i < n) {
        run[i] = s[0]; run[n + i] = s[1]; run[2 * (size_t)n + i] = s[2];
    }
}

// a_i = gscale * (running sum, if any, + the last launch's slots), then the end of the
// step and the drift by the block's first wavefront; gscale = G m_max (the tiles summed
// m_j / m_max), or G m when the tiles left out the common mass m
__global__ void __launch_bounds__(256)
k_grav_finish(const double* __restrict__ part, const double* __restrict__ run, int n,
              mx_grav_slots g, double gscale, mx_kick_params kp, mx_io io) {
    mx_resolve_step(kp);
    const int i = blockIdx.x * GR_BODIES + (threadIdx.x & 63);
    const bool own = threadIdx.x < GR_BODIES && i < n;
    double tval = 0.0;
    mx_atom A;
    if (own) mx_load_atom(i, n, io, A);
    double s[3] = {0.0, 0.0, 0.0};
    if (run != nullptr && own) { s[0] = run[i]; s[1] = run[n + i]; s[2] = run[2 * (size_t)n + i]; }
    grav_add_slots(part, i, n, g, s);
    if (own) {
        double ax = gscale * s[0], ay = gscale * s[1], az = gscale * s[2];
        if (mx_therm_force(kp)) {
            const double cb = mx_berendsen_coeff(kp);
            ax += cb * A.vh[0]; ay += cb * A.vh[1]; az += cb * A.vh[2];
        }
        io.a[i] = ax; io.a[n + i] = ay; io.a[2 * n + i] = az;
        if (kp.do_kick) {
            double v3[3];
            mx_kick_atom(i, ax, ay, az, A, kp, v3);
            if (kp.therm == NBX_THERM_ANDERSEN &&
                nbx_rng_uniform(kp.seed, mx_atom_id(kp, i), kp.step, NBX_RNG_ANDERSEN) < kp.prob)
                mx_andersen_atom(i, kp.m0, kp, v3);
            io.v[i] = v3[0]; io.v[n + i] = v3[1]; io.v[2 * n + i] = v3[2];
            if (io.do_drift) tval = mx_drift_atom(i, n, v3, ax, ay, az, A, kp, io);
        }
    }
    mx_epilogue(tval, io, n);
}

// Launch shape.  Targets per lane: more of them share the rotation and leave fewer source
// slots, fewer give more wavefronts (us per step with 1 / 2 / 4: n = 4,096 15 / 16 / 20,
// n = 6,000 23 / 21 / 24, n = 8,192 48 / 31 / 29).
// Chunks of a tile's ring.  Narrow: one source tile per wavefront, at most about 4,096
// blocks; at one target per lane rounded up to a power of two (idle wavefronts cost less
// there than uneven shares).  Wide: two rounds of the 1,536 blocks that fit the chip (the
// wavefronts of a SIMD finish one after the other, and the next round's blocks fill in:
// n = 65,536 kernel 886 us at 16 chunks, 829 at 24, 779 at 48, 757 at 144, where the
// partials cost more than that wins).
// At most GR_SLOTS offsets per launch bound the partials to (chunks + GR_SLOTS) x 24 n
// bytes: larger rings take several launches with a running sum between them.
#define GR_SLOTS 64
mx_grav_shape mx_gravity_shape(const nbx_ctx* c) {
    mx_grav_shape g{};
    const int64_t n = c->n;
    g.wide = n > 32768;
    g.tpt = c->grav_tpt_set ? c->grav_tpt_set : (n > 6144 ? 4 : (n > 4096 ? 2 : 1));
    g.S = (g.wide ? GR_THREADS : 64) * g.tpt;
    g.tiles = (int)((n + g.S - 1) / g.S);
    const int offsets = g.tiles / 2 + 1;   // with offset 0
    g.passes = (offsets + GR_SLOTS - 1) / GR_SLOTS;
    g.per_pass = (offsets + g.passes - 1) / g.passes;
    const int items = g.per_pass * (g.S / 64);
    if (c->grav_chunks_set) {
        g.chunks = c->grav_chunks_set;
    } else if (g.wide) {
        g.chunks = std::max(1, std::min({3072 / g.tiles, items, 64}));
    } else {
        g.chunks = (items + 3) / 4;
        if (g.tpt == 1) {
            int p = 1;
            while (p < g.chunks) p *= 2;
            g.chunks = p;
        }
        g.chunks = std::max(1, std::min(g.chunks, 4096 / g.tiles));
    }
    g.part_doubles = 3 * (size_t)n * (size_t)(g.chunks + g.per_pass + (g.passes > 1 ? 1 : 0));
    return g;
}

template <int TPT, bool EQM>
static void grav_launch(hipStream_t s, const mx_grav_shape& g, const float4* pos, int n, int o0,
                        int o1, double* part) {
    const dim3 grid(g.tiles, g.chunks);
    if (g.wide)
        hipLaunchKernelGGL((k_grav_tiled<TPT, EQM, true>), grid, dim3(GR_THREADS), 0, s, pos, n,
                           g.tiles, o0, o1, part);
    else
        hipLaunchKernelGGL((k_grav_tiled<TPT, EQM, false>), grid, dim3(GR_THREADS), 0, s, pos, n,
                           g.tiles, o0, o1, part);
}

// ev0/ev1 (optional): HIP events recorded around the k_grav_tiled launches
void mx_launch_gravity(hipStream_t s, const nbx_ctx* c, const void* pos, double G,
                       const mx_kick_params& kp, const mx_io& io, int force_only_kernel,
                       hipEvent_t ev0, hipEvent_t ev1) {
    const int n = (int)c->n;
    if (n <= 0) return;
    const mx_grav_shape g = mx_gravity_shape(c);
    const float4* p4 = (const float4*)pos;
    const bool eqm = c->equal_masses;
    double* const run = g.passes > 1
        ? c->d_part + 3 * (size_t)n * (size_t)(g.chunks + g.per_pass) : nullptr;
    mx_grav_slots sl{};
    sl.tiles = g.tiles;
    sl.S = g.S;
    sl.chunks = g.chunks;
    if (ev0) (void)hipEventRecord(ev0, s);
    for (int p = 0; p < g.passes; ++p) {
        sl.o0 = p * g.per_pass;
        sl.o1 = sl.o0 + g.per_pass;
        if (g.tpt == 4) {
            if (eqm) grav_launch<4, true>(s, g, p4, n, sl.o0, sl.o1, c->d_part);
            else grav_launch<4, false>(s, g, p4, n, sl.o0, sl.o1, c->d_part);
        } else if (g.tpt == 2) {
            if (eqm) grav_launch<2, true>(s, g, p4, n, sl.o0, sl.o1, c->d_part);
            else grav_launch<2, false>(s, g, p4, n, sl.o0, sl.o1, c->d_part);
        } else {
            if (eqm) grav_launch<1, true>(s, g, p4, n, sl.o0, sl.o1, c->d_part);
            else grav_launch<1, false>(s, g, p4, n, sl.o0, sl.o1, c->d_part);
        }
        if (p + 1 < g.passes)
            hipLaunchKernelGGL(k_grav_accumulate, dim3(nbx_blocks(n, GR_BODIES)), dim3(256), 0, s,
                               c->d_part, n, sl, run, p == 0 ? 1 : 0);
    }
    if (ev1) (void)hipEventRecord(ev1, s);
    if (force_only_kernel) return;
    const double scale = eqm ? G * c->h_ms[0] : G / c->mass_wscale;
    hipLaunchKernelGGL(k_grav_finish, dim3(nbx_blocks(n, GR_BODIES)), dim3(256), 0, s, c->d_part, run, n,
                       sl, scale, kp, io);
}

// ---------------------------------------------------------------------------
// All-pairs magnetic dipoles (src/basic_potentials.jl:333-365) in mixed precision: FP32
// pair law on float4 positions and float4 moments staged 256 at a time in LDS, plain FP32
// sums per tile, Kahan across tiles; the per-target sum divided by m_i goes to `part`
// (FP64), and k_grav_finish applies 3 mu/4pi, the kick and the drift.  No boundary
// conditions (as the reference); j == i skipped.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(GR_THREADS)
k_mag_tiled(const float4* __restrict__ pos, const float4* __restrict__ mm, int n,
            double* __restrict__ part) {
    __shared__ float4 tp[GR_TILE];
    __shared__ float4 tm[GR_TILE];
    const int tid = threadIdx.x;
    const int i = blockIdx.x * GR_THREADS + tid;
    const float4 pi = i < n ? pos[i] : make_float4(0.f, 0.f, 0.f, 1.f);
    const float4 mi = i < n ? mm[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    nbx_kahan ax, ay, az;
    ax.init(); ay.init(); az.init();
    for (int base = 0; base < n; base += GR_TILE) {
        const int j = base + tid;
        tp[tid] = j < n ? pos[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        tm[tid] = j < n ? mm[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
        const int lim = (n - base) < GR_TILE ? (n - base) : GR_TILE;
        float sx = 0.f, sy = 0.f, sz = 0.f;
        for (int q = 0; q < lim; ++q) {
            if (base + q == i) continue;
            const float4 pj = tp[q];
            const float4 mj = tm[q];
            const float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
            const float d = rx * rx + ry * ry + rz * rz;
            const float inv = __builtin_amdgcn_rsqf(d);
            const float inv2 = inv * inv;
            const float inv4 = inv2 * inv2;
            const float r1 = rx * inv, r2 = ry * inv, r3 = rz * inv;
            const float mir = mi.x * r1 + mi.y * r2 + mi.z * r3;
            const float mij = mj.x * r1 + mj.y * r2 + mj.z * r3;
            const float dmm = mi.x * mj.x + mi.y * mj.y + mi.z * mj.z;
            const float f5 = 5.0f * mir * mij;
            sx += (mi.x * mij + mj.x * mir + r1 * (dmm - f5)) * inv4;
            sy += (mi.y * mij + mj.y * mir + r2 * (dmm - f5)) * inv4;
            sz += (mi.z * mij + mj.z * mir + r3 * (dmm - f5)) * inv4;
        }
        ax.add(sx); ay.add(sy); az.add(sz);
        __syncthreads();
    }
    if (i < n) {
        const double im = 1.0 / (double)pi.w;
        part[i] = ax.value() * im;
        part[n + i] = ay.value() * im;
        part[2 * n + i] = az.value() * im;
    }
}

void mx_launch_magnetic(hipStream_t s, const nbx_ctx* c, const void* pos, double mu_4pi,
                        const mx_kick_params& kp, const mx_io& io, int force_only_kernel) {
    const int n = (int)c->n;
    if (n <= 0) return;
    hipLaunchKernelGGL(k_mag_tiled, dim3(nbx_blocks(n, GR_THREADS)), dim3(GR_THREADS), 0, s,
                       (const float4*)pos, (const float4*)c->d_mm4, n, c->d_part);
    if (force_only_kernel) return;
    mx_grav_slots one{};   // a single target slot
    one.tiles = 1;
    one.S = n;
    one.chunks = 1;
    hipLaunchKernelGGL(k_grav_finish, dim3(nbx_blocks(n, GR_BODIES)), dim3(256), 0, s, c->d_part,
                       (const double*)nullptr, n, one, 3.0 * mu_4pi, kp, io);
}

// ---------------------------------------------------------------------------
// Plain device-to-device copy: the calibration kernel for HBM byte counters and the
// achievable-bandwidth probe.  Reads `n16` 16-byte words from src, writes them to dst.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_copy_probe(const float4* __restrict__ src,
                                                    float4* __restrict__ dst, int64_t n16) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
        dst[i] = src[i];
}

// VALU issue-rate calibration: 8 independent chains per lane of one instruction, its
// encoding pinned by inline asm (0: v_fmac_f32, 1: v_mul_f32, 2: v_rsq_f32)
#define VP_ITERS 2048
template <int KIND>
__global__ void __launch_bounds__(256) k_valu_probe(float* __restrict__ out, float b0, float c0) {
    float a[8];
    const float b = b0 + threadIdx.x * 1e-9f, cc = c0;
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = 1.0f + threadIdx.x * 1e-3f + k;
    for (int it = 0; it < VP_ITERS; ++it) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (KIND == 0) asm volatile("v_fmac_f32 %0, %1, %2" : "+v"(a[k]) : "v"(b), "v"(cc));
            if (KIND == 1) asm volatile("v_mul_f32 %0, %0, %1" : "+v"(a[k]) : "v"(b));
            if (KIND == 2) asm volatile("v_rsq_f32 %0, %0" : "+v"(a[k]));
        }
    }
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) s += a[k];
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = s;
}

int mx_valu_probe(nbx_ctx* c, int kind, int reps, double* rate) {
    const int blocks = 8192, threads = 256;
    float* out = nullptr;
    if (hipMalloc((void**)&out, sizeof(float) * blocks * threads) != hipSuccess)
        return nbx_fail(c, NBX_ERR_DEVICE, "valu probe: out of memory");
    int cus = 0;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device);
    hipStream_t s = c->stream;
    auto launch = [&]() {
        if (kind == 0) hipLaunchKernelGGL(k_valu_probe<0>, dim3(blocks), dim3(threads), 0, s, out, 0.999f, 1e-3f);
        else if (kind == 1) hipLaunchKernelGGL(k_valu_probe<1>, dim3(blocks), dim3(threads), 0, s, out, 0.999f, 1e-3f);
        else hipLaunchKernelGGL(k_valu_probe<2>, dim3(blocks), dim3(threads), 0, s, out, 0.999f, 1e-3f);
    };
    launch();
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    float best = 0.f;
    hipError_t err = hipSuccess;
    for (int r = 0; r < reps && err == hipSuccess; ++r) {
        (void)hipEventRecord(e0, s);
        launch();
        (void)hipEventRecord(e1, s);
        err = hipEventSynchronize(e1);
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        if (r == 0 || ms < best) best = ms;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(out);
    if (err != hipSuccess) return nbx_fail(c, NBX_ERR_DEVICE, hipGetErrorString(err));
    const double wave_instr = (double)blocks * threads / 64 * VP_ITERS * 8;
    *rate = wave_instr / (4.0 * (cus > 0 ? cus : 256)) / ((double)best * 1e6);
    return NBX_OK;
}

int mx_copy_probe(nbx_ctx* c, int64_t bytes, int iters, double* avg_ms) {
    const int64_t n16 = bytes / 16;
    void* a = nullptr;
    void* b = nullptr;
    if (hipMalloc(&a, n16 * 16) != hipSuccess) return nbx_fail(c, NBX_ERR_DEVICE, "copy probe: out of memory");
    if (hipMalloc(&b, n16 * 16) != hipSuccess) {
        (void)hipFree(a);
        return nbx_fail(c, NBX_ERR_DEVICE, "copy probe: out of memory");
    }
    hipStream_t s = c->stream;
    (void)hipMemsetAsync(a, 0, n16 * 16, s);
    const int blocks = 8192;
    hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, s, (const float4*)a, (float4*)b, n16);
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipEventRecord(e0, s);
    for (int k = 0; k < iters; ++k)
        hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, s, (const float4*)a, (float4*)b,
                           n16);
    (void)hipEventRecord(e1, s);
    hipError_t err = hipEventSynchronize(e1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    if (err != hipSuccess) return nbx_fail(c, NBX_ERR_DEVICE, hipGetErrorString(err));
    *avg_ms = (double)ms / iters;
    return NBX_OK;
}
