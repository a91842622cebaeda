// nbx_api.cpp -- C ABI of libnbx (declared in include/nbx.h): context management,
// argument validation (the reference's BoundsError / MethodError become error codes),
// host <-> device transfers (Julia column-major 3 x n <-> device SoA) and the FP64
// reference-order orchestration of soode_system! (src/nbody_to_ode.jl:474-532) and of
// the velocity-Verlet step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "nbx_internal.h"

static thread_local std::string g_create_error;
void mx_launch_iota(hipStream_t s, int* p, int64_t n);   // nbx_sort.hip

int nbx_fail(nbx_ctx* c, int code, const std::string& msg) {
    if (c) c->err = msg;
    else g_create_error = msg;
    return code;
}

extern "C" const char* nbx_version(void) { return "nbx 0.1 (gfx950)"; }

extern "C" int nbx_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

extern "C" const char* nbx_last_error(const nbx_ctx* c) {
    return c ? c->err.c_str() : g_create_error.c_str();
}

static void free_ptr(void* p) {
    if (p) (void)hipFree(p);
}

static void release(nbx_ctx* c) {
    mx_release(c);
    void* const own[] = {c->d_base, c->d_mm, c->d_mm4, c->d_rdf_work, c->d_frac, c->d_rhs, c->d_water,
                         c->d_frames, c->d_backup, c->d_bins, c->d_sortbuf, c->d_permbuf};
    for (void* p : own) free_ptr(p);
    c->d_base = nullptr;
    c->d_rdf_work = c->d_rhs = c->d_water = c->d_frames = c->d_backup = c->d_permbuf = nullptr;
    c->d_frac = nullptr;
    c->d_bins = nullptr;
    c->d_perm = c->d_iperm = c->d_pmap = nullptr;
    c->d_sortbuf = nullptr;
    c->sortbuf_bytes = 0;
    c->d_mm = nullptr;
    c->d_mm4 = nullptr;
    c->d_x = c->d_v = c->d_a = c->d_vh = c->d_tmp = c->d_ms = c->d_qs = nullptr;
    c->d_red = c->d_scal = nullptr;
    if (c->stream) (void)hipStreamDestroy(c->stream);
    c->stream = nullptr;
}

extern "C" int nbx_create(nbx_ctx** out, int64_t n, int32_t system_kind, const double* masses,
                          const double* charges) {
    if (!out) return nbx_fail(nullptr, NBX_ERR_INVALID, "nbx_create: out is NULL");
    *out = nullptr;
    if (n < 0) return nbx_fail(nullptr, NBX_ERR_INVALID, "nbx_create: n < 0");
    if (system_kind != NBX_SYS_POTENTIAL && system_kind != NBX_SYS_WATER)
        return nbx_fail(nullptr, NBX_ERR_INVALID, "nbx_create: unknown system kind");
    if (system_kind == NBX_SYS_WATER && n % 3 != 0)
        return nbx_fail(nullptr, NBX_ERR_INVALID,
                        "nbx_create: a water system has 3 atoms (O, H1, H2) per molecule");
    if (n > 0 && !masses) return nbx_fail(nullptr, NBX_ERR_INVALID, "nbx_create: masses NULL");
    if (n > (int64_t)1 << 30)
        return nbx_fail(nullptr, NBX_ERR_INVALID, "nbx_create: n above 2^30 atoms");
    for (int64_t i = 0; i < n; ++i)
        if (!(masses[i] > 0.0) || !std::isfinite(masses[i]))
            return nbx_fail(nullptr, NBX_ERR_INVALID,
                            "nbx_create: mass " + std::to_string(i) + " not positive/finite");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return nbx_fail(nullptr, NBX_ERR_DEVICE, "nbx_create: no HIP device visible");
    nbx_ctx* c = new nbx_ctx();
    c->n = n;
    c->sys = system_kind;
    c->h_ms.assign(masses, masses + n);
    c->equal_masses = n > 0 && std::all_of(masses, masses + n,
                                           [&](double m) { return m == masses[0]; });
    if (n > 0) {
        c->mass_wscale = 1.0 / *std::max_element(masses, masses + n);
        c->mass_wmin = 1.0 / *std::min_element(masses, masses + n);
    }
    if (charges) {
        c->h_qs.assign(charges, charges + n);
        c->has_q = true;
    }
    c->bc.kind = NBX_BC_INFINITE;
    for (int k = 0; k < 6; ++k) c->bc.b[k] = (k % 2 == 0) ? -INFINITY : INFINITY;
    if (const char* g = std::getenv("NBX_GRAPH_STEPS")) c->graph_steps = std::max(0, std::atoi(g));
    if (const char* g = std::getenv("NBX_BUILD_EVERY")) {
        const int m = std::atoi(g);
        if (m == 1 || m == 2 || m == 5) {
            c->build_every = m;
            c->every_auto = false;
        }
    }
    if (const char* g = std::getenv("NBX_LANES")) {
        const int l = std::atoi(g);
        if (l == 1 || l == 2 || l == 4 || l == 8 || l == 16 || l == 32) {
            c->nl.lanes = l;
            c->nl.lanes_auto = false;
        }
    }
    // spatial re-sort of the mixed path's state every 10,000 steps from 8,192 atoms on
    // (NBX_SORT_EVERY: another interval for any size, 0 to never sort)
    c->sort_every = n >= 8192 ? 10000 : 0;
    if (const char* g = std::getenv("NBX_SORT_EVERY")) c->sort_every = std::max(0, std::atoi(g));
    hipError_t e = hipGetDevice(&c->device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    // set-up of nbx_rdf_noalloc: the device address of this GPU's histogram array
    if (e == hipSuccess && ref64_rdf_scratch(c->device, &c->d_rdf_hist) != 0)
        e = hipErrorInvalidSymbol;
    // one allocation for the arrays every context needs, each at a 256-byte boundary
    const size_t n1 = (size_t)(n > 0 ? n : 1);
    size_t off = 0;
    const auto part = [&off](size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) / 256 * 256;
        return at;
    };
    const size_t b1 = sizeof(double) * n1, b3 = 3 * b1, bi = sizeof(int) * n1;
    const size_t at3[5] = {part(b3), part(b3), part(b3), part(b3), part(b3)};
    const size_t at_ms = part(b1), at_qs = part(b1), at_red = part(b1 + 8192 * sizeof(double)),
                 at_scal = part(NBX_SCAL_COUNT * sizeof(double)), at_p[3] = {part(bi), part(bi), part(bi)};
    if (e == hipSuccess) e = hipMalloc((void**)&c->d_base, off);
    if (e == hipSuccess) {
        double** const p3[5] = {&c->d_x, &c->d_v, &c->d_a, &c->d_vh, &c->d_tmp};
        int** const pi[3] = {&c->d_perm, &c->d_iperm, &c->d_pmap};
        for (int k = 0; k < 5; ++k) *p3[k] = reinterpret_cast<double*>(c->d_base + at3[k]);
        for (int k = 0; k < 3; ++k) *pi[k] = reinterpret_cast<int*>(c->d_base + at_p[k]);
        c->d_ms = reinterpret_cast<double*>(c->d_base + at_ms);
        c->d_qs = reinterpret_cast<double*>(c->d_base + at_qs);
        c->d_red = reinterpret_cast<double*>(c->d_base + at_red);
        c->d_scal = reinterpret_cast<double*>(c->d_base + at_scal);
        // the finite flag and the Nose-Hoover state start at zero
        ref64_fill(c->stream, c->d_scal, NBX_SCAL_COUNT, 0.0);
        mx_launch_iota(c->stream, c->d_perm, n);
        mx_launch_iota(c->stream, c->d_iperm, n);
        if (n > 0 && !charges) ref64_fill(c->stream, c->d_qs, n, 0.0);
        e = hipGetLastError();
    }
    if (e == hipSuccess && n > 0)
        e = hipMemcpyAsync(c->d_ms, masses, b1, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess && n > 0 && charges)
        e = hipMemcpyAsync(c->d_qs, charges, b1, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) {
        std::string msg = std::string("nbx_create: ") + hipGetErrorString(e);
        release(c);
        delete c;
        return nbx_fail(nullptr, NBX_ERR_DEVICE, msg);
    }
    *out = c;
    return NBX_OK;
}

extern "C" int nbx_destroy(nbx_ctx* c) {
    if (!c) return NBX_OK;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    release(c);
    delete c;
    return NBX_OK;
}

static void invalidate(nbx_ctx* c) {
    c->accel_valid = false;
    c->nl.ready = false;
    c->list_sorted = false;
    c->every_chosen = false;
    c->guarded = false;
    ++c->version;
}

extern "C" int nbx_set_boundary(nbx_ctx* c, int32_t kind, const double* box) {
    if (!c) return NBX_ERR_INVALID;
    nbx_bcv bc{};
    bc.kind = kind;
    if (kind == NBX_BC_INFINITE) {
        for (int k = 0; k < 6; ++k) bc.b[k] = (k % 2 == 0) ? -INFINITY : INFINITY;
    } else if (kind == NBX_BC_CUBIC) {
        if (!box || !(box[0] > 0.0) || !std::isfinite(box[0]))
            return nbx_fail(c, NBX_ERR_INVALID, "cubic box side L must be positive and finite");
        bc.b[0] = box[0];
    } else if (kind == NBX_BC_PERIODIC) {
        if (!box) return nbx_fail(c, NBX_ERR_INVALID, "periodic bounds missing");
        for (int k = 0; k < 3; ++k)
            if (!(box[2 * k + 1] > box[2 * k]) || !std::isfinite(box[2 * k]) ||
                !std::isfinite(box[2 * k + 1]))
                return nbx_fail(c, NBX_ERR_INVALID, "periodic bounds need finite lo < hi");
        for (int k = 0; k < 6; ++k) bc.b[k] = box[k];
    } else {
        return nbx_fail(c, NBX_ERR_INVALID, "unknown boundary condition kind");
    }
    c->bc = bc;
    invalidate(c);
    return NBX_OK;
}

extern "C" int nbx_set_kb(nbx_ctx* c, double kb) {
    if (!c) return NBX_ERR_INVALID;
    if (!(kb > 0.0) || !std::isfinite(kb)) return nbx_fail(c, NBX_ERR_INVALID, "kb must be > 0");
    c->kb = kb;
    invalidate(c);
    return NBX_OK;
}

extern "C" int nbx_set_precision(nbx_ctx* c, int32_t mode) {
    if (!c) return NBX_ERR_INVALID;
    if (mode != NBX_PREC_FP64_REF && mode != NBX_PREC_MIXED)
        return nbx_fail(c, NBX_ERR_INVALID, "unknown precision mode");
    c->prec = mode;
    invalidate(c);
    return NBX_OK;
}

extern "C" int nbx_set_skin(nbx_ctx* c, double skin) {
    if (!c) return NBX_ERR_INVALID;
    if (!(skin >= 0.0) || !std::isfinite(skin))
        return nbx_fail(c, NBX_ERR_INVALID, "skin must be >= 0 and finite");
    c->skin = skin;
    c->skin_set = true;
    invalidate(c);
    return NBX_OK;
}

static int add_term(nbx_ctx* c, int kind, double p0, double p1, double p2) {
    nbx_term t{};
    t.kind = kind;
    t.p[0] = p0; t.p[1] = p1; t.p[2] = p2;
    if (c->sys == NBX_SYS_WATER) {
        if (kind == NBX_TERM_LJ) { c->water_lj = t; c->water_lj_set = true; }
        else if (kind == NBX_TERM_ELEC || kind == NBX_TERM_RF) {
            c->water_elec = t; c->water_elec_set = true;
        } else {
            return nbx_fail(c, NBX_ERR_UNSUPPORTED, "water systems take LJ and electrostatics only");
        }
    } else {
        if (c->terms.size() >= 8) return nbx_fail(c, NBX_ERR_INVALID, "at most 8 potentials");
        c->terms.push_back(t);
    }
    invalidate(c);
    return NBX_OK;
}

extern "C" int nbx_add_lennard_jones(nbx_ctx* c, double eps, double sigma, double R) {
    if (!c) return NBX_ERR_INVALID;
    if (!std::isfinite(eps) || !(sigma > 0.0) || !std::isfinite(sigma) || !(R > 0.0))
        return nbx_fail(c, NBX_ERR_INVALID, "LennardJonesParameters: need finite eps, sigma > 0, R > 0");
    return add_term(c, NBX_TERM_LJ, eps, sigma, R);
}

extern "C" int nbx_add_electrostatic(nbx_ctx* c, double k, double R) {
    if (!c) return NBX_ERR_INVALID;
    if (!c->has_q) return nbx_fail(c, NBX_ERR_INVALID, "electrostatics needs charges");
    if (!std::isfinite(k) || !(R > 0.0))
        return nbx_fail(c, NBX_ERR_INVALID, "ElectrostaticParameters: need finite k and R > 0");
    return add_term(c, NBX_TERM_ELEC, k, R, 0.0);
}

extern "C" int nbx_add_reaction_field(nbx_ctx* c, double k, double R, double eps_rf) {
    if (!c) return NBX_ERR_INVALID;
    if (!c->has_q) return nbx_fail(c, NBX_ERR_INVALID, "reaction field needs charges");
    if (!std::isfinite(k) || !(R > 0.0) || !std::isfinite(R) || !(eps_rf >= 1.0))
        return nbx_fail(c, NBX_ERR_INVALID, "reaction field: need finite k, finite R > 0, eps_rf >= 1");
    return add_term(c, NBX_TERM_RF, k, R, eps_rf);
}

extern "C" int nbx_add_gravitational(nbx_ctx* c, double G) {
    if (!c) return NBX_ERR_INVALID;
    if (!std::isfinite(G)) return nbx_fail(c, NBX_ERR_INVALID, "G must be finite");
    return add_term(c, NBX_TERM_GRAV, G, 0.0, 0.0);
}

static int upload_aos(nbx_ctx* c, const double* host, double* d_soa);

extern "C" int nbx_add_magnetostatic(nbx_ctx* c, double mu_4pi) {
    if (!c) return NBX_ERR_INVALID;
    if (c->sys != NBX_SYS_POTENTIAL)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED, "magnetic dipoles apply to potential systems");
    if (!c->mm_set) return nbx_fail(c, NBX_ERR_INVALID, "magnetostatics needs moments (nbx_set_moments)");
    if (!std::isfinite(mu_4pi)) return nbx_fail(c, NBX_ERR_INVALID, "mu/4pi must be finite");
    return add_term(c, NBX_TERM_MAG, mu_4pi, 0.0, 0.0);
}

extern "C" int nbx_set_moments(nbx_ctx* c, const double* mm) {
    if (!c || !mm) return NBX_ERR_INVALID;
    const int64_t n = c->n;
    if (!nbx_all_finite(mm, 3 * n)) return nbx_fail(c, NBX_ERR_NONFINITE, "moments hold NaN or Inf");
    if (!c->d_mm) NBX_HIP(c, hipMalloc((void**)&c->d_mm, sizeof(double) * 3 * (size_t)std::max<int64_t>(n, 1)));
    if (!c->d_mm4) NBX_HIP(c, hipMalloc(&c->d_mm4, sizeof(float) * 4 * (size_t)std::max<int64_t>(n, 1)));
    if (n > 0) {
        int rc = upload_aos(c, mm, c->d_mm);
        if (rc) return rc;
        std::vector<float> f4((size_t)4 * n);
        for (int64_t i = 0; i < n; ++i) {
            f4[4 * i] = (float)mm[3 * i];
            f4[4 * i + 1] = (float)mm[3 * i + 1];
            f4[4 * i + 2] = (float)mm[3 * i + 2];
            f4[4 * i + 3] = 0.0f;
        }
        NBX_HIP(c, hipMemcpyAsync(c->d_mm4, f4.data(), sizeof(float) * f4.size(),
                                  hipMemcpyHostToDevice, c->stream));
        NBX_HIP(c, hipStreamSynchronize(c->stream));
    }
    c->mm_set = true;
    invalidate(c);
    return NBX_OK;
}

extern "C" int nbx_set_spcfw(nbx_ctx* c, double rOH, double aHOH, double kbond, double kangle) {
    if (!c) return NBX_ERR_INVALID;
    if (c->sys != NBX_SYS_WATER)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED, "SPCFwParameters apply to water systems");
    if (!(rOH > 0.0) || !std::isfinite(aHOH) || !std::isfinite(kbond) || !std::isfinite(kangle))
        return nbx_fail(c, NBX_ERR_INVALID, "SPCFwParameters: need rOH > 0 and finite values");
    c->rOH = rOH; c->aHOH = aHOH; c->kbond = kbond; c->kangle = kangle;
    c->spcfw_set = true;
    invalidate(c);
    return NBX_OK;
}

// the extra coordinate column of the reference's Nose-Hoover state starts at zero
// (gather_bodies_initial_coordinates, src/nbody_to_ode.jl:1-20)
static int reset_nosehoover(nbx_ctx* c) {
    c->nh_advanced = false;
    ref64_fill(c->stream, c->d_scal + NBX_SCAL_ZETA, 2, 0.0);
    NBX_HIP(c, hipGetLastError());
    return NBX_OK;
}

extern "C" int nbx_set_thermostat(nbx_ctx* c, int32_t kind, double T, double param) {
    if (!c) return NBX_ERR_INVALID;
    if (kind < NBX_THERM_NONE || kind > NBX_THERM_NOSEHOOVER)
        return nbx_fail(c, NBX_ERR_INVALID, "unknown thermostat kind");
    if (kind == NBX_THERM_NOSEHOOVER && T <= 0.0)
        return nbx_fail(c, NBX_ERR_INVALID, "Nose-Hoover needs a target temperature > 0");
    if (kind != NBX_THERM_NONE) {
        if (!(T >= 0.0) || !std::isfinite(T))
            return nbx_fail(c, NBX_ERR_INVALID, "thermostat temperature must be >= 0");
        if (!(param > 0.0) || !std::isfinite(param))
            return nbx_fail(c, NBX_ERR_INVALID, "thermostat parameter must be > 0");
    }
    c->therm = kind; c->therm_T = T; c->therm_p = param;
    invalidate(c);
    return reset_nosehoover(c);
}

// ---------------------------------------------------------------------------
// State transfer
// ---------------------------------------------------------------------------

static int upload_aos(nbx_ctx* c, const double* host, double* d_soa) {
    const size_t b = sizeof(double) * (size_t)(3 * c->n);
    NBX_HIP(c, hipMemcpyAsync(c->d_tmp, host, b, hipMemcpyHostToDevice, c->stream));
    ref64_aos_to_soa(c->stream, c->d_tmp, d_soa, c->n);
    NBX_HIP(c, hipGetLastError());
    return NBX_OK;
}

static int download_aos(const nbx_ctx* cc, const double* d_soa, double* host) {
    nbx_ctx* c = const_cast<nbx_ctx*>(cc);
    const size_t b = sizeof(double) * (size_t)(3 * c->n);
    ref64_soa_to_aos(c->stream, d_soa, c->d_tmp, c->n);
    NBX_HIP(c, hipMemcpyAsync(host, c->d_tmp, b, hipMemcpyDeviceToHost, c->stream));
    NBX_HIP(c, hipStreamSynchronize(c->stream));
    return NBX_OK;
}

constexpr int64_t NBX_STAGING_DOUBLES = (int64_t)4 << 20;

// staging of `doubles` doubles for frames on their way to the host
static int frame_staging(nbx_ctx* c, size_t doubles) {
    if (c->frames_doubles >= doubles) return NBX_OK;
    free_ptr(c->d_frames);
    c->d_frames = nullptr;
    c->frames_doubles = 0;
    NBX_HIP(c, hipMalloc((void**)&c->d_frames, sizeof(double) * doubles));
    c->frames_doubles = doubles;
    return NBX_OK;
}

// positions and velocities in the caller's layout: one kernel, two copies, one wait; states
// above the staging's usual 32 MiB go one after the other through d_tmp
static int download_state(nbx_ctx* c, double* u, double* v) {
    const size_t n3 = 3 * (size_t)c->n;
    if (2 * n3 > (size_t)NBX_STAGING_DOUBLES && c->frames_doubles < 2 * n3) {
        int rc = download_aos(c, c->d_x, u);
        return rc ? rc : download_aos(c, c->d_v, v);
    }
    if (int rc = frame_staging(c, 2 * n3)) return rc;
    ref64_save_frame(c->stream, c->d_x, c->d_v, c->d_frames, c->d_frames + n3, c->n);
    NBX_HIP(c, hipMemcpyAsync(u, c->d_frames, sizeof(double) * n3, hipMemcpyDeviceToHost, c->stream));
    NBX_HIP(c, hipMemcpyAsync(v, c->d_frames + n3, sizeof(double) * n3, hipMemcpyDeviceToHost, c->stream));
    NBX_HIP(c, hipStreamSynchronize(c->stream));
    return NBX_OK;
}

extern "C" int nbx_set_state(nbx_ctx* c, const double* u, const double* v) {
    if (!c) return NBX_ERR_INVALID;
    if (c->n == 0) { c->state_set = true; c->steps_taken = 0; return NBX_OK; }
    if (!u) return nbx_fail(c, NBX_ERR_INVALID, "positions are NULL");
    if (!nbx_all_finite(u, 3 * c->n) || (v && !nbx_all_finite(v, 3 * c->n)))
        return nbx_fail(c, NBX_ERR_NONFINITE, "state holds NaN or Inf");
    int rc = upload_aos(c, u, c->d_x);
    if (rc) return rc;
    if (v) {
        rc = upload_aos(c, v, c->d_v);
        if (rc) return rc;
    } else {
        ref64_fill(c->stream, c->d_v, 3 * c->n, 0.0);
    }
    c->state_set = true;
    c->accel_valid = false;
    c->nl.ready = false;
    c->every_chosen = false;
    c->steps_taken = 0;
    if ((rc = mx_reset_order(c))) return rc;
    if ((rc = reset_nosehoover(c))) return rc;
    NBX_HIP(c, hipStreamSynchronize(c->stream));   // the caller's arrays are free again
    return NBX_OK;
}

extern "C" int nbx_get_state(const nbx_ctx* c, double* u, double* v) {
    if (!c) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(const_cast<nbx_ctx*>(c), NBX_ERR_INVALID, "no state set");
    if (c->n == 0) return NBX_OK;
    nbx_ctx* m = const_cast<nbx_ctx*>(c);
    if (u && v) return download_state(m, u, v);
    if (u) return download_aos(c, c->d_x, u);
    return v ? download_aos(c, c->d_v, v) : NBX_OK;
}

extern "C" int64_t nbx_steps_taken(const nbx_ctx* c) { return c ? c->steps_taken : -1; }

// Nose-Hoover extended coordinate and its rate (the reference's u[3n+1] and v[3n+1]) at
// the state; after a mixed run the last drift has already advanced them for the next step,
// and the values before that advance are the state's
extern "C" int nbx_get_thermostat_state(const nbx_ctx* c, double* zeta, double* xi) {
    if (!c) return NBX_ERR_INVALID;
    nbx_ctx* m = const_cast<nbx_ctx*>(c);
    double h[2] = {0.0, 0.0};
    const bool ahead = c->nh_advanced && c->therm == NBX_THERM_NOSEHOOVER;
    const int slot = ahead ? NBX_SCAL_ZETA_PREV : NBX_SCAL_ZETA;
    NBX_HIP(m, hipMemcpyAsync(h, c->d_scal + slot, sizeof(h), hipMemcpyDeviceToHost,
                              c->stream));
    NBX_HIP(m, hipStreamSynchronize(c->stream));
    if (zeta) *zeta = h[0];
    if (xi) *xi = h[1];
    return NBX_OK;
}

// ---------------------------------------------------------------------------
// FP64 reference-order right-hand side
// ---------------------------------------------------------------------------

static int check_config(nbx_ctx* c) {
    if (c->sys == NBX_SYS_WATER) {
        if (!c->water_lj_set || !c->water_elec_set || !c->spcfw_set)
            return nbx_fail(c, NBX_ERR_INVALID,
                            "water needs Lennard-Jones, electrostatic and SPC/Fw parameters");
    }
    for (const nbx_term& t : c->terms)
        if ((t.kind == NBX_TERM_ELEC || t.kind == NBX_TERM_RF) && !c->has_q)
            return nbx_fail(c, NBX_ERR_INVALID, "electrostatics needs charges");
    return NBX_OK;
}

// the pair kernel's form of a term; false for the terms with kernels of their own
// (magnetic dipoles, gravity of many bodies)
static bool ref_pair_term(const nbx_ctx* c, const nbx_term& t, ref64_term* out) {
    if (t.kind == NBX_TERM_MAG || (t.kind == NBX_TERM_GRAV && c->n > NBX_REF_GRAV_WAVES)) return false;
    ref64_term r{};
    r.kind = t.kind;
    for (int k = 0; k < 4; ++k) r.p[k] = t.p[k];
    const int water = c->sys == NBX_SYS_WATER;
    // water's Lennard-Jones: O atoms only, partners = O atoms (src/nbody_to_ode.jl:302-314)
    r.istride = r.jstride = water && t.kind == NBX_TERM_LJ ? 3 : 1;
    r.nj = c->n / r.jstride;
    r.water = water && t.kind != NBX_TERM_LJ;
    r.filter = ref64_filters(r, c->bc);
    *out = r;
    return true;
}

template <class T>
static int ensure(nbx_ctx* c, T** p, size_t count) {
    if (!*p) NBX_HIP(c, hipMalloc((void**)p, sizeof(T) * std::max<size_t>(count, 1)));
    return NBX_OK;
}

// box fractions of x into the given set when a term filters its sources with them
static int ref_fractions(nbx_ctx* c, const double* x, int set) {
    bool any = false;
    ref64_term r;
    if (c->sys == NBX_SYS_WATER) {
        for (const nbx_term* t : {&c->water_elec, &c->water_lj})
            any = any || (t->kind && ref_pair_term(c, *t, &r) && r.filter);
    }
    for (const nbx_term& t : c->terms) any = any || (ref_pair_term(c, t, &r) && r.filter);
    if (!any) return NBX_OK;
    if (int rc = ensure(c, &c->d_frac, 2 * (size_t)c->n)) return rc;
    ref64_fractions(c->stream, x, c->n, c->bc.b[0], c->d_frac + (size_t)set * c->n);
    return NBX_OK;
}

// one potential term's closure for atoms [ib, ie), adding into dv (SoA); set: the box
// fractions of x
static void ref_term(nbx_ctx* c, const nbx_term& t, const double* x, double* dv, int64_t ib,
                     int64_t ie, int set = 0) {
    hipStream_t s = c->stream;
    ref64_term r;
    if (ref_pair_term(c, t, &r)) {
        const int64_t first = (ib + r.istride - 1) / r.istride * r.istride;
        ref64_pairs(s, r, x, c->d_frac ? c->d_frac + (size_t)set * c->n : nullptr, c->d_ms, c->d_qs,
                    c->n, first, ie, c->bc, dv, nullptr);
    } else if (t.kind == NBX_TERM_GRAV) {
        ref64_grav(s, x, dv, c->d_ms, c->n, ib, ie, t.p[0]);
    } else if (t.kind == NBX_TERM_MAG) {
        ref64_mag(s, x, dv, c->d_ms, c->d_mm, c->n, ib, ie, t.p[0]);
    }
}

// soode_system!(dv, v, u): dv overwritten (src/nbody_to_ode.jl:474-488, :502-532)
// xi_out: where the Nose-Hoover rate goes (the context's during runs, scratch otherwise)
static int ref_rhs(nbx_ctx* c, const double* x, const double* v, double* dv, double* xi_out) {
    hipStream_t s = c->stream;
    const int64_t n = c->n;
    ref64_fill(s, dv, 3 * n, 0.0);
    if (int rc = ref_fractions(c, x, 0)) return rc;
    if (c->sys == NBX_SYS_WATER) {
        // per-atom closure order: O = (electrostatic, bond, LJ); H = (electrostatic, bond).
        // Each atom's dv only receives its own closures, so running the terms as
        // whole-array passes in that order reproduces the per-atom sums exactly.
        ref_term(c, c->water_elec, x, dv, 0, n);
        ref64_bond(s, x, dv, c->d_ms, n, 0, n, c->rOH, c->kbond);
        ref_term(c, c->water_lj, x, dv, 0, n);
        ref64_angle(s, x, dv, c->d_ms, n, 0, n / 3, c->aHOH, c->kangle);
    } else {
        for (const nbx_term& t : c->terms) ref_term(c, t, x, dv, 0, n);
    }
    const int64_t Nc = c->sys == NBX_SYS_WATER ? 2 * (n / 3) : 0;
    if (c->therm == NBX_THERM_BERENDSEN) {
        ref64_temperature(s, v, c->d_ms, n, c->kb, Nc, c->d_scal);
        ref64_berendsen(s, dv, v, n, c->d_scal, c->therm_T, 0.5 / c->therm_p);
    } else if (c->therm == NBX_THERM_NOSEHOOVER) {
        // src/thermostats.jl:116-122 (md_temperature over the n atoms, ndf = 3n - Nc)
        ref64_temperature(s, v, c->d_ms, n, c->kb, Nc, c->d_scal);
        ref64_nosehoover(s, dv, v, n, c->d_scal, xi_out, c->therm_T, c->therm_p, 3 * n - Nc);
    }
    NBX_HIP(c, hipGetLastError());
    return NBX_OK;
}

// Scratch triple for calls that must not touch the context state (kept with the context)
struct scratch3 {
    double *x = nullptr, *v = nullptr, *dv = nullptr;
};

static int alloc_scratch(nbx_ctx* c, scratch3& s) {
    const size_t n3 = 3 * (size_t)c->n;
    if (int rc = ensure(c, &c->d_rhs, 3 * n3)) return rc;
    s.x = c->d_rhs;
    s.v = c->d_rhs + n3;
    s.dv = c->d_rhs + 2 * n3;
    return NBX_OK;
}

extern "C" int nbx_rhs(nbx_ctx* c, const double* u, const double* v, double* dv) {
    if (!c) return NBX_ERR_INVALID;
    if (c->n == 0) return NBX_OK;
    if (!u || !dv) return nbx_fail(c, NBX_ERR_INVALID, "u and dv are required");
    int rc = check_config(c);
    if (rc) return rc;
    if (!nbx_all_finite(u, 3 * c->n)) return nbx_fail(c, NBX_ERR_NONFINITE, "u holds NaN or Inf");
    if ((c->therm == NBX_THERM_BERENDSEN || c->therm == NBX_THERM_NOSEHOOVER) && !v)
        return nbx_fail(c, NBX_ERR_INVALID, "the Berendsen / Nose-Hoover term needs v");
    scratch3 s;
    if ((rc = alloc_scratch(c, s))) return rc;
    if ((rc = upload_aos(c, u, s.x))) return rc;
    // v enters through the thermostat terms only
    if (c->therm == NBX_THERM_BERENDSEN || c->therm == NBX_THERM_NOSEHOOVER)
        if ((rc = upload_aos(c, v, s.v))) return rc;
    if ((rc = ref_rhs(c, s.x, s.v, s.dv, c->d_scal + NBX_SCAL_XI_SCRATCH))) return rc;
    return download_aos(c, s.dv, dv);
}

extern "C" int nbx_accelerations(nbx_ctx* c, int32_t term, const double* u, int64_t i_begin,
                                 int64_t i_end, double* dv) {
    if (!c) return NBX_ERR_INVALID;
    if (!u || !dv) return nbx_fail(c, NBX_ERR_INVALID, "u and dv are required");
    if (i_begin < 0 || i_end > c->n || i_begin > i_end)
        return nbx_fail(c, NBX_ERR_BOUNDS,
                        "atom range [" + std::to_string(i_begin) + ", " + std::to_string(i_end) +
                            ") outside 0.." + std::to_string(c->n));
    const int nterms = c->sys == NBX_SYS_WATER ? 4 : (int)c->terms.size();
    if (term < 0 || term >= nterms)
        return nbx_fail(c, NBX_ERR_BOUNDS, "potential term " + std::to_string(term) + " not defined");
    if (c->n == 0 || i_begin == i_end) return NBX_OK;
    if (c->sys == NBX_SYS_WATER) {
        if ((term == 0 && !c->water_elec_set) || (term == 1 && !c->water_lj_set) ||
            (term >= 2 && !c->spcfw_set))
            return nbx_fail(c, NBX_ERR_INVALID, "water term not configured");
    }
    if (!nbx_all_finite(u, 3 * c->n)) return nbx_fail(c, NBX_ERR_NONFINITE, "u holds NaN or Inf");
    scratch3 s;
    int rc;
    if ((rc = alloc_scratch(c, s))) return rc;
    if ((rc = upload_aos(c, u, s.x))) return rc;
    if ((rc = upload_aos(c, dv, s.dv))) return rc;
    if ((rc = ref_fractions(c, s.x, 0))) return rc;
    if (c->sys == NBX_SYS_WATER) {
        if (term == 0) ref_term(c, c->water_elec, s.x, s.dv, i_begin, i_end);
        else if (term == 1) ref_term(c, c->water_lj, s.x, s.dv, i_begin, i_end);
        else if (term == 2) ref64_bond(c->stream, s.x, s.dv, c->d_ms, c->n, i_begin, i_end, c->rOH,
                                       c->kbond);
        else {
            // group closure over molecules whose O index lies in [i_begin, i_end)
            ref64_angle(c->stream, s.x, s.dv, c->d_ms, c->n, (i_begin + 2) / 3, (i_end + 2) / 3,
                        c->aHOH, c->kangle);
        }
    } else {
        ref_term(c, c->terms[term], s.x, s.dv, i_begin, i_end);
    }
    NBX_HIP(c, hipGetLastError());
    return download_aos(c, s.dv, dv);
}

// ---------------------------------------------------------------------------
// Velocity Verlet
// ---------------------------------------------------------------------------

static int save_frame(nbx_ctx* c, int64_t f, double* uf, double* vf) {
    const int64_t n3 = 3 * c->n;
    return download_state(c, uf + f * n3, vf + f * n3);
}

// Frames of an FP64 run: collected on the device in the caller's layout and copied to the
// host many at a time (32 MiB of both arrays at most, one frame at least), not one by one with
// two synchronisations each
struct frame_sink {
    nbx_ctx* c;
    double *uf, *vf;
    int64_t cap = 0, pending = 0, done = 0;

    int open(int64_t frames) {
        const int64_t n3 = 3 * c->n;
        cap = std::max<int64_t>(1, std::min<int64_t>(frames, NBX_STAGING_DOUBLES / 2 / n3));
        return frame_staging(c, 2 * (size_t)(cap * n3));
    }
    int add(const double* x, const double* v) {
        const int64_t n3 = 3 * c->n;
        ref64_save_frame(c->stream, x, v, c->d_frames + pending * n3,
                         c->d_frames + (cap + pending) * n3, c->n);
        return ++pending == cap ? flush() : NBX_OK;
    }
    int flush() {
        const int64_t n3 = 3 * c->n;
        if (pending == 0) return NBX_OK;
        const size_t bytes = sizeof(double) * (size_t)(pending * n3);
        NBX_HIP(c, hipMemcpyAsync(uf + done * n3, c->d_frames, bytes, hipMemcpyDeviceToHost, c->stream));
        NBX_HIP(c, hipMemcpyAsync(vf + done * n3, c->d_frames + cap * n3, bytes, hipMemcpyDeviceToHost,
                                  c->stream));
        NBX_HIP(c, hipStreamSynchronize(c->stream));
        done += pending;
        pending = 0;
        return NBX_OK;
    }
};

// Runs whose steps end inside the kernel that completes the accelerations: water, and
// potential systems whose last term is a pair term, with a thermostat that acts per atom or
// through the temperature of the half-kicked velocities (Nose-Hoover advances its own
// coordinate between the pieces)
static bool ref_fuses(const nbx_ctx* c) {
    if (c->therm == NBX_THERM_NOSEHOOVER) return false;
    if (c->sys == NBX_SYS_WATER) return true;
    ref64_term r;
    return !c->terms.empty() && ref_pair_term(c, c->terms.back(), &r);
}

// nsteps of such a run from (d_x, d_v, d_a): positions alternate between d_x and d_x2
// (a kernel that writes the next positions cannot overwrite those that other targets still
// read), and end in d_x.  Launches per step: one (one more per further potential, two for
// water, one more for Berendsen's temperature) instead of a fill, one per term, kick, drift
// and thermostat.
static int ref_vv_fused(nbx_ctx* c, double dt, int64_t nsteps, uint64_t seed, int64_t save_every,
                        frame_sink* frames) {
    hipStream_t s = c->stream;
    const int64_t n = c->n;
    const bool water = c->sys == NBX_SYS_WATER;
    int rc;
    if ((rc = ensure(c, &c->d_x2, 3 * (size_t)n))) return rc;
    if (water && (rc = ensure(c, &c->d_water, 6 * (size_t)n))) return rc;
    ref64_term last{}, lj{};
    bool filter = false;
    if (water) {
        if (!ref_pair_term(c, c->water_elec, &last) || !ref_pair_term(c, c->water_lj, &lj))
            return nbx_fail(c, NBX_ERR_INVALID, "water takes Lennard-Jones and electrostatics");
        filter = last.filter = lj.filter = last.filter && lj.filter;
    } else {
        (void)ref_pair_term(c, c->terms.back(), &last);
        ref64_term r;
        for (const nbx_term& t : c->terms) filter = filter || (ref_pair_term(c, t, &r) && r.filter);
    }
    if (filter && (rc = ensure(c, &c->d_frac, 2 * (size_t)n))) return rc;
    double* const xb[2] = {c->d_x, c->d_x2};
    float4* const fb[2] = {filter ? c->d_frac : nullptr, filter ? c->d_frac + n : nullptr};
    ref64_step st{};
    st.a = c->d_a;
    st.v = c->d_v;
    st.vh = c->d_vh;
    st.d_T = c->d_scal;
    st.dt = dt;
    st.invL = filter ? 1.0 / c->bc.b[0] : 0.0;
    st.kb = c->kb;
    st.T = c->therm_T;
    st.therm = c->therm;
    st.seed = seed;
    if (c->therm == NBX_THERM_LANGEVIN) {
        st.c1 = std::exp(-c->therm_p * (0.5 * dt));
        st.c2 = std::sqrt(1.0 - st.c1 * st.c1);
    } else if (c->therm == NBX_THERM_ANDERSEN) {
        st.prob = c->therm_p * dt;
    } else if (c->therm == NBX_THERM_BERENDSEN) {
        st.gamma = 0.5 / c->therm_p;
    }
    const int64_t Nc = water ? 2 * (n / 3) : 0;
    const int64_t step0 = c->steps_taken;
    if (c->therm == NBX_THERM_LANGEVIN)
        ref64_langevin_half(s, c->d_v, c->d_ms, n, c->kb, c->therm_T, c->therm_p, dt, seed, step0 + 1,
                            NBX_RNG_LANGEVIN_A);
    ref64_drift(s, xb[0], xb[1], c->d_v, c->d_a, c->d_vh, n, dt, fb[1], c->bc.b[0]);
    for (int64_t k = 1; k <= nsteps; ++k) {
        const int cur = (int)(k & 1);
        if (c->therm == NBX_THERM_BERENDSEN)
            ref64_temperature(s, c->d_vh, c->d_ms, n, c->kb, Nc, c->d_scal);
        st.x_in = xb[cur];
        st.x_out = xb[cur ^ 1];
        st.frac_out = fb[cur ^ 1];
        st.step = step0 + k;
        st.drift = k < nsteps;
        if (water) {
            ref64_water_step(s, last, lj, fb[cur], c->d_ms, c->d_qs, n, c->bc, c->d_water,
                             c->d_water + 3 * n, c->rOH, c->kbond, c->aHOH, c->kangle, st);
        } else {
            if (c->terms.size() > 1) {
                ref64_fill(s, c->d_a, 3 * n, 0.0);
                for (size_t q = 0; q + 1 < c->terms.size(); ++q)
                    ref_term(c, c->terms[q], xb[cur], c->d_a, 0, n, cur);
                st.a_in = c->d_a;
            }
            ref64_pairs(s, last, xb[cur], fb[cur], c->d_ms, c->d_qs, n, 0, n, c->bc, nullptr, &st);
        }
        NBX_HIP(c, hipGetLastError());
        c->steps_taken = step0 + k;
        if (frames && k % save_every == 0 && (rc = frames->add(xb[cur], c->d_v))) return rc;
    }
    if (nsteps & 1)
        NBX_HIP(c, hipMemcpyAsync(c->d_x, c->d_x2, sizeof(double) * 3 * (size_t)n,
                                  hipMemcpyDeviceToDevice, s));
    return NBX_OK;
}

// the small systems whose whole run is one workgroup's (ref64_small_run)
static int ref_vv_small(nbx_ctx* c, double dt, int64_t nsteps, int64_t save_every,
                        frame_sink* frames) {
    std::vector<ref64_term> terms;
    for (const nbx_term& t : c->terms) {
        ref64_term r{};
        if (!ref_pair_term(c, t, &r)) {   // magnetic dipoles
            r.kind = t.kind;
            for (int k = 0; k < 4; ++k) r.p[k] = t.p[k];
        }
        terms.push_back(r);
    }
    const int64_t n3 = 3 * c->n, step0 = c->steps_taken;
    int64_t done = 0;
    while (done < nsteps) {
        // a launch ends after 20,000 steps (some 10 ms), or when the frames fill their buffer
        int64_t m = std::min<int64_t>(nsteps - done, 20000);
        if (frames) m = std::min(m, (frames->cap - frames->pending) * save_every - done % save_every);
        double* const u = frames ? c->d_frames + frames->pending * n3 : nullptr;
        double* const v = frames ? c->d_frames + (frames->cap + frames->pending) * n3 : nullptr;
        ref64_small_run(c->stream, (int)c->n, c->d_x, c->d_v, c->d_a, c->d_ms, c->d_qs,
                        c->mm_set ? c->d_mm : nullptr, terms.data(), (int)terms.size(), c->bc, dt, done,
                        m, frames ? save_every : 0, u, v);
        NBX_HIP(c, hipGetLastError());
        if (frames) {
            frames->pending += (done + m) / save_every - done / save_every;
            if (frames->pending == frames->cap)
                if (int rc = frames->flush()) return rc;
        }
        done += m;
        c->steps_taken = step0 + done;
    }
    return NBX_OK;
}

static int ref_vv(nbx_ctx* c, double dt, int64_t nsteps, uint64_t seed, int64_t save_every,
                  double* uf, double* vf) {
    hipStream_t s = c->stream;
    const int64_t n = c->n;
    int rc;
    frame_sink sink{c, uf, vf};
    frame_sink* const frames = save_every > 0 ? &sink : nullptr;
    if (frames && ((rc = sink.open(1 + nsteps / save_every)) || (rc = sink.add(c->d_x, c->d_v)))) return rc;
    if (c->nh_advanced && c->therm == NBX_THERM_NOSEHOOVER) {
        // a mixed run before this one left zeta and xi advanced for the next step: back to
        // the state's values, which this path advances at its first drift
        NBX_HIP(c, hipMemcpyAsync(c->d_scal + NBX_SCAL_ZETA, c->d_scal + NBX_SCAL_ZETA_PREV,
                                  2 * sizeof(double), hipMemcpyDeviceToDevice, s));
    }
    c->nh_advanced = false;
    if (!c->accel_valid) {
        if ((rc = ref_rhs(c, c->d_x, c->d_v, c->d_a, c->d_scal + NBX_SCAL_XI))) return rc;
        c->accel_valid = true;
    }
    const int water = c->sys == NBX_SYS_WATER;
    if (nsteps > 0 && !water && c->n <= NBX_REF_SMALL && c->therm == NBX_THERM_NONE &&
        !c->terms.empty()) {
        if ((rc = ref_vv_small(c, dt, nsteps, save_every, frames))) return rc;
        return frames ? sink.flush() : NBX_OK;
    }
    if (nsteps > 0 && ref_fuses(c)) {
        if ((rc = ref_vv_fused(c, dt, nsteps, seed, save_every, frames))) return rc;
        return frames ? sink.flush() : NBX_OK;
    }
    for (int64_t k = 1; k <= nsteps; ++k) {
        const int64_t step = c->steps_taken + 1;
        if (c->therm == NBX_THERM_LANGEVIN)
            ref64_langevin_half(s, c->d_v, c->d_ms, n, c->kb, c->therm_T, c->therm_p, dt, seed,
                                step, NBX_RNG_LANGEVIN_A);
        ref64_drift(s, c->d_x, c->d_x, c->d_v, c->d_a, c->d_vh, n, dt, nullptr, 1.0);
        if (c->therm == NBX_THERM_NOSEHOOVER) ref64_nh_drift(s, c->d_scal, dt);
        if ((rc = ref_rhs(c, c->d_x, c->d_vh, c->d_a, c->d_scal + NBX_SCAL_XI))) return rc;
        ref64_kick(s, c->d_v, c->d_vh, c->d_a, n, dt);
        if (c->therm == NBX_THERM_LANGEVIN)
            ref64_langevin_half(s, c->d_v, c->d_ms, n, c->kb, c->therm_T, c->therm_p, dt, seed,
                                step, NBX_RNG_LANGEVIN_B);
        if (c->therm == NBX_THERM_ANDERSEN)
            ref64_andersen(s, c->d_v, c->d_ms, n, water, c->kb, c->therm_T, c->therm_p * dt, seed,
                           step);
        NBX_HIP(c, hipGetLastError());
        c->steps_taken = step;
        if (frames && k % save_every == 0 && (rc = sink.add(c->d_x, c->d_v))) return rc;
    }
    return frames ? sink.flush() : NBX_OK;
}

int mx_vv(nbx_ctx* c, double dt, int64_t nsteps, uint64_t seed, int64_t save_every, double* uf,
          double* vf, int64_t* nframes);
int mx_supported(nbx_ctx* c, std::string* why);

// The end of a run: waits for it and reports a state that became NaN or Inf.  The flag is zero
// until a check sets it, and is cleared when it has been reported.
static int check_finite_state(nbx_ctx* c) {
    int* d_flag = reinterpret_cast<int*>(c->d_scal + 8);
    ref64_check_finite(c->stream, c->d_x, c->d_v, 3 * c->n, d_flag);
    int h = 0;
    NBX_HIP(c, hipMemcpyAsync(&h, d_flag, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    NBX_HIP(c, hipStreamSynchronize(c->stream));
    if (!h) return NBX_OK;
    NBX_HIP(c, hipMemsetAsync(d_flag, 0, sizeof(int), c->stream));
    return nbx_fail(c, NBX_ERR_NONFINITE, "the state became NaN or Inf during the run");
}

extern "C" int nbx_vv_run(nbx_ctx* c, double dt, int64_t nsteps, uint64_t seed,
                          int64_t save_every, double* u_frames, double* v_frames) {
    if (!c) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    if (!(dt > 0.0) || !std::isfinite(dt)) return nbx_fail(c, NBX_ERR_INVALID, "dt must be > 0");
    if (nsteps < 0) return nbx_fail(c, NBX_ERR_INVALID, "nsteps < 0");
    if (save_every > 0 && (!u_frames || !v_frames))
        return nbx_fail(c, NBX_ERR_INVALID, "frames requested but frame buffers are NULL");
    int rc = check_config(c);
    if (rc) return rc;
    if (c->n == 0) { c->steps_taken += nsteps; return NBX_OK; }
    if (c->prec == NBX_PREC_MIXED) {
        int64_t nframes = 0;
        if (save_every > 0) {
            if ((rc = save_frame(c, 0, u_frames, v_frames))) return rc;
            nframes = 1;
        }
        std::string why;
        if (!mx_supported(c, &why)) return nbx_fail(c, NBX_ERR_UNSUPPORTED, why);
        rc = mx_vv(c, dt, nsteps, seed, save_every, u_frames, v_frames, &nframes);
    } else {
        rc = ref_vv(c, dt, nsteps, seed, save_every, u_frames, v_frames);
    }
    if (rc) return rc;
    return check_finite_state(c);
}

// ---------------------------------------------------------------------------
// Euler-Maruyama (the reference's Langevin SDE path)
// ---------------------------------------------------------------------------

static int ref_em(nbx_ctx* c, double dt, int64_t nsteps, uint64_t seed, int64_t save_every,
                  double* uf, double* vf) {
    hipStream_t s = c->stream;
    int rc;
    frame_sink sink{c, uf, vf};
    if (save_every > 0 &&
        ((rc = sink.open(1 + nsteps / save_every)) || (rc = sink.add(c->d_x, c->d_v)))) return rc;
    if (!c->accel_valid) {
        if ((rc = ref_rhs(c, c->d_x, c->d_v, c->d_a, c->d_scal + NBX_SCAL_XI))) return rc;
        c->accel_valid = true;
    }
    const double sigma = std::sqrt(2 * c->therm_p * c->kb * c->therm_T / c->h_ms[0]);
    for (int64_t k = 1; k <= nsteps; ++k) {
        const int64_t step = c->steps_taken + 1;
        ref64_em(s, c->d_x, c->d_v, c->d_a, c->n, dt, c->therm_p, sigma, seed, step);
        if ((rc = ref_rhs(c, c->d_x, c->d_v, c->d_a, c->d_scal + NBX_SCAL_XI))) return rc;
        NBX_HIP(c, hipGetLastError());
        c->steps_taken = step;
        if (save_every > 0 && k % save_every == 0 && (rc = sink.add(c->d_x, c->d_v))) return rc;
    }
    return save_every > 0 ? sink.flush() : NBX_OK;
}

extern "C" int nbx_em_run(nbx_ctx* c, double dt, int64_t nsteps, uint64_t seed,
                          int64_t save_every, double* u_frames, double* v_frames) {
    if (!c) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    if (!(dt > 0.0) || !std::isfinite(dt)) return nbx_fail(c, NBX_ERR_INVALID, "dt must be > 0");
    if (nsteps < 0) return nbx_fail(c, NBX_ERR_INVALID, "nsteps < 0");
    if (save_every > 0 && (!u_frames || !v_frames))
        return nbx_fail(c, NBX_ERR_INVALID, "frames requested but frame buffers are NULL");
    if (c->therm != NBX_THERM_LANGEVIN)
        return nbx_fail(c, NBX_ERR_INVALID,
                        "Euler-Maruyama integrates the Langevin SDE: set the Langevin thermostat");
    if (c->sys == NBX_SYS_WATER)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED,
                        "the Langevin SDE is provided for potential systems only");
    int rc = check_config(c);
    if (rc) return rc;
    if (c->n == 0) { c->steps_taken += nsteps; return NBX_OK; }
    if (c->prec == NBX_PREC_MIXED) {
        int64_t nframes = 0;
        if (save_every > 0) {
            if ((rc = save_frame(c, 0, u_frames, v_frames))) return rc;
            nframes = 1;
        }
        std::string why;
        if (!mx_supported(c, &why)) return nbx_fail(c, NBX_ERR_UNSUPPORTED, why);
        c->em = 1;
        rc = mx_vv(c, dt, nsteps, seed, save_every, u_frames, v_frames, &nframes);
        c->em = 0;
    } else {
        rc = ref_em(c, dt, nsteps, seed, save_every, u_frames, v_frames);
    }
    if (rc) return rc;
    return check_finite_state(c);
}

// ---------------------------------------------------------------------------
// Energies, temperature, RDF
// ---------------------------------------------------------------------------

extern "C" int nbx_energies(nbx_ctx* c, double* ke, double* pe, double* pe_grav) {
    if (!c) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    int rc = check_config(c);
    if (rc) return rc;
    hipStream_t s = c->stream;
    const int64_t n = c->n;
    // every sum is enqueued, then all of them are read at once: out[0] the kinetic energy,
    // then a slot per potential term (the scalars up to the finite flag hold few: more
    // terms are read in several rounds)
    double* out = c->d_scal + 1;
    constexpr int SLOTS = 7;   // d_scal[1..7]
    double h_ke = 0.0, h_pe = 0.0, grav = 0.0;
    struct slot { int at; double factor; double* into; };
    std::vector<slot> want;
    int used = 1;
    const auto collect = [&]() -> int {
        double h[SLOTS];
        NBX_HIP(c, hipGetLastError());
        NBX_HIP(c, hipMemcpyAsync(h, out, sizeof(double) * (size_t)used, hipMemcpyDeviceToHost, s));
        NBX_HIP(c, hipStreamSynchronize(s));
        for (const slot& w : want) *w.into += w.factor * h[w.at];
        want.clear();
        used = 1;
        return NBX_OK;
    };
    const auto take = [&](int count) -> int { return used + count > SLOTS ? collect() : NBX_OK; };
    ref64_ke kin{c->d_v, c->d_ms, out};   // the first pair sum's launch adds it
    const bool pairs = c->sys == NBX_SYS_WATER ||
                       std::any_of(c->terms.begin(), c->terms.end(), [](const nbx_term& t) {
                           return t.kind == NBX_TERM_LJ || t.kind == NBX_TERM_ELEC ||
                                  t.kind == NBX_TERM_RF;
                       });
    if (!pairs || n <= 0) {
        ref64_kinetic(s, c->d_v, c->d_ms, n, out);
        kin.out = nullptr;
    }
    want.push_back({0, 1.0, &h_ke});
    const auto lj_term = [&](const nbx_term& t, int stride, int64_t nj) {
        ref64_lj_pe(s, c->d_x, n, stride, nj, t.p[1], t.p[2], c->bc, c->d_red, out + used, kin);
        kin.out = nullptr;
        want.push_back({used++, 4.0 * t.p[0], &h_pe});
    };
    const auto elec_term = [&](const nbx_term& t, int water) {
        ref64_elec_pe(s, c->d_x, c->d_qs, n, water, t.p[1], t.kind == NBX_TERM_RF, t.p[2], c->bc,
                      c->d_red, out + used, kin);
        kin.out = nullptr;
        want.push_back({used++, t.p[0], &h_pe});
    };
    if (n > 0 && c->sys == NBX_SYS_WATER) {
        // src/nbody_simulation_result.jl:266-291: LJ (O atoms), electrostatic, bonds, angles
        lj_term(c->water_lj, 3, n / 3);
        elec_term(c->water_elec, 1);
        ref64_bonded_pe(s, c->d_x, n, c->rOH, c->kbond, c->aHOH, c->kangle, c->d_tmp, out + used);
        want.push_back({used++, 1.0, &h_pe});
        want.push_back({used++, 1.0, &h_pe});
    } else if (n > 0) {
        // src/nbody_simulation_result.jl:239-264: Lennard-Jones first, then electrostatics;
        // gravity has no potential energy there and is reported separately
        for (const nbx_term& t : c->terms) {
            if (t.kind != NBX_TERM_LJ) continue;
            if ((rc = take(1))) return rc;
            lj_term(t, 1, n);
        }
        for (const nbx_term& t : c->terms) {
            if (t.kind != NBX_TERM_ELEC && t.kind != NBX_TERM_RF) continue;
            if ((rc = take(1))) return rc;
            elec_term(t, 0);
        }
        for (const nbx_term& t : c->terms) {
            if (t.kind != NBX_TERM_GRAV) continue;
            if ((rc = take(1))) return rc;
            ref64_grav_pe(s, c->d_x, c->d_ms, n, t.p[0], c->d_tmp, out + used);
            want.push_back({used++, 1.0, &grav});
        }
    }
    if ((rc = collect())) return rc;
    if (ke) *ke = h_ke;
    if (pe) *pe = h_pe;
    if (pe_grav) *pe_grav = grav;
    return NBX_OK;
}

extern "C" int nbx_temperature(nbx_ctx* c, double* T) {
    if (!c || !T) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    const int64_t Nc = c->sys == NBX_SYS_WATER ? 2 * (c->n / 3) : 0;
    if (c->n == 0) { *T = NAN; return NBX_OK; }
    ref64_temperature(c->stream, c->d_v, c->d_ms, c->n, c->kb, Nc, c->d_scal + 9);
    NBX_HIP(c, hipMemcpyAsync(T, c->d_scal + 9, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    NBX_HIP(c, hipStreamSynchronize(c->stream));
    return NBX_OK;
}

// g(r) and bin centres from the counts of bins 1..maxbin (src/nbody_simulation_result.jl:
// 695-706).  counts may alias gr: count k is read before g k is written.
static void rdf_normalize(const unsigned long long* counts, int64_t nframes, int64_t nj,
                          double L, int64_t maxbin, double* rs, double* gr) {
    const double dr = L / (double)maxbin;
    const double cc = 4.0 / 3.0 * 3.141592653589793 * (double)nj / (L * L * L);
    for (int64_t bin = 1; bin <= maxbin; ++bin) {
        unsigned long long cnt;
        std::memcpy(&cnt, counts + (bin - 1), sizeof(cnt));
        double rl = (double)(bin - 1) * dr;
        double ru = rl + dr;
        double nideal = cc * (ru * ru * ru - rl * rl * rl);
        gr[bin - 1] = ((double)cnt / (double)(nframes * nj)) / nideal;
        rs[bin - 1] = rl + dr / 2.0;
    }
}

extern "C" int nbx_rdf(nbx_ctx* c, const double* frames, int64_t nframes, int64_t maxbin,
                       double* rs, double* gr) {
    if (!c) return NBX_ERR_INVALID;
    if (c->bc.kind != NBX_BC_CUBIC)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED, "rdf needs CubicPeriodicBoundaryConditions");
    if (!frames || nframes <= 0 || maxbin <= 0 || !rs || !gr)
        return nbx_fail(c, NBX_ERR_INVALID, "rdf: frames, maxbin, rs and gr are required");
    const int water = c->sys == NBX_SYS_WATER;
    const int jstride = water ? 3 : 1;
    const int64_t nj = water ? c->n / 3 : c->n;
    const double L = c->bc.b[0];
    // frames go over in batches of at most 32 MiB (one frame at least), each batch one copy
    // and one launch; the workspace stays with the context
    const int64_t n3 = 3 * c->n;
    const int64_t batch = std::max<int64_t>(1, std::min<int64_t>(nframes, ((int64_t)4 << 20) / std::max<int64_t>(n3, 1)));
    const size_t work = (size_t)(batch * n3 + maxbin + 1);
    if (c->rdf_work_doubles < work) {
        free_ptr(c->d_rdf_work);
        c->d_rdf_work = nullptr;
        c->rdf_work_doubles = 0;
        NBX_HIP(c, hipMalloc((void**)&c->d_rdf_work, sizeof(double) * work));
        c->rdf_work_doubles = work;
    }
    auto* d_hist = reinterpret_cast<unsigned long long*>(c->d_rdf_work + batch * n3);
    ref64_zero_u64(c->stream, d_hist, maxbin + 1);
    for (int64_t t = 0; t < nframes; t += batch) {
        const int64_t k = std::min(batch, nframes - t);
        if (n3 > 0)
            NBX_HIP(c, hipMemcpyAsync(c->d_rdf_work, frames + t * n3, sizeof(double) * (size_t)(k * n3),
                                      hipMemcpyHostToDevice, c->stream));
        ref64_rdf_hist(c->stream, c->d_rdf_work, k, c->n, jstride, nj, L, maxbin, d_hist);
    }
    NBX_HIP(c, hipGetLastError());
    std::vector<unsigned long long> h((size_t)maxbin + 1);
    NBX_HIP(c, hipMemcpyAsync(h.data(), d_hist, sizeof(unsigned long long) * h.size(),
                              hipMemcpyDeviceToHost, c->stream));
    NBX_HIP(c, hipStreamSynchronize(c->stream));
    rdf_normalize(h.data() + 1, nframes, nj, L, maxbin, rs, gr);
    return NBX_OK;
}

extern "C" int nbx_rdf_noalloc(nbx_ctx* c, const double* frames, int64_t nframes,
                               int64_t maxbin, double* rs, double* gr) {
    if (!c) return NBX_ERR_INVALID;
    if (c->bc.kind != NBX_BC_CUBIC)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED, "rdf needs CubicPeriodicBoundaryConditions");
    if (!frames || nframes <= 0 || maxbin <= 0 || !rs || !gr)
        return nbx_fail(c, NBX_ERR_INVALID, "rdf: frames, maxbin, rs and gr are required");
    if (maxbin > NBX_RDF_NOALLOC_MAXBIN)
        return nbx_fail(c, NBX_ERR_CAPACITY,
                        "nbx_rdf_noalloc: maxbin " + std::to_string(maxbin) + " exceeds " +
                            std::to_string(NBX_RDF_NOALLOC_MAXBIN) +
                            ", the size of its fixed histogram (use nbx_rdf)");
    if (!c->d_rdf_hist) return nbx_fail(c, NBX_ERR_DEVICE, "rdf histogram address not set up");
    const int water = c->sys == NBX_SYS_WATER;
    const int jstride = water ? 3 : 1;
    const int64_t nj = water ? c->n / 3 : c->n;
    const double L = c->bc.b[0];
    unsigned long long* hist = c->d_rdf_hist;
    ref64_zero_u64(c->stream, hist, maxbin + 1);
    const size_t b = sizeof(double) * (size_t)(3 * c->n);
    for (int64_t t = 0; t < nframes; ++t) {
        NBX_HIP(c, hipMemcpyAsync(c->d_tmp, frames + t * 3 * c->n, b, hipMemcpyHostToDevice,
                                  c->stream));
        ref64_rdf_hist(c->stream, c->d_tmp, 1, c->n, jstride, nj, L, maxbin, hist);
    }
    NBX_HIP(c, hipGetLastError());
    // the counts of bins 1..maxbin land in gr (8 bytes each) and are turned into g(r) there,
    // so no host buffer is allocated either
    static_assert(sizeof(double) == sizeof(unsigned long long), "bin counts are 8 bytes");
    NBX_HIP(c, hipMemcpyAsync(gr, hist + 1, sizeof(unsigned long long) * (size_t)maxbin,
                              hipMemcpyDeviceToHost, c->stream));
    NBX_HIP(c, hipStreamSynchronize(c->stream));
    rdf_normalize(reinterpret_cast<const unsigned long long*>(gr), nframes, nj, L, maxbin, rs, gr);
    return NBX_OK;
}

extern "C" int nbx_time_force_kernel(nbx_ctx* c, int32_t iters, double* avg_ms,
                                     const char** name) {
    if (!c || !avg_ms) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    if (iters <= 0) return nbx_fail(c, NBX_ERR_INVALID, "iters must be > 0");
    if (c->prec != NBX_PREC_MIXED)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED, "kernel timing is provided for the mixed path");
    return mx_time_force(c, iters, avg_ms, name);
}

extern "C" int nbx_set_kernel_timing(nbx_ctx* c, int32_t enable) {
    if (!c) return NBX_ERR_INVALID;
    c->kt_on = enable != 0;
    c->kt_sum_ms = 0.0;
    c->kt_launches = 0;
    c->kt_used = 0;
    return NBX_OK;
}

extern "C" int nbx_get_kernel_timing(nbx_ctx* c, double* avg_ms, int64_t* launches,
                                     const char** name) {
    if (!c || !avg_ms || !launches) return NBX_ERR_INVALID;
    *launches = c->kt_launches;
    *avg_ms = c->kt_launches > 0 ? c->kt_sum_ms / (double)c->kt_launches : 0.0;
    if (name) *name = mx_force_kernel_name(c);
    return NBX_OK;
}

extern "C" int nbx_copy_probe(nbx_ctx* c, int64_t bytes, int32_t iters, double* avg_ms) {
    if (!c || !avg_ms) return NBX_ERR_INVALID;
    if (bytes < 16 || iters <= 0) return nbx_fail(c, NBX_ERR_INVALID, "bytes >= 16 and iters > 0 required");
    return mx_copy_probe(c, bytes, iters, avg_ms);
}

extern "C" int nbx_valu_probe(nbx_ctx* c, int32_t kind, int32_t reps, double* rate) {
    if (!c || !rate) return NBX_ERR_INVALID;
    if (kind < 0 || kind > 2 || reps <= 0)
        return nbx_fail(c, NBX_ERR_INVALID, "kind 0..2 and reps > 0 required");
    return mx_valu_probe(c, kind, reps, rate);
}

static int learn_ready(nbx_ctx* c) {
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    if (c->prec != NBX_PREC_MIXED)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED, "the learned stride runs on the mixed-precision path");
    return NBX_OK;
}

extern "C" int nbx_features(nbx_ctx* c, double* feats, double* frames) {
    if (!c) return NBX_ERR_INVALID;
    int rc;
    if ((rc = learn_ready(c))) return rc;
    return mx_features(c, feats, frames);
}

extern "C" int nbx_learn_energy(nbx_ctx* c, double* ke, double* pe) {
    if (!c || !ke || !pe) return NBX_ERR_INVALID;
    int rc;
    if ((rc = learn_ready(c))) return rc;
    return mx_learn_energy(c, ke, pe);
}

extern "C" int nbx_learn_collect(nbx_ctx* c, nbx_model* m, double dt, int32_t stride,
                                 int64_t nframes, int32_t atoms_per_frame, uint64_t seed) {
    if (!c || !m) return NBX_ERR_INVALID;
    int rc;
    if ((rc = learn_ready(c))) return rc;
    if (!(dt > 0.0) || !std::isfinite(dt)) return nbx_fail(c, NBX_ERR_INVALID, "dt must be > 0");
    if (stride < 1 || stride > 64) return nbx_fail(c, NBX_ERR_INVALID, "stride must be in 1..64");
    if (nframes < 0) return nbx_fail(c, NBX_ERR_INVALID, "nframes must be >= 0");
    if (atoms_per_frame < 1 || atoms_per_frame > c->n)
        return nbx_fail(c, NBX_ERR_INVALID, "atoms_per_frame must be in 1..n");
    if (nframes == 0) return NBX_OK;
    return mx_learn_collect(c, m, dt, stride, nframes, atoms_per_frame, seed);
}

extern "C" int nbx_learned_run(nbx_ctx* c, const nbx_model* m, double dt, int32_t stride,
                               int64_t nsteps, double drift_tol, int32_t check_every,
                               double* report) {
    if (!c || !m) return NBX_ERR_INVALID;
    int rc;
    if ((rc = learn_ready(c))) return rc;
    if (!(dt > 0.0) || !std::isfinite(dt)) return nbx_fail(c, NBX_ERR_INVALID, "dt must be > 0");
    if (stride < 1 || stride > 64) return nbx_fail(c, NBX_ERR_INVALID, "stride must be in 1..64");
    if (nsteps < 0) return nbx_fail(c, NBX_ERR_INVALID, "nsteps must be >= 0");
    if (!(drift_tol > 0.0)) return nbx_fail(c, NBX_ERR_INVALID, "drift_tol must be > 0");
    if (check_every < 1) return nbx_fail(c, NBX_ERR_INVALID, "check_every must be >= 1");
    return mx_learned_run(c, m, dt, stride, nsteps, drift_tol, check_every, report);
}

extern "C" int nbx_autotune(nbx_ctx* c, double dt, int32_t trial_steps, double* out,
                            int32_t nout) {
    if (!c || (nout > 0 && !out) || nout < 0 || nout > 6) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    if (c->prec != NBX_PREC_MIXED)
        return nbx_fail(c, NBX_ERR_UNSUPPORTED, "autotuning is provided for the mixed path");
    if (!(dt > 0.0) || !std::isfinite(dt)) return nbx_fail(c, NBX_ERR_INVALID, "dt must be > 0");
    if (trial_steps < 1) return nbx_fail(c, NBX_ERR_INVALID, "trial_steps must be >= 1");
    return mx_autotune(c, dt, trial_steps, out, nout);
}

extern "C" int nbx_get_stats(nbx_ctx* c, int64_t* out, int32_t nout) {
    if (!c || !out || nout < 0 || nout > 8) return NBX_ERR_INVALID;
    int64_t v[8] = {0, c->nl.cap, c->nl.ncell, c->nl.lanes, c->graph_steps,
                    c->every_auto && c->guarded ? 1 : c->build_every, c->stale_replays,
                    c->sorts_applied};
    if (c->nl.d_flags) {
        int h[8] = {0};
        NBX_HIP(c, hipMemcpyAsync(h, c->nl.d_flags, sizeof(h), hipMemcpyDeviceToHost, c->stream));
        NBX_HIP(c, hipStreamSynchronize(c->stream));
        v[0] = h[2];
    }
    for (int k = 0; k < nout; ++k) out[k] = v[k];
    return NBX_OK;
}

extern "C" int nbx_count_pairs(nbx_ctx* c, int64_t* pairs) {
    if (!c || !pairs) return NBX_ERR_INVALID;
    if (!c->state_set) return nbx_fail(c, NBX_ERR_INVALID, "no state set");
    return mx_count_pairs(c, pairs);
}
