// C ABI of libdrifter_hip: context lifecycle, right-hand side, time stepping,
// CFL reduction and mode splitting.  Host code only; kernels live in *.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "drf_internal.hpp"
#include "lincomb.hpp"

namespace drf {
int g_rhs_per_cu[2][3][kMaxN][2] = {};
}

namespace drf {

static thread_local std::string g_last_error;

void set_error(const std::string &msg) { g_last_error = msg; }

drf_status fail(drf_status code, const std::string &msg)
{
    g_last_error = msg;
    return code;
}

} // namespace drf

using namespace drf;

namespace {

#define DRF_REQUIRE(cond, code, msg)                                                         \
    do {                                                                                     \
        if (!(cond))                                                                         \
            return ::drf::fail((code), (msg));                                               \
    } while (0)

// Device entry points run on the caller's stream exactly as given; NULL is
// HIP's null (default) stream, as everywhere in the HIP API.
hipStream_t pick_stream(drf_ctx *c, void *s)
{
    (void)c;
    return (hipStream_t)s;
}

size_t elem_size(const drf_ctx *c) { return c->precision == DRF_PREC_FP64 ? 8 : 4; }

int64_t state_len(const drf_ctx *c, int layout = DRF_LAYOUT_PACKED)
{
    return layout_state_len(layout, c->E, c->n, 5);
}

drf_status ensure_work(drf_ctx *c, size_t bytes)
{
    if (c->work_bytes >= bytes)
        return DRF_OK;
    if (c->d_work)
        DRF_HIP_CHECK(hipFree(c->d_work));
    c->d_work = nullptr;
    c->work_bytes = 0;
    DRF_HIP_CHECK(hipMalloc(&c->d_work, bytes));
    c->work_bytes = bytes;
    return DRF_OK;
}

drf_status check_ready(const drf_ctx *c)
{
    DRF_REQUIRE(c, DRF_ERR_ARG, "null context");
    DRF_REQUIRE(c->E > 0 && c->d_h, DRF_ERR_STATE, "drf_initialize has not been called");
    return DRF_OK;
}

template <class T> View<T> view(void *p, int layout, const drf_ctx *c)
{
    View<T> v{(T *)p, 0, 0, 0, 0};
    layout_strides(layout, c->E, c->n, 5, v.fs, v.es, v.ls, v.is, v.bs, v.bb);
    return v;
}

template <class T> View<const T> cview(const void *p, int layout, const drf_ctx *c)
{
    View<const T> v{(const T *)p, 0, 0, 0, 0};
    layout_strides(layout, c->E, c->n, 5, v.fs, v.es, v.ls, v.is, v.bs, v.bb);
    return v;
}

// Per-node coefficient arrays (bathymetry, Coriolis) live on the device in
// the LINES layout whatever layout the state uses.
template <class T> View<const T> coef_view(const T *p, const drf_ctx *c)
{
    return cview<T>(p, DRF_LAYOUT_LINES, c);
}

bool valid_layout(int layout)
{
    return layout == DRF_LAYOUT_PACKED || layout == DRF_LAYOUT_SOA ||
           layout == DRF_LAYOUT_LINES || layout == DRF_LAYOUT_BLOCKS;
}

// element-major reference order h[e*nd + i + n L] -> LINES order
template <class T> std::vector<T> to_lines(const double *h, int64_t E, int n)
{
    const int64_t n2 = (int64_t)n * n, nd = n2 * n;
    std::vector<T> out(E * nd);
    for (int64_t e = 0; e < E; ++e)
        for (int64_t L = 0; L < n2; ++L)
            for (int i = 0; i < n; ++i)
                out[i * (E * n2) + e * n2 + L] = (T)h[e * nd + L * n + i];
    return out;
}

// The volume kernel addresses each field through a 32-bit per-lane byte
// offset (element and line part); it must fit for every view of the call.
bool lane_offsets_fit(const drf_ctx *c, int layout)
{
    View<const char> v{nullptr, 0, 0, 0, 0};
    layout_strides(layout, c->E, c->n, 5, v.fs, v.es, v.ls, v.is, v.bs, v.bb);
    const int64_t n2 = (int64_t)c->n * c->n;
    const int64_t max_off =
        (elem_offset(v, c->E - 1) + (n2 - 1) * v.ls + 1) * (int64_t)elem_size(c);
    return max_off < (int64_t(1) << 32);
}

// A Runge-Kutta step of the volume kernel: the scheme's EpiMode and
// coefficients (Epi).
struct StepCoefs {
    int mode, nst;
    double c1[kMaxStages], c2[kMaxStages], c3[kMaxStages], q[kMaxStages];
    const double *dtp;
};

// One volume-kernel launch at the context's precision: the right-hand side of
// U into R, or with step the state after a step (R may be U).
// faces: the context precision's VolFaces (the fused conforming face term
// of the plain RHS) or null.
template <class T>
hipError_t volume_t(drf_ctx *c, const void *U, void *R, int layout, hipStream_t s,
                    const StepCoefs *step, const VolFaces<T> *faces, const T *h, const T *f,
                    hipError_t (*launch)(int, const VolGeom<T> &, const Ops &, const Phys &,
                                         View<const T>, const Epi<T> &, hipStream_t))
{
    Epi<T> epi{};
    epi.mode = EPI_RHS;
    epi.R = view<T>(R, layout, c);
    if (step) {
        epi.mode = step->mode;
        epi.nst = step->nst;
        for (int k = 0; k < kMaxStages; ++k) {
            epi.c1[k] = step->c1[k];
            epi.c2[k] = step->c2[k];
            epi.c3[k] = step->c3[k];
            epi.q[k] = step->q[k];
        }
        epi.dtp = step->dtp;
    }
    VolGeom<T> geo{c->E, coef_view<T>(h, c), coef_view<T>(f, c),
                   c->f0, c->wg_per_cu, c->xcd_remap, c->wg_lines};
    if (faces)
        geo.faces = *faces;
    return launch(c->order, geo, c->ops, c->phys, cview<T>(U, layout, c), epi, s);
}

drf_status volume(drf_ctx *c, const void *U, void *R, int layout, hipStream_t s,
                  const StepCoefs *step = nullptr, const void *faces = nullptr)
{
    DRF_REQUIRE(lane_offsets_fit(c, layout), DRF_ERR_UNSUPPORTED,
                "mesh too large for 32-bit per-field offsets in this layout (use LINES or SOA)");
    const hipError_t err =
        c->precision == DRF_PREC_FP64
            ? volume_t<double>(c, U, R, layout, s, step, (const VolFaces<double> *)faces, c->d_h,
                               c->d_f, launch_volume_fp64)
            : volume_t<float>(c, U, R, layout, s, step, (const VolFaces<float> *)faces, c->d_h32,
                              c->d_f32, launch_volume_fp32);
    if (err != hipSuccess)
        return fail(DRF_ERR_HIP, std::string("volume kernel launch: ") + hipGetErrorString(err));
    return DRF_OK;
}

drf_status rhs_into(drf_ctx *c, const void *U, void *R, int layout, hipStream_t s)
{
    // An attached face plan's conforming interfaces go into the volume
    // kernel where the plan allows it; its mortars follow.
    VolFaces<double> f64{};
    VolFaces<float> f32{};
    const bool fused = c->faces && (c->precision == DRF_PREC_FP64
                                        ? volume_faces<double>(c->faces, layout, &f64)
                                        : volume_faces<float>(c->faces, layout, &f32));
    const void *vf = !fused ? nullptr : c->precision == DRF_PREC_FP64 ? (const void *)&f64
                                                                       : (const void *)&f32;
    drf_status st = volume(c, U, R, layout, s, nullptr, vf);
    if (st || !c->faces)
        return st;
    return fused ? face_term_mortars(c->faces, U, R, layout, s) : face_term(c->faces, U, R, layout, s);
}

// Un-fused stepping: the reference's sequence of RHS evaluations and vector
// updates (FP64 only).
drf_status rk_unfused(drf_ctx *c, int scheme, double dt, double *U, int layout, hipStream_t s)
{
    DRF_REQUIRE(c->precision == DRF_PREC_FP64, DRF_ERR_UNSUPPORTED,
                "un-fused stepping is the FP64 baseline only");
    const int64_t len = state_len(c, layout);
    drf_status st = ensure_work(c, sizeof(double) * len * 7);
    if (st)
        return st;
    double *w = (double *)c->d_work;
    double *k[6] = {w, w + len, w + 2 * len, w + 3 * len, w + 4 * len, w + 5 * len};
    double *Ut = w + 6 * len;
    auto V = [&](double *p) { return view<double>(p, layout, c); };
    auto CV = [&](const double *p) { return cview<double>(p, layout, c); };
    auto lin = [&](double *Y, const double *X0, double alpha, const double *X1, double beta,
                   double gamma, std::initializer_list<std::pair<const double *, double>> ks) {
        LinComb lc{};
        lc.Y = V(Y);
        lc.X0 = CV(X0);
        lc.X1 = CV(X1);
        lc.alpha = alpha;
        lc.beta = beta;
        lc.gamma = gamma;
        lc.nk = 0;
        for (auto &kc : ks) {
            lc.K[lc.nk] = CV(kc.first);
            lc.c[lc.nk] = kc.second;
            ++lc.nk;
        }
        hipError_t e = launch_lincomb(c->E, c->n, lc, s);
        return e == hipSuccess ? DRF_OK : fail(DRF_ERR_HIP, hipGetErrorString(e));
    };
#define TRY(x)                                                                               \
    do {                                                                                     \
        drf_status t_ = (x);                                                                 \
        if (t_)                                                                              \
            return t_;                                                                       \
    } while (0)
    switch (scheme) {
    case DRF_RK_EULER: // :14-18
        TRY(rhs_into(c, U, k[0], layout, s));
        TRY(lin(U, U, 1.0, nullptr, 1.0, dt, {{k[0], 1.0}}));
        break;
    case DRF_RK_RK2: // :33-47
        TRY(rhs_into(c, U, k[0], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, 0.5 * dt, {{k[0], 1.0}}));
        TRY(rhs_into(c, Ut, k[1], layout, s));
        TRY(lin(U, U, 1.0, nullptr, 1.0, dt, {{k[1], 1.0}}));
        break;
    case DRF_RK_SSPRK3: // :64-80 (U1 in Ut, U2 in k[1])
        TRY(rhs_into(c, U, k[0], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, dt, {{k[0], 1.0}}));
        TRY(rhs_into(c, Ut, k[0], layout, s));
        TRY(lin(k[1], U, 0.75, Ut, 0.25, dt, {{k[0], 1.0}}));
        TRY(rhs_into(c, k[1], k[0], layout, s));
        TRY(lin(U, U, 1.0 / 3.0, k[1], 2.0 / 3.0, dt, {{k[0], 1.0}}));
        break;
    case DRF_RK_RK4: // :88-112
        TRY(rhs_into(c, U, k[0], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, 0.5 * dt, {{k[0], 1.0}}));
        TRY(rhs_into(c, Ut, k[1], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, 0.5 * dt, {{k[1], 1.0}}));
        TRY(rhs_into(c, Ut, k[2], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, dt, {{k[2], 1.0}}));
        TRY(rhs_into(c, Ut, k[3], layout, s));
        TRY(lin(U, U, 1.0, nullptr, 1.0, dt / 6.0,
                {{k[0], 1.0}, {k[1], 2.0}, {k[2], 2.0}, {k[3], 1.0}}));
        break;
    case DRF_RK_LSRK45: { // :126-143
        static const double A[5] = {0.0, -0.4178904745, -1.192151694643, -1.697784692471,
                                    -1.514183444257};
        static const double B[5] = {0.1496590219993, 0.3792103129999, 0.8229550293869,
                                    0.6994504559488, 0.1530572479681};
        // The reference zeroes the residual first; A[0] = 0 so stage 0 is
        // res = 0 * 0 + dt k = dt k, written directly (no memset is recorded).
        double *res = k[1];
        for (int st5 = 0; st5 < 5; ++st5) {
            TRY(rhs_into(c, U, k[0], layout, s));
            TRY(lin(res, st5 == 0 ? nullptr : res, A[st5], nullptr, 1.0, dt, {{k[0], 1.0}}));
            TRY(lin(U, U, 1.0, nullptr, 1.0, B[st5], {{res, 1.0}}));
        }
        break;
    }
    case DRF_RK_DP45: // :151-189
        TRY(rhs_into(c, U, k[0], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, dt / 5.0, {{k[0], 1.0}}));
        TRY(rhs_into(c, Ut, k[1], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, dt, {{k[0], 3.0 / 40.0}, {k[1], 9.0 / 40.0}}));
        TRY(rhs_into(c, Ut, k[2], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, dt,
                {{k[0], 44.0 / 45.0}, {k[1], -56.0 / 15.0}, {k[2], 32.0 / 9.0}}));
        TRY(rhs_into(c, Ut, k[3], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, dt,
                {{k[0], 19372.0 / 6561.0},
                 {k[1], -25360.0 / 2187.0},
                 {k[2], 64448.0 / 6561.0},
                 {k[3], -212.0 / 729.0}}));
        TRY(rhs_into(c, Ut, k[4], layout, s));
        TRY(lin(Ut, U, 1.0, nullptr, 1.0, dt,
                {{k[0], 9017.0 / 3168.0},
                 {k[1], -355.0 / 33.0},
                 {k[2], 46732.0 / 5247.0},
                 {k[3], 49.0 / 176.0},
                 {k[4], -5103.0 / 18656.0}}));
        TRY(rhs_into(c, Ut, k[5], layout, s));
        TRY(lin(U, U, 1.0, nullptr, 1.0, dt,
                {{k[0], 35.0 / 384.0},
                 {k[2], 500.0 / 1113.0},
                 {k[3], 125.0 / 192.0},
                 {k[4], -2187.0 / 6784.0},
                 {k[5], 11.0 / 84.0}}));
        break;
    default:
        return fail(DRF_ERR_ARG, "unknown Runge-Kutta scheme " + std::to_string(scheme));
    }
    return DRF_OK;
}

// Fused stepping: one launch runs every stage of the step, in place.
// Every dt-proportional coefficient is (m dt) / q; with dtp (device dt) the
// kernel forms it from *dtp with the same operations, so both give the same
// bits for the same dt.
drf_status rk_fused(drf_ctx *c, int scheme, double dt, void *U, int layout, hipStream_t s,
                    const double *dtp = nullptr)
{
    DRF_REQUIRE(!c->faces, DRF_ERR_UNSUPPORTED,
                "fused Runge-Kutta stages carry no face term: step a context with a face plan "
                "un-fused");
    if (scheme == DRF_RK_DP45) {
        if (dtp)
            return fail(DRF_ERR_UNSUPPORTED, "device time steps need a fused scheme (not DP45)");
        return rk_unfused(c, scheme, dt, (double *)U, layout, s);
    }
    StepCoefs k{};
    k.dtp = dtp;
    // appends a stage whose dt coefficient is m dt / q
    auto stage = [&](double m, double q, double c2, double c3) {
        k.c1[k.nst] = dtp ? m : (m * dt) / q;
        k.q[k.nst] = q;
        k.c2[k.nst] = c2;
        k.c3[k.nst] = c3;
        ++k.nst;
    };
    switch (scheme) {
    case DRF_RK_EULER:
        k.mode = EPI_STAGE;
        stage(1.0, 1.0, 0, 0);
        break;
    case DRF_RK_RK2:
        k.mode = EPI_STAGE;
        stage(0.5, 1.0, 0, 0);
        stage(1.0, 1.0, 0, 0);
        break;
    case DRF_RK_SSPRK3:
        k.mode = EPI_SSP3;
        stage(1.0, 1.0, 0, 0);
        stage(1.0, 1.0, 0.75, 0.25);
        stage(1.0, 1.0, 1.0 / 3.0, 2.0 / 3.0);
        break;
    case DRF_RK_RK4:
        k.mode = EPI_RK4;
        stage(0.5, 1.0, 1.0, 0);
        stage(0.5, 1.0, 2.0, 0);
        stage(1.0, 1.0, 2.0, 0);
        stage(1.0, 6.0, 1.0, 0);
        break;
    case DRF_RK_LSRK45: {
        static const double Ac[5] = {0.0, -0.4178904745, -1.192151694643, -1.697784692471,
                                     -1.514183444257};
        static const double Bc[5] = {0.1496590219993, 0.3792103129999, 0.8229550293869,
                                     0.6994504559488, 0.1530572479681};
        k.mode = EPI_LSRK;
        for (int i = 0; i < 5; ++i)
            stage(1.0, 1.0, Ac[i], Bc[i]);
        break;
    }
    default:
        return fail(DRF_ERR_ARG, "unknown Runge-Kutta scheme " + std::to_string(scheme));
    }
    return volume(c, U, U, layout, s, &k);
}

drf_status wave_speed(drf_ctx *c, const void *U, int layout, double *out, hipStream_t s)
{
    DRF_REQUIRE(c->precision == DRF_PREC_FP64, DRF_ERR_UNSUPPORTED,
                "wave speed on the FP64 state only");
    const int64_t npart = wave_speed_parts(c->order, c->E);
    hipError_t e = launch_wave_speed(c->order, c->E, cview<double>(U, layout, c),
                                     coef_view<double>(c->d_h, c), c->d_red + 1, npart, s);
    if (e == hipSuccess)
        e = launch_max_reduce(c->d_red + 1, npart, c->d_red, s);
    if (e == hipSuccess)
        e = hipMemcpyAsync(out, c->d_red, sizeof(double), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    if (e != hipSuccess)
        return fail(DRF_ERR_HIP, std::string("wave speed: ") + hipGetErrorString(e));
    return DRF_OK;
}

// SimulationDriver::step without leaving the device: the wave-speed maximum
// of U into d_red[0], dt and time on the device, then the fused RK step that
// reads dt from *dt_dev.
drf_status adaptive_step(drf_ctx *c, int scheme, double cfl, double dx_min, double dt_min,
                         double dt_max, void *U, int layout, double *dt_dev, double *t_dev,
                         hipStream_t s)
{
    const int64_t npart = wave_speed_parts(c->order, c->E);
    hipError_t e = launch_wave_speed(c->order, c->E, cview<double>(U, layout, c),
                                     coef_view<double>(c->d_h, c), c->d_red + 1, npart, s);
    if (e == hipSuccess)
        e = launch_adaptive_dt(c->d_red + 1, npart, c->d_red, dx_min, cfl, dt_min, dt_max, dt_dev,
                               t_dev, s);
    if (e != hipSuccess)
        return fail(DRF_ERR_HIP, std::string("adaptive dt: ") + hipGetErrorString(e));
    return rk_fused(c, scheme, 0.0, U, layout, s, dt_dev);
}

drf_status check_adaptive(drf_ctx *c, int scheme, void *U, int layout, void *dt_dev)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U && dt_dev, DRF_ERR_ARG, "null state or dt pointer");
    DRF_REQUIRE(valid_layout(layout), DRF_ERR_ARG, "unknown layout");
    DRF_REQUIRE(scheme >= DRF_RK_EULER && scheme < DRF_RK_DP45, DRF_ERR_UNSUPPORTED,
                "device time steps need a fused scheme (Euler, RK2, SSPRK3, RK4, LSRK45)");
    DRF_REQUIRE(c->precision == DRF_PREC_FP64, DRF_ERR_UNSUPPORTED,
                "device time steps on FP64 contexts (the wave speed is FP64)");
    return DRF_OK;
}

} // namespace


// A captured sequence of steps.  The graph owns the workspace its kernels
// use, so later growth of the context's own workspace cannot leave it
// pointing at freed memory.
struct drf_graph {
    int device;
    hipGraph_t graph;
    hipGraphExec_t exec;
    void *work;
};

drf_status drf_graph_destroy_impl(drf_graph *g);

namespace {

template <class Body>
drf_status capture_graph(drf_ctx *c, size_t work_bytes, int n_steps, drf_graph **out, Body body)
{
    DRF_HIP_CHECK(hipSetDevice(c->device));
    drf_graph *g = new drf_graph{c->device, nullptr, nullptr, nullptr};
    if (work_bytes && hipMalloc(&g->work, work_bytes) != hipSuccess) {
        delete g;
        return fail(DRF_ERR_HIP, "graph workspace allocation failed");
    }
    hipStream_t cs = nullptr;
    if (hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess) {
        (void)hipFree(g->work);
        delete g;
        return fail(DRF_ERR_HIP, "capture stream creation failed");
    }
    // route the context's workspace to the graph's own buffer while capturing
    void *saved = c->d_work;
    const size_t saved_bytes = c->work_bytes;
    if (work_bytes) {
        c->d_work = g->work;
        c->work_bytes = work_bytes;
    }
    drf_status st = DRF_OK;
    hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeRelaxed);
    if (e != hipSuccess)
        st = fail(DRF_ERR_HIP, std::string("begin capture: ") + hipGetErrorString(e));
    for (int i = 0; i < n_steps && st == DRF_OK && e == hipSuccess; ++i)
        st = body(cs);
    if (e == hipSuccess) {
        hipGraph_t graph = nullptr;
        const hipError_t e2 = hipStreamEndCapture(cs, &graph);
        if (st == DRF_OK && e2 != hipSuccess)
            st = fail(DRF_ERR_HIP, std::string("end capture: ") + hipGetErrorString(e2));
        g->graph = graph;
    }
    c->d_work = saved;
    c->work_bytes = saved_bytes;
    (void)hipStreamDestroy(cs);
    if (st == DRF_OK) {
        e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
        if (e != hipSuccess)
            st = fail(DRF_ERR_HIP, std::string("graph instantiate: ") + hipGetErrorString(e));
    }
    if (st != DRF_OK) {
        drf_graph_destroy_impl(g);
        return st;
    }
    *out = g;
    return DRF_OK;
}

} // namespace

drf_status drf_graph_destroy_impl(drf_graph *g)
{
    if (!g)
        return DRF_OK;
    (void)hipSetDevice(g->device);
    if (g->exec)
        (void)hipGraphExecDestroy(g->exec);
    if (g->graph)
        (void)hipGraphDestroy(g->graph);
    if (g->work)
        (void)hipFree(g->work);
    delete g;
    return DRF_OK;
}

extern "C" {

void drf_default_physics(drf_physics *p)
{
    if (!p)
        return;
    p->g = 9.81;
    p->nu_h = 1.0;
    p->nu_v = 1e-4;
    p->kappa_v_T = 1e-5;
    p->kappa_v_S = 1e-5;
    p->rho_0 = 1025.0;
    p->alpha = 2e-4;
    p->beta = 7.6e-4;
}

const char *drf_last_error(void) { return g_last_error.c_str(); }

drf_status drf_basis(int order, double *nodes, double *weights, double *D)
{
    DRF_REQUIRE(order >= 1 && order + 1 <= kMaxN, DRF_ERR_ARG,
                "order must be in [1, 8], got " + std::to_string(order));
    double x[kMaxN], w[kMaxN], Dm[kMaxN * kMaxN];
    if (lgl_nodes(order + 1, x, w))
        return fail(DRF_ERR_ARG, "LGL requires at least 2 nodes");
    derivative_matrix(order + 1, x, Dm);
    const int n = order + 1;
    if (nodes)
        std::memcpy(nodes, x, sizeof(double) * n);
    if (weights)
        std::memcpy(weights, w, sizeof(double) * n);
    if (D)
        std::memcpy(D, Dm, sizeof(double) * n * n);
    return DRF_OK;
}

drf_status drf_create(int order, int precision, int device, drf_ctx **out)
{
    DRF_REQUIRE(out, DRF_ERR_ARG, "null output pointer");
    *out = nullptr;
    DRF_REQUIRE(order >= 1 && order + 1 <= kMaxN, DRF_ERR_UNSUPPORTED,
                "order must be in [1, 8], got " + std::to_string(order));
    DRF_REQUIRE(precision == DRF_PREC_FP64 || precision == DRF_PREC_MIXED, DRF_ERR_ARG,
                "unknown precision " + std::to_string(precision));
    int ndev = 0;
    DRF_HIP_CHECK(hipGetDeviceCount(&ndev));
    DRF_REQUIRE(device >= 0 && device < ndev, DRF_ERR_ARG,
                "device " + std::to_string(device) + " not present");
    DRF_HIP_CHECK(hipSetDevice(device));
    {
        const drf_status st = register_scratch(device);
        if (st)
            return st;
    }
    drf_ctx *c = new drf_ctx();
    c->order = order;
    c->n = order + 1;
    c->nh = c->n * c->n;
    c->nd = c->nh * c->n;
    c->precision = precision;
    c->device = device;
    double x[kMaxN], w[kMaxN];
    lgl_nodes(c->n, x, w);
    derivative_matrix(c->n, x, c->ops.D);
    for (int k = 0; k < c->n; ++k)
        c->ops.sw[k] = 0.5 * w[k]; // sigma_weights_, primitive_equations.cpp:116-121
    drf_physics p;
    drf_default_physics(&p);
    c->phys = Phys{p.g, p.nu_h, p.nu_v, p.kappa_v_T, p.kappa_v_S, p.rho_0, p.alpha, p.beta};
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete c;
        return fail(DRF_ERR_HIP, std::string("hipStreamCreate: ") + hipGetErrorString(e));
    }
    e = hipMalloc(&c->d_red, sizeof(double) * (kMaxWaveParts + 1));
    if (e != hipSuccess) {
        (void)hipStreamDestroy(c->stream);
        delete c;
        return fail(DRF_ERR_HIP, std::string("reduction buffer: ") + hipGetErrorString(e));
    }
    *out = c;
    return DRF_OK;
}

void drf_destroy(drf_ctx *c)
{
    if (!c)
        return;
    (void)hipSetDevice(c->device);
    if (c->stream)
        (void)hipStreamSynchronize(c->stream);
    (void)drf_set_face_plan(c, nullptr);
    (void)hipFree(c->d_h);
    (void)hipFree(c->d_f);
    (void)hipFree(c->d_h32);
    (void)hipFree(c->d_f32);
    (void)hipFree(c->d_work);
    (void)hipFree(c->d_red);
    if (c->stream)
        (void)hipStreamDestroy(c->stream);
    delete c;
}

drf_status drf_set_physics(drf_ctx *c, const drf_physics *p)
{
    DRF_REQUIRE(c && p, DRF_ERR_ARG, "null argument");
    c->phys = Phys{p->g, p->nu_h, p->nu_v, p->kappa_v_T, p->kappa_v_S, p->rho_0, p->alpha, p->beta};
    return DRF_OK;
}

drf_status drf_initialize(drf_ctx *c, int64_t E, const double *h, const double *dh_dx,
                          const double *dh_dy, double f0, double beta, double y0,
                          const double *y)
{
    (void)dh_dx;
    (void)dh_dy;
    DRF_REQUIRE(c, DRF_ERR_ARG, "null context");
    DRF_REQUIRE(E > 0, DRF_ERR_ARG, "number of elements must be positive");
    DRF_REQUIRE(h, DRF_ERR_ARG, "bathymetry is required");
    DRF_REQUIRE(y || beta == 0.0, DRF_ERR_ARG, "y_positions are required when beta != 0");
    DRF_HIP_CHECK(hipSetDevice(c->device));
    (void)drf_set_face_plan(c, nullptr); // a plan belongs to the mesh it was built on
    const int64_t len = E * c->nd;
    (void)hipFree(c->d_h);
    (void)hipFree(c->d_f);
    (void)hipFree(c->d_h32);
    (void)hipFree(c->d_f32);
    c->d_h = c->d_f = nullptr;
    c->d_h32 = c->d_f32 = nullptr;
    c->E = E;
    c->f0 = f0;
    {
        std::vector<double> hl = to_lines<double>(h, E, c->n);
        DRF_HIP_CHECK(hipMalloc(&c->d_h, sizeof(double) * len));
        DRF_HIP_CHECK(hipMemcpy(c->d_h, hl.data(), sizeof(double) * len, hipMemcpyHostToDevice));
        if (c->precision == DRF_PREC_MIXED) {
            std::vector<float> h32 = to_lines<float>(h, E, c->n);
            DRF_HIP_CHECK(hipMalloc(&c->d_h32, sizeof(float) * len));
            DRF_HIP_CHECK(
                hipMemcpy(c->d_h32, h32.data(), sizeof(float) * len, hipMemcpyHostToDevice));
        }
    }
    if (beta != 0.0) {
        // CoriolisParameter::compute, primitive_equations.hpp:65-70
        std::vector<double> f(len);
        for (int64_t i = 0; i < len; ++i)
            f[i] = f0 + beta * (y[i] - y0);
        std::vector<double> fl = to_lines<double>(f.data(), E, c->n);
        DRF_HIP_CHECK(hipMalloc(&c->d_f, sizeof(double) * len));
        DRF_HIP_CHECK(hipMemcpy(c->d_f, fl.data(), sizeof(double) * len, hipMemcpyHostToDevice));
        if (c->precision == DRF_PREC_MIXED) {
            std::vector<float> f32 = to_lines<float>(f.data(), E, c->n);
            DRF_HIP_CHECK(hipMalloc(&c->d_f32, sizeof(float) * len));
            DRF_HIP_CHECK(
                hipMemcpy(c->d_f32, f32.data(), sizeof(float) * len, hipMemcpyHostToDevice));
        }
    }
    return DRF_OK;
}

drf_status drf_rhs_dev(drf_ctx *c, double t, const void *U, void *dUdt, int layout, void *stream)
{
    (void)t; // the reference RHS does not depend on time
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U && dUdt, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(valid_layout(layout), DRF_ERR_ARG, "unknown layout");
    return rhs_into(c, U, dUdt, layout, pick_stream(c, stream));
}

drf_status drf_set_launch(drf_ctx *c, int wg_per_cu, int xcd_remap, int wg_lines)
{
    DRF_REQUIRE(c, DRF_ERR_ARG, "null context");
    DRF_REQUIRE(wg_per_cu >= 0 && wg_per_cu <= 64, DRF_ERR_ARG, "wg_per_cu must be 0..64");
    DRF_REQUIRE(wg_lines == 0 || wg_lines == 128 || wg_lines == 256 || wg_lines == 512,
                DRF_ERR_ARG, "wg_lines must be 0, 128, 256 or 512");
    c->wg_per_cu = wg_per_cu;
    c->xcd_remap = xcd_remap ? 1 : 0;
    c->wg_lines = wg_lines ? wg_lines : 128;
    return DRF_OK;
}

int drf_layout_block_elements(int order) { return layout_block_elements(order); }

int64_t drf_state_len(const drf_ctx *c, int layout)
{
    if (!c || c->E <= 0 || !valid_layout(layout))
        return 0;
    return state_len(c, layout);
}

drf_status drf_get_launch(const drf_ctx *c, int *wg_per_cu, int *xcd_remap, int *wg_lines)
{
    DRF_REQUIRE(c && wg_per_cu && xcd_remap && wg_lines, DRF_ERR_ARG, "null argument");
    *wg_per_cu = c->wg_per_cu;
    *xcd_remap = c->xcd_remap;
    *wg_lines = c->wg_lines;
    return DRF_OK;
}

drf_status drf_autotune(drf_ctx *c, const void *U, void *dUdt, int layout, int reps,
                        void *stream, float *best_us)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U && dUdt, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(valid_layout(layout), DRF_ERR_ARG, "unknown layout");
    DRF_REQUIRE(reps >= 1 && reps <= 1000, DRF_ERR_ARG, "reps must be 1..1000");
    DRF_HIP_CHECK(hipSetDevice(c->device));
    hipStream_t s = pick_stream(c, stream);
    hipEvent_t e0, e1;
    DRF_HIP_CHECK(hipEventCreate(&e0));
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail(DRF_ERR_HIP, "hipEventCreate failed");
    }
    // The trials cycle over the caller's state and output and kNset - 1
    // temporary copies (1.3 GB at 64x64x8, N = 4, FP64), so that every timed
    // launch reads its state from HBM, as a solver's stages do, rather than
    // from what the previous launch left in the 256 MB last-level cache.  If
    // the copies cannot be allocated, the trials run on the caller's buffers.
    constexpr int kNset = 4;
    const size_t bytes = elem_size(c) * (size_t)state_len(c, layout);
    const void *Us[kNset] = {U};
    void *Rs[kNset] = {dUdt};
    int nset = 1;
    drf_status res = DRF_OK;
    for (; nset < kNset; ++nset) {
        void *u = nullptr, *r = nullptr;
        if (hipMalloc(&u, bytes) != hipSuccess || hipMalloc(&r, bytes) != hipSuccess) {
            (void)hipGetLastError();
            if (u)
                (void)hipFree(u);
            break;
        }
        Us[nset] = u;
        Rs[nset] = r;
        if (hipMemcpyAsync(u, U, bytes, hipMemcpyDeviceToDevice, s) != hipSuccess) {
            res = fail(DRF_ERR_HIP, "hipMemcpyAsync failed");
            ++nset;
            break;
        }
    }
    // workgroup size x resident workgroups per CU (values above the occupancy
    // limit clamp to it; wider workgroups hold fewer per CU) x XCD-aware
    // batch order.  Orders above 4 have the 128-line workgroup only.
    static const int kWpc[] = {1, 2, 3, 4, 5, 6, 8};
    static const int kLines[] = {128, 256, 512};
    const int nlines = c->order <= 4 ? 3 : 1;
    float best = 1e30f;
    int bw = c->wg_per_cu, br = c->xcd_remap, bl = c->wg_lines;
    for (int li = 0; li < nlines && res == DRF_OK; ++li)
    for (int remap = 0; remap < 2 && res == DRF_OK; ++remap)
        for (int wpc : kWpc) {
            if (kLines[li] * wpc > 2048) // beyond a CU's 32 waves
                continue;
            c->wg_lines = kLines[li];
            c->wg_per_cu = wpc;
            c->xcd_remap = remap;
            for (int k = 0; k < nset && res == DRF_OK; ++k) // warm-up
                res = rhs_into(c, Us[k], Rs[k], layout, s);
            if (res == DRF_OK && hipEventRecord(e0, s) != hipSuccess)
                res = fail(DRF_ERR_HIP, "hipEventRecord failed");
            for (int r = 0; r < reps && res == DRF_OK; ++r)
                res = rhs_into(c, Us[r % nset], Rs[r % nset], layout, s);
            float ms = 0.f;
            if (res == DRF_OK && (hipEventRecord(e1, s) != hipSuccess ||
                                  hipEventSynchronize(e1) != hipSuccess ||
                                  hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
                res = fail(DRF_ERR_HIP, "event timing failed");
            if (res != DRF_OK)
                break;
            const float us = ms * 1000.f / reps;
            if (us < best) {
                best = us;
                bw = wpc;
                br = remap;
                bl = kLines[li];
            }
        }
    (void)hipStreamSynchronize(s);
    for (int k = 1; k < nset; ++k) {
        (void)hipFree(const_cast<void *>(Us[k]));
        (void)hipFree(Rs[k]);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    // report the shape as it runs: a request above the occupancy limit runs at it
    {
        VolFaces<double> f64{};
        VolFaces<float> f32{};
        const bool fused = c->faces && (c->precision == DRF_PREC_FP64
                                            ? volume_faces<double>(c->faces, layout, &f64)
                                            : volume_faces<float>(c->faces, layout, &f32));
        const int li = bl == 128 ? 0 : bl == 256 ? 1 : 2;
        const int lim = (c->order < kMaxN)
                            ? g_rhs_per_cu[c->precision == DRF_PREC_FP64 ? 0 : 1][li][c->order]
                                          [fused ? 1 : 0]
                            : 0;
        if (lim > 0 && bw > lim)
            bw = lim;
    }
    c->wg_per_cu = bw;
    c->xcd_remap = br;
    c->wg_lines = bl;
    if (best_us)
        *best_us = best;
    return res;
}

drf_status drf_rhs(drf_ctx *c, double t, const double *U, double *dUdt)
{
    (void)t;
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U && dUdt, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(c->precision == DRF_PREC_FP64, DRF_ERR_UNSUPPORTED,
                "host-pointer RHS is provided for FP64 contexts");
    const int64_t len = state_len(c);
    st = ensure_work(c, sizeof(double) * len * 2);
    if (st)
        return st;
    double *dU = (double *)c->d_work, *dR = dU + len;
    hipStream_t s = c->stream;
    DRF_HIP_CHECK(hipMemcpyAsync(dU, U, sizeof(double) * len, hipMemcpyHostToDevice, s));
    st = rhs_into(c, dU, dR, DRF_LAYOUT_PACKED, s);
    if (st)
        return st;
    DRF_HIP_CHECK(hipMemcpyAsync(dUdt, dR, sizeof(double) * len, hipMemcpyDeviceToHost, s));
    DRF_HIP_CHECK(hipStreamSynchronize(s));
    return DRF_OK;
}

drf_status drf_rk_step_dev(drf_ctx *c, int scheme, double t, double dt, void *U, int layout,
                           int fused, void *stream)
{
    (void)t;
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(valid_layout(layout), DRF_ERR_ARG, "unknown layout");
    DRF_REQUIRE(scheme >= DRF_RK_EULER && scheme <= DRF_RK_DP45, DRF_ERR_ARG,
                "unknown Runge-Kutta scheme " + std::to_string(scheme));
    hipStream_t s = pick_stream(c, stream);
    if (fused)
        return rk_fused(c, scheme, dt, U, layout, s);
    return rk_unfused(c, scheme, dt, (double *)U, layout, s);
}

drf_status drf_rk_step_adaptive_dev(drf_ctx *c, int scheme, double cfl, double dx_min,
                                    double dt_min, double dt_max, void *U, int layout,
                                    void *dt_dev, void *time_dev, void *stream)
{
    drf_status st = check_adaptive(c, scheme, U, layout, dt_dev);
    if (st)
        return st;
    return adaptive_step(c, scheme, cfl, dx_min, dt_min, dt_max, U, layout, (double *)dt_dev,
                         (double *)time_dev, pick_stream(c, stream));
}

drf_status drf_rk_step(drf_ctx *c, int scheme, double t, double dt, double *U)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(c->precision == DRF_PREC_FP64, DRF_ERR_UNSUPPORTED,
                "host-pointer stepping is provided for FP64 contexts");
    const int64_t len = state_len(c);
    double *dU = nullptr;
    DRF_HIP_CHECK(hipMalloc(&dU, sizeof(double) * len));
    hipStream_t s = c->stream;
    hipError_t e = hipMemcpyAsync(dU, U, sizeof(double) * len, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        st = drf_rk_step_dev(c, scheme, t, dt, dU, DRF_LAYOUT_PACKED, 1, s);
        if (st == DRF_OK) {
            e = hipMemcpyAsync(U, dU, sizeof(double) * len, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess)
                e = hipStreamSynchronize(s);
        }
    }
    (void)hipFree(dU);
    if (st)
        return st;
    if (e != hipSuccess)
        return fail(DRF_ERR_HIP, std::string("drf_rk_step: ") + hipGetErrorString(e));
    return DRF_OK;
}

drf_status drf_max_wave_speed_dev(drf_ctx *c, const void *U, int layout, double *c_max,
                                  void *stream)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U && c_max, DRF_ERR_ARG, "null argument");
    DRF_REQUIRE(valid_layout(layout), DRF_ERR_ARG, "unknown layout");
    return wave_speed(c, U, layout, c_max, pick_stream(c, stream));
}

drf_status drf_max_wave_speed(drf_ctx *c, const double *U, double *c_max)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U && c_max, DRF_ERR_ARG, "null argument");
    const int64_t len = state_len(c);
    st = ensure_work(c, sizeof(double) * len);
    if (st)
        return st;
    DRF_HIP_CHECK(
        hipMemcpyAsync(c->d_work, U, sizeof(double) * len, hipMemcpyHostToDevice, c->stream));
    return wave_speed(c, c->d_work, DRF_LAYOUT_PACKED, c_max, c->stream);
}

drf_status drf_max_wave_speed_derived_dev(drf_ctx *c, const void *H, const void *u,
                                          const void *v, int64_t es, double *c_max, void *stream)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(H && u && v && c_max, DRF_ERR_ARG, "null argument");
    hipStream_t s = pick_stream(c, stream);
    const int64_t npart = std::min<int64_t>(kMaxWaveParts, (c->E + 3) / 4);
    hipError_t e = launch_wave_speed_derived(c->order, c->E, (const double *)H, (const double *)u,
                                             (const double *)v, es, c->d_red + 1, npart, s);
    if (e == hipSuccess)
        e = launch_max_reduce(c->d_red + 1, npart, c->d_red, s);
    if (e == hipSuccess)
        e = hipMemcpyAsync(c_max, c->d_red, sizeof(double), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    if (e != hipSuccess)
        return fail(DRF_ERR_HIP, std::string("wave speed: ") + hipGetErrorString(e));
    return DRF_OK;
}

double drf_compute_dt(double cmax, double dx_min, double cfl, double dt_min, double dt_max)
{
    // AdaptiveTimeController::compute_dt, src/solver/time_stepper.cpp:261-268
    if (cmax < 1e-14)
        return dt_max;
    return std::clamp(cfl * dx_min / cmax, dt_min, dt_max);
}

drf_status drf_mode_split_step_dev(drf_ctx *c, double dt3, int nsub, void *full, void *stream)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(full, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(nsub >= 1, DRF_ERR_ARG, "subcycles must be >= 1");
    hipError_t e = launch_mode_split(c->order, c->E, dt3, nsub, (double *)full,
                                     coef_view<double>(c->d_h, c), coef_view<double>(c->d_f, c),
                                     c->f0, c->ops, c->phys, pick_stream(c, stream));
    if (e != hipSuccess)
        return fail(DRF_ERR_HIP, std::string("mode split launch: ") + hipGetErrorString(e));
    return DRF_OK;
}

drf_status drf_mode_split_step(drf_ctx *c, double dt3, int nsub, double *full)
{
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(full, DRF_ERR_ARG, "null state pointer");
    const int64_t len = c->E * 12 * (int64_t)c->nd;
    st = ensure_work(c, sizeof(double) * len);
    if (st)
        return st;
    hipStream_t s = c->stream;
    DRF_HIP_CHECK(hipMemcpyAsync(c->d_work, full, sizeof(double) * len, hipMemcpyHostToDevice, s));
    st = drf_mode_split_step_dev(c, dt3, nsub, c->d_work, s);
    if (st)
        return st;
    DRF_HIP_CHECK(hipMemcpyAsync(full, c->d_work, sizeof(double) * len, hipMemcpyDeviceToHost, s));
    DRF_HIP_CHECK(hipStreamSynchronize(s));
    return DRF_OK;
}

double drf_rhs_bytes(const drf_ctx *c)
{
    if (!c)
        return 0.0;
    // 5 state reads + 1 bathymetry read + 5 tendency writes per node (+ Coriolis
    // when it varies per node).
    const double s = (c->precision == DRF_PREC_FP64) ? 8.0 : 4.0;
    const double arrays = 11.0 + ((c->d_f || c->d_f32) ? 1.0 : 0.0);
    return (double)c->E * c->nd * arrays * s;
}

int64_t drf_num_elements(const drf_ctx *c) { return c ? c->E : 0; }
int drf_order(const drf_ctx *c) { return c ? c->order : 0; }

// ---------------- HIP graphs of repeated steps ----------------

drf_status drf_graph_rk_adaptive(drf_ctx *c, int scheme, double cfl, double dx_min,
                                 double dt_min, double dt_max, void *U, int layout, int n_steps,
                                 void *dt_dev, void *time_dev, drf_graph **out)
{
    DRF_REQUIRE(out, DRF_ERR_ARG, "null output");
    *out = nullptr;
    drf_status st = check_adaptive(c, scheme, U, layout, dt_dev);
    if (st)
        return st;
    DRF_REQUIRE(n_steps >= 1 && n_steps <= 100000, DRF_ERR_ARG, "n_steps must be 1..100000");
    return capture_graph(c, 0, n_steps, out, [&](hipStream_t cs) {
        return adaptive_step(c, scheme, cfl, dx_min, dt_min, dt_max, U, layout,
                             (double *)dt_dev, (double *)time_dev, cs);
    });
}

drf_status drf_graph_rk(drf_ctx *c, int scheme, double dt, void *U, int layout, int fused,
                        int n_steps, drf_graph **out)
{
    DRF_REQUIRE(out, DRF_ERR_ARG, "null output");
    *out = nullptr;
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(U, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(valid_layout(layout), DRF_ERR_ARG, "unknown layout");
    DRF_REQUIRE(scheme >= DRF_RK_EULER && scheme <= DRF_RK_DP45, DRF_ERR_ARG,
                "unknown Runge-Kutta scheme " + std::to_string(scheme));
    DRF_REQUIRE(n_steps >= 1 && n_steps <= 100000, DRF_ERR_ARG, "n_steps must be 1..100000");
    DRF_REQUIRE(fused || c->precision == DRF_PREC_FP64, DRF_ERR_UNSUPPORTED,
                "un-fused stepping is the FP64 baseline only");
    const bool uses_lincomb = !fused || scheme == DRF_RK_DP45;
    const size_t bytes = uses_lincomb ? sizeof(double) * state_len(c, layout) * 7 : 0;
    return capture_graph(c, bytes, n_steps, out, [&](hipStream_t cs) {
        return fused ? rk_fused(c, scheme, dt, U, layout, cs)
                     : rk_unfused(c, scheme, dt, (double *)U, layout, cs);
    });
}

drf_status drf_graph_mode_split(drf_ctx *c, double dt_3d, int n_sub, void *full, int n_steps,
                                drf_graph **out)
{
    DRF_REQUIRE(out, DRF_ERR_ARG, "null output");
    *out = nullptr;
    drf_status st = check_ready(c);
    if (st)
        return st;
    DRF_REQUIRE(full, DRF_ERR_ARG, "null state pointer");
    DRF_REQUIRE(n_sub >= 1, DRF_ERR_ARG, "subcycles must be >= 1");
    DRF_REQUIRE(n_steps >= 1 && n_steps <= 100000, DRF_ERR_ARG, "n_steps must be 1..100000");
    return capture_graph(c, 0, n_steps, out, [&](hipStream_t cs) -> drf_status {
        hipError_t e = launch_mode_split(c->order, c->E, dt_3d, n_sub, (double *)full,
                                         coef_view<double>(c->d_h, c),
                                         coef_view<double>(c->d_f, c), c->f0, c->ops, c->phys, cs);
        if (e != hipSuccess)
            return fail(DRF_ERR_HIP, std::string("mode split launch: ") + hipGetErrorString(e));
        return DRF_OK;
    });
}

drf_status drf_graph_launch(drf_graph *g, void *stream)
{
    DRF_REQUIRE(g, DRF_ERR_ARG, "null graph");
    DRF_HIP_CHECK(hipSetDevice(g->device));
    DRF_HIP_CHECK(hipGraphLaunch(g->exec, (hipStream_t)stream));
    return DRF_OK;
}

void drf_graph_destroy(drf_graph *g) { (void)drf_graph_destroy_impl(g); }

} // extern "C"
