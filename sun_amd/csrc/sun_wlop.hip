// sun_wlop.hip -- operator-basis Wilson loops on a resident lattice (host code): the
// Sigma_g_plus measurement object (include/meas/wloopex.h:13-36) and the fieldOp /
// wloop pair of include/meas/wlop.h.  The A0 family (src/wl/calcop_dg_A0.cu, 10
// operators) and the 33 family (src/wl/calcop_dg_33.cu, 25 operators) build one
// 18-real operator field per slot; the correlator (src/wl/wilsonloop_dg_A0.cu,
// wilsonloop_dg.cu) accumulates every slot pair into an FP64 device array.  The
// reference's block reductions end in floating-point atomics (run-to-run order
// varies); here every (pair, T) is a fixed-order sum of per-workgroup partials.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "sun_internal.hpp"

using namespace sun;

struct sun_wlop {
    sun_lattice* lat = nullptr;
    int family = 0, nop = 0, tmax = 0;
    size_t lb = 0;          // bytes of one 18-real entry
    size_t stride = 0;      // bytes of one slot (V entries)
    size_t held = 0;        // bytes of the block that all the following lie in
    void* ops = nullptr;    // nop slots
    void* aux = nullptr;    // scratch slots of the 33 family's shared products, or none
    double* partials = nullptr;
    int nb = 0, rows = 0;   // workgroups of the fallback and of the matrix-core correlator
    bool direct = false;    // few T, or no memory for them: without time lines
    bool planes() const { return wlop_planes(direct, lat->d.nc, lat->d.precision == SUN_PREC_F64, nop); }
    double* lines = nullptr;   // time lines: X3 + tmax times of every spatial site
    double* inverses = nullptr;  // their inverses, X3 times
    int* state = nullptr;   // per block of lines, what they allow
    double* acc = nullptr;  // nop^2 (tmax + 1), (i nop + j)(tmax + 1) + T
    int r = -1, mu = -1;    // radius and direction of the current operator field
};

namespace {

int wlop_nops(int family) { return family == SUN_WLOP_A0 ? 10 : (family == SUN_WLOP_33 ? 25 : 0); }

void release(sun_wlop* h) {
    if (!h) return;
    if (h->ops) {
        if (hipDeviceSynchronize() == hipSuccess)
            h->lat->ctx->spare.give(h->ops, h->held);
        else
            hipFree(h->ops);
    }
    delete h;
}

// Few T: multiplying every link out takes less time than moving the operators along time
// lines.  us per correlator, multiplied out / moved, around the rule's line:
//   A0 FP64   SU(3) 8^3 x 16 61 / 64 for seven T, 69 / 64 for eight; 12^4 92 / 90 for seven; 16^3 x
//             32 264 / 306 for four, 330 / 310 for five; 24^3 x 32 698 / 890 for three, 987 / 889
//             for four; SU(4) 12^3 x 24 211 / 253 for four, 264 / 254 for five
//   A0 FP32   16^4 140 / 143 for seven, 158 / 142 for eight (16^3 x 32 279 / 275, 8^3 x 16 69 / 76)
//   33 FP64   16^3 x 32 530 / 619 for two, 795 / 642 for three; 24^3 x 32 1742 / 1820 for two
//   33 FP32   16^3 x 32 593 / 665 for five, 710 / 665 for six; 24^3 x 32 2230 / 2052 for five; SU(4) 770 /
//             963 for two, 1150 / 964 for three
bool wlop_direct(int nop, int T1, const sun_lattice* lat) {
    const bool f64 = lat->d.precision == SUN_PREC_F64;
    const int V = lat->g.V;
    if (nop > 16) return T1 <= (f64 || lat->d.nc > 3 ? 2 : V > (1 << 18) ? 4 : 5);
    if (f64) return T1 <= (V > (1 << 18) ? 3 : V > 25000 ? 4 : V > 10000 ? 6 : 7);
    return T1 <= (V <= 10000 ? 8 : 7);
}

int check_radius(const sun_wlop* h, int r, int mu, const char* what) {
    const Geom& g = h->lat->g;
    if (mu < 0 || mu > 2) return fail(SUN_ERR_INVALID, "%s: mu %d is not a spatial direction", what, mu);
    if (r < 1 || r > g.X[mu]) return fail(SUN_ERR_INVALID, "%s: radius %d outside 1..%d", what, r, g.X[mu]);
    return SUN_OK;
}

}  // namespace

// shared: the fields will come from shared products (fields())
static int create(sun_lattice* lat, int family, int tmax, bool shared, sun_wlop** out) {
    if (!out) return fail(SUN_ERR_INVALID, "sun_wlop_create: NULL handle pointer");
    *out = nullptr;
    if (!lat) return fail(SUN_ERR_INVALID, "sun_wlop_create: NULL lattice");
    if (lat->external) return fail(SUN_ERR_STATE, "sun_wlop_create: not available on a server job's lattice");
    const int nop = wlop_nops(family);
    if (!nop) return fail(SUN_ERR_INVALID, "sun_wlop_create: family %d (use SUN_WLOP_A0 or SUN_WLOP_33)", family);
    const Geom& g = lat->g;
    if (tmax < 0 || tmax > g.X[3]) return fail(SUN_ERR_INVALID, "sun_wlop_create: tmax %d outside 0..%d", tmax, g.X[3]);
    HIP_TRY(hipSetDevice(lat->ctx->device));
    sun_wlop* h = new (std::nothrow) sun_wlop();
    if (!h) return fail(SUN_ERR_NOMEM, "sun_wlop_create: host allocation");
    h->lat = lat;
    h->family = family;
    h->nop = nop;
    h->tmax = tmax;
    h->lb = (size_t)2 * lat->d.nc * lat->d.nc * (size_t)lat->d.precision;
    h->stride = (size_t)g.V * h->lb;
    h->nb = monitor_blocks(g);
    h->rows = wlop_corr_blocks(g);
    h->direct = wlop_direct(nop, tmax + 1, lat);
    // scratch slots for the 33 family's shared products, which FP64 fields that are handed out are not
    bool aux = family == SUN_WLOP_33 && (shared || lat->d.precision == SUN_PREC_F32);
    const size_t nout = (size_t)nop * nop * (tmax + 1);
    const size_t npart = nout * (size_t)std::max(h->nb, h->rows);
    const size_t line = (size_t)2 * lat->d.nc * lat->d.nc * sizeof(double), vs = (size_t)g.str[3];
    // the parts of a block: without one counted, then with it
    auto lay_out = [&](char* base) {
        size_t total = 0;
        auto part = [&](size_t bytes) {
            char* p = base + total;
            total += (bytes + 255) & ~(size_t)255;
            return p;
        };
        part((size_t)nop * h->stride);
        h->partials = (double*)part(npart * sizeof(double));
        h->acc = (double*)part(nout * sizeof(double));
        h->aux = aux ? part((size_t)kWlopAuxSlots * h->stride) : nullptr;
        if (!h->direct) {
            h->lines = (double*)part(vs * (g.X[3] + tmax) * line);
            h->inverses = (double*)part(vs * g.X[3] * line);
            h->state = (int*)part(line_blocks(g) * sizeof(int));
        }
        return total;
    };
    hipError_t e = lat->ctx->spare.take(lay_out(nullptr), &h->ops, &h->held);
    if (e == hipErrorOutOfMemory && (aux || !h->direct)) {
        // the operators and sums alone: the fields multiplied out path by path, the correlators link by link
        hipGetLastError();
        aux = false;
        h->direct = true;
        e = lat->ctx->spare.take(lay_out(nullptr), &h->ops, &h->held);
    }
    HIP_TRY_CLEANUP(e, release(h));
    char* base = static_cast<char*>(h->ops);
    lay_out(base);
    if (family == SUN_WLOP_A0)  // slot 9 is zero throughout
        HIP_TRY_CLEANUP(hipMemset(base + 9 * h->stride, 0, h->stride), release(h));
    HIP_TRY_CLEANUP(hipMemset(h->acc, 0, nout * sizeof(double)), release(h));
    HIP_TRY_CLEANUP(hipStreamSynchronize(nullptr), release(h));  // the handle's streams do not wait for it
    *out = h;
    return SUN_OK;
}

extern "C" int sun_wlop_create(sun_lattice* lat, int family, int tmax, sun_wlop** out) {
    return create(lat, family, tmax, false, out);
}

extern "C" int sun_wlop_destroy(sun_wlop* h) {
    if (!h) return SUN_OK;
    hipSetDevice(h->lat->ctx->device);
    release(h);
    return SUN_OK;
}

extern "C" int sun_wlop_nops(const sun_wlop* h) { return h ? h->nop : 0; }

// exact: FP64 fields equal the products multiplied one by one, bit for bit
static int fields(sun_wlop* h, int r, int mu, bool exact, hipStream_t s) {
    sun_lattice* lat = h->lat;
    HIP_TRY(lat->ops->wlop_fields(lat->f, (char*)h->ops, (char*)h->aux, h->stride, lat->g, h->family, r, mu,
                                  2.0 * std::sqrt(2.0), exact, h->planes(), s));
    h->r = r;
    h->mu = mu;
    return SUN_OK;
}

extern "C" int sun_wlop_fields(sun_wlop* h, int r, int mu, void* stream) {
    if (!h) return fail(SUN_ERR_INVALID, "sun_wlop_fields: NULL handle");
    SUN_TRY(check_radius(h, r, mu, "sun_wlop_fields"));
    hipStream_t s = pick_stream(h->lat, stream);
    HIP_TRY(hipSetDevice(h->lat->ctx->device));
    return fields(h, r, mu, true, s);
}

// Time lines that are inverted, FP32 and FP64 lattices (whose X and Y are formed in FP32 and
// FP64): up to the condition numbers at which rounding errors, which grow with their square,
// stay those of the links multiplied out (measured for Wilson loops, sun_meas.hip).  X and Y
// stay within the range times the operators (Y within its square past the lattice's end),
// far from the limits of FP32.
constexpr LineLimits kLines[2] = {{1.2, 1e8}, {2.0, 1e60}};

// the time lines of the lattice's present temporal links
static int time_lines(sun_wlop* h, hipStream_t s) {
    if (h->direct) return SUN_OK;
    const sun_lattice* lat = h->lat;
    HIP_TRY(lat->ops->time_lines(lat->f, lat->g, lat->g.X[3] + h->tmax, false,
                                 kLines[lat->d.precision == SUN_PREC_F64], h->lines, h->inverses, h->state, s));
    return SUN_OK;
}

// the correlators of the current operator field, the time lines being there
static int correlate(sun_wlop* h, int r, int mu, hipStream_t s) {
    sun_lattice* lat = h->lat;
    HIP_TRY(lat->ops->wlop_corr(lat->f, (char*)h->ops, h->stride, lat->g, h->nop, r, mu, h->tmax, h->lines, h->inverses,
                                h->direct ? nullptr : h->state, h->partials, s));
    HIP_TRY(launch_wlop_finalize(h->partials, h->rows, h->nb, h->nop, h->tmax + 1,
                                 h->direct ? nullptr : h->state, line_blocks(lat->g), h->acc, s));
    return SUN_OK;
}

extern "C" int sun_wlop_correlate(sun_wlop* h, int r, int mu, void* stream) {
    if (!h) return fail(SUN_ERR_INVALID, "sun_wlop_correlate: NULL handle");
    SUN_TRY(check_radius(h, r, mu, "sun_wlop_correlate"));
    if (h->r < 0) return fail(SUN_ERR_STATE, "sun_wlop_correlate: no operator field yet (call sun_wlop_fields)");
    sun_lattice* lat = h->lat;
    hipStream_t s = pick_stream(lat, stream);
    HIP_TRY(hipSetDevice(lat->ctx->device));
    SUN_TRY(time_lines(h, s));
    return correlate(h, r, mu, s);
}

extern "C" int sun_wlop_clear(sun_wlop* h, void* stream) {
    if (!h) return fail(SUN_ERR_INVALID, "sun_wlop_clear: NULL handle");
    hipStream_t s = pick_stream(h->lat, stream);
    HIP_TRY(hipSetDevice(h->lat->ctx->device));
    HIP_TRY(hipMemsetAsync(h->acc, 0, (size_t)h->nop * h->nop * (h->tmax + 1) * sizeof(double), s));
    return SUN_OK;
}

extern "C" int sun_wlop_read(sun_wlop* h, double* out, void* stream) {
    if (!h || !out) return fail(SUN_ERR_INVALID, "sun_wlop_read: NULL argument");
    hipStream_t s = pick_stream(h->lat, stream);
    HIP_TRY(hipSetDevice(h->lat->ctx->device));
    HIP_TRY(hipMemcpyAsync(out, h->acc, (size_t)h->nop * h->nop * (h->tmax + 1) * sizeof(double),
                           hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return SUN_OK;
}

static int sun_wlop_read_blocks_body(sun_wlop* h, int ncomp, const int* comps, const int* pos, double* out,
                                     void* stream) {
    if (!h || !out || ncomp < 0 || (ncomp > 0 && (!comps || !pos)))
        return fail(SUN_ERR_INVALID, "sun_wlop_read_blocks: bad arguments");
    for (int c = 0; c < ncomp; c++)
        if (comps[c] < 0 || pos[c] < 0 || pos[c] + comps[c] > h->nop)
            return fail(SUN_ERR_INVALID, "sun_wlop_read_blocks: component %d (%d operators from slot %d) outside %d slots",
                        c, comps[c], pos[c], h->nop);
    const int T1 = h->tmax + 1;
    std::vector<double> all((size_t)h->nop * h->nop * T1);
    SUN_TRY(sun_wlop_read(h, all.data(), stream));
    size_t id = 0;
    for (int c = 0; c < ncomp; c++)
        for (int a = 0; a < comps[c]; a++)
            for (int b = 0; b < comps[c]; b++, id++) {
                const int i = pos[c] + a, j = pos[c] + b;
                memcpy(out + id * T1, all.data() + (size_t)(i * h->nop + j) * T1, T1 * sizeof(double));
            }
    return SUN_OK;
}

extern "C" int sun_wlop_read_blocks(sun_wlop* h, int ncomp, const int* comps, const int* pos, double* out,
                                    void* stream) {
    return guard_alloc("sun_wlop_read_blocks",
                       [&] { return sun_wlop_read_blocks_body(h, ncomp, comps, pos, out, stream); });
}

static int sun_wlop_fields_to_host_body(sun_wlop* h, double* out) {
    if (!h || !out) return fail(SUN_ERR_INVALID, "sun_wlop_fields_to_host: NULL argument");
    if (h->r < 0) return fail(SUN_ERR_STATE, "sun_wlop_fields_to_host: no operator field yet");
    sun_lattice* lat = h->lat;
    HIP_TRY(hipSetDevice(lat->ctx->device));
    HIP_TRY(hipStreamSynchronize(pick_stream(lat, nullptr)));
    HIP_TRY(hipDeviceSynchronize());
    const size_t V = (size_t)lat->g.V;
    const int nreal = 2 * lat->d.nc * lat->d.nc;
    const bool f32 = lat->d.precision == SUN_PREC_F32;
    std::vector<float> raw(f32 ? V * nreal : 0);
    std::vector<double> planes(h->planes() ? h->stride / sizeof(double) : 0);
    for (int k = 0; k < h->nop; k++) {
        double* dst = out + (size_t)k * V * nreal;
        if (h->planes()) {  // of 16 bytes: real q of site l
            const size_t per = f32 ? 4 : 2;
            HIP_TRY(hipMemcpy(planes.data(), (char*)h->ops + (size_t)k * h->stride, h->stride, hipMemcpyDeviceToHost));
            const float* p32 = (const float*)planes.data();
            for (size_t q = 0; q < (size_t)nreal; q++)
                for (size_t l = 0; l < V; l++) {
                    const size_t at = (q / per * V + l) * per + q % per;
                    dst[l * nreal + q] = f32 ? p32[at] : planes[at];
                }
            continue;
        }
        if (!f32) {
            HIP_TRY(hipMemcpy(dst, (char*)h->ops + (size_t)k * h->stride, h->stride, hipMemcpyDeviceToHost));
            continue;
        }
        HIP_TRY(hipMemcpy(raw.data(), (char*)h->ops + (size_t)k * h->stride, h->stride, hipMemcpyDeviceToHost));
        for (size_t q = 0; q < V * nreal; q++) dst[q] = raw[q];
    }
    return SUN_OK;
}

extern "C" int sun_wlop_fields_to_host(sun_wlop* h, double* out) {
    return guard_alloc("sun_wlop_fields_to_host", [&] { return sun_wlop_fields_to_host_body(h, out); });
}

// test.cpp:273-298 with the operator basis of `family`: for r = 2..rmax the
// correlators of every slot pair summed over mu < 3, divided by 3 N V
static int sun_wilson_loops_ops_body(sun_lattice* lat, int family, int rmax, int tmax, double* out, void* stream) {
    if (!lat || !out) return fail(SUN_ERR_INVALID, "sun_wilson_loops_ops: NULL argument");
    const Geom& g = lat->g;
    if (rmax < 2 || rmax > g.X[0] || rmax > g.X[1] || rmax > g.X[2])
        return fail(SUN_ERR_INVALID, "sun_wilson_loops_ops: rmax %d outside 2..(smallest spatial extent)", rmax);
    sun_wlop* h = nullptr;
    SUN_TRY(create(lat, family, tmax, true, &h));
    const size_t n = (size_t)h->nop * h->nop * (tmax + 1);
    const double norm = (double)g.V * 3.0 * lat->d.nc;  // test.cpp:290
    const hipStream_t s = pick_stream(lat, stream);
    int rc = time_lines(h, s);
    for (int r = 2; r <= rmax && rc == SUN_OK; r++) {
        rc = sun_wlop_clear(h, stream);
        for (int mu = 0; mu < 3 && rc == SUN_OK; mu++) {
            rc = fields(h, r, mu, false, s);
            if (rc == SUN_OK) rc = correlate(h, r, mu, s);
        }
        if (rc == SUN_OK) rc = sun_wlop_read(h, out + (size_t)(r - 2) * n, stream);
        if (rc == SUN_OK)
            for (size_t k = 0; k < n; k++) out[(size_t)(r - 2) * n + k] /= norm;
    }
    sun_wlop_destroy(h);
    return rc;
}

extern "C" int sun_wilson_loops_ops(sun_lattice* lat, int family, int rmax, int tmax, double* out, void* stream) {
    return guard_alloc("sun_wilson_loops_ops",
                       [&] { return sun_wilson_loops_ops_body(lat, family, rmax, tmax, out, stream); });
}
