// sun_meas.hip -- the reference's measurement chain on a resident lattice (host
// code): APE smearing (smear/ape.cu:198-264), stout smearing (smear/stout.cu:687-766),
// HYP smearing (smear/hyp.cu:277-368), spatial multihit (smear/multihitsp.cu:246-266),
// multihit of temporal links (smear/multihit.cu:291-333), extended multihit
// (smear/multihitext.cu:395-459) and Wilson loops (meas/wilsonloop.cu:494-516).
// Scratch (the ping-pong field of APE, the Wilson lines and partial sums) is the
// context's, taken for the length of a call.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "sun_internal.hpp"

using namespace sun;

namespace {

int check_lattice(const sun_lattice* lat, const char* what) {
    if (!lat) return fail(SUN_ERR_INVALID, "%s: NULL lattice", what);
    if (lat->external) return fail(SUN_ERR_STATE, "%s: not available on a server job's lattice", what);
    return SUN_OK;
}

}  // namespace

extern "C" int sun_ape_smear(sun_lattice* lat, double w, int steps, int nhit, double tol, int time_dir,
                             void* stream) {
    SUN_TRY(check_lattice(lat, "sun_ape_smear"));
    if (steps < 0 || nhit < 0 || !(w >= 0.0) || (time_dir != 0 && time_dir != 1))
        return fail(SUN_ERR_INVALID, "sun_ape_smear: steps %d, nhit %d, w %g, time_dir %d", steps, nhit, w,
                    time_dir);
    if (steps == 0) return SUN_OK;
    hipStream_t s = pick_stream(lat, stream);
    HIP_TRY(hipSetDevice(lat->ctx->device));
    CallScratch tmp(lat->ctx, s);
    HIP_TRY(tmp.take(lat->bytes));
    // ping-pong between the lattice and a copy: every direction of a step reads the
    // field of the previous step (ape.cu:209-214); the directions a step does not
    // smear are equal in both buffers
    HIP_TRY(hipMemcpyAsync(tmp.at(), lat->buf, lat->bytes, hipMemcpyDeviceToDevice, s));
    const Field other = make_field(tmp.at(), 4 * (size_t)lat->g.V, link_bytes(&lat->d));
    for (int st = 0; st < steps; st++) {
        const Field& src = (st & 1) ? other : lat->f;
        const Field& dst = (st & 1) ? lat->f : other;
        for (int mu = time_dir ? 3 : 0; mu < (time_dir ? 4 : 3); mu++)
            HIP_TRY(lat->ops->ape(src, dst, lat->g, mu, w, nhit, tol, s));
    }
    if (steps & 1) HIP_TRY(hipMemcpyAsync(lat->buf, tmp.at(), lat->bytes, hipMemcpyDeviceToDevice, s));
    HIP_TRY(tmp.sync());
    return SUN_OK;
}

extern "C" int sun_stout_smear(sun_lattice* lat, double rho, int steps, int time_dir, void* stream) {
    SUN_TRY(check_lattice(lat, "sun_stout_smear"));
    if (!lat->ops->stout) return fail(SUN_ERR_UNSUPPORTED, "sun_stout_smear: SU(3) only (N = %d)", lat->d.nc);
    if (steps < 0 || !(rho >= 0.0) || (time_dir != 0 && time_dir != 1))
        return fail(SUN_ERR_INVALID, "sun_stout_smear: steps %d, rho %g, time_dir %d", steps, rho, time_dir);
    if (steps == 0) return SUN_OK;
    hipStream_t s = pick_stream(lat, stream);
    HIP_TRY(hipSetDevice(lat->ctx->device));
    CallScratch tmp(lat->ctx, s);
    HIP_TRY(tmp.take(lat->bytes));
    // the ping-pong of sun_ape_smear: every direction of a step reads the previous
    // step's field (stout.cu:697-705)
    HIP_TRY(hipMemcpyAsync(tmp.at(), lat->buf, lat->bytes, hipMemcpyDeviceToDevice, s));
    const Field other = make_field(tmp.at(), 4 * (size_t)lat->g.V, link_bytes(&lat->d));
    for (int st = 0; st < steps; st++) {
        const Field& src = (st & 1) ? other : lat->f;
        const Field& dst = (st & 1) ? lat->f : other;
        for (int mu = time_dir ? 3 : 0; mu < (time_dir ? 4 : 3); mu++)
            HIP_TRY(lat->ops->stout(src, dst, lat->g, mu, rho, s));
    }
    if (steps & 1) HIP_TRY(hipMemcpyAsync(lat->buf, tmp.at(), lat->bytes, hipMemcpyDeviceToDevice, s));
    HIP_TRY(tmp.sync());
    return SUN_OK;
}

extern "C" int sun_hyp_smear(sun_lattice* lat, double alpha1, double alpha2, double alpha3, int steps, int nhit,
                             double tol, int time_dir, void* stream) {
    SUN_TRY(check_lattice(lat, "sun_hyp_smear"));
    if (steps < 0 || nhit < 0 || (time_dir != 0 && time_dir != 1) || !(alpha1 >= 0.0) || !(alpha2 >= 0.0) ||
        !(alpha3 >= 0.0))
        return fail(SUN_ERR_INVALID, "sun_hyp_smear: steps %d, nhit %d, alphas %g %g %g, time_dir %d", steps, nhit,
                    alpha1, alpha2, alpha3, time_dir);
    if (steps == 0) return SUN_OK;
    hipStream_t s = pick_stream(lat, stream);
    HIP_TRY(hipSetDevice(lat->ctx->device));
    const size_t full = (size_t)2 * lat->d.nc * lat->d.nc * (size_t)lat->d.precision;  // 18-real record
    const size_t one = (size_t)lat->g.V * full;  // one pair's field
    Field views[24];
    const size_t at_tab = (lat->bytes + 255) & ~(size_t)255, at_pairs = at_tab + ((sizeof(views) + 255) & ~(size_t)255);
    CallScratch tmp(lat->ctx, s);
    HIP_TRY(tmp.take(at_pairs + 24 * one));
    // 12 separate V-link fields per level (site-indexed plane views), as a device table
    for (int p = 0; p < 24; p++) views[p] = make_field(tmp.at(at_pairs + p * one), (size_t)lat->g.V, full);
    HIP_TRY(hipMemcpyAsync(tmp.at(at_tab), views, sizeof(views), hipMemcpyHostToDevice, s));
    const Field* fb = (const Field*)tmp.at(at_tab);
    const Field* ft = fb + 12;
    // the ping-pong of sun_ape_smear (hyp.cu:291-313): each step reads the previous field
    HIP_TRY(hipMemcpyAsync(tmp.at(), lat->buf, lat->bytes, hipMemcpyDeviceToDevice, s));
    const Field other = make_field(tmp.at(), 4 * (size_t)lat->g.V, link_bytes(&lat->d));
    for (int st = 0; st < steps; st++) {
        const Field& src = (st & 1) ? other : lat->f;
        const Field& dst = (st & 1) ? lat->f : other;
        HIP_TRY(lat->ops->hyp(src, fb, ft, dst, lat->g, time_dir ? 3 : 0, time_dir ? 4 : 3, alpha1, alpha2, alpha3,
                              nhit, tol, s));
    }
    if (steps & 1) HIP_TRY(hipMemcpyAsync(lat->buf, tmp.at(), lat->bytes, hipMemcpyDeviceToDevice, s));
    HIP_TRY(tmp.sync());
    return SUN_OK;
}

// the output of a multihit: another lattice, same context, N, precision and extents,
// 18-real storage (a mean of SU(N) matrices is not in SU(N))
static int check_average_output(const sun_lattice* in, const sun_lattice* out, const char* what) {
    SUN_TRY(check_lattice(in, what));
    SUN_TRY(check_lattice(out, what));
    if (in == out) return fail(SUN_ERR_INVALID, "%s: the output must be another lattice", what);
    if (out->d.storage != 18)
        return fail(SUN_ERR_INVALID, "%s: the output lattice must use 18-real storage (the averaged links are not "
                                     "in SU(N))", what);
    if (in->ctx != out->ctx || in->d.nc != out->d.nc || in->d.precision != out->d.precision)
        return fail(SUN_ERR_INVALID, "%s: input and output differ in context, N or precision", what);
    for (int i = 0; i < 4; i++)
        if (in->d.dims[i] != out->d.dims[i]) return fail(SUN_ERR_INVALID, "%s: the extents differ", what);
    return SUN_OK;
}

extern "C" int sun_multihit_space(sun_lattice* in, sun_lattice* out, int nhit, void* stream) {
    SUN_TRY(check_average_output(in, out, "sun_multihit_space"));
    if (nhit < 1) return fail(SUN_ERR_INVALID, "sun_multihit_space: nhit %d (the mean needs at least one)", nhit);
    hipStream_t s = pick_stream(in, stream);
    HIP_TRY(hipSetDevice(in->ctx->device));
    HIP_TRY(in->ops->multihit_space(in->f, out->f, in->g, nhit, s));
    HIP_TRY(hipStreamSynchronize(s));
    return SUN_OK;
}

extern "C" int sun_multihit(sun_lattice* in, sun_lattice* out, uint64_t seed, int nhit, void* stream) {
    SUN_TRY(check_average_output(in, out, "sun_multihit"));
    if (nhit < 0) return fail(SUN_ERR_INVALID, "sun_multihit: nhit %d", nhit);
    hipStream_t s = pick_stream(in, stream);
    HIP_TRY(hipSetDevice(in->ctx->device));
    HIP_TRY(in->ops->multihit(in->f, out->f, in->g, seed, nhit, in->d.beta / (double)in->d.nc, s));
    HIP_TRY(hipStreamSynchronize(s));
    return SUN_OK;
}

extern "C" int sun_multihit_ext(sun_lattice* in, sun_lattice* out, uint64_t seed, int nhit, void* stream) {
    SUN_TRY(check_average_output(in, out, "sun_multihit_ext"));
    if (nhit < 1) return fail(SUN_ERR_INVALID, "sun_multihit_ext: nhit %d (the mean needs at least one)", nhit);
    hipStream_t s = pick_stream(in, stream);
    HIP_TRY(hipSetDevice(in->ctx->device));
    HIP_TRY(in->ops->multihit_ext(in->f, out->f, in->g, seed, nhit, in->d.beta / (double)in->d.nc, s));
    HIP_TRY(hipStreamSynchronize(s));
    return SUN_OK;
}

// Wilson loops by planes (sun_ops.hpp PlaneShape): the time lines, then radii in groups
// whose partial sums fit what there is
namespace {

struct WlPlanes {
    PlaneShape ps[2];  // time lines near to unitary, others
    size_t off, lines, per_radius;  // bytes: of the lines, with what they are off unitary, of the sums of a radius
    bool fits() const { return ps[0].sites && ps[1].sites; }
};

WlPlanes wl_planes(const sun_lattice* lat, int tmax) {
    const Geom& g = lat->g;
    const size_t reals = (size_t)2 * lat->d.nc * lat->d.nc;
    WlPlanes w;
    const bool f64 = lat->d.precision == SUN_PREC_F64;
    w.ps[0] = plane_shape(g, tmax + 1, (int)(reals * lat->d.precision), lat->d.nc == 2 || (lat->d.nc == 3 && !f64));
    w.ps[1] = plane_shape(g, tmax + 1, (int)(reals * sizeof(double)), lat->d.nc == 2);
    w.off = ((size_t)g.str[3] * (g.X[3] + 1) * reals * sizeof(double) + 255) & ~(size_t)255;
    w.lines = w.off + (((size_t)g.V * (reals / 2 + 3) * lat->d.precision + 255) & ~(size_t)255);
    w.per_radius = (size_t)3 * (tmax + 1) * std::max(w.ps[0].blocks, w.ps[1].blocks) * sizeof(double2);
    return w;
}

// of sun_wilson_loops_noalloc: the line field and the partial sums of the multiplied-out loops
size_t wl_line_bytes(const sun_lattice* lat) {
    return (3 * (size_t)lat->g.V * 2 * lat->d.nc * lat->d.nc * (size_t)lat->d.precision + 255) & ~(size_t)255;
}
size_t wl_part_bytes(const sun_lattice* lat, int tmax) {
    return (size_t)3 * (tmax + 1) * monitor_blocks(lat->g) * sizeof(double2);
}

bool wl_fits_noalloc(const sun_lattice* lat, int tmax) {
    return wl_line_bytes(lat) + wl_part_bytes(lat, tmax) <= kNoAllocScratchBytes;
}

// Planes cost the time lines, a chain over the lattice's times; multiplied out, every radius and
// T costs its products.  Estimates of both, us: a launch's latency, and per time, radius, T and
// 2^20 sites what calls of 4^4 to 32^4 with r <= 8 and T <= 16 take (rows N = 2, 3, 4, FP32 and FP64;
// fitted to 1458 calls by either route).  The route so chosen takes 0.7 % more than the better
// one on the average, at most 8 % more than multiplied out before there were planes (SU(3) FP32
// r, T <= 1: 4^3 x 128 219 us by planes, 52 multiplied out; 24^3 x 32 r = 4, T = 0 366 and 352, r = 8 549
// and 616; r, T <= 2 at 16^4 102 and 103).
struct WlCost {
    double time, site, radius, radius_site, loop_site;       // planes
    double p_radius, p_loop, p_site, p_loop_site;            // products
};
constexpr WlCost kWlCost[3][2] = {
    {{0.44, 68, 2.7, 33, 2.0, 2.7, 0.9, 63, 18}, {0.51, 82, 2.8, 53, 2.8, 2.8, 1.1, 117, 38}},
    {{1.2, 153, 4.8, 97, 4.8, 2.7, 1.7, 122, 45}, {1.5, 235, 5.6, 167, 8.5, 3.5, 2.6, 270, 128}},
    {{2.4, 326, 10, 329, 13, 3.4, 2.8, 257, 106}, {3.0, 398, 18, 649, 45, 2.9, 4.4, 582, 302}}};
bool wl_planes_faster(const sun_lattice* lat, int rmax, int tmax) {
    const Geom& g = lat->g;
    const WlCost& c = kWlCost[lat->d.nc - 2][lat->d.precision == SUN_PREC_F64];
    const double sites = (double)g.V / (1 << 20);
    double planes = 56 + c.time * g.X[3] + c.site * sites;
    planes += rmax * (c.radius + sites * (c.radius_site + c.loop_site * (tmax + 1)));
    // the launches of sun_wilson_loops_noalloc's other route, which find nothing to do
    if (wl_fits_noalloc(lat, tmax)) planes += 3.6 * (rmax + 1);
    const double radius = c.p_radius + c.p_loop * (tmax + 1) + sites * (c.p_site + c.p_loop_site * tmax);
    return planes < 24 + (rmax + 1) * radius;
}

// Both entry points take the same route, for the same bits: by planes where they fit LDS and are
// the faster ones, except sizes that sun_wilson_loops_noalloc accepts but whose time lines its
// array does not hold
bool wl_takes_planes(const sun_lattice* lat, const WlPlanes& w, int rmax, int tmax) {
    if (!w.fits() || !wl_planes_faster(lat, rmax, tmax)) return false;
    if (!wl_fits_noalloc(lat, tmax)) return true;
    return w.lines + w.per_radius <= kNoAllocScratchBytes && line_blocks(lat->g) * sizeof(int) <= kNoAllocStateBytes;
}

double wl_scale(const sun_lattice* lat) { return 1.0 / (3.0 * lat->d.nc * (double)lat->g.V); }  // wilsonloop.cu:512

// Time lines that are inverted (FP64 arithmetic), FP32 and FP64 lattices.  Rounding errors
// grow with the square of the condition number: FP32 lattices have that to spare (1e-10 at
// 1e3).  FP64 ones have not: against multiplied-out links the errors of single loops (SU(3),
// 32 times) are 1.1 to 2.4 times as large for T = 16 to 0 up to 1.6, 1.4 to 2.5 times at 2.8, 2
// to 5 times at 10 and 15 to 41 times at 63, so they take lines up to 2.
constexpr LineLimits kWlLines[2] = {{1e3, 1e60}, {2.0, 1e60}};

int wl_by_planes(sun_lattice* lat, const WlPlanes& w, int rmax, int tmax, double* P, double2* part, size_t part_bytes,
                 int* state, double2* res, hipStream_t s) {
    const Geom& g = lat->g;
    void* E = (char*)P + w.off;
    HIP_TRY(lat->ops->time_lines(lat->f, g, g.X[3] + 1, true, kWlLines[lat->d.precision == SUN_PREC_F64], P, E, state, s));
    const int group = (int)std::min<size_t>((size_t)rmax + 1, part_bytes / w.per_radius);
    const int nb[3] = {w.ps[0].blocks, w.ps[1].blocks, 0};
    for (int r = 0; r <= rmax; r += group) {
        const int hi = std::min(rmax + 1, r + group);
        HIP_TRY(lat->ops->wl_plane(lat->f, g, r, hi, tmax + 1, g.X[3] + 1, P, E, state, w.ps, part, s));
        HIP_TRY(launch_wl_finalize(part, nb, hi - r, tmax, wl_scale(lat), state, line_blocks(g),
                                   res + (size_t)r * (tmax + 1), s));
    }
    return SUN_OK;
}

// Every product multiplied out, in `bytes` bytes at base; where state is given, only if it is
// kLinesBad.  Two line fields where sun_wilson_loops_noalloc's array holds them (for both entry
// points: the same bits), so that a radius is one launch and the sums of several radii another.
bool wl_two_fields(const sun_lattice* lat, int tmax) {
    return 2 * wl_line_bytes(lat) + wl_part_bytes(lat, tmax) <= kNoAllocScratchBytes;
}
size_t wl_products_bytes(const sun_lattice* lat, int rmax, int tmax) {
    const size_t part = wl_part_bytes(lat, tmax);
    if (!wl_two_fields(lat, tmax)) return wl_line_bytes(lat) + part;
    return std::min(2 * wl_line_bytes(lat) + (rmax + 1) * part, kNoAllocScratchBytes);
}
int wl_by_products(sun_lattice* lat, int rmax, int tmax, char* base, size_t bytes, const int* state, double2* res,
                   hipStream_t s) {
    const Geom& g = lat->g;
    const size_t full = (size_t)2 * lat->d.nc * lat->d.nc * (size_t)lat->d.precision;  // 18-real record
    const size_t line = wl_line_bytes(lat), part_bytes = wl_part_bytes(lat, tmax);
    const bool two = wl_two_fields(lat, tmax);
    const size_t sites = 3 * (size_t)g.V;
    const Field lines[2] = {make_field(base, sites, full), make_field(base + (two ? line : 0), sites, full)};
    const size_t at_part = two ? 2 * line : line;
    double2* part = reinterpret_cast<double2*>(base + at_part);
    const int nb[3] = {0, 0, monitor_blocks(g)};
    const int group = two ? (int)std::min<size_t>((size_t)rmax + 1, (bytes - at_part) / part_bytes) : 1;
    for (int lo = 0; lo <= rmax; lo += group) {
        const int hi = std::min(rmax + 1, lo + group);
        for (int r = lo; r < hi; r++) {
            double2* p = part + (r - lo) * (part_bytes / sizeof(double2));
            if (!two) HIP_TRY(lat->ops->wl_lines(lat->f, lines[0], g, r, state, s));
            HIP_TRY(lat->ops->wl_loops(lat->f, lines[two ? r & 1 : 0], two ? &lines[~r & 1] : nullptr, r == rmax, g, r, tmax,
                                       state, p, s));
        }
        HIP_TRY(launch_wl_finalize(part, nb, hi - lo, tmax, wl_scale(lat), state, line_blocks(g),
                                   res + (size_t)lo * (tmax + 1), s));
    }
    return SUN_OK;
}

}  // namespace

static int sun_wilson_loops_body(sun_lattice* lat, int rmax, int tmax, double* out, void* stream) {
    SUN_TRY(check_lattice(lat, "sun_wilson_loops"));
    if (!out) return fail(SUN_ERR_INVALID, "sun_wilson_loops: NULL output");
    const Geom& g = lat->g;
    if (rmax < 0 || tmax < 0 || rmax > g.X[0] || rmax > g.X[1] || rmax > g.X[2] || tmax > g.X[3])
        return fail(SUN_ERR_INVALID, "sun_wilson_loops: rmax %d, tmax %d outside the lattice", rmax, tmax);
    hipStream_t s = pick_stream(lat, stream);
    HIP_TRY(hipSetDevice(lat->ctx->device));
    const size_t nres = (size_t)(rmax + 1) * (tmax + 1), res_bytes = (nres * sizeof(double2) + 255) & ~(size_t)255;
    std::vector<double2> h(nres);
    const WlPlanes w = wl_planes(lat, tmax);
    bool done = false;
    if (wl_takes_planes(lat, w, rmax, tmax)) {
        constexpr size_t kPartBytes = size_t(64) << 20;  // of partial sums at a time
        const size_t part = std::max(w.per_radius, std::min(w.per_radius * (rmax + 1), kPartBytes));
        std::vector<int> st(line_blocks(g));
        CallScratch mem(lat->ctx, s);
        const hipError_t e = mem.take(w.lines + part + res_bytes + st.size() * sizeof(int));
        if (e == hipErrorOutOfMemory) {  // the other route may do with less
            hipGetLastError();
        } else {
            HIP_TRY(e);
            char* p = mem.at();
            double2* res = (double2*)(p + w.lines);
            int* state = (int*)(p + w.lines + res_bytes + part);
            SUN_TRY(wl_by_planes(lat, w, rmax, tmax, (double*)p, (double2*)(p + w.lines + res_bytes), part, state, res, s));
            HIP_TRY(hipMemcpyAsync(h.data(), res, nres * sizeof(double2), hipMemcpyDeviceToHost, s));
            HIP_TRY(hipMemcpyAsync(st.data(), state, st.size() * sizeof(int), hipMemcpyDeviceToHost, s));
            HIP_TRY(mem.sync());
            done = std::find(st.begin(), st.end(), kLinesBad) == st.end();
        }
    }
    if (!done) {
        const size_t at_res = wl_products_bytes(lat, rmax, tmax);
        CallScratch mem(lat->ctx, s);
        HIP_TRY(mem.take(at_res + res_bytes));
        SUN_TRY(wl_by_products(lat, rmax, tmax, mem.at(), at_res, nullptr, (double2*)mem.at(at_res), s));
        HIP_TRY(hipMemcpyAsync(h.data(), mem.at(at_res), nres * sizeof(double2), hipMemcpyDeviceToHost, s));
        HIP_TRY(mem.sync());
    }
    for (size_t i = 0; i < nres; i++) {
        out[2 * i] = h[i].x;
        out[2 * i + 1] = h[i].y;
    }
    return SUN_OK;
}

extern "C" int sun_wilson_loops(sun_lattice* lat, int rmax, int tmax, double* out, void* stream) {
    return guard_alloc("sun_wilson_loops", [&] { return sun_wilson_loops_body(lat, rmax, tmax, out, stream); });
}

// The same kernels with the lines and the partial sums in the device's scratch array (its
// address from sun_init) and the results written straight to the caller's device buffer:
// no allocation and no host synchronisation, so both routes are launched and the state of
// the time lines decides on the device which one does anything.  Everything is written
// before it is read, so nothing left in the array by an earlier call is used.
extern "C" int sun_wilson_loops_noalloc(sun_lattice* lat, int rmax, int tmax, double* dev_out, void* stream) {
    SUN_TRY(check_lattice(lat, "sun_wilson_loops_noalloc"));
    if (!dev_out || (reinterpret_cast<uintptr_t>(dev_out) & 15u) != 0)
        return fail(SUN_ERR_INVALID, "sun_wilson_loops_noalloc: dev_out must be a 16-byte aligned device pointer");
    const Geom& g = lat->g;
    if (rmax < 0 || tmax < 0 || rmax > g.X[0] || rmax > g.X[1] || rmax > g.X[2] || tmax > g.X[3])
        return fail(SUN_ERR_INVALID, "sun_wilson_loops_noalloc: rmax %d, tmax %d outside the lattice", rmax, tmax);
    if (!lat->ctx->scratch) return fail(SUN_ERR_STATE, "sun_wilson_loops_noalloc: no scratch array on this device");
    const size_t line_bytes = wl_line_bytes(lat), part_bytes = wl_part_bytes(lat, tmax);
    if (line_bytes + part_bytes > kNoAllocScratchBytes)
        return fail(SUN_ERR_BUDGET,
                    "sun_wilson_loops_noalloc: needs %zu bytes of scratch (line field %zu + partials %zu), the "
                    "array holds %zu; use sun_wilson_loops",
                    line_bytes + part_bytes, line_bytes, part_bytes, kNoAllocScratchBytes);
    hipStream_t s = pick_stream(lat, stream);
    HIP_TRY(hipSetDevice(lat->ctx->device));
    unsigned char* base = static_cast<unsigned char*>(lat->ctx->scratch);
    double2* res = reinterpret_cast<double2*>(dev_out);
    const WlPlanes w = wl_planes(lat, tmax);
    int* state = nullptr;
    if (wl_takes_planes(lat, w, rmax, tmax)) {
        state = reinterpret_cast<int*>(base + kNoAllocScratchBytes);
        SUN_TRY(wl_by_planes(lat, w, rmax, tmax, reinterpret_cast<double*>(base),
                             reinterpret_cast<double2*>(base + w.lines), kNoAllocScratchBytes - w.lines, state, res, s));
    }
    return wl_by_products(lat, rmax, tmax, reinterpret_cast<char*>(base), kNoAllocScratchBytes, state, res, s);
}
