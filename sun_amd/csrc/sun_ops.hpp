// sun_ops.hpp -- the per-variant launcher table shared by the kernel translation
// units and the C-ABI layer.  One table exists for every (N, storage, precision)
// combination the engine supports; the C-ABI picks the table of a lattice once at
// creation.
#pragma once

#include <hip/hip_runtime.h>

#include "sun_field.hpp"

namespace sun {

// Launch shape chosen by the autotuner.
struct LaunchCfg {
    int block = 256;
    // dynamic LDS reserved per workgroup and not used by the kernel: caps the
    // workgroups resident per CU (160 KB of LDS per CU), i.e. the lattice volume in
    // flight per XCD, which decides whether neighbour links are still in L2 when
    // the next staple direction needs them
    int lds = 0;
    // brick mapping (brick_site) when b1 >= 0: log2 of the rows per workgroup along
    // x1, x2, x3; b1 < 0: linear mapping with `block` threads
    int b1 = -1, b2 = 0, b3 = 0;
    // 1: the software-pipelined overrelaxation kernel (where the variant has one)
    int piped = 0;
    // the kernel that shares a link's staple among waves, whatever the rest says: of small
    // lattices (default_launch) for which nobody has set a shape
    bool split = false;
};

// Brick mapping of workgroups to lattice sites.  The sites of one parity form rows
// of L = X0/2 consecutive ids (fixed x1, x2, x3).  Workgroup b takes a brick of
// 2^b1 x 2^b2 x 2^b3 rows along (x1, x2, x3) -- L * 2^(b1+b2+b3) threads, row
// index x1-fastest inside the brick, bricks numbered x1-fastest -- so the sites
// whose staples share links sit in one workgroup, on one CU, at the same time.
// Returns the site id within the parity of thread t of workgroup b.
SUN_HD int brick_site(const Geom& g, int b, int t, int b1, int b2, int b3) {
    const int L = g.X[0] >> 1;
    const int row = (int)g.dxh.div((uint32_t)t);
    const int s = t - row * L;
    const int i1 = row & ((1 << b1) - 1);
    const int i2 = (row >> b1) & ((1 << b2) - 1);
    const int i3 = row >> (b1 + b2);
    const int n1 = g.X[1] >> b1, n2 = g.X[2] >> b2;
    const int B23 = b / n1, B1 = b - B23 * n1;
    const int B3 = B23 / n2, B2 = B23 - B3 * n2;
    const int x1 = (B1 << b1) + i1, x2 = (B2 << b2) + i2, x3 = (B3 << b3) + i3;
    return ((x3 * g.X[2] + x2) * g.X[1] + x1) * L + s;
}

constexpr int kReduceBlock = 256;   // threads of every reduction block

// site (0 <= idd < V, parity-major) of thread t of reduction workgroup lb of a
// lattice: workgroups 2k and 2k+1 take brick k of parity 0 and of parity 1 (whose
// links are each other's neighbours, so they run on the same XCD and share its L2);
// linear when the geometry has no reduction brick.  The single-lattice and the
// batched plaquette kernels share it, so their per-workgroup partial sums agree.
SUN_HD int reduce_site(const Geom& g, int lb, int t) {
    if (g.rb1 < 0) return lb * kReduceBlock + t;
    const int parity = lb & 1;
    return parity * g.half + brick_site(g, lb >> 1, t, g.rb1, g.rb2, g.rb3);
}

// threads per workgroup of a brick shape on this geometry, or 0 when the brick does
// not tile the lattice or the workgroup is not whole wavefronts within max_block
inline int brick_block(const Geom& g, int b1, int b2, int b3, int max_block) {
    if (b1 < 0 || b2 < 0 || b3 < 0 || b1 > 6 || b2 > 6 || b3 > 6) return 0;
    if ((g.X[1] % (1 << b1)) || (g.X[2] % (1 << b2)) || (g.X[3] % (1 << b3))) return 0;
    const long long block = (long long)(g.X[0] / 2) << (b1 + b2 + b3);
    if (block < 64 || block > max_block || (block % 64)) return 0;
    return (int)block;
}

// One lattice of a batched launch.  `first_block` is the prefix sum of the blocks
// of the preceding lattices; a block finds its lattice by binary search.  Each
// kind of batched launch (update, reunitarisation, plaquette, Polyakov loop) has
// its own table because the blocks per lattice differ.
struct BatchEntry {
    Field f;
    Geom g;
    uint64_t seed;
    double bnc;          // beta / N
    uint32_t sweep;      // heatbath sweep counter of this lattice
    int first_block;
    int nblocks;
    double2* partials;   // this lattice's per-block reduction scratch (nblocks entries)
    double scale;        // normalisation of the reduced sum
    double2* hist;       // observable history: {plaquette, polyakov} per iteration
    uint32_t hist_iter;  // next history row
    int ub1, ub2, ub3;   // update brick (ub1 < 0: none)
    int spt;             // 256-thread workgroups per update brick (the brick holds 256 spt sites)
};

// The update brick of a batched lattice: 256 * spt sites = (X0/2) * 2^k rows, taken by
// spt consecutive 256-thread workgroups (same XCD, side by side; every workgroup of a
// batch does the same work, so the XCDs' contiguous ranges stay balanced).  spt = 1
// where rows of X0/2 tile 256 sites: the k doublings go to x1, x3, x1, x3 (the tuned
// single-lattice shape at 32^4 is such a (2, 0, 2) brick), then x2, x2, then
// round-robin, each only where the extent stays divisible.  Else spt = 3 where rows
// tile 768 sites (X0/2 = 12: 24^4, 64 rows), doublings x1, x3, x1, x3, x1, x3 (8 x 1 x
// 8 rows at 24^4: in the cache-sized chunks of a batch the best of five shapes
// measured, 4 x 2 x 8 and 4 x 4 x 4 rows 1-2% slower).  b1 < 0 (spt = 1) when no brick
// tiles the lattice.
inline void batch_brick(const Geom& g, int& b1, int& b2, int& b3, int& spt) {
    b1 = -1;
    b2 = b3 = 0;
    spt = 1;
    const int L = g.X[0] / 2;
    if (L <= 0 || L > 768) return;
    int m = 0;
    if (256 % L == 0) m = 1;
    else if (768 % L == 0 && ((768 / L) & (768 / L - 1)) == 0) m = 3;
    if (!m) return;
    int k = 0;
    while ((L << k) < 256 * m) k++;
    static const int seq1[] = {1, 3, 1, 3, 2, 2, 1, 3, 2, 1, 3, 2, 1, 3, 2, 1, 3, 2};
    static const int seq3[] = {1, 3, 1, 3, 1, 3, 2, 2, 1, 3, 2, 1, 3, 2, 1, 3, 2, 2};
    const int* seq = m == 1 ? seq1 : seq3;
    int c[4] = {0, 0, 0, 0};
    for (int i = 0; i < 18 && k > 0; i++) {
        const int d = seq[i];
        if (g.X[d] % (2 << c[d]) == 0) {
            c[d]++;
            k--;
        }
    }
    if (k > 0) return;
    b1 = c[1];
    b2 = c[2];
    b3 = c[3];
    spt = m;
}

// Wilson loops in (mu, t) planes: a workgroup of 256 threads takes `sites` spatial sites
// with all times, two per thread, and T in chunks.  LDS: the moved lines of `extent` times
// of each site (the lattice's and, going on around it, those that the last chunk reaches)
// and the waves' sums.
struct PlaneShape {
    int sites, blocks, chunk, extent;
    int sums, lds;  // bytes before the sums, and in all
};
// the shape for matrices of `bytes` bytes, or sites = 0 where the times do not fit
inline PlaneShape plane_shape(const Geom& g, int T1, int bytes, bool two_wgs) {
    constexpr int kThreads = 256, kLds = 156 * 1024;
    PlaneShape p{};
    // chunks of 5, 7 or 9 T (compiled kernels), as few as possible, then as small as possible
    const int n = (T1 + 8) / 9, need = (T1 + n - 1) / n;
    p.chunk = need <= 5 ? 5 : need <= 7 ? 7 : 9;
    p.extent = g.X[3] + (n * p.chunk + 1) / 2 * 2;
    const long long sums = 8ll * kThreads / 64 * 2 * T1;
    const long long most = (kLds - sums) / ((long long)p.extent * bytes);
    // two workgroups a CU where they fit and registers allow two (FP64 SU(4), which they do not: half of
    // the threads were without a site; SU(3) 13 sites for 16)
    const long long two = (kLds / 2 - sums) / ((long long)p.extent * bytes);
    long long sites = 2 * kThreads / g.X[3];
    if (sites > most) sites = most;
    if (two_wgs && two >= 1 && two < sites) sites = two;
    if (sites < 1 || g.X[3] > 2 * kThreads) return p;
    p.sites = (int)sites;
    p.blocks = (g.str[3] + p.sites - 1) / p.sites;
    p.sums = (p.extent * p.sites * bytes + 15) / 16 * 16;
    p.lds = p.sums + (int)sums;
    return p;
}

// What time lines may be inverted (sun_transport.inc): condition number and norms
struct LineLimits {
    double cond, range;
};

struct OpsTable {
    int nc, storage, real_bytes;
    // one (parity, mu) heatbath (hb=true) or overrelaxation launch
    // sweep_dev, when not null, overrides sweep with a device-resident counter (graph replay)
    hipError_t (*update)(const Field&, const Geom&, int parity, int mu, bool hb, uint32_t sweep,
                         const uint32_t* sweep_dev, double bnc, uint64_t seed, const LaunchCfg&, hipStream_t);
    hipError_t (*cold_start)(const Field&, int nlinks, hipStream_t);
    hipError_t (*hot_start)(const Field&, const Geom&, uint64_t seed, hipStream_t);
    hipError_t (*reunitarize)(const Field&, int nlinks, hipStream_t);
    // per-block partial sums (double2) of the plaquette (spatial, temporal) and of
    // the Polyakov loop (re, im); the number of partials is *_blocks(geom)
    hipError_t (*plaquette_partial)(const Field&, const Geom&, double2* partials, hipStream_t);
    hipError_t (*polyakov_partial)(const Field&, const Geom&, double2* partials, hipStream_t);
    hipError_t (*to_canonical)(const Field&, int nlinks, double* out, hipStream_t);
    hipError_t (*from_canonical)(const Field&, int nlinks, const double* in, hipStream_t);
    // batched: every lattice of the table, one (parity, mu) launch; piped 0 plain,
    // 1 / 2 software-pipelined staple (only where has_piped); brick: the entries'
    // update bricks (ub1 >= 0) instead of the linear site order; lds: unused dynamic
    // LDS per workgroup (occupancy cap)
    hipError_t (*batch_update)(const BatchEntry* dev_table, int nlat, int total_blocks, int parity,
                               int mu, bool hb, int piped, int brick, int lds, hipStream_t);
    hipError_t (*batch_reunitarize)(const BatchEntry* dev_table, int nlat, int total_blocks, hipStream_t);
    hipError_t (*batch_plaquette_partial)(const BatchEntry* dev_table, int nlat, int total_blocks, hipStream_t);
    hipError_t (*batch_polyakov_partial)(const BatchEntry* dev_table, int nlat, int total_blocks, hipStream_t);
    // link trace / determinant sums and unitarity deviations, 3 * monitor_blocks(geom) partials
    hipError_t (*monitor_partial)(const Field&, const Geom&, double2* partials, hipStream_t);
    // plaquette partials at [0, plaquette_blocks) and Polyakov partials after them,
    // in one launch
    hipError_t (*measure_partial)(const Field&, const Geom&, double2* partials, hipStream_t);
    // measurement chain: one APE direction in -> out; multihit in -> out (18-real
    // field of the same N and precision); Wilson lines of radius r (3V-entry 18-real
    // field, r = 0 sets the identity) and the loops of radius r, tmax + 1 extents in
    // time, 3 * (tmax + 1) * monitor_blocks(geom) partials
    hipError_t (*ape)(const Field& in, const Field& out, const Geom&, int mu, double w, int nhit, double tol,
                      hipStream_t);
    // one stout direction in -> out (SU(3) variants; null otherwise)
    hipError_t (*stout)(const Field& in, const Field& out, const Geom&, int mu, double rho, hipStream_t);
    // HYP: level-1 and level-2 fields (device tables of 12 plane views of V 18-real
    // links each) from in, then the directions [mu_lo, mu_hi) of out
    hipError_t (*hyp)(const Field& in, const Field* bar, const Field* til, const Field& out, const Geom&, int mu_lo,
                      int mu_hi, double a1, double a2, double a3, int nhit, double tol, hipStream_t);
    hipError_t (*multihit)(const Field& in, const Field& out, const Geom&, uint64_t seed, int nhit, double bnc,
                           hipStream_t);
    // spatial links -> mean of nhit overrelaxation steps, temporal copied (out 18-real)
    hipError_t (*multihit_space)(const Field& in, const Field& out, const Geom&, int nhit, hipStream_t);
    // temporal links -> mean of the centre of nhit heatbath sweeps of each site's 3^3
    // box of temporal links, spatial copied (out 18-real)
    hipError_t (*multihit_ext)(const Field& in, const Field& out, const Geom&, uint64_t seed, int nhit, double bnc,
                               hipStream_t);
    // Wilson loops of radii [r_lo, r_hi) and T < T1, moved along time lines (planes, next =
    // X3 + 1 times): 3 T1 blocks partials per radius, of the shape's blocks, ps[0] where the
    // lines are near to unitary, ps[1] where not; nothing where they are kLinesBad
    hipError_t (*wl_plane)(const Field& f, const Geom&, int r_lo, int r_hi, int T1, int next, const double* P,
                           const void* E, const int* state, const PlaneShape ps[2], double2* partials, hipStream_t);
    // the same with the links multiplied out: the Wilson lines of radius r, then its loops, or, with
    // a second field `next`, the loops and there the lines of r + 1 (none after the last radius);
    // where state is given, only if it is kLinesBad
    hipError_t (*wl_lines)(const Field& f, const Field& lines, const Geom&, int r, const int* state, hipStream_t);
    hipError_t (*wl_loops)(const Field& f, const Field& lines, const Field* next, bool last, const Geom&, int r, int tmax,
                           const int* state, double2* partials, hipStream_t);
    // operator-basis Wilson loops: the operator fields of direction mu at radius r
    // (family 0: 10 slots, 1: 25; slot k, V matrices of 2 N^2 reals one after another or, where
    // `planes`, like the links, at ops + k * stride; rt8 = 2 sqrt 2).  exact: FP64 fields with the reference's products one
    // by one (33 also where aux is null), otherwise from shared products (33: in kWlopAuxSlots more slots at aux; A0: slot
    // 9 is left as it is)
    hipError_t (*wlop_fields)(const Field& f, char* ops, char* aux, size_t stride, const Geom&, int family, int r,
                              int mu, double rt8, bool exact, bool planes, hipStream_t);
    // time lines of every spatial site: P of `next` times, inverses Q of X3 times, FP64 N x N
    // matrices; where `planes`, P element by element and Q the N^2 reals of the links'
    // precision by which P P^+ is off 1; state[line_blocks(geom)]: per block whether its lines
    // are near to unitary (0), within the limits (1) or not (kLinesBad)
    hipError_t (*time_lines)(const Field& f, const Geom&, int next, bool planes, const LineLimits& lim, double* P, void* Q,
                             int* state, hipStream_t);
    // the correlator of every slot pair; time lines of next = X3 + tmax times.  Partials:
    // [wlop_corr_blocks][T][i][j], or, where a state is kLinesBad,
    // [(i nop + j)(tmax + 1) + T][monitor_blocks]; state null: the latter, without lines
    hipError_t (*wlop_corr)(const Field& f, char* ops, size_t stride, const Geom&, int nop, int r, int mu,
                            int tmax, const double* P, const double* Q, const int* state, double* partials, hipStream_t);
    int max_block;   // largest workgroup the update kernels are compiled for
    int has_piped;   // the variant has the software-pipelined overrelaxation kernel
    int piped_max_block;
    int split_groups;  // workgroups of 64 links up to which the shared-staple kernel is the faster one
};

// The launch shape of a lattice's updates unless the tuner or the caller has one (kernel 0
// heatbath, 1 overrelaxation).  us per overrelaxation launch, 256 threads in linear order /
// the rule's shape:
// - Links that decode in registers run best software-pipelined by half-directions (12-real
//   FP32 at 20^4: 9.3 / 8.1; 8-real FP32 at 28^4: 30.4 / 28.0), except the 8-real heatbath of
//   large lattices (48^4: 252 / more than 260).
// - Up to 2^18 sites the chip is not full: one wavefront per workgroup spreads over more
//   CUs (FP64 SU(3) at 16^3 x 18: 17.7 / 16.0, at 20^4: 32.0 / 29.0, SU(4) FP32 at 8^4: 15.1 /
//   13.5; at 2^18 sites no difference).
// - Above, bricks of 16 rows (8 from X0 = 48 on), two apart in x1 and x3, keep the links that
//   neighbours share in the L2, with no more than two workgroups a CU (FP64 SU(3) at
//   24^3 x 48: 120 / 104, SU(4) FP32 at 32^4: 169 / 150, FP32 12-real at 32^4: 52.6 / 38.7;
//   no gain at 2^18 sites, nor below 2^19 for 32-byte links).  Where no brick tiles, linear
//   (40 x 32^3, 28^4: no shape is faster).
// - Decoding FP64 links is arithmetic: linear, one wavefront per workgroup (12-real heatbath
//   at 48^4: 989 / 903), but bricks for 12-real overrelaxation where they are workgroups of 256,
//   which rows of 16 and 32 sites make (32^4: 162 / 153, 64 x 32^3: 337 / 307; the 192 threads of
//   rows of 12 or 24 sites are slower than linear, 24 x 32^3 129 / 116, 48 x 32^3 269 / 241, the 128
//   of 8 sites no faster).
inline LaunchCfg default_launch(const OpsTable* ops, const Geom& g, int kernel) {
    LaunchCfg c;
    const bool f64 = ops->real_bytes == 8, full = ops->storage == 18, hb = kernel == 0;
    const int rows = g.X[0] / 2;
    c.split = (g.half + 63) / 64 <= ops->split_groups;
    const bool large = g.V > (1 << 18);
    if (ops->has_piped && (ops->storage == 12 || !hb || g.V <= (1 << 19))) c.piped = 2;
    if (!large || (f64 && !full) || (ops->storage == 8 && c.piped)) c.block = 64;
    bool brick = large && ops->storage != 8;
    if (f64 && !full) brick = brick && !hb;
    if (full && ops->nc == 2 && !f64) brick = brick && g.V >= (1 << 19);
    if (!brick) return c;
    const int b1 = rows <= 16 ? 2 : 1;
    const int block = brick_block(g, b1, 0, 2, 256);
    if (!block || (f64 && !full && block != 256)) return c;
    c.b1 = b1;
    c.b2 = 0;
    c.b3 = 2;
    c.block = block;
    c.lds = 54272;
    return c;
}

// The launch shape of batched updates unless the caller picks one (kernel 0
// heatbath, 1 overrelaxation).  Staple kernel (0 plain, 1 / 2 direction /
// half-direction pipelined): measured over 64 FP32 SU(3) lattices of 8^4..24^4 and a
// 32^4 lattice alone, half-direction pipelining is the fastest for both kernels with
// 12-real links (+3% and +17% over plain); with 8-real links for the
// overrelaxation only (+13% over 64 lattices), the pipelined heatbath being slower.
inline int default_batch_piped(const OpsTable* ops, int kernel) {
    if (!ops->has_piped) return 0;
    if (ops->storage == 12) return 2;
    return kernel == 0 ? 0 : 2;
}
// Bricks (where a 256-thread brick tiles a lattice): a 32^4 lattice runs 12% faster
// with them (its workgroups' shared neighbour links stay in one L2); over the
// 64-lattice mix they change the rate by -0.8..+1.8%.
inline int default_batch_brick(const OpsTable*, int) { return 1; }
inline int default_batch_lds(const OpsTable*, int) { return 0; }

// gfx950 dispatches workgroup b of a grid to XCD (b mod 8); each XCD has its own
// 4 MB L2.  xcd_remap turns the dispatch order into a contiguous range of tiles per
// XCD, so the lattice neighbours that share links (+-1 site, +-1 row, +-1 plane) run
// on the same L2.  A bijection of [0, nblocks) for any nblocks.
constexpr int kXcds = 8;

SUN_HD int xcd_remap(int b, int nblocks) {
    const int xcd = b % kXcds, local = b / kXcds;
    const int per = nblocks / kXcds, rem = nblocks % kXcds;
    return xcd * per + (xcd < rem ? xcd : rem) + local;
}

inline int plaquette_blocks(const Geom& g) { return (g.V + kReduceBlock - 1) / kReduceBlock; }
// Polyakov loop workgroups: kReduceBlock threads = kPolySites spatial sites x
// kPolySegs segments of each time line
constexpr int kPolySegs = 4;
constexpr int kPolySites = kReduceBlock / kPolySegs;
inline int polyakov_blocks(const Geom& g) {
    int ts = g.X[0] * g.X[1] * g.X[2];
    return (ts + kPolySites - 1) / kPolySites;
}
// maximum that keeps a NaN (fmax drops it): a monitor must not report a field that
// went non-finite as an exact one
SUN_HD double nan_max(double a, double b) {
    if (a != a) return a;
    if (b != b) return b;
    return b > a ? b : a;
}

// link monitor workgroups (one site per thread) and the partials every reduction of
// a lattice needs: the monitor writes three segments of monitor_blocks entries
inline int monitor_blocks(const Geom& g) { return (g.V + kReduceBlock - 1) / kReduceBlock; }
inline int partial_slots(const Geom& g) {
    const int a = 3 * monitor_blocks(g), b = plaquette_blocks(g) + polyakov_blocks(g);
    return a > b ? a : b;
}
// scratch slots of the 33 family's fields from shared products
constexpr int kWlopAuxSlots = 14;
// whether the operator fields of a handle have the links' plane layout (sun_wlop.inc): FP64 and
// SU(4) fields of A0 handles that multiply every link out (`direct`)
constexpr bool wlop_planes(bool direct, int nc, bool f64, int nop) { return direct && (f64 || nc == 4) && nop <= 16; }
// state of time lines that the measurement kernels cannot invert
constexpr int kLinesBad = 2;
// workgroups of the time-line kernel (64 spatial sites each)
inline int line_blocks(const Geom& g) { return (g.str[3] + 63) / 64; }
// workgroups of the matrix-core correlator, one per CU (its LDS), each with an equal share
// of the spatial sites
inline int wlop_corr_blocks(const Geom& g) { return g.str[3] < 256 ? g.str[3] : 256; }
inline int update_blocks(const Geom& g, int block) { return (g.half + block - 1) / block; }
inline int link_blocks(const Geom& g) { return (4 * g.V + kReduceBlock - 1) / kReduceBlock; }

// sum of partials[0..n) in a fixed order, times `scale`, into out (device)
hipError_t launch_finalize(const double2* partials, int n, double scale0, double scale1, double2* out,
                           hipStream_t s);
// end of a measured generation iteration, one workgroup: plaquette (partials
// [0, pb)) and Polyakov loop (partials [pb, pb + qb)) summed as launch_finalize sums,
// scaled into out[0], out[1], recorded in history row ctr - first, then ctr += 1
hipError_t launch_finalize_iteration(const double2* partials, int pb, int qb, double s_plaq, double s_poly,
                                     double2* out, double2* history, uint32_t* ctr, uint32_t first, hipStream_t s);
// Wilson loops of nr radii: out[r (tmax + 1) + T] = scale * sum over mu < 3 and the partials
// of (r, mu, T), T = 0..tmax, in a fixed order.  nb[i]: the workgroups of time lines in state
// i; where nb[i] is 0 nothing is done.  state null: nb[kLinesBad].
hipError_t launch_wl_finalize(const double2* partials, const int nb[3], int nr, int tmax, double scale,
                              const int* state, int nstate, double2* out, hipStream_t s);
// accum[(i nop + j) T1 + T] += the sum of the correlator's partials in a fixed order:
// [rows][T][i][j], or [(i nop + j) T1 + T][nb] where one of the nstate states is kLinesBad or
// state is null
hipError_t launch_wlop_finalize(const double* partials, int rows, int nb, int nop, int T1, const int* state,
                                int nstate, double* accum, hipStream_t s);
// link monitor: out[0] = trace sum * scale_tr, out[1] = determinant sum * scale_det,
// out[2] = (max deviation, max |det - 1|) from the three segments of n partials
hipError_t launch_monitor_finalize(const double2* partials, int n, double scale_tr, double scale_det, double2* out,
                                   hipStream_t s);
// finalize for every lattice of a batch table: out[i] = (sum of entry i's partials)
// * entry i's scale, in the same order as launch_finalize
hipError_t launch_batch_finalize(const BatchEntry* table, int nlat, double2* out, hipStream_t s);
// plaquette and Polyakov finalize, history record and sweep advance of a group whose
// members' plaquette and Polyakov partials are separate buffers, in one launch
hipError_t launch_group_close(BatchEntry* t_plaq, const BatchEntry* t_poly, BatchEntry* t_update, int nlat,
                              double2* plaq, double2* poly, hipStream_t s);
// entry i's history row hist_iter <- {plaq[i], poly[i]}; hist_iter += 1
hipError_t launch_batch_record(BatchEntry* table, int nlat, const double2* plaq, const double2* poly,
                               hipStream_t s);

const OpsTable* ops_n2_f18_r4();
const OpsTable* ops_n2_f18_r8();
const OpsTable* ops_n3_f18_r4();
const OpsTable* ops_n3_f18_r8();
const OpsTable* ops_n3_f12_r4();
const OpsTable* ops_n3_f12_r8();
const OpsTable* ops_n3_f8_r4();
const OpsTable* ops_n3_f8_r8();
const OpsTable* ops_n4_f18_r4();
const OpsTable* ops_n4_f18_r8();

inline const OpsTable* find_ops(int nc, int storage, int real_bytes) {
    const OpsTable* all[] = {ops_n2_f18_r4(), ops_n2_f18_r8(), ops_n3_f18_r4(), ops_n3_f18_r8(),
                             ops_n3_f12_r4(), ops_n3_f12_r8(), ops_n3_f8_r4(),  ops_n3_f8_r8(),
                             ops_n4_f18_r4(), ops_n4_f18_r8()};
    for (const OpsTable* t : all)
        if (t->nc == nc && t->storage == storage && t->real_bytes == real_bytes) return t;
    return nullptr;
}

}  // namespace sun
