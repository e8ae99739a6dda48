// k_fstrength.hip -- lattice field strengths F_munu(x) = TA(sum of closed loops at x) and what
// is measured from them: the topological charge density with the plaquette, clover and 2x1
// rectangle loop sets (improved = 5/3 clover - 1/12 rectangle) and the clover energy density.
//
// Reference: _plaquette/_clover/_rectangle_field_strengths and the matching
// *_topological_charge_density (AbstractGaugefields.jl:1195-1397), make_cloverloops
// (autostaples/wilsonloops.jl:166-177), calculate_energy_density
// (samples/measurements/energydensity.jl:32-76).
//
// With F = sum_a c_a i lambda_a / 2, tr(F F') = -(1/2) c . c', so
//   sum_{mu nu rho sigma} eps tr(F_munu F_rhosigma) = -4 (c01.c23 - c02.c13 + c03.c12)
// and the density -norm Re(...) / (32 pi^2 n_loops^2) = norm (c01.c23 - c02.c13 + c03.c12) /
// (8 pi^2 n_loops^2); the clover energy sum_{mu != nu} -tr(F F)/2 / 16 = sum_planes |c|^2 / 32.
//
// Loops through x in the plane (a, b), a < b, come in pairs: with S_up(x), S_low(x) the open paths from
// x + a back to x above and below the link U_a(x), the two loops that leave x along +a are U_a S_up and
// (U_a S_low)^dag, and TA(M^dag) = -TA(M), so their sum is TA(U_a K), K = S_up - S_low; the two that come
// back along +a, through z = x - a, are TA(K(z) U_a(z)).  A site therefore forms K once, for itself (near)
// and for x + a (far): clover leaves 6 products instead of 12, a x 2b rectangles (paths of height 2) 10
// instead of 20, 2a x b rectangles (the double link D = U_a(x) U_a(x+a) in place of U_a, far site x + 2a) 9
// instead of 20.  k_loops stores near and far coefficients, k_charge adds near(x) and far(x - a) and
// contracts the planes.  No step goes along t, so both run over blocks of whole t-slices, which bounds the
// buffer between them (256 MB: 24^3x48 FP64 clover / improved charge 296 / 821 us; 128 MB 312 / 876, 512 MB
// 324 / 830; 32^4 475 / 1283, 493 / 1327, 495 / 1286).  Against walking every loop from x in one kernel, clover /
// improved charge with the readback: 32^4 FP64 533 / 2030 -> 475 / 1283 us, 24^3x48 334 / 1290 -> 296 / 821, 20^3x10
// 94 / 238 -> 49 / 107, 8^4 37 / 66 -> 23 / 30; FP32 links 32^4 562 / 2047 -> 403 / 1286.  k_loops is bound by the L2
// reads of links up to two steps away and by the products.
// Products are evaluated in double for both storage precisions.
#include <algorithm>

#include "internal.hpp"

namespace gf {

namespace {

// Product of links along a path.  FP64 links are SU(3) to double rounding, so every partial product is too:
// only its rows 0 and 1 are formed (72 instead of 108 FMAs per product) and row 2 rebuilt where the next
// step needs it.  FP32-stored links are unitary only to float rounding, which the cross product would
// carry into every partial product: there the full products are formed.  Links are widened to double
// before row 2 is rebuilt, as in every FP64 sum over FP32-stored links.
template <typename T>
struct Path;
template <>
struct Path<double> {
    R6<double> r;
    __device__ __forceinline__ void start(const R6<double>& l) { r = l; }
    __device__ __forceinline__ void mul(const R6<double>& l) { r = rows_of(su3_mul(r, full_of(l))); }
    __device__ __forceinline__ void mul_dag(const R6<double>& l) { r = rows_of(su3_mul_nd(r, full_of(l))); }
    // this^dag l
    __device__ __forceinline__ void dag_mul(const R6<double>& l) {
        r = rows_of(su3_mul(rows_of(dag(full_of(r))), full_of(l)));
    }
    __device__ __forceinline__ M3<double> get() const { return full_of(r); }
};
template <>
struct Path<float> {
    M3<double> m;
    static __device__ __forceinline__ M3<double> wide(const R6<float>& l) { return full_of(r6_f64(l)); }
    __device__ __forceinline__ void start(const R6<float>& l) { m = wide(l); }
    __device__ __forceinline__ void mul(const R6<float>& l) { m = gf::mul(m, wide(l)); }
    __device__ __forceinline__ void mul_dag(const R6<float>& l) { m = mul_nd(m, wide(l)); }
    __device__ __forceinline__ void dag_mul(const R6<float>& l) { m = mul_dn(m, wide(l)); }
    __device__ __forceinline__ M3<double> get() const { return m; }
};

__device__ __forceinline__ void plane_dirs(int pl, int& a, int& b) {
    a = pl < 3 ? 0 : (pl < 5 ? 1 : 2);
    b = pl < 3 ? pl + 1 : (pl < 5 ? pl - 1 : 3);
}

// Coefficient fields of a block of sites: field f of plane pl holds 4 pair planes of n sites.
// Plaquette; clover near, far; rectangles near (both kinds), far of a x 2b, far of 2a x b
template <int SETS>
constexpr int kFields = (SETS & 1) + 2 * ((SETS >> 1) & 1) + 3 * ((SETS >> 2) & 1);
template <int SETS>
constexpr int kClover = SETS & 1;
template <int SETS>
constexpr int kRect = (SETS & 1) + 2 * ((SETS >> 1) & 1);

__device__ __forceinline__ void st_coeffs(double2* __restrict__ at, unsigned n, unsigned i, const double c[8]) {
#pragma unroll
    for (int e = 0; e < 4; e++) at[(size_t)e * n + i] = double2{c[2 * e], c[2 * e + 1]};
}
__device__ __forceinline__ void add_coeffs(const double2* __restrict__ at, unsigned n, unsigned i, double c[8]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const double2 v = at[(size_t)e * n + i];
        c[2 * e] += v.x;
        c[2 * e + 1] += v.y;
    }
}

}  // namespace

// The r-th 64-site group to visit of a block of n sites in t-slices of `slice`: where eight divides the groups of a
// slice, each eighth of the order (an XCD's part, xcd_block) is an eighth of the slice followed through the
// block's t, so that the links of neighbouring slices are still in the XCD's L2; linear otherwise.
__device__ __forceinline__ int block_group(int r, int n, int slice) {
    if (slice % 512 != 0) return r;
    const int part = slice / 512, run = part * (n / slice);
    const int k = r / run, m = r % run;
    return (m / part) * (slice / 64) + k * part + m % part;
}
// sites i and j of a block are lanes of one wave
__device__ __forceinline__ bool same_wave(int i, int j) { return (i >> 6) == (j >> 6); }

// One wave per 64 sites of the block [s0, s0 + n), plane and path type (clover and plaquette; rectangles).  The
// links of a path are loaded one ahead of their use, as in staple_sigma_pipe.  In the planes (0, b) the far
// site is mostly one of the wave's own (the sites are consecutive along x): its part is then added to the
// near one there, through LDS, and only what leaves the wave is stored.  FP32 links hold whole products (Path): two
// waves per SIMD without spills instead of three with (32^4 improved charge 1309 -> 1286 us).
template <typename T, int SETS>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && (SETS & 4) ? 2 : 3))) void
k_loops(Geo g, const T* __restrict__ U, int s0, int n, double2* __restrict__ fields) {
    __shared__ C8Lds<double> sh[kBlock / 64], park[(SETS & 4) ? kBlock / 64 : 1];
    constexpr int NT = ((SETS & 3) ? 1 : 0) + ((SETS & 4) ? 1 : 0), FIRST = (SETS & 3) ? 0 : 1;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
    const int task = (int)xcd_block() * (kBlock / 64) + w;
    const int type = task % NT + FIRST, pl = (task / NT) % 6;
    const int i = block_group(task / (6 * NT), n, g.st[3]) * 64 + lane;
    if (i >= n) return;
    const int s = s0 + i;
    int x[4];
    decode(g, s, x);
    const unsigned V = g.V;
    int a, b;
    plane_dirs(pl, a, b);
    int xa = sel4(a, x[0], x[1], x[2], x[3]), xb = sel4(b, x[0], x[1], x[2], x[3]);
    // offset of d steps along a direction (periodic; extents may be smaller than d)
    auto off = [&](int dir, int xd, int d) {
        const int e = g.n[dir];
        int y = xd + d;
#pragma unroll
        for (int k = 0; k < 2; k++) y = y >= e ? y - e : (y < 0 ? y + e : y);
        return (y - xd) * g.st[dir];
    };
    auto ld = [&](int dir, int da, int db) {
        int t = s;
        if (da) t += off(a, xa, da);
        if (db) t += off(b, xb, db);
        return ldr(U, V, dir, (unsigned)t);
    };
    double2* const f0 = fields + (size_t)pl * kFields<SETS> * 4 * n;
    auto field = [&](int k) { return f0 + (size_t)k * 4 * n; };
    Path<T> p;
    M3<double> K;
    R6<T> cur, nxt;
    // the next link asked for before the arithmetic on the current one
#define GF_STEP(OP, NEXT)                     \
    nxt = NEXT;                               \
    __builtin_amdgcn_sched_barrier(0);        \
    p.OP(cur);                                \
    cur = nxt;
    auto minus = [&](const M3<double>& m) {
#pragma unroll
        for (int e = 0; e < 9; e++) {
            K.m[e].r -= m.m[e].r;
            K.m[e].i -= m.m[e].i;
        }
    };
    // near[] and the coefficients of m for the site d steps along a (field k): added to that site's near part if
    // it is in the wave (a = 0), else stored
    double near_[8];
    auto far_part = [&](const M3<double>& m, int d, int k) {
        double c[8];
        ta_coeffs(m, c);
        bool store = true;
        if (a == 0) {
            const int to = i + off(0, xa, d), from = i + off(0, xa, -d);
            put_c8(&sh[w], lane, c);
            wave_exchange();
            if (same_wave(i, from)) {
                double t[8];
                get_c8(&sh[w], from & 63, t);
#pragma unroll
                for (int e = 0; e < 8; e++) near_[e] += t[e];
            }
            wave_exchange();
            store = !same_wave(i, to);
        }
        if (store) st_coeffs(field(k), n, i, c);
    };
    if ((SETS & 3) && type == 0) {
        cur = ld(b, 1, 0);
        GF_STEP(start, ld(a, 0, 1))
        GF_STEP(mul_dag, ld(b, 0, 0))
        GF_STEP(mul_dag, ld(a, 0, -1))
        K = p.get();
        if constexpr (SETS & 1) {
            ta_coeffs(mul(full_of(r6_f64(ld(a, 0, 0))), K), near_);
            st_coeffs(field(0), n, i, near_);
        }
        if constexpr (SETS & 2) {
            GF_STEP(start, ld(b, 1, -1))
            GF_STEP(mul, ld(b, 0, -1))
            GF_STEP(dag_mul, ld(a, 0, 0))
            minus(p.get());
            const M3<double> u = full_of(r6_f64(cur));
            ta_coeffs(mul(u, K), near_);
            far_part(mul(K, u), 1, kClover<SETS> + 1);
            st_coeffs(field(kClover<SETS>), n, i, near_);
        }
    } else if (SETS & 4) {
        cur = ld(b, 1, 0);
        GF_STEP(start, ld(b, 1, 1))
        GF_STEP(mul, ld(a, 0, 2))
        GF_STEP(mul_dag, ld(b, 0, 1))
        GF_STEP(mul_dag, ld(b, 0, 0))
        GF_STEP(mul_dag, ld(a, 0, -2))
        K = p.get();
        GF_STEP(start, ld(b, 1, -2))
        GF_STEP(mul, ld(b, 1, -1))
        GF_STEP(mul, ld(b, 0, -2))
        GF_STEP(dag_mul, ld(b, 0, -1))
        GF_STEP(mul, ld(a, 0, 0))
        minus(p.get());
        {
            const M3<double> u = full_of(r6_f64(cur));
            ta_coeffs(mul(u, K), near_);
            far_part(mul(K, u), 1, kRect<SETS> + 1);
            put_c8(&park[w], lane, near_);
        }
        // the second kind's first link and site offsets are not formed before this (spills: 32^4 1375 -> 1294 us, and the
        // first launch of a spilling kernel on a stream waits 130 us for its private segment)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+v"(xa), "+v"(xb));
        cur = ld(b, 2, 0);
        GF_STEP(start, ld(a, 1, 1))
        GF_STEP(mul_dag, ld(a, 0, 1))
        GF_STEP(mul_dag, ld(b, 0, 0))
        GF_STEP(mul_dag, ld(a, 0, -1))
        K = p.get();
        GF_STEP(start, ld(a, 1, -1))
        GF_STEP(mul, ld(b, 2, -1))
        GF_STEP(mul, ld(b, 0, -1))
        GF_STEP(dag_mul, ld(a, 0, 0))
        minus(p.get());
        GF_STEP(start, ld(a, 1, 0))
        p.mul(cur);
        const M3<double> D = p.get();
        double c[8];
        ta_coeffs(mul(D, K), c);
        get_c8(&park[w], lane, near_);
#pragma unroll
        for (int e = 0; e < 8; e++) near_[e] += c[e];
        far_part(mul(K, D), 2, kRect<SETS> + 2);
        st_coeffs(field(kRect<SETS>), n, i, near_);
    }
#undef GF_STEP
}

// TA coefficients of the plaquette U_a(x) U_b(x+a) U_a(x+b)^dag U_b(x)^dag
template <typename T>
__device__ __forceinline__ void plaquette_coeffs(const Geo& g, const T* __restrict__ U, int s, const int x[4], int pl,
                                                 double c[8]) {
    int a, b;
    plane_dirs(pl, a, b);
    const unsigned V = g.V;
    int fw[4];
#pragma unroll
    for (int d = 0; d < 4; d++) fw[d] = s + dlt(g, x, d, 1);
    const R6<T> l0 = ldr(U, V, a, (unsigned)s), l1 = ldr(U, V, b, (unsigned)sel4(a, fw[0], fw[1], fw[2], fw[3])),
                l2 = ldr(U, V, a, (unsigned)sel4(b, fw[0], fw[1], fw[2], fw[3])), l3 = ldr(U, V, b, (unsigned)s);
    Path<T> p;
    p.start(l0);
    p.mul(l1);
    p.mul_dag(l2);
    p.mul_dag(l3);
    ta_coeffs(p.get(), c);
}

// The densities of the block's sites: wave j contracts the planes (01)(23), (02)(13), (03)(12).  Partial sums per
// workgroup at partial[k * stride + base + workgroup]: k = 0 clover energy (sum |c|^2 / 32), 1 plaquette q,
// 2 clover q, 3 rectangle q.  dens (optional): density of method dens_method per site.  The plaquette set alone
// has no far parts and is evaluated in place (U; fields not used).
template <typename T, int SETS>
__global__ __launch_bounds__(192) void k_charge(Geo g, const T* __restrict__ U, const double2* __restrict__ fields,
                                                int s0, int n,
                                                double* __restrict__ partial, int stride, int base,
                                                double* __restrict__ dens, int dens_method) {
    __shared__ double q[3][3][64];
    const int j = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
    const int i = (SETS == 1 ? group_of_block(g) : (int)xcd_block()) * 64 + lane;
    double e = 0.0, dot[3] = {0.0, 0.0, 0.0};
    if (i < n) {
        const int s = s0 + i;
        int x[4];
        decode(g, s, x);
        double c[2][3][8];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int pl = h == 0 ? j : 5 - j;
            int a, b;
            plane_dirs(pl, a, b);
            const double2* const f0 = fields + (size_t)pl * kFields<SETS> * 4 * n;
            const int xa = sel4(a, x[0], x[1], x[2], x[3]), ea = g.n[a];
            const int m1 = xa == 0 ? ea - 1 : xa - 1, m2 = m1 == 0 ? ea - 1 : m1 - 1;
            const unsigned i1 = (unsigned)(i + (m1 - xa) * g.st[a]), i2 = (unsigned)(i + (m2 - xa) * g.st[a]);
            auto field = [&](int k) { return f0 + (size_t)k * 4 * n; };
#pragma unroll
            for (int k = 0; k < 8; k++) c[h][0][k] = c[h][1][k] = c[h][2][k] = 0.0;
            if constexpr (SETS == 1)
                plaquette_coeffs(g, U, s, x, pl, c[h][0]);
            else if constexpr (SETS & 1)
                add_coeffs(field(0), n, i, c[h][0]);
            const bool far1 = a > 0 || !same_wave(i, (int)i1), far2 = a > 0 || !same_wave(i, (int)i2);
            if (SETS & 2) {
                add_coeffs(field(kClover<SETS>), n, i, c[h][1]);
                if (far1) add_coeffs(field(kClover<SETS> + 1), n, i1, c[h][1]);
            }
            if (SETS & 4) {
                add_coeffs(field(kRect<SETS>), n, i, c[h][2]);
                if (far1) add_coeffs(field(kRect<SETS> + 1), n, i1, c[h][2]);
                if (far2) add_coeffs(field(kRect<SETS> + 2), n, i2, c[h][2]);
            }
        }
#pragma unroll
        for (int t = 0; t < 3; t++)
#pragma unroll
            for (int k = 0; k < 8; k++) dot[t] = fma(c[0][t][k], c[1][t][k], dot[t]);
        if (SETS & 2) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int k = 0; k < 8; k++) e = fma(c[h][1][k], c[h][1][k], e);
            e *= 1.0 / 32.0;
        }
    }
    const double k8 = 1.0 / (8.0 * 3.14159265358979323846 * 3.14159265358979323846), sg = j == 1 ? -1.0 : 1.0;
    const double v[3] = {sg * k8 * dot[0], sg * k8 / 16.0 * dot[1], sg * 2.0 * k8 / 64.0 * dot[2]};
    if (dens) {
#pragma unroll
        for (int t = 0; t < 3; t++) q[t][j][lane] = v[t];
        __syncthreads();
        if (j == 0 && i < n) {
            double d[3];
#pragma unroll
            for (int t = 0; t < 3; t++) d[t] = q[t][0][lane] + q[t][1][lane] + q[t][2][lane];
            dens[s0 + i] = dens_method == 0   ? d[0]
                           : dens_method == 1 ? d[1]
                           : dens_method == 2 ? (5.0 / 3.0) * d[1] + (-1.0 / 12.0) * d[2]
                                              : d[2];
        }
    }
    double* const p = partial + base;
    block_sum_store<192>(e, p);
#pragma unroll
    for (int t = 0; t < 3; t++) {
        __syncthreads();
        block_sum_store<192>(v[t], p + (size_t)(t + 1) * stride);
    }
}

static int fields_of(int sets) { return (sets & 1) + 2 * ((sets >> 1) & 1) + 3 * ((sets >> 2) & 1); }
// Blocks of whole t-slices: as many as keep the fields of a block near kFieldBytes, evenly, at least one; all
// of them where there are no fields (the plaquette set alone, whose sites are then visited as the stencil
// kernels visit theirs)
constexpr double kFieldBytes = 256e6;
static size_t slice_bytes(const Geo& g, int sets) { return (size_t)(g.V / g.n[3]) * 6 * 64 * fields_of(sets); }
static int slices_per_block(const Geo& g, int sets, size_t bytes) {
    if (sets == 1) return g.n[3];
    const int most = std::max(1, (int)((double)bytes / (double)slice_bytes(g, sets)));
    const int blocks = (g.n[3] + most - 1) / most;
    return (g.n[3] + blocks - 1) / blocks;
}
// the block of these sets, and no less than the blocks of the other sets take where a t-slice of theirs fits into
// kFieldBytes: a density and then an energy of one context grow the buffer once
size_t field_strength_bytes(const Geo& g, int sets, size_t most) {
    if (sets == 1) return 0;
    most = std::min(most, (size_t)kFieldBytes);
    return std::max(slices_per_block(g, sets, most) * slice_bytes(g, sets),
                    std::min(most, g.n[3] * slice_bytes(g, 7)));
}

template <typename T, int SETS>
void launch_sets(const Geo& g, const T* U, double2* fields, int per, double* partial, int stride, double* dens, int dens_method,
                 hipStream_t st) {
    constexpr int NT = ((SETS & 3) ? 1 : 0) + ((SETS & 4) ? 1 : 0);
    const int slice = g.V / g.n[3];
    int base = 0;
    for (int t = 0; t < g.n[3]; t += per) {
        const int n = slice * std::min(per, g.n[3] - t), groups = (n + 63) / 64;
        if constexpr (SETS != 1)
            k_loops<T, SETS><<<(groups * 6 * NT + 3) / 4, kBlock, 0, st>>>(g, U, slice * t, n, fields);
        k_charge<T, SETS><<<groups, 192, 0, st>>>(g, U, fields, slice * t, n, partial, stride, base, dens,
                                                  dens_method);
        base += groups;
    }
}

// partial: 4 (V / 64 + NT + 1) doubles
template <typename T>
hipError_t launch_field_strength(const Geo& g, const T* U, int sets, void* fields, size_t bytes, double* partial,
                                 double* out4, double* dens, int dens_method, hipStream_t st) {
    const int slice = g.V / g.n[3], per = slices_per_block(g, sets, std::min(bytes, (size_t)kFieldBytes));
    int stride = 0;
    for (int t = 0; t < g.n[3]; t += per) stride += (slice * std::min(per, g.n[3] - t) + 63) / 64;
    double2* const f = (double2*)fields;
    switch (sets) {
        case 1: launch_sets<T, 1>(g, U, f, per, partial, stride, dens, dens_method, st); break;
        case 2: launch_sets<T, 2>(g, U, f, per, partial, stride, dens, dens_method, st); break;
        case 4: launch_sets<T, 4>(g, U, f, per, partial, stride, dens, dens_method, st); break;
        case 6: launch_sets<T, 6>(g, U, f, per, partial, stride, dens, dens_method, st); break;
        case 7: launch_sets<T, 7>(g, U, f, per, partial, stride, dens, dens_method, st); break;
        default: return hipErrorInvalidValue;
    }
    return launch_sum_partials(partial, stride, 4, out4, st);
}

#define GF_INST_FS(T)                                                                                            \
    template hipError_t launch_field_strength<T>(const Geo&, const T*, int, void*, size_t, double*, double*, double*,  \
                                                 int, hipStream_t);
GF_INST_FS(double)
GF_INST_FS(float)
#undef GF_INST_FS

}  // namespace gf
