// k_flow_stout.hip -- Luscher RK3 Wilson-flow stage, stout smearing forward and backward.
#include <utility>

#include "internal.hpp"

namespace gf {

// the 8 coefficients of a link in a workgroup's LDS (an array [..][4][..] of pairs)
template <typename T, typename A>
__device__ __forceinline__ void put_c8(A* a, int k, int l, const T c[8]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        T2<T> v;
        v.x = c[2 * e];
        v.y = c[2 * e + 1];
        a[k][e][l] = v;
    }
}
template <typename T, typename A>
__device__ __forceinline__ void get_c8(const A* a, int k, int l, T c[8]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const T2<T> v = a[k][e][l];
        c[2 * e] = v.x;
        c[2 * e + 1] = v.y;
    }
}

// ---------------------------------------------------------------------------
// K7: one RK3 stage (flow!, gradientflow.jl:171-238, in the low-storage form):
//   F = TA(W_mu V_mu^dag)                  (add_force! plaqonly, AbstractGaugefields.jl:2717-2762)
//   A = alpha F + beta A
//   Wout_mu = exp(A_mu) W_mu               (exp_aF_U!, AbstractGaugefields.jl:2810-2841)
// stages (alpha, beta) = (-eps/4, 0), (-8eps/9, -17/9), (-3eps/4, -1)
// ---------------------------------------------------------------------------
// ST: form of the stencil (stencil_form).  At most 168 VGPRs: three waves per SIMD.
template <typename T, int ST>
__global__ __launch_bounds__(stencil_threads(ST)) __attribute__((amdgpu_waves_per_eu(3))) void k_flow_stage(
    Geo g, const T* __restrict__ W, T* __restrict__ Wout, T* __restrict__ A, double alpha, double beta) {
    int s, mu;
    R6<T> own;
    T c[8];
    if (!ta_force<ST>(g, W, s, mu, own, c)) return;
    const unsigned V = g.V;
    const M3<T> w = full_of(own);
    if (beta != T(0)) {
        T a[8];
        ldp<T, GF_LD_NT>(A, V, mu, s, a);
#pragma unroll
        for (int k = 0; k < 8; k++) c[k] = (T)fma(alpha, (double)c[k], beta * (double)a[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) c[k] = scale1(alpha, c[k]);
    }
    stp<T, GF_ST_NT>(A, V, mu, s, c);
    const M3<T> wn = exp_coeffs_times(c, 1.0, w);
    stu<T, GF_ST_NT>(Wout, V, mu, s, wn);
}

// ---------------------------------------------------------------------------
// K5: stout forward level (forward!, stout_fast.jl:250-274; calc_C! :603-624)
//   C_mu = rho V_mu = rho Sigma_mu^dag,  Q_mu = TA(C_mu U_mu^dag) = -rho TA(U_mu Sigma_mu),
//   Uout_mu = exp(Q_mu) U_mu
// so the level is the force kernel's stencil with a link update on top (32^4 FP64: 0.50 ms when it formed
// the whole staple sum and stored C).  WHAT: STOUT_LINKS the smeared links, STOUT_Q the 8 coefficients of
// Q_mu, which are all the backward pass of a force needs of the level besides its links.
// The coefficients are formed and summed in double for FP32 links too, from staples in float: a level's links at rho = 1
// lie 5.2e-8 ... 5.4e-8 RMS from the FP64 level's (with float products and sums 7.2e-8 ... 8.0e-8, and 8.8e-8 with C kept
// rounded to float), for 17 % of the kernel's time (32^4 FP32, three levels 665 -> 777 us; force 2.29 -> 2.41 ms).
// ---------------------------------------------------------------------------
enum { STOUT_LINKS = 1, STOUT_Q = 2 };
template <typename T, int WHAT, int ST>
__global__ __launch_bounds__(stencil_threads(ST)) __attribute__((amdgpu_waves_per_eu(3))) void k_stout_forward(
    Geo g, const T* __restrict__ Uin, T* __restrict__ Uout, T* __restrict__ Qst, double rho) {
    int s, mu;
    R6<T> own;
    double c[8];
    if (!ta_force<ST>(g, Uin, s, mu, own, c)) return;
    const unsigned V = g.V;
    if constexpr (WHAT & STOUT_LINKS) stu<T, GF_ST_NT>(Uout, V, mu, s, exp_coeffs_times(c, -rho, full_of(own)));
    if constexpr (WHAT & STOUT_Q) {
        T q[8];
#pragma unroll
        for (int k = 0; k < 8; k++) q[k] = (T)(-rho * c[k]);
        stp<T, GF_ST_NT>(Qst, V, mu, s, q);
    }
}

// ---------------------------------------------------------------------------
// Backward pass of a stout force.  The action depends on a level's links only through the group, so
// what a level hands down is not dS/dU (18 reals) but F = TA(U dS/dU) (8), and what it keeps is Q (8)
// instead of C (18).  Per level, from F' of its output links:
//   site-local (stout_local): Lam = derivative with respect to Q, Floc = derivative at fixed Q
//   staples: dQ_mu(x) = -rho dTA(U_mu Sigma_mu); summed over links, sum Re tr(Lam dQ) is -rho d of
//     sum over plaquettes of Re tr(Z P),  P = U_a(z) U_b(z+a) U_a(z+b)^dag U_b(z)^dag  (a < b),
//     Z = Lam_a + G - G' - Lam_b,  G = U_a Lam_b(z+a) U_a^dag,  G' = U_b Lam_a(z+b) U_b^dag,
//   so each plaquette gives its four links
//     U_a(z):    TA(P Z + G P - P G)          U_b(z+a): U_a^dag TA(P Z) U_a
//     U_b(z):   -TA(Z P + G' P - P G')        U_a(z+b): -U_b^dag TA(Z P) U_b
//   times -rho.
// k_stout_pair evaluates every plaquette once: the sums at the near links (z) are added to Floc, the two
// far ones are stored at z (3 momentum-shaped fields: field j of direction mu holds the contribution
// to U_mu(z + b), b = j + (j >= mu)); k_stout_gather reads those back at z = y - b and goes on to the
// next level's site-local step or to the force.  The start of the chain, F' of the top level (coeff
// TA(U Sigma)) and its site-local step, is k_stout_top.
// (Replaces a gather that evaluated every plaquette once per link, 3258 instead of 1390 x 6/4 FMAs per
// link and four times the loads, and carried dS/dU and C.)
// ---------------------------------------------------------------------------
// FP32: four waves per SIMD (force with three levels 32^4 2.34 -> 2.32 ms).
template <typename T, int ST>
__global__ __launch_bounds__(stencil_threads(ST)) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 3 : 4))) void k_stout_top(
    Geo g, const T* __restrict__ Utop, double coeff, const T* __restrict__ Qst, T* __restrict__ Lc,
    T* __restrict__ Fl) {
    int s, mu;
    R6<T> own;
    T c[8];
    __shared__ ForceShare<T, ST, T> sh;
    if (!ta_force<ST>(g, Utop, s, mu, own, c, sh)) return;
    const unsigned V = g.V;
    T q[8], lam[8], fl[8];
#pragma unroll
    for (int k = 0; k < 8; k++) c[k] = scale1(coeff, c[k]);
    // F' waits for its second use in LDS that only this wave still uses: in registers it would spill some, and the
    // first launch of a spilling kernel on a stream waits 130 us for its private segment (first force of a context, two
    // levels, 8^4 203 -> 71 us, 16^4 356 -> 229)
    int lane = (int)(threadIdx.x & 63u);
    if constexpr (ST == ST_WIDE)
        put_c8<T>(sh.tp, 0, lane, c);
    else
        put_c8<T>(sh.ol, mu, lane, c);
    ldp<T, GF_LD_NT>(Qst, V, mu, s, q);
    stout_local(q, c, lam, fl, [&](T f[8]) {
        asm volatile("" : "+v"(lane));
        if constexpr (ST == ST_WIDE)
            get_c8(sh.tp, 0, lane, f);
        else
            get_c8(sh.ol, mu, lane, f);
    });
    stp(Lc, V, mu, s, lam);
    stp(Fl, V, mu, s, fl);
}

// One workgroup = 64 sites, NW wavefronts for the six pairs (a, b).  NW = 4: two waves take two, another
// two in every other workgroup; three workgroups fit a CU.  (With six waves a CU holds one workgroup: its
// first two SIMDs get two waves of 168 VGPRs and have no room for the next one's two.  32^4 FP64: 0.79
// against 0.64 ms.)  NW = 6 on small lattices, one pair each.  The waves work by themselves (what three
// pairs of a site share comes from L1) up to one exchange in LDS of the near contributions.  Three waves
// per SIMD are too few to hide memory behind each other, so a wave asks for a pair's inputs at once: the
// four links and the site's two Lam into registers, the neighbours' Lam straight into LDS, where the near
// contributions will go.  The far contribution to U_b(z + x) of the pairs (0, b) mostly goes to a site of the
// workgroup and is added to the near ones there: up to a quarter of the far fields less, also where the groups
// cut the rows (force with three levels, FP64 24^4 1.40 -> 1.36 ms, 24x24x16x12 475 -> 459 us; FP32 24^4 774 -> 760).
__device__ __forceinline__ bool same_group(int s, int r) { return (s >> 6) == (r >> 6); }
template <typename T, bool ROWS, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(3))) void k_stout_pair(
    Geo g, const T* __restrict__ U, const T* __restrict__ Lc, T* __restrict__ Fl, T* __restrict__ far, double rho) {
    __shared__ C8Lds<T> near_[12];
    const SiteMu sm = site_mu_index(g);
    const int w = sm.mu, s = stencil_site<ROWS>(g, sm);
    const int lane = (int)(threadIdx.x & 63u);
    const unsigned V = g.V;
    int x[4], fw[4];
    decode(g, s, x);
#pragma unroll
    for (int d = 0; d < 4; d++) fw[d] = s + dlt(g, x, d, 1);
    const int first = NW == 4 ? w ^ (int)((blockIdx.x >> 2) & 2u) : w;
#pragma unroll 1
    for (int p = first; p < 6; p += NW) {
        const int a = p < 3 ? 0 : (p < 5 ? 1 : 2), b = p < 3 ? p + 1 : (p < 5 ? p - 1 : 3);
        const int sa = sel4(a, fw[0], fw[1], fw[2], fw[3]), sb = sel4(b, fw[0], fw[1], fw[2], fw[3]);
        M3<T> P;
        Herm<T> G, Gp, Z;
        {
            const R6<T> nb = ldr(U, V, b, (unsigned)sa), na = ldr(U, V, a, (unsigned)sb);
            const R6<T> ra = ldr(U, V, a, (unsigned)s), rb = ldr(U, V, b, (unsigned)s);
            T ca[8], cb[8];
            ldp(Lc, V, a, (unsigned)s, ca);
            ldp(Lc, V, b, (unsigned)s, cb);
            ldp_lds(Lc, V, a, (unsigned)sb, &near_[2 * p]);
            ldp_lds(Lc, V, b, (unsigned)sa, &near_[2 * p + 1]);
            __builtin_amdgcn_sched_barrier(0);
            P = su3_mul(ra, su3_mul_nd(nb, full_of(na)));
#pragma unroll
            for (int k = 0; k < 8; k++) ca[k] -= cb[k];
            Z = herm_of_coeffs(ca);
            const M3<T> ub = full_of(rb);
            P = su3_mul_nd(rows_of(P), ub);
            wait_lds_loads();
            T h[8];
            get_c8(&near_[2 * p], lane, h);
            Gp = herm_conj(ub, herm_of_coeffs(h));
            get_c8(&near_[2 * p + 1], lane, h);
            G = herm_conj(full_of(ra), herm_of_coeffs(h));
        }
        T fa[8], fb[8];  // TA(i Z P), TA(i P Z)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            Z.d[k] += G.d[k] - Gp.d[k];
            Z.u[k].r += G.u[k].r - Gp.u[k].r;
            Z.u[k].i += G.u[k].i - Gp.u[k].i;
        }
        ta_coeffs_i(mul_mh(P, Z), fb);
        ta_coeffs_i(mul_hm(Z, P), fa);
        T c[8];
        ta_coeffs_i(herm_comm(G, P), c);
#pragma unroll
        for (int k = 0; k < 8; k++) c[k] += fb[k];
        put_c8(&near_[2 * p], lane, c);
        ta_coeffs_i(herm_comm(Gp, P), c);  // TA(i (P G' - G' P)) is minus this
#pragma unroll
        for (int k = 0; k < 8; k++) c[k] = -(c[k] + fa[k]);
        // the far links; U_a and U_b again from L1 rather than held
        int s1 = s;
        asm volatile("" : "+v"(s1));
        const R6<T> ra = ldr(U, V, a, (unsigned)s1), rb = ldr(U, V, b, (unsigned)s1);
        T t[8];
        coeffs_of_herm(herm_conj_dag(full_of(ra), herm_of_coeffs(fb)), t);
        bool store = in_lattice<ROWS>(g, sm);
        if (a == 0) {
            // the contribution to the lane of x + 1, through this wave's place in LDS (its lanes in step)
            const int from = s + dlt(g, x, 0, -1);
            put_c8(&near_[2 * p + 1], lane, t);
            wave_exchange();
            if (ROWS || same_group(from, s)) {
                T n[8];
                get_c8(&near_[2 * p + 1], from & 63, n);
#pragma unroll
                for (int k = 0; k < 8; k++) c[k] += n[k];
            }
            wave_exchange();
            store = !ROWS && store && !same_group(fw[0], s);
        }
        if (store) stp<T, GF_ST_NT>(far + (size_t)a * 32 * V, V, b, (unsigned)s, t);
        put_c8(&near_[2 * p + 1], lane, c);
#pragma unroll
        for (int k = 0; k < 8; k++) fa[k] = -fa[k];
        coeffs_of_herm(herm_conj_dag(full_of(rb), herm_of_coeffs(fa)), t);
        if (in_lattice<ROWS>(g, sm)) stp<T, GF_ST_NT>(far + (size_t)(b - 1) * 32 * V, V, a, (unsigned)s, t);
    }
    T f[8];
    if (w < 4) ldp<T, GF_LD_NT>(Fl, V, w, (unsigned)s, f);
    __syncthreads();  // every pair's near contributions are in LDS
    if (w < 4 && in_lattice<ROWS>(g, sm)) {
        T c[8], t[8];
#pragma unroll
        for (int k = 0; k < 8; k++) c[k] = T(0);
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int nu = j + (j >= w ? 1 : 0);
            get_c8(&near_[2 * pair_index(w < nu ? w : nu, w < nu ? nu : w) + (w < nu ? 0 : 1)], lane, t);
#pragma unroll
            for (int k = 0; k < 8; k++) c[k] += t[k];
        }
#pragma unroll
        for (int k = 0; k < 8; k++) f[k] = fma1(-rho, c[k], f[k]);
        stp<T, GF_ST_NT>(Fl, V, w, (unsigned)s, f);
    }
}

// F of a level's input links: Floc and near contributions (Fl, as k_stout_pair left it) plus the far
// contributions of the three plaquettes below.  OUT < 0: the site-local step of the next level down (Qst its
// Q), Lam and Floc in place.  Otherwise the thin-link level of a force, -(1/3) F, as k_force's modes
// (test/HMCstout_test_nowing.jl:99-118).  Streaming: a thread per link; workgroups of one wave on small
// lattices, to reach more CUs.
template <typename T, int OUT, bool ROWS>
__global__ __launch_bounds__(kBlock) void k_stout_gather(Geo g, const T* __restrict__ far, T* __restrict__ Fl,
                                                         double rho, const T* __restrict__ Qst, T* __restrict__ Lc,
                                                         const T* __restrict__ U, T* __restrict__ FP,
                                                         T* __restrict__ Unew, double fac, double eps_u, double eps_p,
                                                         double* __restrict__ U64) {
    int s, mu;
    if (blockDim.x == 64u) {
        const unsigned b = xcd_block();
        s = (int)((b >> 2) * 64u + threadIdx.x);
        mu = (int)(b & 3u);
    } else {
        const SiteMu sm = site_mu_index(g);
        s = sm.s;
        mu = sm.mu;
    }
    if (s >= g.V) return;
    const unsigned V = g.V;
    int x[4];
    decode(g, s, x);
    T f[8], c[8], t[3][8];
    ldp<T, GF_LD_NT>(Fl, V, mu, (unsigned)s, f);
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const int nu = j + (j >= mu ? 1 : 0), from = s + dlt(g, x, nu, -1);
        if (j == 0) {
#pragma unroll
            for (int k = 0; k < 8; k++) t[0][k] = T(0);
            if (mu > 0 && (ROWS || same_group(from, s))) continue;  // in Fl
        }
        ldp(far + (size_t)j * 32 * V, V, mu, (unsigned)from, t[j]);
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        c[k] = t[1][k] + t[2][k];
        if (!ROWS || mu == 0) c[k] += t[0][k];
        c[k] = fma1(-rho, c[k], f[k]);
    }
    if constexpr (OUT < 0) {
        T q[8], lam[8], fl[8];
        ldp<T, GF_LD_NT>(Qst, V, mu, (unsigned)s, q);
        stout_local(q, c, lam, fl);
        stp(Lc, V, mu, (unsigned)s, lam);
        stp(Fl, V, mu, (unsigned)s, fl);
    } else {
        force_out<T, OUT>(c, [&] { return ldu<T, GF_LD_NT>(U, V, mu, (unsigned)s); }, V, mu, s, FP, Unew, fac, eps_u,
                          eps_p, U64);
    }
}

// ---------------------------------------------------------------------------
// K6a: stout backward, site-local part (backward_dSdUαUβρ_add!, stout_fast.jl:317-407):
//   Din_mu = Dout_mu e^{Q_mu} + (Lam_mu C_mu)^dag,   Lam_mu = TA(CdexpQdQ(U_mu Dout_mu, Q_mu))
// Lam_mu (traceless anti-Hermitian) is stored as its 8 su(3) coefficients; the staple part
// uses G_mu = U_mu^dag Lam_mu (= dS/dC_mu) without storing it.
// (Used by the explicit backward pass, whose dS/dU_in is wanted as a matrix; the forces take the algebra form
// above.)  Where the smearing has kept Q_mu, it is read (back_local_q), and (Lam C)^dag = -rho Sigma Lam is left to the
// staple part, which walks the staples of Sigma anyway: a streaming step without a stencil, done by the staple part's
// kernel of the level above.  Otherwise, and on small lattices, C_mu is formed from the staples again (back_local).
// Two levels, us, C formed again / Q read: FP64 16^4 197 / 165, 20^3x10 234 / 198, 24^4 888 / 748, 32^4 2953 / 2380; FP32
// 116 / 96, 133 / 116, 500 / 418, 1555 / 1211.
// ---------------------------------------------------------------------------
// A 3x3 field element kept in the wave's own LDS slice between two uses (each lane reads back what
// it wrote: no barrier), instead of being held in registers or read from memory twice.
template <typename T>
using MStage = T2<T> (*)[64];
template <typename T>
__device__ __forceinline__ M3<T> stage_m3(MStage<T> st, int lane, const M3<T>& m) {
#pragma unroll
    for (int e = 0; e < 9; e++) {
        T2<T> v;
        v.x = m.m[e].r;
        v.y = m.m[e].i;
        st[e][lane] = v;
    }
    return m;
}
template <typename T>
__device__ __forceinline__ M3<T> staged_m3(MStage<T> st, int lane) {
    // an opaque copy of the index, so that the compiler reads LDS rather than forwarding the
    // stored value (which would keep it live in registers)
    asm volatile("" : "+v"(lane));
    M3<T> m;
#pragma unroll
    for (int e = 0; e < 9; e++) {
        const T2<T> v = st[e][lane];
        m.m[e].r = v.x;
        m.m[e].i = v.y;
    }
    return m;
}
// from the staple sum and the link: Din and Lam of the level (dout() is Dout_mu(s); dst the lane's staging)
template <typename T, typename D>
__device__ __forceinline__ void back_local(const M3<T>& sig, const R6<T>& own, D&& dout, T* __restrict__ Din,
                                           T* __restrict__ Lc, double rho, unsigned V, int mu, int s, int lane,
                                           MStage<T> dst) {
    const M3<T> C = round_link<T>(scal(rho, dag(to_f64(sig))));
    M3<T> E, L;
    {
        const M3<T> u = full_of(own);
        exp_dexp(ta_mat(mul_nd(C, u)), mul(u, stage_m3<T>(dst, lane, dout())), E, L);
    }
    const M3<T> Lam = ta_mat(L);
    {
        T c[8];
        ta_coeffs(Lam, c);
        stp<T, GF_ST_NT>(Lc, V, mu, s, c);
    }
    M3<T> D2 = mul(staged_m3<T>(dst, lane), E);
    acc_dag(D2, mul(Lam, C));
    stm<T, GF_ST_NT>(Din, V, mu, s, D2);
}
template <typename T, int ST>
__global__ __launch_bounds__(stencil_threads(ST)) void k_stout_back_local(Geo g, const T* __restrict__ Uin,
                                                                          const T* Dout, T* Din, T* __restrict__ Lc,
                                                                          double rho) {
    // the staples' exchange, then Dout_mu, which is used before and after exp_dexp: kept in LDS in between
    __shared__ T2<T> xs[ST == ST_WIDE ? 1 : 6][6][64];
    __shared__ T2<T> dst[ST == ST_WIDE ? 2 : 4][9][64];
    const int lane = (int)(threadIdx.x & 63u);
    const unsigned V = g.V;
    int s, mu, x[4];
    R6<T> own;
    M3<T> sig;
    bool valid;
    if constexpr (ST == ST_WIDE) {
        const WideIndex wi = wide_index(g);
        s = wi.s;
        mu = wi.mu;
        decode(g, s, x);
        sig = staples_of_plane(g, Uin, V, s, x, mu, wi.j + (wi.j >= mu ? 1 : 0), own);
        valid = wide_sum(sig, wi.j, dst) && wi.site < g.V;
    } else {
        const SiteMu sm = site_mu_index(g);
        s = stencil_site<ST == ST_ROWS>(g, sm);
        mu = sm.mu;
        decode(g, s, x);
        sig = staple_sigma_shared(g, Uin, V, s, x, mu, own, xs);
        valid = in_lattice<ST == ST_ROWS>(g, sm);
    }
    if (!valid) return;
    back_local<T>(sig, own, [&] { return ldm<T, GF_LD_NT>(Dout, V, mu, s); }, Din, Lc, rho, V, mu, s, lane,
                  dst[ST == ST_WIDE ? 0 : mu]);
}
// Lam and Din without (Lam C)^dag, from Q, the link and Dout
template <typename T>
__device__ __forceinline__ void back_local_q(const T q[8], const M3<T>& u, const M3<T>& dout, T* __restrict__ Din,
                                             T* __restrict__ Lc, unsigned V, int mu, int s, int lane, MStage<T> dst) {
    M3<T> E, L;
    {
        const Herm<T> h = herm_of_coeffs(q);
        M3<T> Q;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const cx<T> e = herm_el(h, i, j);
                Q.m[3 * i + j].r = -e.i;
                Q.m[3 * i + j].i = e.r;
            }
        exp_dexp(Q, mul(u, stage_m3<T>(dst, lane, dout)), E, L);
    }
    T c[8];
    ta_coeffs(L, c);
    stp<T, GF_ST_NT>(Lc, V, mu, s, c);
    stm<T, GF_ST_NT>(Din, V, mu, s, mul(staged_m3<T>(dst, lane), E));
}
// a thread per link
template <typename T>
__global__ __launch_bounds__(kBlock) void k_stout_back_local_q(Geo g, const T* __restrict__ U, const T* __restrict__ Qst,
                                                               const T* __restrict__ Dout, T* __restrict__ Din, T* __restrict__ Lc) {
    __shared__ T2<T> dst[4][9][64];
    const SiteMu sm = site_mu_index(g);
    const int s = sm.s, mu = sm.mu;
    if (s >= g.V) return;
    const unsigned V = g.V;
    T q[8];
    ldp<T, GF_LD_NT>(Qst, V, mu, s, q);
    back_local_q<T>(q, ldu<T, GF_LD_NT>(U, V, mu, s), ldm<T, GF_LD_NT>(Dout, V, mu, s), Din, Lc, V, mu, s,
                    (int)(threadIdx.x & 63u), dst[mu]);
}
// ---------------------------------------------------------------------------
// K6b: stout backward, staple-derivative part (calc_dSdUν_fromdSCμ_add!, stout_fast.jl:712-785):
// for output direction a at site y and each plane b != a, with G = U^dag Lam,
//   Din_a(y) += rho [ U_b(y+a) (G_a(y+b) U_b(y)^dag + U_a(y+b)^dag G_b(y))
//                   + U_b(y-b+a)^dag (G_a(y-b) U_b(y-b) + U_a(y-b)^dag G_b(y-b)^dag)
//                   + G_b(y+a)^dag U_a(y+b)^dag U_b(y)^dag
//                   + G_b(y+a-b) U_a(y-b)^dag U_b(y-b) ]
// evaluated with Lam directly (Lam^dag = -Lam): with X = U_b(y+a) U_a(y+b)^dag, S = X U_b(y)^dag,
// Z = U_a(y-b)^dag U_b(y-b),
//   upper = X Lam_a(y+b) U_b(y)^dag + S Lam_b(y) - Lam_b(y+a) S
//   lower = U_b(y+a-b)^dag [U_a(y-b)^dag (Lam_a(y-b) - Lam_b(y-b)) U_b(y-b) + Lam_b(y+a-b) Z]
//         = U_b(y+a-b)^dag [U_a(y-b)^dag (Lam_a(y-b) - Lam_b(y-b)) + Lam_b(y+a-b) U_a(y-b)^dag] U_b(y-b)
// Six links and six 8-real Lam per plane instead of ten links and six 18-real G.  Lam = i H with
// H Hermitian (its 8 coefficients): products with Lam are i times Hermitian-structured products.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ Herm<T> herm_at(const T* __restrict__ Lc, unsigned V, int mu, unsigned s) {
    T c[8];
    ldp(Lc, V, mu, s, c);
    return herm_of_coeffs(c);
}
// c += SG i m h  (SG = +1 or -1), each product element accumulated as it is formed
template <typename T, int SG>
__device__ __forceinline__ void acc_i_mh(M3<T>& c, const M3<T>& m, const Herm<T>& h) {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            cx<T> t;
            t.r = m.m[3 * i + j].r * h.d[j];
            t.i = m.m[3 * i + j].i * h.d[j];
#pragma unroll
            for (int k = 0; k < 3; k++)
                if (k != j) cmac(t, m.m[3 * i + k], herm_off(h, k, j));
            c.m[3 * i + j].r -= T(SG) * t.i;
            c.m[3 * i + j].i += T(SG) * t.r;
        }
}
// c += SG i h m
template <typename T, int SG>
__device__ __forceinline__ void acc_i_hm(M3<T>& c, const Herm<T>& h, const M3<T>& m) {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            cx<T> t;
            t.r = h.d[i] * m.m[3 * i + j].r;
            t.i = h.d[i] * m.m[3 * i + j].i;
#pragma unroll
            for (int k = 0; k < 3; k++)
                if (k != i) cmac(t, herm_off(h, i, k), m.m[3 * k + j]);
            c.m[3 * i + j].r -= T(SG) * t.i;
            c.m[3 * i + j].i += T(SG) * t.r;
        }
}
// c += h m^dag
template <typename T>
__device__ __forceinline__ void acc_hd(M3<T>& c, const Herm<T>& h, const M3<T>& m) {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            cx<T>& t = c.m[3 * i + j];
            t.r = fma(h.d[i], m.m[3 * j + i].r, t.r);
            t.i = fma(-h.d[i], m.m[3 * j + i].i, t.i);
#pragma unroll
            for (int k = 0; k < 3; k++)
                if (k != i) cmac_nc(t, herm_off(h, i, k), m.m[3 * j + k]);
        }
}

// Plane b of K6b added into acc.  SH: U_b(y) and Lam_b(y) come from the workgroup's LDS copies (ul, hl);
// A0 (a = 0) and B0 (b = 0): the x-neighbour links and Lam at y + 1 and y - 1 (xr) as well.  SL adds the plane's
// part of -Sigma_a Lam_a: of the staples S and U_b(y+a-b)^dag U_a(y-b)^dag U_b(y-b) times H_a(y), by H_b(y) - H_a(y) in
// place of H_b(y) and H_d - U_b(y-b) H_a(y) U_b(y-b)^dag in place of H_d.
template <typename T, bool SL, bool SH, bool A0, bool B0>
__device__ __forceinline__ void back_plane(const Geo& g, const T* __restrict__ U, const T* __restrict__ Lc, unsigned V,
                                           int y, const int x[4], int a, int b, int ypa, M3<T>& acc, XLinks<T> ul,
                                           XCoefs<T> hl, int lane, const XRow& xr) {
    const int ypb0 = y + dlt(g, x, b, 1);
    // each group loads its links through its own opaque index copies, so the compiler
    // issues them group by group instead of hoisting all of them
    {  // upper: i X H_a(y+b) U_b(y)^dag + i [S H_b(y) - H_b(y+a) S],  S = X U_b(y)^dag
        int y1 = ypa, ypb = ypb0;
        asm volatile("" : "+v"(y1), "+v"(ypb));
        const R6<T> uby = A0 ? shared_link<T>(ul, b, xr.p) : ldr(U, V, b, y1);                // U_b(y+a)
        const M3<T> X = su3_mul_nd(uby, full_of(B0 ? shared_link<T>(ul, a, xr.p) : ldr(U, V, a, ypb)));  // U_a(y+b)
        T c[8];
        if (B0) get_c8(hl, a, xr.p, c);  // Lam_a(y+b)
        else ldp(Lc, V, a, ypb, c);
        const M3<T> XH = times_i(mul_mh(X, herm_of_coeffs(c)));
        const M3<T> ub = full_of(SH ? shared_link<T>(ul, b, lane) : ldr(U, V, b, (unsigned)y));        // U_b(y)
        acc_mul_nd(acc, XH, ub);
        const M3<T> S = su3_mul_nd(rows_of(X), ub);
        if (SH) get_c8(hl, b, lane, c);  // Lam_b(y)
        else ldp(Lc, V, b, (unsigned)y, c);
        if (SL) {
            T own[8];
            get_c8(hl, a, lane, own);
#pragma unroll
            for (int k = 0; k < 8; k++) c[k] -= own[k];
        }
        acc_i_mh<T, 1>(acc, S, herm_of_coeffs(c));
        if (A0) get_c8(hl, b, xr.p, c);  // Lam_b(y+a)
        else ldp(Lc, V, b, y1, c);
        acc_i_hm<T, -1>(acc, herm_of_coeffs(c), S);
    }
    {  // lower: U_b(y+a-b)^dag i [U_a(y-b)^dag H_d + H_b(y+a-b) U_a(y-b)^dag] U_b(y-b),
       // H_d = H_a(y-b) - H_b(y-b)
        // opaque: the offset is formed here, not kept through the upper staple (registers)
        int xb = sel4(b, x[0], x[1], x[2], x[3]);
        asm volatile("" : "+v"(xb));
        const int dmb = (xb == 0 ? sel4(b, g.n[0], g.n[1], g.n[2], g.n[3]) - 1 : -1) * sel4(b, g.st[0], g.st[1], g.st[2], g.st[3]);
        int ymb = y + dmb, ypamb = ypa + dmb;
        asm volatile("" : "+v"(ymb), "+v"(ypamb));
        Herm<T> hd;
        {
            T ca[8], cb[8];
            if (B0) {
                get_c8(hl, a, xr.m, ca);
                get_c8(hl, 0, xr.m, cb);
            } else {
                ldp(Lc, V, a, ymb, ca);
                ldp(Lc, V, b, ymb, cb);
            }
#pragma unroll
            for (int k = 0; k < 8; k++) ca[k] -= cb[k];
            hd = herm_of_coeffs(ca);
        }
        if (SL) {
            T own[8];
            get_c8(hl, a, lane, own);
            const Herm<T> t = herm_conj(full_of(B0 ? shared_link<T>(ul, 0, xr.m) : ldr(U, V, b, ymb)), herm_of_coeffs(own));
#pragma unroll
            for (int k = 0; k < 3; k++) {
                hd.d[k] -= t.d[k];
                hd.u[k].r -= t.u[k].r;
                hd.u[k].i -= t.u[k].i;
            }
            // formed before the links below are loaded (registers)
#pragma unroll
            for (int k = 0; k < 3; k++) asm volatile("" : "+v"(hd.d[k]), "+v"(hd.u[k].r), "+v"(hd.u[k].i));
            asm volatile("" : "+v"(ymb), "+v"(ypamb));
        }
        const M3<T> ua = full_of(B0 ? shared_link<T>(ul, a, xr.m) : ldr(U, V, a, ymb));  // U_a(y-b)
        M3<T> A = mul_dh(ua, hd);
        acc_hd(A, herm_at(Lc, V, b, ypamb), ua);
        const M3<T> ubm = full_of(B0 ? shared_link<T>(ul, 0, xr.m) : ldr(U, V, b, ymb));  // U_b(y-b)
        acc_mul_dn(acc, ldu(U, V, b, ypamb), times_i(mul(A, ubm)));
    }
}

// The staple part of K6b for output direction a at site y (all planes b != a).  U(y) and Lam(y) of
// the workgroup's sites and of their x-neighbours go through LDS (per wave 12 link and 6 Lam loads
// fewer than from memory); one workgroup barrier after filling ul/hl.
template <bool ROWS, bool SL, typename T>
__device__ __forceinline__ M3<T> back_stencil_acc(const Geo& g, const T* __restrict__ U, const T* __restrict__ Lc,
                                                  int y, const int x[4], int a, int lane, XLinks<T> ul,
                                                  XCoefs<T> hl) {
    const unsigned V = g.V;
    const XRow xr = xrow_of<ROWS>(g, y, x[0], lane);
    {
        T c[8];
        const R6<T> u = ldr(U, V, a, (unsigned)y);
        ldp(Lc, V, a, (unsigned)y, c);
        share_links<ROWS, T>(ul, U, V, a, lane, xr, u);
        put_c8(hl, a, lane, c);
        if (!ROWS && xr.halo >= 0) {
            ldp(Lc, V, a, (unsigned)xr.halo, c);
            put_c8(hl, a, 64 + lane, c);
        }
        __syncthreads();
    }
    M3<T> acc = zero3<T>();
    const int ypa = y + dlt(g, x, a, 1);
    if (a == 0) {
#pragma unroll 1
        for (int b = 1; b < 4; b++) back_plane<T, SL, true, true, false>(g, U, Lc, V, y, x, a, b, ypa, acc, ul, hl, lane, xr);
    } else {
        back_plane<T, SL, true, false, true>(g, U, Lc, V, y, x, a, 0, ypa, acc, ul, hl, lane, xr);
#pragma unroll 1
        for (int b = 1; b < 4; b++) {
            if (b == a) continue;
            back_plane<T, SL, true, false, false>(g, U, Lc, V, y, x, a, b, ypa, acc, ul, hl, lane, xr);
        }
    }
    return acc;
}
// Din_a(y) + rho * (staple part)
template <typename T>
__device__ __forceinline__ M3<T> back_din(const T* __restrict__ Din, unsigned V, int a, int y, double rho,
                                          const M3<T>& acc) {
    M3<T> dn = ldm<T, GF_LD_NT>(Din, V, a, y);
#pragma unroll
    for (int k = 0; k < 9; k++) {
        dn.m[k].r = fma1(rho, acc.m[k].r, dn.m[k].r);
        dn.m[k].i = fma1(rho, acc.m[k].i, dn.m[k].i);
    }
    return dn;
}
// K6b: Din += rho (staple part; SL: and -Sigma Lam).  LOCAL: followed by K6a of the level below (Uprev its input links,
// Qprev its Q), whose Dout this Din is: not stored and read back (1152 B a site in FP64).  Lout is another buffer than Lc,
// whose entries at neighbour sites other workgroups still read.  At most 168 VGPRs (FP64), so that three waves fit per
// SIMD; with K6a two.
template <typename T, bool ROWS, bool SL, bool LOCAL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(LOCAL && sizeof(T) == 8 ? 2 : 3))) void
k_stout_back_stencil(Geo g, const T* __restrict__ U, const T* __restrict__ Lc, T* __restrict__ Din, double rho,
                     const T* __restrict__ Uprev, const T* __restrict__ Qprev, T* __restrict__ Lout) {
    // links and Lam of the sites and their x-neighbours; then Dout of the level below
    __shared__ __align__(16) unsigned char sh[4 * 10 * kXW * sizeof(T2<T>)];
    XLinks<T> ul = reinterpret_cast<XLinks<T>>(sh);
    XCoefs<T> hl = reinterpret_cast<XCoefs<T>>(sh + 4 * 6 * kXW * sizeof(T2<T>));
    const unsigned V = g.V;
    const int lane = (int)(threadIdx.x & 63u);
    const SiteMu sm = site_mu_index(g);
    const int a = sm.mu, y = stencil_site<ROWS>(g, sm);
    int x[4];
    decode(g, y, x);
    const M3<T> acc = back_stencil_acc<ROWS, SL>(g, U, Lc, y, x, a, lane, ul, hl);
    if constexpr (LOCAL) __syncthreads();  // every wave is done with ul and hl
    if (!in_lattice<ROWS>(g, sm)) return;
    const M3<T> dn = back_din(Din, V, a, y, rho, acc);
    if constexpr (LOCAL) {
        MStage<T> dst = reinterpret_cast<T2<T>(*)[9][64]>(sh)[a];
        T q[8];
        ldp<T, GF_LD_NT>(Qprev, V, a, y, q);
        back_local_q<T>(q, ldu<T, GF_LD_NT>(Uprev, V, a, y), dn, Din, Lout, V, a, y, lane, dst);
    } else {
        stm<T, GF_ST_NT>(Din, V, a, y, dn);
    }
}
template <typename T>
__global__ __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(2))) void k_stout_back_stencil_wide(
    Geo g, const T* __restrict__ U, const T* __restrict__ Lc, T* __restrict__ Din, double rho) {
    __shared__ T2<T> red[2][9][64];
    const WideIndex wi = wide_index(g);
    const int y = wi.s, a = wi.mu;
    int x[4];
    decode(g, y, x);
    M3<T> acc = zero3<T>();
    back_plane<T, false, false, false, false>(g, U, Lc, (unsigned)g.V, y, x, a, wi.j + (wi.j >= a ? 1 : 0), y + dlt(g, x, a, 1),
                                       acc, nullptr, nullptr, (int)(threadIdx.x & 63u), XRow{});
    if (!wide_sum(acc, wi.j, red) || wi.site >= g.V) return;
    stm<T, GF_ST_NT>(Din, (unsigned)g.V, a, y, back_din(Din, (unsigned)g.V, a, y, rho, acc));
}

// K6b of a level and K6a of the one below (Uprev its input links) in one launch, on small lattices: the
// three waves form their planes' parts of both stencils.  Lout is another buffer than Lc, whose entries
// at neighbour sites other workgroups still read.
template <typename T>
__global__ __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(1))) void k_stout_back_chain_wide(
    Geo g, const T* __restrict__ U, const T* __restrict__ Lc, T* __restrict__ Din, double rho,
    const T* __restrict__ Uprev, T* __restrict__ Lout) {
    __shared__ T2<T> red[2][2][9][64];
    const unsigned V = g.V;
    const int lane = (int)(threadIdx.x & 63u);
    const WideIndex wi = wide_index(g);
    const int a = wi.mu, b = wi.j + (wi.j >= a ? 1 : 0);
    int x[4];
    decode(g, wi.s, x);
    R6<T> own;
    M3<T> sig = staples_of_plane(g, Uprev, V, wi.s, x, a, b, own);
#pragma unroll
    for (int e = 0; e < 9; e++) asm volatile("" : "+v"(sig.m[e].r), "+v"(sig.m[e].i));  // one stencil after the other
    M3<T> acc = zero3<T>();
    back_plane<T, false, false, false, false>(g, U, Lc, V, wi.s, x, a, b, wi.s + dlt(g, x, a, 1), acc, nullptr, nullptr, lane,
                                       XRow{});
    const bool first = wide_sum(sig, wi.j, red[0]);
    wide_sum(acc, wi.j, red[1]);
    if (!first || wi.site >= g.V) return;
    back_local<T>(sig, own, [&] { return back_din(Din, V, a, wi.s, rho, acc); }, Din, Lout, rho, V, a, wi.s, lane,
                  red[0][0]);
}

// ---------------------------------------------------------------------------
template <typename T>
hipError_t launch_flow_stage(const Geo& g, const T* W, T* Wout, T* A, double alpha, double beta, hipStream_t st) {
    by_form<T>(g, [&](auto f) {
        k_flow_stage<T, decltype(f)::value><<<stencil_groups(f, grid_sites_mu(g.V)), stencil_threads(f), 0, st>>>(g, W, Wout, A, alpha, beta);
    });
    return hipGetLastError();
}
// Uout / Qst null: not written (one of them is wanted)
template <typename T>
hipError_t launch_stout_forward(const Geo& g, const T* Uin, T* Uout, T* Qst, double rho, hipStream_t st) {
    by_form<T>(g, [&](auto f) {
        const int nb = stencil_groups(f, grid_sites_mu(g.V)), nt = stencil_threads(f);
        if (Uout && Qst)
            k_stout_forward<T, STOUT_LINKS | STOUT_Q, decltype(f)::value><<<nb, nt, 0, st>>>(g, Uin, Uout, Qst, rho);
        else if (Uout)
            k_stout_forward<T, STOUT_LINKS, decltype(f)::value><<<nb, nt, 0, st>>>(g, Uin, Uout, Qst, rho);
        else
            k_stout_forward<T, STOUT_Q, decltype(f)::value><<<nb, nt, 0, st>>>(g, Uin, Uout, Qst, rho);
    });
    return hipGetLastError();
}
template <typename T>
hipError_t launch_stout_top(const Geo& g, const T* Utop, double coeff, const T* Qst, T* Lc, T* Fl, hipStream_t st) {
    by_form<T>(g, [&](auto f) {
        k_stout_top<T, decltype(f)::value><<<stencil_groups(f, grid_sites_mu(g.V)), stencil_threads(f), 0, st>>>(
            g, Utop, coeff, Qst, Lc, Fl);
    });
    return hipGetLastError();
}
// Six waves a group, one pair each, up to 256 groups, a workgroup per CU; four above.  Kernel, six / four waves, us: FP64 64
// groups 10.9 / 12.6, 256 12.8 / 13.8, 282 19.9 / 18.6, 384 21.5 / 19.8, 1024 48.0 / 37.0; FP32 64 8.1 / 10.4, 256 9.7 / 12.2,
// 384 13.5 / 13.6, 512 13.8 / 14.4, 648 16.3 / 16.0, 1024 27.6 / 21.3.
template <typename T>
hipError_t launch_stout_pair(const Geo& g, const T* U, const T* Lc, T* Fl, T* far, double rho, hipStream_t st) {
    const int groups = grid_sites_mu(g.V);
    by_rows(g, [&](auto rows) {
        if (groups <= 256)
            k_stout_pair<T, decltype(rows)::value, 6><<<groups, 384, 0, st>>>(g, U, Lc, Fl, far, rho);
        else
            k_stout_pair<T, decltype(rows)::value, 4><<<groups, 256, 0, st>>>(g, U, Lc, Fl, far, rho);
    });
    return hipGetLastError();
}
// Workgroups of one wave up to 512 groups, of four above.  Kernel, one / four waves, us: FP64 64 groups 4.8 / 5.3, 256 8.5 /
// 7.8, 384 11.3 / 11.0, 512 11.6 / 12.8, 768 17.8 / 18.2, 1250 25.7 / 26.2; FP32 64 4.8 / 5.2, 256 5.5 / 5.5, 512 10.4 / 9.5, 648
// 10.8 / 10.8, 1024 14.9 / 16.8, 1250 17.6 / 16.9: it matters below 100 groups only.
template <typename T>
hipError_t launch_stout_gather(const Geo& g, const T* far, T* Fl, double rho, const T* Qst, T* Lc, hipStream_t st,
                               int fmode, const T* U, T* FP, double eps_p, T* Unew, double eps_u, double* U64) {
    const int groups = grid_sites_mu(g.V);
    const bool small = groups <= 512;
    const int nb = small ? 4 * groups : groups, nt = small ? 64 : kBlock;
    const double fac = -1.0 / 3.0;
    auto go = [&](auto out) {
        constexpr int OUT = decltype(out)::value;
        const bool s64 = OUT == FORCE_KICK_S64 || OUT == FORCE_KICK_EXP_S64;
        by_rows(g, [&](auto rows) {
            k_stout_gather<T, OUT, decltype(rows)::value><<<nb, nt, 0, st>>>(
                g, far, Fl, rho, Qst, Lc, U, FP, Unew, OUT == FORCE_KICK || OUT == FORCE_KICK_EXP ? fac * eps_p : fac,
                eps_u, s64 ? eps_p : 0.0, U64);
        });
    };
    switch (fmode) {
        case FORCE_STORE: go(std::integral_constant<int, FORCE_STORE>{}); break;
        case FORCE_KICK: go(std::integral_constant<int, FORCE_KICK>{}); break;
        case FORCE_KICK_EXP: go(std::integral_constant<int, FORCE_KICK_EXP>{}); break;
        case FORCE_KICK_S64:
        case FORCE_KICK_EXP_S64:
            if constexpr (sizeof(T) == 4) {  // FP32 force kernels only
                if (fmode == FORCE_KICK_S64)
                    go(std::integral_constant<int, FORCE_KICK_S64>{});
                else
                    go(std::integral_constant<int, FORCE_KICK_EXP_S64>{});
                break;
            } else {
                return hipErrorInvalidValue;
            }
        default: go(std::integral_constant<int, -1>{});
    }
    return hipGetLastError();
}
template <typename T>
hipError_t launch_stout_backward(const Geo& g, const T* const* Uin, const T* const* Q, int nlev, const T* D, T* D2,
                                 T* Lc, T* Lc2, double rho, hipStream_t st) {
    const int groups = grid_sites_mu(g.V), top = nlev - 1;
    T *la = Lc, *lb = Lc2;
    if (stencil_form<T>(g) == ST_WIDE) {
        const int nb = stencil_groups(ST_WIDE, groups), nt = stencil_threads(ST_WIDE);
        k_stout_back_local<T, ST_WIDE><<<nb, nt, 0, st>>>(g, Uin[top], D, D2, la, rho);
        for (int l = top; l >= 1; l--, std::swap(la, lb))
            k_stout_back_chain_wide<T><<<nb, nt, 0, st>>>(g, Uin[l], la, D2, rho, Uin[l - 1], lb);
        k_stout_back_stencil_wide<T><<<nb, nt, 0, st>>>(g, Uin[0], la, D2, rho);
        return hipGetLastError();
    }
    by_rows(g, [&](auto rows) {
        constexpr bool R = decltype(rows)::value;
        if (Q) {
            k_stout_back_local_q<T><<<groups, kBlock, 0, st>>>(g, Uin[top], Q[top], D, D2, la);
            for (int l = top; l >= 1; l--, std::swap(la, lb))
                k_stout_back_stencil<T, R, true, true><<<groups, kBlock, 0, st>>>(g, Uin[l], la, D2, rho, Uin[l - 1], Q[l - 1], lb);
            k_stout_back_stencil<T, R, true, false><<<groups, kBlock, 0, st>>>(g, Uin[0], la, D2, rho, nullptr, nullptr, nullptr);
            return;
        }
        constexpr int ST = R ? ST_ROWS : ST_CUT;
        for (int l = top; l >= 0; l--) {
            k_stout_back_local<T, ST><<<groups, kBlock, 0, st>>>(g, Uin[l], l == top ? D : D2, D2, la, rho);
            k_stout_back_stencil<T, R, false, false><<<groups, kBlock, 0, st>>>(g, Uin[l], la, D2, rho, nullptr, nullptr, nullptr);
        }
    });
    return hipGetLastError();
}

#define GF_INST2(T)                                                                                       \
    template hipError_t launch_flow_stage<T>(const Geo&, const T*, T*, T*, double, double, hipStream_t);  \
    template hipError_t launch_stout_forward<T>(const Geo&, const T*, T*, T*, double, hipStream_t);       \
    template hipError_t launch_stout_top<T>(const Geo&, const T*, double, const T*, T*, T*, hipStream_t); \
    template hipError_t launch_stout_pair<T>(const Geo&, const T*, const T*, T*, T*, double, hipStream_t); \
    template hipError_t launch_stout_gather<T>(const Geo&, const T*, T*, double, const T*, T*, hipStream_t, int, \
                                               const T*, T*, double, T*, double, double*);                \
    template hipError_t launch_stout_backward<T>(const Geo&, const T* const*, const T* const*, int, const T*, T*,  \
                                                 T*, T*, double, hipStream_t);

GF_INST2(double)
GF_INST2(float)

}  // namespace gf
