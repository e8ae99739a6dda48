// internal.hpp -- host-side declarations shared by the kernel translation units and the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <type_traits>

#include "lattice.hpp"

namespace gf {

constexpr int kBlock = 256;

inline int grid_for(int V, int block = kBlock) { return (V + block - 1) / block; }
// gridDim.y of the streaming link kernels: threads per site (4: one per link) on lattices of so few
// workgroups of sites that CUs stay empty (4^4: 5.2 -> 3.5 us, 12^3x8: 7.6 -> 3.7; 16^4: 12.4 -> 12.9, hence
// the limit between)
inline int link_dirs(int V) { return grid_for(V) <= 128 ? 4 : 1; }
// grid of the (site, direction) kernels: one 256-thread workgroup per 64 sites
inline int grid_sites_mu(int V) { return (V + 63) / 64; }

// f(std::true_type) where every 64-site group is whole x-rows (rows_whole), f(std::false_type) otherwise
template <typename F>
inline void by_rows(const Geo& g, F&& f) {
    if (rows_whole(g))
        f(std::true_type{});
    else
        f(std::false_type{});
}
// f(std::integral_constant<int, ST>) of the lattice's stencil form for fields of T
template <typename T, typename F>
inline void by_form(const Geo& g, F&& f) {
    const int form = stencil_form<T>(g);
    if (form == ST_WIDE)
        f(std::integral_constant<int, ST_WIDE>{});
    else if (form == ST_ROWS)
        f(std::integral_constant<int, ST_ROWS>{});
    else
        f(std::integral_constant<int, ST_CUT>{});
}

// force kernel modes
enum ForceMode { FORCE_STORE = 0, FORCE_KICK = 1, FORCE_KICK_EXP = 2, FORCE_KICK_S64 = 3, FORCE_KICK_EXP_S64 = 4 };
// FORCE_KICK_S64 / FORCE_KICK_EXP_S64 (FP32 kernels over an FP64 MD state): the FP32 force kicks the
// FP64 momenta, and the FP64 links are updated in place, their float rounding written to Unew

// What a force kernel does with fac * c, c = TA coefficients of a link (MODE: ForceMode; link() is U_mu(s),
// read only by the modes that update it)
template <typename T, int MODE, typename L>
__device__ __forceinline__ void force_out(T c[8], L&& link, unsigned V, int mu, int s, T* __restrict__ FP,
                                          T* __restrict__ Unew, double fac, double eps_u, double eps_p,
                                          double* __restrict__ U64) {
    if constexpr (MODE == FORCE_KICK_S64 || MODE == FORCE_KICK_EXP_S64) {
        double* P64 = reinterpret_cast<double*>(FP);
        double p[8];
        ldp<double, GF_LD_NT>(P64, V, mu, s, p);
#pragma unroll
        for (int a = 0; a < 8; a++) p[a] = fma(eps_p, (double)scale1(fac, c[a]), p[a]);
        stp<double, GF_ST_NT>(P64, V, mu, s, p);
        if constexpr (MODE == FORCE_KICK_EXP_S64) {
            const M3<double> un = exp_coeffs_times(p, eps_u, ldu<double, GF_LD_NT>(U64, V, mu, s));
            stu<double, GF_ST_NT>(U64, V, mu, s, un);
            stu<T, GF_ST_NT>(Unew, V, mu, s, round_link<T>(un));
        }
    } else if constexpr (MODE == FORCE_STORE) {
#pragma unroll
        for (int a = 0; a < 8; a++) c[a] = scale1(fac, c[a]);
        stp<T, GF_ST_NT>(FP, V, mu, s, c);
    } else {
        const M3<T> u = MODE == FORCE_KICK_EXP ? link() : M3<T>{};
        T p[8];
        ldp<T, GF_LD_NT>(FP, V, mu, s, p);
#pragma unroll
        for (int a = 0; a < 8; a++) p[a] = fma1(fac, c[a], p[a]);
        stp<T, GF_ST_NT>(FP, V, mu, s, p);
        if constexpr (MODE == FORCE_KICK_EXP) stu<T, GF_ST_NT>(Unew, V, mu, s, exp_coeffs_times(p, eps_u, u));
    }
}

// ---- k_gauge.hip ----
// dst = src, bytes a multiple of 16 (streaming copy: the measured HBM ceiling)
hipError_t launch_stream_copy(const void* src, void* dst, size_t bytes, hipStream_t st);
// FP64 link rows 0-1 (optionally SU(3)-projected first) and/or momenta rounded to float in place
hipError_t launch_round_f32(double* U, double* P, int V, bool links, bool project, bool momenta, hipStream_t st);
// out[0] = sum of partial[0..n) (one workgroup, fixed order)
hipError_t launch_sum_partials(const double* partial, int n, int sums, double* out, hipStream_t st);
// out null: the per-workgroup partials (grid_sites_mu(V) of them) only
template <typename T>
hipError_t launch_plaquette(const Geo& g, const T* U, double* partial, double* out, hipStream_t st);
template <typename T>
hipError_t launch_action_untraced(const Geo& g, const T* U, double coeff, double* ref, hipStream_t st);
template <typename T>
hipError_t launch_momenta_dot(const Geo& g, const T* P, double* partial, double* out, hipStream_t st);
template <typename T>
hipError_t launch_dsdu(const Geo& g, const T* U, double coeff, T* D, hipStream_t st);
// MODE FORCE_STORE: F = -(coeff/3) TA(U Sigma)
// MODE FORCE_KICK : P += eps_p * F
// MODE FORCE_KICK_EXP : P += eps_p * F;  Unew = exp(eps_u P) U
// MODE FORCE_KICK_S64, FORCE_KICK_EXP_S64 (float): the same on the FP64 momenta (FP) and links
//   (U64) of an FP64 state, with Unew the updated links rounded to float
template <typename T>
hipError_t launch_force(int mode, const Geo& g, const T* U, T* FP, T* Unew, double coeff, double eps_p,
                        double eps_u, hipStream_t st, double* U64 = nullptr);
template <typename T>
hipError_t launch_exp_update(const Geo& g, const T* Uin, T* Uout, const T* P, double eps, hipStream_t st);
// reference-layout (column-major 3x3 per link) <-> device field; general = false: SU(3) link
// field (rows 0 and 1 kept, row 2 rebuilt on the way out), true: general matrix field
hipError_t launch_links_widen(const float* Uf, double* Ud, int V, hipStream_t st);
// FP32 forces over an FP64 MD state (k_state64_step): mode 1 exp update of U64 (and its float
// rounding into U32), 3 rounding only
hipError_t launch_state64_step(int mode, const Geo& g, const double* P64, double* U64, float* U32, double eps_u,
                               hipStream_t st);
template <typename T>
hipError_t launch_links_from_ref(const double* ref, T* soa, int V, bool general, int q0, int nq, hipStream_t st);
template <typename T>
hipError_t launch_links_to_ref(const T* soa, double* ref, int V, bool general, int q0, int nq, hipStream_t st);
template <typename T>
hipError_t launch_momenta_from_ref(const double* ref, T* soa, int V, int q0, int nq, hipStream_t st);
template <typename T>
hipError_t launch_momenta_to_ref(const T* soa, double* ref, int V, int q0, int nq, hipStream_t st);
template <typename T>
hipError_t launch_set_identity(T* U, int V, hipStream_t st);
template <typename T>
hipError_t launch_fill(T* p, size_t n, T v, hipStream_t st);

// ---- k_fstrength.hip ----
// Field strengths of the loop sets in `sets` (bit 0 plaquette, 1 clover, 2 rectangle); out4 =
// {clover energy sum, plaquette Q, clover Q, rectangle Q}; dens (device, V) if
// non-null receives the density of dens_method (0 plaquette, 1 clover, 2 improved, 3 rectangle).
// fields: scratch of `bytes`, field_strength_bytes for the speed it is meant to have and at least that for
// most = 1 (one t-slice); partial: 4 (V / 64 + NT + 1) doubles
size_t field_strength_bytes(const Geo& g, int sets, size_t most);
template <typename T>
hipError_t launch_field_strength(const Geo& g, const T* U, int sets, void* fields, size_t bytes, double* partial,
                                 double* out4, double* dens, int dens_method, hipStream_t st);

// ---- k_random.hip ----
template <typename T>
hipError_t launch_gaussian_momenta(const Geo& g, T* P, double sigma, unsigned long long seed,
                                   unsigned long long sweep, hipStream_t st);
template <typename T>
hipError_t launch_hot_links(const Geo& g, T* U, unsigned long long seed, hipStream_t st);

// heatbath (mode 0) or overrelaxation (mode 1) sweep: mu = 0..3, colours even then odd;
// failures (device double) = links a heatbath left unchanged.  partial: >= 8 * (V/2 + 255)/256
template <typename T>
hipError_t launch_heatbath(const Geo& g, T* U, int mode, double beta, unsigned long long seed,
                           unsigned long long sweep, int itmax, double* partial, double* failures, hipStream_t st);

// ---- k_flow_stout.hip ----
// A = alpha * TA(W V^dag) + beta * A ; Wout = exp(A) W
template <typename T>
hipError_t launch_flow_stage(const Geo& g, const T* W, T* Wout, T* A, double alpha, double beta,
                             hipStream_t st);

// one smearing level: the smeared links (Uout) and / or the coefficients of Q (Qst); null: not wanted
template <typename T>
hipError_t launch_stout_forward(const Geo& g, const T* Uin, T* Uout, T* Qst, double rho, hipStream_t st);
// the backward pass of a stout force in the algebra (k_flow_stout.hip): F' of the top links and the top
// level's site-local step: Lam into Lc, Floc into Fl
template <typename T>
hipError_t launch_stout_top(const Geo& g, const T* Utop, double coeff, const T* Qst, T* Lc, T* Fl, hipStream_t st);
// the plaquettes of a level (U its input links): near contributions added to Fl, far ones (3 momentum fields)
template <typename T>
hipError_t launch_stout_pair(const Geo& g, const T* U, const T* Lc, T* Fl, T* far, double rho, hipStream_t st);
// F of the level's input links; fmode < 0: the site-local step of the level below (Qst its Q) into Lc
// and Fl; otherwise the force -(1/3) F as launch_force's modes, U the thin links
template <typename T>
hipError_t launch_stout_gather(const Geo& g, const T* far, T* Fl, double rho, const T* Qst, T* Lc, hipStream_t st,
                               int fmode = -1, const T* U = nullptr, T* FP = nullptr, double eps_p = 0.0,
                               T* Unew = nullptr, double eps_u = 0.0, double* U64 = nullptr);
// explicit backward pass of nlev levels: D2 = dS/dU_bare from D = dS/dU of the top level (general matrix fields).
// Uin[l] the input links of level l, Q[l] its Q; Q null: C formed from the staples again (as in any case where
// stout_backward_reads_q is false); Lc, Lc2: scratch momentum fields
inline bool stout_backward_reads_q(const Geo& g, bool f64) {
    return (f64 ? stencil_form<double>(g) : stencil_form<float>(g)) != ST_WIDE;
}
template <typename T>
hipError_t launch_stout_backward(const Geo& g, const T* const* Uin, const T* const* Q, int nlev, const T* D, T* D2,
                                 T* Lc, T* Lc2, double rho, hipStream_t st);

}  // namespace gf
