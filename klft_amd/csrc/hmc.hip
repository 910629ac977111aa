// HMC for the Wilson gauge action: momentum refresh, fused force + momentum
// update, link exponential update, kinetic / gauge action sums and the
// leapfrog trajectory with FP64 accept/reject.
//
// Semantics follow the reference's HMC stack (HMC.hpp:48-71,
// Integrator.hpp:26-53, GaugeMonomial.hpp:19-37, HamiltonianField.hpp:23-60,
// AdjointGroup.hpp), generalised to one formula for U(1), SU(2), SU(3):
//   P = sum_a p_a T_a, p_a ~ N(0,1);  H_kin = 1/2 sum p_a^2;
//   H_g = -(beta/Nc) sum_x sum_{mu<nu} Re Tr U_munu(x);
//   F_a(x,mu) = (beta/Nc) Im Tr(T_a U_mu(x) Sigma_mu(x));
//   P <- P - dtau F;  U <- exp(i dtau P) U.
// Momenta are stored structure-of-arrays: P[(mu * NGEN + a) * V + s] in the
// link precision, s the sublattice-major device index.
#include <hip/hip_runtime.h>

#include <cmath>
#include <utility>
#include <vector>

#include "internal.hpp"

using namespace kd;
namespace ki = klft_internal;

struct klft_hmc_s {
  klft_field_t f = nullptr;
  klft_hmc_params p{};
  void *P = nullptr;       // momenta (R)
  // the leapfrog's two link buffers: a trajectory reads the field's links
  // and alternates between these, then hands the final buffer to the field
  // and keeps the starting one, which a rejected trajectory hands back
  void *Ubuf[2] = {nullptr, nullptr};
  double *Fdbg = nullptr;  // force in host (AoS) order, for klft_hmc_force
  double *stage = nullptr; // host-order FP64 momenta for upload / download
};

template <typename R, int NC, int ND>
__global__ __launch_bounds__(256) void k_refresh(R *P, Geom g, uint64_t seed, uint32_t traj,
                                                  double *partials) {
  __shared__ double lds[8];
  constexpr int NG = Ngen<NC>::value;
  const long long s = (long long)blockIdx.x * 256 + threadIdx.x;  // device order
  double k = 0.0;
  if (s < g.V) {
    int x[ND];
    dev_coords<ND>(g, s, x);
    const uint32_t site = (uint32_t)lex_index<ND>(g, x);
#pragma unroll
    for (int mu = 0; mu < ND; ++mu) {
      klft_rng::Stream st(seed, klft_rng::TAG_MOMENTA, site, traj, 0, 0, (uint32_t)mu);
      double z[NG + 1];
#pragma unroll
      for (int a = 0; a < NG; a += 2) {
        const double u1 = 1.0 - st.u01(), u2 = st.u01();
        const double r = sqrt(-2.0 * log(u1)), t = 2.0 * KLFT_PI * u2;
        z[a] = r * cos(t);
        z[a + 1] = r * sin(t);
      }
      double n2 = 0.0;
#pragma unroll
      for (int a = 0; a < NG; ++a) {
        const R v = (R)z[a];
        P[((long long)mu * NG + a) * g.V + s] = v;
        n2 += (double)v * (double)v;
      }
      k += 0.5 * n2;
    }
  }
  block_partial<256>(k, lds, partials);
}

// P -= dtau * F with F recomputed from the current links.  Fout (optional):
// write F in host AoS order instead of updating P.  kin (optional): also
// reduce 1/2 sum p^2 of the updated momenta.
template <typename R, int NC, bool COMP, int ND, bool LOWREG>
__global__ __launch_bounds__(256) void k_force(Links<R, NC, COMP> f, R *P, Geom g,
                                                                     R coef, R dtau, double *Fout,
                                                                     double *partials) {
  f.nd = ND;
  __shared__ double lds[8];
  constexpr int NG = Ngen<NC>::value;
  const unsigned int lb = xcd_block(blockIdx.x, gridDim.x);
  int x[ND], mu;
  long long s;
  double k = 0.0;
  if (link_site<ND>(g, lb, x, &s, &mu)) {
    const Nbr<ND> nb = make_nbr<ND>(g, x, s);
    Mat<R, NC> S;
    if constexpr (LOWREG)
      S = staple_lowreg<R, NC, COMP, ND>(f, nb, mu);
    else
      S = staple<R, NC, COMP, ND>(f, nb, mu);
    const Mat<R, NC> M = mul(f.load(s, mu), S);
    R F[NG];
    project(M, coef, F);
    if (Fout) {
      const long long site = lex_index<ND>(g, x);
#pragma unroll
      for (int a = 0; a < NG; ++a) Fout[(site * ND + mu) * NG + a] = (double)F[a];
    } else {
      double n2 = 0.0;
#pragma unroll
      for (int a = 0; a < NG; ++a) {
        R *q = P + ((long long)mu * NG + a) * g.V + s;
        const R v = *q - dtau * F[a];
        *q = v;
        n2 += (double)v * (double)v;
      }
      k = 0.5 * n2;
    }
  }
  if (partials) block_partial<256>(k, lds, partials);
}

// loads and stores past the caches (NT), for arrays that a launch touches once
template <bool NT, typename R>
__device__ __forceinline__ R load_stream(const R *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  return *p;
}
template <bool NT, typename R>
__device__ __forceinline__ void store_stream(R *p, R v) {
  if constexpr (NT)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// One leapfrog step with the momentum and link updates fused and the links
// double-buffered: F from the links in src, P <- P - dtp F, and
// dst(x,mu) = exp(i dtu P(x,mu)) src(x,mu) (FP32 links reunitarised).  The
// staples read src only, so no link is written while another thread may
// still read it; the arithmetic is that of k_force followed by
// k_update_gauge, so the result is the same.  One thread per link as in
// k_force: a block holds one 64-site chunk, wave w taking direction w.  For the
// SU(3) lattices where a step lasts as long as one thread (directions_per_thread);
// the others take k_step_dirs.  Past the caches (NT) by request and in tuning only:
// the rule's lattices fit them.
template <typename R, int NC, bool COMP, int ND, bool NT>
__global__ __launch_bounds__(256) void k_md_step(Links<R, NC, COMP> src, Links<R, NC, COMP> dst, R *P, Geom g,
                                                  R coef, R dtp, R dtu) {
  src.nd = ND;
  dst.nd = ND;
  constexpr int NG = Ngen<NC>::value;
  const unsigned int lb = xcd_block(blockIdx.x, gridDim.x);
  int x[ND], mu;
  long long s;
  if (!link_site<ND>(g, lb, x, &s, &mu)) return;
  R pm[NG];
#pragma unroll
  for (int a = 0; a < NG; ++a) pm[a] = load_stream<NT>(P + ((long long)mu * NG + a) * g.V + s);
  const Mat<R, NC> S = staple<R, NC, COMP, ND>(src, make_nbr<ND>(g, x, s), mu);
  const Mat<R, NC> U = src.load(s, mu);
  R v[NG];
  project(mul(U, S), coef, v);
#pragma unroll
  for (int a = 0; a < NG; ++a) {
    const R pn = pm[a] - dtp * v[a];
    store_stream<NT>(P + ((long long)mu * NG + a) * g.V + s, pn);
    v[a] = dtu * pn;
  }
  const Mat<R, NC> e = exp_iq(v, (Mat<R, NC> *)nullptr);
  Mat<R, NC> u = mul(e, U);
  if constexpr (sizeof(R) == 4) reunitarize(u);
  if constexpr (NT)
    dst.store_stream(s, mu, u);
  else
    dst.store(s, mu, u);
}

// The step (GAUGE) and the force (P only; Fout and kin as in k_force) with K
// directions per thread: a block holds 64 sites, wave h taking the directions
// h K .. h K + K - 1.  Bound by the L1: a CU keeps about 60 requests of 128
// bytes in flight, and nearly each one waits for the memory-side cache or HBM, so
// the time goes with the number of link loads, 19 a link with a thread per
// link, 15 with two directions per thread, 11 with four (staples_of).
// SU(3) 28x24x20x32 FP32 170 -> 145 us per step, 32^4 FP32 454 -> 340,
// FP64 (two directions, 256 registers and 8 spilled, 14 in the force; four need 488,
// one wave per SIMD) 860 -> 731, SU(2) 16^4 FP64 32 -> 17.
// With ND directions the next term's links are in flight while a term is
// multiplied; with two, twice the waves do the same and the registers
// that takes would cost one (SU(3) FP64 32^4 950 us).
constexpr int step_waves(int rbytes, int nc, int k) { return rbytes == 8 && nc == 3 && k > 2 ? 1 : 2; }
template <typename R, int NC, bool COMP, int ND, int K, bool NT, bool GAUGE>
__global__ __launch_bounds__(64 * ND / K, step_waves(sizeof(R), NC, K)) void k_step_dirs(
    Links<R, NC, COMP> src, Links<R, NC, COMP> dst, R *P, Geom g, R coef, R dtp, R dtu, double *Fout,
    double *partials) {
  src.nd = ND;
  dst.nd = ND;
  constexpr int NG = Ngen<NC>::value, NSUB = 1 << ND, NW = ND / K;
  const unsigned int lb = xcd_block(blockIdx.x, gridDim.x);
  const int sub = (int)(lb % NSUB), h = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // lanes past the sublattice repeat its last site, with the same stores: a
  // wave that runs with 16 lanes or fewer takes longer than a full one (SU(3)
  // 10x8x10x8, whose last blocks hold 16 sites, FP64 23.5 instead of 18.9 us per
  // step, two rows 24.8 instead of 15.2; 4^4 FP64 23.5 instead of 16.1)
  const long long rl = (long long)(lb / NSUB) * 64 + (threadIdx.x & 63), r = rl < g.Vh ? rl : g.Vh - 1;
  double kin = 0.0;
  {
    int x[ND];
    sub_coords<ND>(g, sub, r, x);
    const long long s = (long long)sub * g.Vh + r;
    R pm[2][NG];
    auto load_p = [&](int k, R *o) {
#pragma unroll
      for (int a = 0; a < NG; ++a) o[a] = load_stream<NT>(P + ((long long)(h * K + k) * NG + a) * g.V + s);
    };
    Mat<R, NC> U[K], S[K];
    const Nbr<ND> nb = make_nbr<ND>(g, x, s);
    if (NW == 1 || h == 0)
      staples_of<R, NC, COMP, ND, 0, K, K == ND>(src, nb, U, S);
    else
      staples_of<R, NC, COMP, ND, ND - K, K, K == ND>(src, nb, U, S);
    // the next direction's momenta are in flight while this one is updated
    load_p(0, pm[0]);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k + 1 < K) load_p(k + 1, pm[(k + 1) & 1]);
      const int mu = h * K + k;
      R v[NG];
      project(mul(U[k], S[k]), coef, v);
      if constexpr (!GAUGE) {
        if (Fout) {
          const long long site = lex_index<ND>(g, x);
#pragma unroll
          for (int a = 0; a < NG; ++a) Fout[(site * ND + mu) * NG + a] = (double)v[a];
          continue;
        }
      }
      double n2 = 0.0;
#pragma unroll
      for (int a = 0; a < NG; ++a) {
        const R pn = pm[k & 1][a] - dtp * v[a];
        store_stream<NT>(P + ((long long)mu * NG + a) * g.V + s, pn);
        if constexpr (!GAUGE) n2 += (double)pn * (double)pn;
        v[a] = dtu * pn;
      }
      kin += rl < g.Vh ? 0.5 * n2 : 0.0;
      if constexpr (GAUGE) {
        Mat<R, NC> u = mul(exp_iq(v, (Mat<R, NC> *)nullptr), U[k]);
        if constexpr (sizeof(R) == 4) reunitarize(u);
        if constexpr (NT)
          dst.store_stream(s, mu, u);
        else
          dst.store(s, mu, u);
      }
      asm volatile("" ::: "memory");
    }
  }
  if constexpr (!GAUGE) {
    __shared__ double lds[NW];
    if (partials) block_partial<64 * NW>(kin, lds, partials);
  }
}

// U <- exp(i dtau P) U; FP32 links are reunitarised after the update
template <typename R, int NC, bool COMP, int ND>
__global__ __launch_bounds__(256) void k_update_gauge(Links<R, NC, COMP> f, const R *__restrict__ P,
                                                       Geom g, R dtau) {
  f.nd = ND;
  constexpr int NG = Ngen<NC>::value;
  const long long s = (long long)blockIdx.x * 256 + threadIdx.x;
  if (s >= g.V) return;
#pragma unroll 1
  for (int mu = 0; mu < ND; ++mu) {
    R v[NG];
#pragma unroll
    for (int a = 0; a < NG; ++a) v[a] = dtau * P[((long long)mu * NG + a) * g.V + s];
    const Mat<R, NC> e = exp_iq(v, (Mat<R, NC> *)nullptr);
    Mat<R, NC> u = mul(e, f.load(s, mu));
    if constexpr (sizeof(R) == 4) reunitarize(u);
    f.store(s, mu, u);
  }
}

template <typename R, int NG>
__global__ __launch_bounds__(256) void k_kinetic_soa(const R *__restrict__ P, long long V, int nd,
                                                      double *partials, unsigned int *ticket,
                                                      double *out) {
  __shared__ double lds[8];
  const long long s = (long long)blockIdx.x * 256 + threadIdx.x;
  double k = 0.0;
  if (s < V) {
    for (int mu = 0; mu < nd; ++mu) {
      double n2 = 0.0;
#pragma unroll
      for (int a = 0; a < NG; ++a) {
        const double v = (double)P[((long long)mu * NG + a) * V + s];
        n2 += v * v;
      }
      k += 0.5 * n2;
    }
  }
  const double bt = block_sum<256>(k, lds);
  grid_finish<256>(bt, partials, ticket, out, lds);
}

template <typename R, int NG, int ND>
__global__ __launch_bounds__(256) void k_mom_io(R *P, Geom g, double *host_img, int upload) {
  const long long s = (long long)blockIdx.x * 256 + threadIdx.x;  // lexicographic
  if (s >= g.V) return;
  int x[ND];
  lex_coords<ND>(g, s, x);
  const long long d = dev_index<ND>(g, x);
  for (int mu = 0; mu < ND; ++mu)
#pragma unroll
    for (int a = 0; a < NG; ++a) {
      R *q = P + ((long long)mu * NG + a) * g.V + d;
      double *h = host_img + ((size_t)s * ND + mu) * NG + a;
      if (upload)
        *q = (R)*h;
      else
        *h = (double)*q;
    }
}

namespace {

int ngen(int nc) { return nc == 1 ? 1 : (nc == 2 ? 3 : 8); }

int check_hmc(klft_hmc_t h) {
  if (!h || !h->P) return ki::set_error(KLFT_E_ARG, "null or destroyed HMC handle");
  return ki::check_field(h->f);
}

int enqueue_refresh(klft_hmc_t h, uint64_t traj, int slot) {
  klft_field_t f = h->f;
  return ki::dispatch(f->storage, f->nc, f->nd, [&](auto rt, auto nct, auto ct, auto ndt) -> int {
    KLFT_UNPACK(rt, nct, ct, ndt);
    (void)COMP;
    const unsigned nb = ki::blocks_for(f->g.V, 256);
    if ((long long)nb > f->max_partials) return ki::set_error(KLFT_E_ARG, "lattice too large for reduction");
    hipLaunchKernelGGL((k_refresh<R, NC, ND>), dim3(nb), dim3(256), 0, ki::stream(), (R *)h->P, f->g,
                       h->p.seed, (uint32_t)traj, f->partials);
    KLFT_HIP(hipGetLastError());
    return ki::enqueue_sum_blocks(f->partials, nb, f->result + slot);
  });
}

// Directions per thread of k_step_dirs (1: a thread per link, k_md_step and
// k_force).
// Four dimensions: FP64 SU(3) takes two (746 against 787 us with one and 1300
// with four at 32^4; 25.0, 33.6 and 58.6 at 12^4).  SU(3) with one block of
// 17 to 64 sites per sublattice takes one, as a step lasts as long as one thread
// there (FP64 4^3 x 8 14.0 against 15.5 us with two, 4^2 x 8^2 14.4 against 15.9, two
// rows 11.8 against 13.9 and 11.9 against 14.0; above, 8^4 FP64 17.4 against 16.6;
// below, where a thread per link runs short waves, 4^4 15.2 against 15.4 and 2^4
// 23.1 against 14.7).  The others take all four once
// the waves of two would wait for one another: U(1) and SU(2) from a wave per
// SIMD on (SU(2) FP64 16^4 17.3 against 18.4 us, 12^4 14.1 against 13.8, 8^4 10.6
// against 9.0; U(1) 32^4 54 against 65), FP32 SU(3), with two waves per SIMD at
// most, where the fields no longer fit the memory-side cache (32^4 345 against
// 372, 28x24x20x32 145 both, 20^4 60 against 53, 12^4 23.6 against 19.5).
// Fewer dimensions: all of them, but for SU(3) with less than a wave per CU, where
// a step lasts as long as one thread (16^3 FP64 19.1 against 14.3 us with one
// direction, 64^2 8.7 against 6.9; 32^3 23.1 against 28.7).
int directions_per_thread(const klft_field_s *f, bool streams) {
  if (f->nd < 4) return f->nc == 3 && f->g.V < 64 * 256 ? 1 : f->nd;
  if (f->nc == 3 && f->g.Vh > 16 && f->g.Vh <= 64) return 1;
  if (f->nc == 3) return f->storage == KLFT_STORAGE_F64 || !streams ? 2 : 4;
  return f->g.V < 64 * 1024 ? 2 : 4;
}

// Links read, links written (`links` buffers in all) and momenta beyond 300 MiB
// (the memory-side cache holds 256 MB): what a launch touches once goes past
// the caches (SU(3) 32^4 FP64 776 -> 746 us per step, FP32 363 -> 345, SU(2) FP32,
// 304 MiB, 137 -> 129); below that the next launch finds it there (SU(3)
// 28x24x20x32 FP32, 289 MiB, 145 both, 16^4 FP64 46 against 50, U(1) 32^4 54
// against 70).  KLFT_VARIANT="md_stream=0|1" forces one.
bool past_caches(const klft_field_s *f, int links) {
  const int forced = ki::forced_variant("md_stream");
  if (forced >= 0) return forced != 0;
  const size_t rbytes = f->storage == KLFT_STORAGE_F64 ? 8 : 4;
  return links * f->link_bytes + (size_t)f->g.V * f->nd * ngen(f->nc) * rbytes > (size_t)300 << 20;
}

// variants: 0 one thread per link, one-term-at-a-time staple; 4 the same with
// all staple loads in flight at once (full staple); 5 a thread for all
// directions of a site; 6 for two (four dimensions)
constexpr int kForceVariants = 7;

int launch_force(klft_hmc_t h, double dtau, double *Fout, int kin_slot, int variant) {
  klft_field_t f = h->f;
  if (variant != 0 && variant < 4) return ki::set_error(KLFT_E_ARG, "force variant %d is not built", variant);
  // with a kinetic slot, every block writes a partial; k_sum_blocks adds them
  double *parts = kin_slot >= 0 ? f->partials : nullptr;
  return ki::dispatch(f->storage, f->nc, f->nd, [&](auto rt, auto nct, auto ct, auto ndt) -> int {
    KLFT_UNPACK(rt, nct, ct, ndt);
    const auto links = ki::links_of<R, NC, COMP>(f);
    const R coef = (R)(h->p.beta / (double)NC);
    const long long nb = link_blocks<ND>(f->g);
    if (nb > f->max_partials) return ki::set_error(KLFT_E_ARG, "lattice too large for reduction");
    {
      ki::ProfScope prof("force", "derivative+update_momentum");
      auto dirs = [&](auto kt, auto ntt) {
        constexpr int K = decltype(kt)::value;
        hipLaunchKernelGGL((k_step_dirs<R, NC, COMP, ND, K, decltype(ntt)::value != 0, false>), dim3((unsigned)nb),
                           dim3(64 * ND / K), 0, ki::stream(), links, links, (R *)h->P, f->g, coef, (R)dtau, R(0), Fout,
                           parts);
      };
      auto go = [&](auto ntt) {
        if (variant == 5)
          dirs(ki::ic<ND>{}, ntt);
        else if (variant == 6)
          dirs(ki::ic<ND == 4 ? 2 : ND>{}, ntt);
        else if (variant == 4)
          hipLaunchKernelGGL((k_force<R, NC, COMP, ND, false>), dim3((unsigned)nb), dim3(64 * ND), 0, ki::stream(),
                             links, (R *)h->P, f->g, coef, (R)dtau, Fout, parts);
        else
          hipLaunchKernelGGL((k_force<R, NC, COMP, ND, true>), dim3((unsigned)nb), dim3(64 * ND), 0, ki::stream(),
                             links, (R *)h->P, f->g, coef, (R)dtau, Fout, parts);
      };
      if (past_caches(f, 1))
        go(ki::ic<1>{});
      else
        go(ki::ic<0>{});
      KLFT_HIP(hipGetLastError());
    }
    if (parts) return ki::enqueue_sum_blocks(parts, nb, f->result + kin_slot);
    return KLFT_OK;
  });
}

// the tuning launcher uses dtau = 0, which leaves the momenta unchanged
int enqueue_force(klft_hmc_t h, double dtau, double *Fout, int kin_slot) {
  const int k = directions_per_thread(h->f, past_caches(h->f, 1)), dflt = k == 1 ? 4 : (k == 2 && h->f->nd == 4 ? 6 : 5);
  const int v = ki::pick_variant("force", h->f, kForceVariants, dflt,
                                 [&](int var) { return launch_force(h, 0.0, nullptr, -1, var); });
  return launch_force(h, dtau, Fout, kin_slot, v);
}

int enqueue_gauge(klft_hmc_t h, double dtau) {
  klft_field_t f = h->f;
  return ki::dispatch(f->storage, f->nc, f->nd, [&](auto rt, auto nct, auto ct, auto ndt) -> int {
    KLFT_UNPACK(rt, nct, ct, ndt);
    ki::ProfScope prof("update_gauge", "update_gauge");
    hipLaunchKernelGGL((k_update_gauge<R, NC, COMP, ND>), dim3(ki::blocks_for(f->g.V, 256)), dim3(256),
                       0, ki::stream(), ki::links_of<R, NC, COMP>(f), (const R *)h->P, f->g, (R)dtau);
    KLFT_HIP(hipGetLastError());
    return KLFT_OK;
  });
}

int enqueue_kinetic(klft_hmc_t h, int slot) {
  klft_field_t f = h->f;
  return ki::dispatch(f->storage, f->nc, f->nd, [&](auto rt, auto nct, auto ct, auto ndt) -> int {
    KLFT_UNPACK(rt, nct, ct, ndt);
    (void)COMP;
    (void)ND;
    if ((long long)ki::blocks_for(f->g.V, 256) > f->max_partials)
      return ki::set_error(KLFT_E_ARG, "lattice too large for reduction");
    hipLaunchKernelGGL((k_kinetic_soa<R, Ngen<NC>::value>), dim3(ki::blocks_for(f->g.V, 256)), dim3(256),
                       0, ki::stream(), (const R *)h->P, f->g.V, f->nd, f->partials, f->ticket,
                       f->result + slot);
    KLFT_HIP(hipGetLastError());
    return KLFT_OK;
  });
}

// variants: 1 a thread per link, 2 a thread for all directions of a site, 3 for
// two directions (four dimensions).  0 (a thread per link with one term of
// the staple at a time) never won and runs as 1.
constexpr int kMdVariants = 4;

int launch_md_step(klft_hmc_t h, void *src, void *dst, double dtp, double dtu, int variant) {
  klft_field_t f = h->f;
  return ki::dispatch(f->storage, f->nc, f->nd, [&](auto rt, auto nct, auto ct, auto ndt) -> int {
    KLFT_UNPACK(rt, nct, ct, ndt);
    auto ls = ki::links_of<R, NC, COMP>(f), ld = ls;
    ls.p = reinterpret_cast<cx<R> *>(src);
    ld.p = reinterpret_cast<cx<R> *>(dst);
    const unsigned nb = (unsigned)link_blocks<ND>(f->g);
    const R coef = (R)(h->p.beta / (double)NC);
    ki::ProfScope prof("md_step", "derivative+update_momentum+update_gauge");
    auto dirs = [&](auto kt, auto ntt) {
      constexpr int K = decltype(kt)::value;
      hipLaunchKernelGGL((k_step_dirs<R, NC, COMP, ND, K, decltype(ntt)::value != 0, true>), dim3(nb),
                         dim3(64 * ND / K), 0, ki::stream(), ls, ld, (R *)h->P, f->g, coef, (R)dtp, (R)dtu, nullptr,
                         nullptr);
    };
    auto go = [&](auto ntt) {
      if (variant == 2)
        dirs(ki::ic<ND>{}, ntt);
      else if (variant == 3)
        dirs(ki::ic<ND == 4 ? 2 : ND>{}, ntt);
      else
        hipLaunchKernelGGL((k_md_step<R, NC, COMP, ND, decltype(ntt)::value != 0>), dim3(nb), dim3(64 * ND), 0,
                           ki::stream(), ls, ld, (R *)h->P, f->g, coef, (R)dtp, (R)dtu);
    };
    if (past_caches(f, 2))
      go(ki::ic<1>{});
    else
      go(ki::ic<0>{});
    KLFT_HIP(hipGetLastError());
    return KLFT_OK;
  });
}

// Leapfrog::integrate (Integrator.hpp:26-53): dtau = tau/n; half momentum
// step, gauge step, n x (momentum, gauge), half momentum step, restoreGauge.
// Each momentum step and the gauge step after it are one fused launch that
// writes the new links to the other buffer: field -> Ubuf[0] -> Ubuf[1] ->
// Ubuf[0] ...  The final buffer is then swapped into the field, and the
// starting links stay in the handle (slot `*start_slot`).
int enqueue_leapfrog(klft_hmc_t h, int kin_slot, int *start_slot) {
  const double dtau = h->p.tau / (double)h->p.nsteps;
  klft_field_t f = h->f;
  const int k = directions_per_thread(f, past_caches(f, 2)), dflt = k == 1 ? 1 : (k == 2 && f->nd == 4 ? 3 : 2);
  const int v = ki::pick_variant("md_step", f, kMdVariants, dflt, [&](int var) {
    return launch_md_step(h, f->links, h->Ubuf[0], 0.0, 0.0, var);  // dtp = 0: P unchanged
  });
  void *cur = f->links;
  int nxt = 0, rc = KLFT_OK;
  for (int i = 0; i <= h->p.nsteps && !rc; ++i) {
    rc = launch_md_step(h, cur, h->Ubuf[nxt], i == 0 ? dtau / 2.0 : dtau, dtau, v);
    cur = h->Ubuf[nxt];
    nxt ^= 1;
  }
  if (rc) return rc;
  // the field takes the final links; the buffer it held takes their slot
  const int fin = nxt ^ 1;
  h->Ubuf[fin] = f->links;
  f->links = cur;
  if (start_slot) *start_slot = fin;
  rc = enqueue_force(h, dtau / 2.0, nullptr, kin_slot);
  if (!rc) rc = ki::enqueue_reunit(h->f);
  return rc;
}

int momenta_io(klft_hmc_t h, double *host, int upload) {
  klft_field_t f = h->f;
  const size_t n = (size_t)f->g.V * f->nd * ngen(f->nc) * sizeof(double);
  if (!h->stage) KLFT_HIP(hipMalloc(&h->stage, n));  // kept with the handle
  double *stage = h->stage;
  hipError_t e = hipSuccess;
  if (upload) e = hipMemcpyAsync(stage, host, n, hipMemcpyHostToDevice, ki::stream());
  int rc = KLFT_OK;
  if (e == hipSuccess)
    rc = ki::dispatch(f->storage, f->nc, f->nd, [&](auto rt, auto nct, auto ct, auto ndt) -> int {
      KLFT_UNPACK(rt, nct, ct, ndt);
      (void)COMP;
      hipLaunchKernelGGL((k_mom_io<R, Ngen<NC>::value, ND>), dim3(ki::blocks_for(f->g.V, 256)), dim3(256), 0,
                         ki::stream(), (R *)h->P, f->g, stage, upload);
      KLFT_HIP(hipGetLastError());
      return KLFT_OK;
    });
  if (e == hipSuccess && !rc && !upload) e = hipMemcpyAsync(host, stage, n, hipMemcpyDeviceToHost, ki::stream());
  if (e == hipSuccess) e = hipStreamSynchronize(ki::stream());
  if (e != hipSuccess) return ki::hip_fail(e, "momenta transfer");
  return rc;
}

}  // namespace

extern "C" int klft_hmc_create(klft_field_t f, const klft_hmc_params *p, klft_hmc_t *out) {
  if (!out || !p) return ki::set_error(KLFT_E_ARG, "null argument");
  *out = nullptr;
  int rc = ki::check_field(f);
  if (rc) return rc;
  if (p->nsteps < 1) return ki::set_error(KLFT_E_ARG, "n_steps must be >= 1");
  if (!(p->tau > 0.0)) return ki::set_error(KLFT_E_ARG, "tau must be > 0");
  klft_hmc_s *h = new klft_hmc_s();
  h->f = f;
  h->p = *p;
  const size_t rbytes = f->storage == KLFT_STORAGE_F64 ? 8 : 4;
  const size_t pbytes = (size_t)f->g.V * f->nd * ngen(f->nc) * rbytes;
  hipError_t e = hipMalloc(&h->P, pbytes);
  for (int i = 0; i < 2 && e == hipSuccess; ++i) e = hipMalloc(&h->Ubuf[i], f->link_bytes);
  // cleared on the (non-blocking) library stream, where the kernels that
  // read P run, and waited for
  if (e == hipSuccess) e = hipMemsetAsync(h->P, 0, pbytes, ki::stream());
  if (e == hipSuccess) e = hipStreamSynchronize(ki::stream());
  if (e != hipSuccess) {
    if (h->P) (void)hipFree(h->P);
    for (void *b : h->Ubuf)
      if (b) (void)hipFree(b);
    delete h;
    return ki::set_error(KLFT_E_NOMEM, "HMC workspace allocation failed");
  }
  *out = h;
  return KLFT_OK;
}

extern "C" int klft_hmc_destroy(klft_hmc_t h) {
  if (!h) return KLFT_OK;
  (void)ki::sync_stream();
  if (h->P) (void)hipFree(h->P);
  for (void *b : h->Ubuf)
    if (b) (void)hipFree(b);
  if (h->Fdbg) (void)hipFree(h->Fdbg);
  if (h->stage) (void)hipFree(h->stage);
  h->P = nullptr;
  delete h;
  return KLFT_OK;
}

extern "C" int klft_hmc_refresh_momenta(klft_hmc_t h, uint64_t traj) {
  int rc = check_hmc(h);
  if (!rc) rc = enqueue_refresh(h, traj, 1);
  if (rc) return rc;
  return ki::sync_stream();
}

extern "C" int klft_hmc_momenta_upload(klft_hmc_t h, const double *host) {
  int rc = check_hmc(h);
  if (rc) return rc;
  if (!host) return ki::set_error(KLFT_E_ARG, "null host buffer");
  return momenta_io(h, const_cast<double *>(host), 1);
}

extern "C" int klft_hmc_momenta_download(klft_hmc_t h, double *host) {
  int rc = check_hmc(h);
  if (rc) return rc;
  if (!host) return ki::set_error(KLFT_E_ARG, "null host buffer");
  return momenta_io(h, host, 0);
}

extern "C" int klft_hmc_force(klft_hmc_t h, double *host_force) {
  int rc = check_hmc(h);
  if (rc) return rc;
  if (!host_force) return ki::set_error(KLFT_E_ARG, "null host buffer");
  klft_field_t f = h->f;
  const size_t n = (size_t)f->g.V * f->nd * ngen(f->nc);
  if (!h->Fdbg) KLFT_HIP(hipMalloc(&h->Fdbg, n * sizeof(double)));
  rc = enqueue_force(h, 0.0, h->Fdbg, -1);
  if (rc) return rc;
  KLFT_HIP(hipMemcpyAsync(host_force, h->Fdbg, n * sizeof(double), hipMemcpyDeviceToHost, ki::stream()));
  return ki::sync_stream();
}

extern "C" int klft_hmc_update_momentum(klft_hmc_t h, double dtau) {
  int rc = check_hmc(h);
  if (!rc) rc = enqueue_force(h, dtau, nullptr, -1);
  if (rc) return rc;
  return ki::sync_stream();
}

extern "C" int klft_hmc_update_gauge(klft_hmc_t h, double dtau) {
  int rc = check_hmc(h);
  if (!rc) rc = enqueue_gauge(h, dtau);
  if (rc) return rc;
  return ki::sync_stream();
}

extern "C" int klft_hmc_kinetic(klft_hmc_t h, double *out) {
  int rc = check_hmc(h);
  if (rc) return rc;
  if (!out) return ki::set_error(KLFT_E_ARG, "null output");
  rc = enqueue_kinetic(h, 1);
  if (rc) return rc;
  return ki::read_results(h->f, 1, 1, out);
}

extern "C" int klft_gauge_action(klft_field_t f, double beta, double *out) {
  int rc = ki::check_field(f);
  if (rc) return rc;
  if (!out) return ki::set_error(KLFT_E_ARG, "null output");
  rc = ki::plaquette_raw(f, 2, nullptr);
  double raw = 0.0;
  if (!rc) rc = ki::read_results(f, 2, 1, &raw);
  if (rc) return rc;
  *out = -(beta / (double)f->nc) * raw;  // GaugeMonomial.hpp:19-25
  return KLFT_OK;
}

extern "C" int klft_hmc_integrate(klft_hmc_t h) {
  int rc = check_hmc(h);
  if (!rc) rc = enqueue_leapfrog(h, -1, nullptr);
  if (rc) return rc;
  return ki::sync_stream();
}

// HMC::hmc_step (HMC.hpp:48-71) with the monomials in the order of
// lib/HMC_SU2.cpp:46-47 (kinetic, then gauge).
extern "C" int klft_hmc_trajectory(klft_hmc_t h, uint64_t traj, double *dH, int *accepted) {
  int rc = check_hmc(h);
  if (rc) return rc;
  klft_field_t f = h->f;
  rc = enqueue_refresh(h, traj, 4);  // K_old
  if (rc) return rc;
  rc = ki::plaquette_raw(f, 5, nullptr);  // G_old (raw)
  int start = -1;                         // handle slot of the starting links
  if (!rc) rc = enqueue_leapfrog(h, 6, &start);  // K_new fused into the last half step
  if (!rc) rc = ki::plaquette_raw(f, 7, nullptr);
  double r[4];
  if (!rc) rc = ki::read_results(f, 4, 4, r);
  if (rc) return rc;
  const double c = -(h->p.beta / (double)f->nc);
  const double K0 = r[0], G0 = c * r[1], K1 = r[2], G1 = c * r[3];
  double d = 0.0;
  d += K1 - K0;
  d += G1 - G0;
  int acc = 1;
  if (d > 0.0) {
    klft_rng::Stream st(h->p.seed, klft_rng::TAG_ACCEPT, 0, (uint32_t)traj, 0, 0, 0);
    if (st.u01() > std::exp(-d)) acc = 0;
  }
  if (!acc) std::swap(f->links, h->Ubuf[start]);  // the starting links, untouched
  if (dH) *dH = d;
  if (accepted) *accepted = acc;
  return KLFT_OK;
}
