// One sublattice pass with a link's hits in parallel, for passes whose sites
// do not fill the GPU.
//
// There the time of a pass is one block's chain of dependent work, so it is
// taken apart.  What does not depend on the site's own links is done up
// front, spread over the lanes: the first product of every staple term
// (U_nu(x+mu) U_mu(x+nu)^+ and U_nu(x+mu-nu)^+ U_mu(x-nu)^+), and the proposals,
// each drawn from its hit's own stream.  A block of W waves holds 64 / G sites
// with G lanes per site in each wave.  The waves take the directions in turn:
// the wave of direction mu draws its proposals, one hit a lane, and sums its
// staple, one entry a lane, all but the term through U_{mu-1}(x), while the wave
// of direction mu - 1 judges its hits; then it adds that term, forms M = S U and
// judges its own.
//
// SU(3): all G hits are judged at once against the same M.  The first accepted
// one is final (and so are the rejected ones before it); M becomes M r and the
// hits after it are judged again, so a link costs 1 + (accepted hits) rounds (of
// the reference's SU(3) proposals 3 % are accepted at beta = 6; hits_in_parallel
// keeps this kernel from sizes where many rounds lose).  U(1) and SU(2):
// most hits are accepted, so the lanes step through the hits, the proposals
// handed over through LDS, the even lanes multiplying M and the odd ones U.
//
// Every decision is the one the serial chain takes, from the same stream
// words, products and term order (ILV: that of ws_pass), so links and counts
// are those of the site-wave kernel bit for bit (FP64 U(1) to the last bit or
// two of a link).
//
// What bounds it: the chain (8^4 SU(3) FP64: 13 us per launch, of which about
// 8 are launch, loads, products and staples and 4 the proposals, against 75
// for the site waves); above 16^4 the register file (FP64 SU(3): 154
// registers, three waves per SIMD) and its instructions.
#pragma once
#include "metro_kernels.hpp"

namespace klft_metro {

// LDS slots of one site, NM = NC^2 entries each
template <int ND>
struct HitSlots {
  static constexpr int NU = (ND - 1) + (ND - 1) * (ND - 2);  // upper first products (the deferred ones are adjoints)
  static constexpr int NL = ND * (ND - 1);                   // lower first products
  static constexpr int C = NU + NL;                          // U_d(x - d)
  static constexpr int U = C + ND;                           // U_d(x)
  static constexpr int N = U + ND;
  // slot of the first product of direction mu's j-th upper / lower term
  __host__ __device__ static constexpr int upper(int mu, int j) {
    return mu == 0 ? j : (ND - 1) + (mu - 1) * (ND - 2) + (j < mu - 1 ? j : j - 1);
  }
  __host__ __device__ static constexpr int lower(int mu, int j) { return NU + mu * (ND - 1) + j; }
  // slots that nothing reads once direction mu's staple is summed: M's, and an
  // accepted proposal's
  __host__ __device__ static constexpr int m_slot(int mu) { return lower(mu, 0); }
  __host__ __device__ static constexpr int r_slot(int mu) { return ND > 2 ? lower(mu, 1) : C + 1 - mu; }
};
// reals of a proposal's record in LDS, the accept uniform included (U(1),
// SU(2): the first row; SU(3) proposals stay in registers)
template <int NC>
constexpr int hit_record() {
  return NC == 1 ? 3 : (NC == 2 ? 5 : 0);
}
// reals of one site's LDS region: the matrices, an odd number of entries so
// that the sites of a wave start in different banks, and the records of the
// block's W waves (G hits each)
template <int NC, int ND, int W>
__host__ __device__ inline int hit_stride(int G) {
  return 2 * (HitSlots<ND>::N * NC * NC | 1) + ((W * G * hit_record<NC>() + 1) & ~1);
}
// lanes per site for nhits hits: the hits in as few equal rounds of at most 10
// as possible, and at least a lane per staple entry
__host__ __device__ inline int hit_lanes(int nc, int nhits) {
  const int lo = nc == 3 ? 9 : (nc == 2 ? 6 : 4);
  const int rounds = nhits > 10 ? (nhits + 9) / 10 : 1;
  const int g = (nhits + rounds - 1) / rounds;
  return g < lo ? lo : g;
}

// LDS written by one lane and read by another of the same wave: the LDS
// serves a wave's accesses in order, so only the compiler must keep them so
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The pass for positions t0 .. t0 + 64 / G - 1 of the sublattice, by a block
// of W waves; returns the lane's accepted hits.  `lds`: 64 / G regions of
// hit_stride reals.  SYM as in ws_pass.
template <typename R, int NC, bool COMP, int ND, int W, bool ILV, bool SYM>
__device__ __forceinline__ unsigned int hits_pass(const Links<R, NC, COMP> &f, const Geom &g, int pass,
                                                  long long t0, int G, int nhits, R beta_nc, R delta, uint64_t seed,
                                                  uint32_t sweep, uint32_t chain, int *visit, R *lds) {
  using SL = HitSlots<ND>;
  constexpr int NM = NC * NC, RS = hit_record<NC>();
  constexpr int NIT = SL::NU + SL::NL + 2 * ND;  // items of a site: products and link copies
  const int lane = (int)(threadIdx.x & 63), w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int NS = 64 / G;
  const int gi = lane / G, e = lane - gi * G;
  const long long t = t0 + gi;
  const bool active = gi < NS && t < g.Vh;
  R *region = lds + (gi < NS ? gi : 0) * hit_stride<NC, ND, W>(G);
  cx<R> *base = reinterpret_cast<cx<R> *>(region);
  auto at = [&](int slot, int i, int j) -> cx<R> & { return base[slot * NM + i * NC + j]; };
  auto put = [&](int slot, const Mat<R, NC> &m) {
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j) at(slot, i, j) = m.m[i][j];
  };
  auto get = [&](int slot) {
    Mat<R, NC> m;
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j) m.m[i][j] = at(slot, i, j);
    return m;
  };
  R *rec = region + 2 * (SL::N * NM | 1) + w * G * RS;  // the wave's proposal records
  uint32_t site = 0, s = 0;
  // neighbour offsets in 32 bits (fields hold < 2^32 sites), picked by value: a
  // select over an indexed array would put it in scratch
  uint32_t p0 = 0, p1 = 0, p2 = 0, p3 = 0, m0 = 0, m1 = 0, m2 = 0, m3 = 0;
  int x[ND];
#pragma unroll
  for (int k = 0; k < ND; ++k) x[k] = 0;
  if (active) {
    sub_coords<ND>(g, pass, t, x);
    site = (uint32_t)lex_index<ND>(g, x);
    if (visit && e == 0 && w == 0) visit[site] = pass;
    const Nbr<ND> nb = make_nbr<ND>(g, x, (long long)pass * g.Vh + t);
    s = (uint32_t)nb.s;
    p0 = (uint32_t)nb.dp[0];
    m0 = (uint32_t)nb.dm[0];
    p1 = (uint32_t)nb.dp[1];
    m1 = (uint32_t)nb.dm[1];
    if constexpr (ND > 2) {
      p2 = (uint32_t)nb.dp[2];
      m2 = (uint32_t)nb.dm[2];
    }
    if constexpr (ND > 3) {
      p3 = (uint32_t)nb.dp[3];
      m3 = (uint32_t)nb.dm[3];
    }
  }
  auto pick = [](int k, uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3) {
    return k < 0 ? 0u : (k == 0 ? v0 : (k == 1 ? v1 : (k == 2 ? v2 : v3)));
  };
  // the link in direction dir at x + e_dp - e_dm (-1: none)
  auto link = [&](int dp, int dm, int dir) -> Mat<R, NC> {
    return f.load((long long)(s + pick(dp, p0, p1, p2, p3) + pick(dm, m0, m1, m2, m3)), dir);
  };
  // items: the upper products, one link copy, the lower products, the other
  // copies (with ten lanes a wave's round holds one kind of product)
  if (active) {
#pragma unroll 1
    for (int it = w * G + e; it < NIT; it += W * G) {
      if (it < SL::NU) {
        int mu = 0, j = it;
        if constexpr (ND > 2) {
          if (it >= ND - 1) {
            const int q = it - (ND - 1);
            mu = 1 + q / (ND - 2);
            const int k = q % (ND - 2);
            j = k < mu - 1 ? k : k + 1;
          }
        }
        const int nu = j < mu ? j : j + 1;
        const Mat<R, NC> ia = link(mu, -1, nu), ib = link(nu, -1, mu);
        put(it, mul_ad(ia, ib));
      } else if (it > SL::NU && it <= SL::NU + SL::NL) {
        const int l = it - SL::NU - 1;
        const int mu = l / (ND - 1), j = l % (ND - 1);
        const int nu = j < mu ? j : j + 1;
        const Mat<R, NC> ia = link(mu, nu, nu), ib = link(-1, nu, mu);
        put(SL::NU + l, mul_dd(ia, ib));
      } else {
        const int k = it == SL::NU ? 0 : it - SL::NU - SL::NL;  // 0 .. 2 ND - 1
        const bool own = k < ND;
        const int dir = own ? k : k - ND;
        put((own ? SL::U : SL::C) + dir, link(-1, own ? -1 : dir, dir));
      }
    }
  }
  // barriers met by this wave: the first when the products are in place, the
  // next ones when U_0(x), U_1(x), ... are final
  int met = 0;
  auto meet = [&](int upto) {
    for (; met < upto; ++met) __syncthreads();
  };
  const int ei = e / NC, ej = e - ei * NC;  // the lane's staple entry (e < NM)
  const bool entry = active && e < NM;
  unsigned int n = 0;
#pragma unroll 1
  for (int mu = w; mu < ND; mu += W) {
    const int mslot = SL::m_slot(mu);
    // NC <= 2: the even lanes of a site carry M, the odd ones U
    const bool odd = (e & 1) != 0;
    Mat<R, NC> X = zero<R, NC>();
    R trM = R(0);
    bool changed = false;  // uniform over the site's lanes
    int h0 = 0;
    do {
      Mat<R, NC> r;  // the lane's proposal
      R u = R(0);
      if (active && h0 + e < nhits) {
        propose_law<R, NC, SYM>(seed, site, sweep, (uint32_t)(h0 + e), chain, (uint32_t)mu, delta, r, u);
        if constexpr (NC <= 2) {
          R *o = rec + e * RS;
#pragma unroll
          for (int j = 0; j < NC; ++j) {
            o[2 * j] = r.m[0][j].re;
            o[2 * j + 1] = r.m[0][j].im;
          }
          o[2 * NC] = u;
        }
      }
      if (h0 == 0) {
        // the staple, one entry a lane: all but the term through U_{mu-1}(x)
        // once U_{mu-2}(x) is final, while the wave of direction mu - 1 judges
        // its hits
        auto up = [&](int j, cx<R> v) -> cx<R> {
          const int nu = j < mu ? j : j + 1, sl = SL::upper(mu, j);
#pragma unroll
          for (int k = 0; k < NC; ++k) v = cfma_c(at(sl, ei, k), at(SL::U + nu, ej, k), v);
          __builtin_amdgcn_sched_barrier(0);
          return v;
        };
        auto lo = [&](int j, cx<R> v) -> cx<R> {
          const int nu = j < mu ? j : j + 1, sl = SL::lower(mu, j);
#pragma unroll
          for (int k = 0; k < NC; ++k) v = cfma(at(sl, ei, k), at(SL::C + nu, k, ej), v);
          __builtin_amdgcn_sched_barrier(0);
          return v;
        };
        meet(mu > 0 ? mu : 1);
        cx<R> v = mk<R>(0, 0);
        if (entry) {
          if (mu == 0) {
            cx<R> v2 = v;
            v = up(0, v);
#pragma unroll
            for (int j = 1; j < ND - 1; ++j) v = lo(j, v);
            if constexpr (ILV) v2 = lo(0, v2);
#pragma unroll
            for (int j = 1; j < ND - 1; ++j) v2 = up(j, v2);
            if constexpr (!ILV) v2 = lo(0, v2);
            v = v + v2;
          } else if constexpr (ILV) {
#pragma unroll
            for (int j = 0; j < ND - 1; ++j) {
              if (j != mu - 1) v = up(j, v);
              v = lo(j, v);
            }
          } else {
#pragma unroll
            for (int j = 0; j < ND - 1; ++j)
              if (j != mu - 1) v = up(j, v);
#pragma unroll
            for (int j = 0; j < ND - 1; ++j) v = lo(j, v);
          }
        }
        meet(mu + 1);
        if (entry && mu > 0) {
          // its first product is the adjoint of direction mu - 1's with mu
          const int sl = SL::upper(mu - 1, mu - 1);
#pragma unroll
          for (int k = 0; k < NC; ++k) v = cfma_c(conj(at(sl, k, ei)), at(SL::U + mu - 1, ej, k), v);
        }
        wave_lds_fence();
        if (entry) at(mslot, ei, ej) = v;
        wave_lds_fence();
        cx<R> me = mk<R>(0, 0);
        if (entry) {
          me = cmul1(at(mslot, ei, 0), at(SL::U + mu, 0, ej));
#pragma unroll
          for (int k = 1; k < NC; ++k) me = cfma(at(mslot, ei, k), at(SL::U + mu, k, ej), me);
        }
        wave_lds_fence();
        if (entry) at(mslot, ei, ej) = me;
        wave_lds_fence();
        if constexpr (NC <= 2) {
          X = get(odd ? SL::U + mu : mslot);
          trM = retrace(X);
        }
      }
      if constexpr (NC <= 2) {
        wave_lds_fence();
        const int hn = nhits - h0 < G ? nhits - h0 : G;
        R nxt[RS];
#pragma unroll
        for (int k = 0; k < RS; ++k) nxt[k] = rec[k];
#pragma unroll 1
        for (int h = 0; h < hn; ++h) {
          Mat<R, NC> p;
          p.m[0][0] = mk(nxt[0], nxt[1]);
          if constexpr (NC == 2) {
            p.m[0][1] = mk(nxt[2], nxt[3]);
            complete_row1(p);
          }
          const R ua = nxt[2 * NC];
          const int hq = h + 1 < hn ? h + 1 : h;
#pragma unroll
          for (int k = 0; k < RS; ++k) nxt[k] = rec[hq * RS + k];
          // the decision is lane 0's; both products with p are one instruction
          // stream, and only U is restored
          const bool acc = active && metro_accept(-beta_nc * (retr_mul(p, X) - trM), ua);
          if ((__ballot(acc) >> (gi * G)) & 1ull) {
            changed = true;
            if (e == 0) ++n;
            X = mul(X, p);
            trM = retrace(X);
            Mat<R, NC> un = X;
            reunitarize(un);
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
              for (int j = 0; j < NC; ++j) {
                X.m[i][j].re = odd ? un.m[i][j].re : X.m[i][j].re;
                X.m[i][j].im = odd ? un.m[i][j].im : X.m[i][j].im;
              }
          }
        }
        wave_lds_fence();
      } else {
        Mat<R, NC> M = get(mslot);
        trM = retrace(M);
        const int gsh = gi * G;
        const unsigned int gmask = (1u << G) - 1u;
        bool live = active && h0 + e < nhits;
#pragma unroll 1
        for (;;) {
          const bool acc = live && metro_accept(-beta_nc * (retr_mul(r, M) - trM), u);
          const unsigned long long any = __ballot(acc);
          if (!any) break;
          const unsigned int mine = active ? (unsigned int)(any >> gsh) & gmask : 0u;
          const int fst = __builtin_ctz(mine | 0x80000000u);
          // M <- M r and U <- U r, one entry a lane
          cx<R> *rs = &at(SL::r_slot(mu), 0, 0);
          if (mine) {
            changed = true;
            if (e <= fst) live = false;
            if (e == fst) {
              ++n;
#pragma unroll
              for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int j = 0; j < NC; ++j) rs[i * NC + j] = r.m[i][j];
            }
          }
          wave_lds_fence();
          cx<R> me = mk<R>(0, 0), ue = me;
          if (mine && entry) {
            me = cmul1(at(mslot, ei, 0), rs[ej]);
            ue = cmul1(at(SL::U + mu, ei, 0), rs[ej]);
#pragma unroll
            for (int k = 1; k < NC; ++k) {
              me = cfma(at(mslot, ei, k), rs[k * NC + ej], me);
              ue = cfma(at(SL::U + mu, ei, k), rs[k * NC + ej], ue);
            }
          }
          wave_lds_fence();
          if (mine && entry) {
            at(mslot, ei, ej) = me;
            at(SL::U + mu, ei, ej) = ue;
          }
          wave_lds_fence();
          if (mine && e == 0) {
            Mat<R, NC> un = get(SL::U + mu);
            reunitarize(un);
            put(SL::U + mu, un);
          }
          wave_lds_fence();
          // every lane, so that M is not held across the lines above
          M = get(mslot);
          trM = retrace(M);
        }
      }
      h0 += G;
    } while (h0 < nhits);
    if constexpr (NC <= 2) {
      if (changed && e == 1) put(SL::U + mu, X);
      wave_lds_fence();
    }
    // only a link with an accepted hit has changed
    if (changed && e < Links<R, NC, COMP>::NCOMP)
      f.p[f.comp_index((long long)pass * g.Vh + t, mu, e)] = at(SL::U + mu, ei, ej);
  }
  meet(ND);
  return n;
}

template <typename R, int NC, int ND, int W>
inline size_t hit_lds_bytes(int G) {
  return (size_t)(64 / G) * hit_stride<NC, ND, W>(G) * sizeof(R);
}

// block total of the accepted hits into *nacc
template <int W>
__device__ __forceinline__ void hits_count(unsigned int n, unsigned int *red, unsigned long long *nacc) {
  n = (unsigned int)wave_sum_u64(n);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long b = 0;
#pragma unroll
    for (int i = 0; i < W; ++i) b += red[i];
    if (b) atomicAdd(nacc, b);
  }
}

// waves per SIMD asked of the register allocator
template <typename R, int NC>
struct HitOcc {
  static constexpr int value = (sizeof(R) == 8 && NC > 1) ? 2 : 4;
};

// pass2 >= 0: two independent passes in one launch, as in k_metropolis_ws
template <typename R, int NC, bool COMP, int ND, int W, bool ILV, bool SYM>
__global__ __launch_bounds__(64 * W, (HitOcc<R, NC>::value)) void k_metropolis_hits(
    Links<R, NC, COMP> f, Geom g, int pass, int pass2, int G, int nhits, R beta_nc, R delta, uint64_t seed,
    uint32_t sweep, uint32_t sweep2, uint32_t chain, unsigned long long *nacc, unsigned long long *nacc2,
    int nacc_row, int *visit) {
  f.nd = ND;
  extern __shared__ __align__(16) unsigned char hits_smem[];
  __shared__ unsigned int red[W];
  unsigned int lb = xcd_block(blockIdx.x, gridDim.x);
  if (pass2 >= 0) {
    if (lb & 1u) {
      pass = pass2;
      sweep = sweep2;
      nacc = nacc2;
    }
    lb >>= 1;
  }
  const unsigned int n = hits_pass<R, NC, COMP, ND, W, ILV, SYM>(
      f, g, pass, (long long)lb * (64 / G), G, nhits, beta_nc, delta, seed, sweep, chain, visit,
      reinterpret_cast<R *>(hits_smem));
  hits_count<W>(n, red, nacc + (size_t)(blockIdx.x % kCounterRows) * nacc_row);
}

}  // namespace klft_metro
