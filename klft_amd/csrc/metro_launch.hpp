// The launcher of the Metropolis sweep kernels (metro_kernels.hpp,
// metro_hits.hpp), instantiated per link storage in metropolis_f64.hip,
// metropolis_f32.hip and metropolis_f32rows.hip (the three translation units
// compile in parallel).
#pragma once
#include "metro_hits.hpp"
#include "metro_kernels.hpp"

namespace klft_metro {

// Sweep variants (numbers kept stable for tuning caches): 0 one lane per
// site; 4 one lane, low-register staple, >= 2 waves per SIMD; 7 one lane,
// next direction's staple loaded during the hits; 11 one lane, the site's own
// links kept in registers; 12 site waves fed by staple waves; 13 the same with
// each direction's upper and lower staple terms back to back; 14, 15: 12, 13
// with the symmetric SU(3) proposal; 16, 17: the hits of a link in parallel,
// staple terms in the order of 12, 13; 18, 19: those with the symmetric
// proposal.  1-3, 5, 6, 8-10 (four or two lanes per
// site, proposals drawn in pairs, LDS-staged staple terms) never won at
// 16^4 - 48^4 and were removed.
template <typename RR, bool CC>
int launch_passes_typed(klft_field_t f, void *links, int variant, int p0, int p1,
                        const klft_metropolis_params *p, uint64_t sweep, int nsweeps, uint32_t chain,
                        Counters counter, int *visit) {
  return dispatch_typed<RR, CC>(f->nc, f->nd, [&](auto rt, auto nct, auto ct, auto ndt) -> int {
    KLFT_UNPACK(rt, nct, ct, ndt);
    Links<R, NC, COMP> l;
    l.p = reinterpret_cast<cx<R> *>(links);
    l.V = f->g.V;
    l.nd = f->nd;
    const R beta_nc = (R)(p->beta / (double)NC);
    const unsigned nb = blocks_for(f->g.Vh, kMetroBlock);
    switch (variant) {
      case 0: case 4: case 7: case 11: case 12: case 13: case 14: case 15:
      case 16: case 17: case 18: case 19: break;
      default: return set_error(KLFT_E_ARG, "sweep variant %d is not built", variant);
    }
    // acceptance counter of sweep i of the run (relative to `sweep`)
    auto cnt = [&](int i) { return counter.base + (long long)i * counter.per_sweep; };
    const unsigned nws = blocks_for(f->g.Vh, kWsSites);
    // launch the site-wave kernel on one pass (pb < 0), or on two
    // independent ones, each with its own sweep and counter
    auto ws = [&](auto kern, int pa, int sa, int pb, int sb) {
      hipLaunchKernelGGL(kern, dim3(pb >= 0 ? 2 * nws : nws), dim3(kWsBlock), 0, stream(), l, f->g, pa, pb,
                         p->nhits, beta_nc, (R)p->delta, p->seed, (uint32_t)(sweep + sa), (uint32_t)(sweep + sb),
                         chain, cnt(sa), cnt(sb), counter.row, visit);
    };
    // the hit-parallel kernel (metro_hits.hpp) likewise
    const int G = hit_lanes(NC, p->nhits);
    const unsigned nhb = blocks_for(f->g.Vh, 64 / G);
    auto hits_w = [&](auto wt, auto ilv, auto sym, int pa, int sa, int pb, int sb) {
      constexpr int W = decltype(wt)::value;
      constexpr bool ILV = decltype(ilv)::value != 0, SYM = decltype(sym)::value != 0;
      const size_t lds = hit_lds_bytes<R, NC, ND, W>(G);
      hipLaunchKernelGGL((k_metropolis_hits<R, NC, COMP, ND, W, ILV, SYM>),
                         dim3(pb >= 0 ? 2 * nhb : nhb), dim3(64 * W), lds, stream(), l, f->g, pa, pb, G, p->nhits, beta_nc, (R)p->delta, p->seed, (uint32_t)(sweep + sa),
                         (uint32_t)(sweep + sb), chain, cnt(sa), cnt(sb), counter.row, visit);
    };
    // One wave per direction while the blocks of a pass are few: it has the
    // shortest chain (SU(3) 8^4 115 us per sweep against 143 with two waves);
    // beyond that two waves in turn, which keep more sites resident (16^4 226
    // against 237, U(1) 16^4 219 against 293).
    const int fw = forced_variant("hits_waves");
    const bool wide = fw > 0 ? fw != 2 : f->g.Vh <= (NC == 3 ? 10LL : 8LL) * cu_count();
    auto hits = [&](auto ilv, auto sym, int pa, int sa, int pb, int sb) {
      if (wide)
        hits_w(ic<ND>{}, ilv, sym, pa, sa, pb, sb);
      else
        hits_w(ic<2>{}, ilv, sym, pa, sa, pb, sb);
    };
    auto launch_ws = [&](int pa, int sa, int pb, int sb) -> int {
      switch (variant) {
        case 16: hits(ic<0>{}, ic<0>{}, pa, sa, pb, sb); break;
        case 17: hits(ic<1>{}, ic<0>{}, pa, sa, pb, sb); break;
        case 12: ws(k_metropolis_ws<R, NC, COMP, ND, false>, pa, sa, pb, sb); break;
        case 13: ws(k_metropolis_ws<R, NC, COMP, ND, true>, pa, sa, pb, sb); break;
        default:
          // the symmetric SU(3) proposal: site waves, terms as in 12 / 13
          if constexpr (NC == 3) {
            switch (variant) {
              case 14: ws(k_metropolis_ws<R, NC, COMP, ND, false, true>, pa, sa, pb, sb); break;
              case 15: ws(k_metropolis_ws<R, NC, COMP, ND, true, true>, pa, sa, pb, sb); break;
              case 18: hits(ic<0>{}, ic<1>{}, pa, sa, pb, sb); break;
              default: hits(ic<1>{}, ic<1>{}, pa, sa, pb, sb); break;
            }
          } else {
            return set_error(KLFT_E_ARG, "the symmetric proposal variants are SU(3) only");
          }
      }
      return KLFT_OK;
    };
    // whole sweeps run their independent passes in pairs when both passes'
    // blocks fit on the GPU at once (KLFT_VARIANT=metropolis_pairs=0: never);
    // a run of several sweeps also pairs passes of consecutive sweeps
    // (run_schedule)
    bool pair = false;
    if (variant >= 12 && p0 == 0 && p1 == (1 << ND) && forced_variant("metropolis_pairs") != 0) {
      const void *kern = nullptr;
      switch (variant) {
        case 12: kern = reinterpret_cast<const void *>(&k_metropolis_ws<R, NC, COMP, ND, false>); break;
        case 13: kern = reinterpret_cast<const void *>(&k_metropolis_ws<R, NC, COMP, ND, true>); break;
        case 14: kern = reinterpret_cast<const void *>(&k_metropolis_ws<R, NC, COMP, ND, false, true>); break;
        case 15: kern = reinterpret_cast<const void *>(&k_metropolis_ws<R, NC, COMP, ND, true, true>); break;
        default: break;
      }
      // the hit-parallel kernel's blocks are small enough to queue: always
      pair = !kern || 2LL * nws <= (long long)cu_count() * blocks_per_cu(kern, kWsBlock);
    }
    if (pair) {
      int rc = KLFT_OK;
      for_each_run_launch(ND, nsweeps, [&](const RunLaunch &L) {
        if (rc) return;
        const int pa = L.pass[0], pb = L.pass[1];
        char label[56];
        if (pb >= 0)
          snprintf(label, sizeof label, "sweep_Metropolis_GaugeField_sublat_%d_%d", pa, pb);
        else
          snprintf(label, sizeof label, "sweep_Metropolis_GaugeField_sublat_%d", pa);  // Metropolis.hpp:161
        ProfScope prof(pb >= 0 ? "metropolis_pass_pair" : "metropolis_pass", label);
        rc = launch_ws(pa, L.sweep[0], pb, pb >= 0 ? L.sweep[1] : L.sweep[0]);
      });
      if (rc) return rc;
    } else {
      for (int i = 0; i < nsweeps; ++i) {
        for (int pass = p0; pass < p1; ++pass) {
          char label[48];
          snprintf(label, sizeof label, "sweep_Metropolis_GaugeField_sublat_%d", pass);  // Metropolis.hpp:161
          ProfScope prof("metropolis_pass", label);
          if (variant >= 12) {
            const int rc = launch_ws(pass, i, -1, i);
            if (rc) return rc;
          } else {
            auto one_lane = [&](auto kern) {
              hipLaunchKernelGGL(kern, dim3(nb), dim3(kMetroBlock), 0, stream(), l, f->g, pass, p->nhits, beta_nc,
                                 (R)p->delta, p->seed, (uint32_t)(sweep + i), chain, cnt(i), visit);
            };
            switch (variant) {
              case 4: one_lane(k_metropolis_pass<R, NC, COMP, ND, true, 2>); break;
              case 7: one_lane(k_metropolis_pipe<R, NC, COMP, ND>); break;
              case 11: one_lane(k_metropolis_own<R, NC, COMP, ND>); break;
              default: one_lane(k_metropolis_pass<R, NC, COMP, ND, false, 1>); break;
            }
          }
        }
      }
    }
    KLFT_HIP(hipGetLastError());
    return KLFT_OK;
  });
}

}  // namespace klft_metro
