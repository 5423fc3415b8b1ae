// mh_sweep.hip -- launch sequences of the remap (sweeps in the rotated direction order,
// finalize) for single meshes, and of a whole iteration for a batched ensemble group.
// Compiled once per environment count: -DMH_TU_M=1..4.
#include <algorithm>

#include "mh_kernels.h"
#include "mh_host.h"

#ifndef MH_TU_M
#error "MH_TU_M (environment count of this unit) must be defined"
#endif

// Cell part of one sweep direction (computeGradPhiFace ... computeUremap).
// Slots shared out over gridDim.y groups of vper: as many groups as bring the launch to
// `target` wavefronts, at least one.
struct SlotSplit {
  int groups, vper;
};
inline SlotSplit slot_split(long waves, long target, int nv) {
  const long g = std::max(1L, std::min((long)nv, (target + waves / 2) / std::max(1L, waves)));
  const int vper = (int)((nv + g - 1) / g);
  return {(nv + vper - 1) / vper, vper};
}
template <int DIM, int M>
void launch_cell_x(MhHandle* h, int sel, int first) {
  const MhDev& S = h->dev;
  // One thread runs a cell's 3m+1 slots one after the other, some 1 us each where nothing else
  // fills the wait: up to about 4000 wavefronts (4 per SIMD) the slots are shared out (two
  // environments: 7.9 -> 5.0 us on 100x5x5 cells, 7.7 -> 5.8 us on 181x181, 13.1 -> 11.6 us on
  // 362x362); beyond that the repeated geometry costs more (512x512: 16.0 us, split 16.2).
  const SlotSplit p = slot_split((long)row_blocks(h) * (MH_BLOCK / 64), 4000, 3 * M + 1);
  if (p.groups > 1 && !S.pm[0])  // (the presence byte of a cell is written with its last slot)
    MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL, (k_sweep_cell_row_slots<DIM, M, LIM>), dim3(row_blocks(h), p.groups), MH_BLOCK,
                       S, sel, first, p.vper));
  else
    MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL, (k_sweep_cell_row<DIM, M, LIM>), row_blocks(h), MH_BLOCK, S, sel, first));
}
template <int DIM, int D, int M>
void launch_cell_yz(MhHandle* h, int sel, int first) {
  const MhDev& S = h->dev;
  if (seg_sweep(h)) {
    // the slots of a segment as in launch_cell_x, up to about 2000 wavefronts of 2-cell segments
    const SlotSplit p = slot_split((long)seg_blocks(h, D, MH_SEG_L) * (MH_BLOCK / 64), 2048, 3 * M + 1);
    MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL + D, (k_sweep_cell_seg<DIM, D, M, LIM, MH_SEG_L>),
                       dim3(seg_blocks(h, D, MH_SEG_L), p.groups), MH_BLOCK, S, sel, first, p.vper));
  } else if (MH_CM_HAS(DIM, M) && cell_march(h)) {
    if constexpr (MH_CM_HAS(DIM, M))
      MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL + D, (k_sweep_cell_march<DIM, D, M, LIM>), cell_march_blocks(h, D), MH_BLOCK,
                         S, sel, first));
  } else {
    MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL + D, (k_sweep_cell_tile<DIM, D, M, LIM>), tile_blocks(h, D), MH_BLOCK, S, sel,
                       first));
  }
}
template <int DIM, int D, int M>
void launch_cell3(MhHandle* h, int sel, int first) {
  const int nb = seg_blocks(h, D, MH_O3_L);
  const SlotSplit p = slot_split((long)nb * (MH_BLOCK / 64), 2048, M + 1);
  LAUNCH(h, KN_SWEEP_CELL + D, (k_sweep_cell3<DIM, D, M>), dim3(nb, p.groups), MH_BLOCK, h->dev, sel, first, p.vper);
}
template <int DIM, int M>
void launch_cell_part(MhHandle* h, int D, int sel, int first, bool gen, bool o3) {
  const MhDev& S = h->dev;
  const bool flat = h->sweep_mode == MH_SWEEP_FLAT;
  if (gen) {
    if (D == 0) LAUNCH(h, KN_SWEEP_CELL + 0, (k_sweep_cell_gen<DIM, 0, M>), gen_blocks(h, 0), MH_BLOCK, S, sel, first);
    else if (D == 1) LAUNCH(h, KN_SWEEP_CELL + 1, (k_sweep_cell_gen<DIM, 1, M>), gen_blocks(h, 1), MH_BLOCK, S, sel, first);
    else if constexpr (DIM == 3) LAUNCH(h, KN_SWEEP_CELL + 2, (k_sweep_cell_gen<3, 2, M>), gen_blocks(h, 2), MH_BLOCK, S, sel, first);
  } else if (o3) {
    if (D == 0) launch_cell3<DIM, 0, M>(h, sel, first);
    else if (D == 1) launch_cell3<DIM, 1, M>(h, sel, first);
    else if constexpr (DIM == 3) launch_cell3<3, 2, M>(h, sel, first);
  } else if (D == 0) {
    if (flat) MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL, (k_sweep_cell<DIM, 0, M, LIM>), h->nblk_c, MH_BLOCK, S, sel, first));
    else launch_cell_x<DIM, M>(h, sel, first);
  } else if (D == 1) {
    if (flat) MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL + 1, (k_sweep_cell<DIM, 1, M, LIM>), h->nblk_c, MH_BLOCK, S, sel, first));
    else launch_cell_yz<DIM, 1, M>(h, sel, first);
  } else if constexpr (DIM == 3) {
    if (flat) MH_LIMSW(h, LAUNCH(h, KN_SWEEP_CELL + 2, (k_sweep_cell<3, 2, M, LIM>), h->nblk_c, MH_BLOCK, S, sel, first));
    else launch_cell_yz<3, 2, M>(h, sel, first);
  }
}

// Dual part of one sweep direction (computeDualUremap), then the dual kinetic energy when
// the total energy is conserved.  None in advection mode (withDualProjection, PrepareRemap.cc:211).
template <int DIM, int M>
void launch_dual_part(MhHandle* h, int D, int sel, int prev, int last, bool gen, bool o3) {
  const MhDev& S = h->dev;
  if (S.sans_lagrange) return;
  const bool flat = h->sweep_mode == MH_SWEEP_FLAT;
  const bool march = !flat && !o3 && march_sweep(h);  // y / z: threads march over segments of nodes
  if (gen) {
    if (D == 0) LAUNCH(h, KN_SWEEP_NODE, (k_sweep_node<DIM, 0, M, MH_LIM_ANY>), h->nblk_n, MH_BLOCK, S, sel, prev, last);
    else if (D == 1) LAUNCH(h, KN_SWEEP_NODE + 1, (k_sweep_node<DIM, 1, M, MH_LIM_ANY>), h->nblk_n, MH_BLOCK, S, sel, prev, last);
    else if constexpr (DIM == 3) LAUNCH(h, KN_SWEEP_NODE + 2, (k_sweep_node<3, 2, M, MH_LIM_ANY>), h->nblk_n, MH_BLOCK, S, sel, prev, last);
  } else if (D == 0) {
    if (flat) MH_LIMSW(h, LAUNCH(h, KN_SWEEP_NODE, (k_sweep_node<DIM, 0, M, LIM>), h->nblk_n, MH_BLOCK, S, sel, prev, last));
    else MH_LIMSW(h, LAUNCH(h, KN_SWEEP_NODE, (k_sweep_node_row<DIM, M, LIM>), node_row_blocks(h), MH_BLOCK, S, sel, prev, last));
  } else if (D == 1) {
    if (march)
      MH_LIMSW(h, LAUNCH(h, KN_SWEEP_NODE + 1, (k_sweep_node_march<DIM, 1, M, LIM>), node_march_blocks(h, 1), MH_BLOCK, S, sel, prev, last));
    else
      MH_LIMSW(h, LAUNCH(h, KN_SWEEP_NODE + 1, (k_sweep_node<DIM, 1, M, LIM>), h->nblk_n, MH_BLOCK, S, sel, prev, last));
  } else if constexpr (DIM == 3) {
    if (march)
      MH_LIMSW(h, LAUNCH(h, KN_SWEEP_NODE + 2, (k_sweep_node_march<3, 2, M, LIM>), node_march_blocks(h, 2), MH_BLOCK, S, sel, prev, last));
    else
      MH_LIMSW(h, LAUNCH(h, KN_SWEEP_NODE + 2, (k_sweep_node<3, 2, M, LIM>), h->nblk_n, MH_BLOCK, S, sel, prev, last));
  }
  if (S.dec) {  // conservation-energie-totale: the dual kinetic energy of this sweep
    if (D == 0) LAUNCH(h, KN_SWEEP_KE, (k_sweep_ke<DIM, 0, M>), h->nblk_n, MH_BLOCK, S, sel, prev);
    else if (D == 1) LAUNCH(h, KN_SWEEP_KE, (k_sweep_ke<DIM, 1, M>), h->nblk_n, MH_BLOCK, S, sel, prev);
    else if constexpr (DIM == 3) LAUNCH(h, KN_SWEEP_KE, (k_sweep_ke<3, 2, M>), h->nblk_n, MH_BLOCK, S, sel, prev);
  }
}

// The remap of one iteration (RemapADIService::appliRemap, RemapADIService.cc:15-90, and
// remapVariables).
template <int DIM, int M>
void launch_sweeps_t(MhHandle* h) {
  const MhDev& S = h->dev;
  const int dim = DIM;
  int dirs[3], nd = 0;
  for (int i = 0; i < dim; ++i) {
    const int idir = (i + h->sens) % dim;
    const int ncell = idir == 0 ? h->g.nx : idir == 1 ? h->g.ny : h->g.nz;
    if (ncell == 1) continue;  // RemapADIService.cc:27
    dirs[nd++] = idir;
  }
  const bool o3 = S.order2 == 2;
  // pente-borne or generalised limiters: one thread per face and per node, limiter read at run time
  const bool gen = !o3 && (S.pb || (S.order2 && S.limiter >= MH_MINMOD_G));
  if (S.csts) LAUNCH(h, KN_NODE_FWD, (k_node_fwd<DIM>), h->nblk_n, MH_BLOCK, S);  // PrepareRemap.cc:210
  if (S.hc && nd > 0) LAUNCH(h, KN_HCELL, (k_hcell<DIM>), h->nblk_c, MH_BLOCK, S);
  int prev = 0;  // directions swept so far
  for (int s = 0; s < nd; ++s) {
    const int first = s == 0, last = (s == nd - 1) && !first, sel = s & 1;
    const int D = dirs[s];
    launch_cell_part<DIM, M>(h, D, sel, first, gen, o3);
    launch_dual_part<DIM, M>(h, D, sel, prev, last, gen, o3);
    prev |= 1 << D;
  }
  if (S.dec && nd == 0) LAUNCH(h, KN_SWEEP_KE, (k_dual_init<DIM>), h->nblk_n, MH_BLOCK, S);
  if (nd <= 1 && !S.sans_lagrange)
    LAUNCH(h, KN_NODE_VEL, (k_node_velocity<DIM>), h->nblk_n, MH_BLOCK, S, prev);
  if (S.dec) LAUNCH(h, KN_CONS_EC, (k_cons_ec<DIM>), h->nblk_c, MH_BLOCK, S, nd > 0 ? (nd - 1) & 1 : 0);
  LAUNCH(h, KN_FINAL, (k_finalize<DIM, M>), h->nblk_c, MH_BLOCK, S, nd & 1);
  h->sens = (h->sens + 1) % dim;
}

// ---- batched ensembles: one persistent launch per phase and batch group --------------------
#define MH_LIST(l) (l).d, (l).d_n

// One sweep direction of a batch group (cell part, then dual part).
template <int DIM, int D, int M, int LIM>
void ens_sweep(const EnsGroup& g, const MhDev* tab, hipStream_t st, dim3 G, int sel, int prev, int last) {
  const int first = prev == 0;
  const dim3 B(MH_BLOCK);
  if constexpr (LIM < 0) {  // order 3 or pente-borne / generalised limiters
    const EnsList& dir = D == 0 ? g.rcmap : g.tmap[D == 0 ? 0 : D - 1];
    if (g.gen) {
      hipLaunchKernelGGL((k_sweep_cell_gen_batch<DIM, D, M>), G, B, 0, st, tab, MH_LIST(dir), sel, first);
      if (!g.adv)
        hipLaunchKernelGGL((k_sweep_node_batch<DIM, D, M, MH_LIM_ANY>), G, B, 0, st, tab, MH_LIST(g.nmap), sel, prev, last);
    } else {
      hipLaunchKernelGGL((k_sweep_cell3_batch<DIM, D, M>), G, B, 0, st, tab, MH_LIST(dir), sel, first);
      if (!g.adv)
        hipLaunchKernelGGL((k_sweep_node_batch<DIM, D, M, -1>), G, B, 0, st, tab, MH_LIST(g.nmap), sel, prev, last);
    }
  } else if (g.rows && D == 0) {
    hipLaunchKernelGGL((k_sweep_cell_row_batch<DIM, M, LIM>), G, B, 0, st, tab, MH_LIST(g.rcmap), sel, first);
    if (!g.adv)
      hipLaunchKernelGGL((k_sweep_node_row_batch<DIM, M, LIM>), G, B, 0, st, tab, MH_LIST(g.rnmap), sel, prev, last);
  } else if (g.rows) {
    constexpr int DT = D == 0 ? 1 : D;
    if (MH_CM_HAS(DIM, M) && g.cmarch) {
      if constexpr (MH_CM_HAS(DIM, M))
        hipLaunchKernelGGL((k_sweep_cell_march_batch<DIM, DT, M, LIM>), G, B, 0, st, tab, MH_LIST(g.tmap[DT - 1]), sel, first);
    } else {
      hipLaunchKernelGGL((k_sweep_cell_tile_batch<DIM, DT, M, LIM>), G, B, 0, st, tab, MH_LIST(g.tmap[DT - 1]), sel, first);
    }
    if (!g.adv && !g.o3)  // threads march along D over segments of nodes
      hipLaunchKernelGGL((k_sweep_node_march_batch<DIM, (D == 0 ? 1 : D), M, LIM>), G, B, 0, st, tab,
                         MH_LIST(g.mmap[D == 0 ? 0 : D - 1]), sel, prev, last);
    else if (!g.adv)
      hipLaunchKernelGGL((k_sweep_node_batch<DIM, D, M, LIM>), G, B, 0, st, tab, MH_LIST(g.nmap), sel, prev, last);
  } else {
    hipLaunchKernelGGL((k_sweep_cell_batch<DIM, D, M, LIM>), G, B, 0, st, tab, MH_LIST(g.cmap), sel, first);
    if (!g.adv)
      hipLaunchKernelGGL((k_sweep_node_batch<DIM, D, M, LIM>), G, B, 0, st, tab, MH_LIST(g.nmap), sel, prev, last);
  }
}

// One iteration of every case of a batch group: a fixed grid of E->ncu * g.bpc blocks per
// launch walks the group's work lists.
template <int DIM, int M, int LIM>
void ens_group_cycle_l(MhEnsembleImpl* E, const EnsGroup& g) {
  const int par = (int)(E->launched & 1);
  const MhDev* tab = E->d_tab[par];
  hipStream_t st = E->stream;
  const dim3 G((unsigned)(E->ncu * g.bpc)), B(MH_BLOCK);
  if (g.adv) hipLaunchKernelGGL((k_node_adv_batch<DIM>), G, B, 0, st, tab, MH_LIST(g.nmap));
  else if (DIM == 3 && g.ntile) hipLaunchKernelGGL((k_node_lag3_tiled_batch<>), G, B, 0, st, tab, MH_LIST(g.ntmap));
  else hipLaunchKernelGGL((k_node_lag_batch<DIM>), G, B, 0, st, tab, MH_LIST(g.nmap));
  if (g.lc) hipLaunchKernelGGL((k_cell_length_batch<DIM>), G, B, 0, st, tab, MH_LIST(g.cmap));
  if (g.csts) hipLaunchKernelGGL((k_cell_lag_csts_batch<DIM, M>), G, B, 0, st, tab, MH_LIST(g.cmap));
  else if (g.adv) hipLaunchKernelGGL((k_cell_lag_batch<DIM, M>), G, B, 0, st, tab, MH_LIST(g.cmap));
  else hipLaunchKernelGGL((k_cell_lag_remap_batch<DIM, M>), G, B, 0, st, tab, MH_LIST(g.cmap));
  if (g.csts) hipLaunchKernelGGL((k_node_fwd_batch<DIM>), G, B, 0, st, tab, MH_LIST(g.nmap));
  const int sens = (int)(E->launched % DIM);
  if (g.o3 || g.gen) hipLaunchKernelGGL((k_hcell_batch<DIM>), G, B, 0, st, tab, MH_LIST(g.cmap));
  int prev = 0;  // directions swept so far
  for (int s = 0; s < DIM; ++s) {
    const int D = (s + sens) % DIM, last = s == DIM - 1, sel = s & 1;
    if (D == 0) ens_sweep<DIM, 0, M, LIM>(g, tab, st, G, sel, prev, last);
    else if (D == 1) ens_sweep<DIM, 1, M, LIM>(g, tab, st, G, sel, prev, last);
    else if constexpr (DIM == 3) ens_sweep<3, 2, M, LIM>(g, tab, st, G, sel, prev, last);
    if (g.cons) {  // the dual kinetic energy of this sweep
      if (D == 0) hipLaunchKernelGGL((k_sweep_ke_batch<DIM, 0, M>), G, B, 0, st, tab, MH_LIST(g.nmap), sel, prev);
      else if (D == 1) hipLaunchKernelGGL((k_sweep_ke_batch<DIM, 1, M>), G, B, 0, st, tab, MH_LIST(g.nmap), sel, prev);
      else if constexpr (DIM == 3)
        hipLaunchKernelGGL((k_sweep_ke_batch<3, 2, M>), G, B, 0, st, tab, MH_LIST(g.nmap), sel, prev);
    }
    prev |= 1 << D;
  }
  if (g.cons) hipLaunchKernelGGL((k_cons_ec_batch<DIM>), G, B, 0, st, tab, MH_LIST(g.cmap), (DIM - 1) & 1);
  hipLaunchKernelGGL((k_finalize_batch<DIM, M>), G, B, 0, st, tab, MH_LIST(g.cmap), DIM & 1);
  hipLaunchKernelGGL((k_dt_batch<>), dim3((unsigned)E->ncu), dim3(MH_DT_BLOCK), 0, st, tab, g.d_list, g.d_nlist);
}

template <int DIM, int M>
void ens_group_cycle(MhEnsembleImpl* E, const EnsGroup& g) {
  switch (g.lim) {
    case 0: ens_group_cycle_l<DIM, M, 0>(E, g); break;
    case 1: ens_group_cycle_l<DIM, M, 1>(E, g); break;
    case 2: ens_group_cycle_l<DIM, M, 2>(E, g); break;
    case 3: ens_group_cycle_l<DIM, M, 3>(E, g); break;
    default: ens_group_cycle_l<DIM, M, -1>(E, g); break;
  }
}

template void launch_sweeps_t<2, MH_TU_M>(MhHandle*);
template void launch_sweeps_t<3, MH_TU_M>(MhHandle*);
template void ens_group_cycle<2, MH_TU_M>(MhEnsembleImpl*, const EnsGroup&);
template void ens_group_cycle<3, MH_TU_M>(MhEnsembleImpl*, const EnsGroup&);
