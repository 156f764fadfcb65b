// The device view of a graph that the expansion launchers take.
#pragma once

#include "common.h"
#include "kernels.h"

namespace ibfs {

inline HubSplit hub_split(const HubCut &h) { return HubSplit{h.deg, h.tie, h.cut}; }

inline GraphDev graph_dev(const ibfs_graph_s *g, const ibfs_config &c, const HubCut &h) {
  return GraphDev{g->d_beg,   g->d_adj,   g->d_tadj,
                  reinterpret_cast<const int4 *>(g->heads->d), g->Vt,
                  c.lrg_shed, __builtin_ctz((unsigned)c.td_chunk), hub_split(h)};
}

}  // namespace ibfs
