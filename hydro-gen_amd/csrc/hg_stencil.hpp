// hg_stencil.hpp — the heights of a droplet's 2x2 stencil, from what the lanes
// of its group loaded.  Apart from the kernel (hg_particle.hip), so that a host
// program can check it for any values of the lanes.
#pragma once

namespace hgk {

// v: lane g of a group of 16 has layer g & 1 of corner (g >> 1) & 3, the corners
// being (0,0), (1,0), (0,1), (1,1).  h..: the corners' rock + dirt, in every lane
// of the group those of lanes 0, 2, 4 and 6.  Lanes 8-15 hold loads of their own
// of the same cells, which other droplets change meanwhile; two lanes may see
// different values, and a group whose lanes hold different heights would go
// different ways.
// Lanes::other_layer(v): the value of the lane beside, g ^ 1; Lanes::lane<L>(v):
// the value of lane L of the group.
template <class Lanes, class V>
__device__ __forceinline__ void corner_heights(V v, V& h00, V& h10, V& h01, V& h11) {
    const V h = v + Lanes::other_layer(v);
    h00 = Lanes::template lane<0>(h);
    h10 = Lanes::template lane<2>(h);
    h01 = Lanes::template lane<4>(h);
    h11 = Lanes::template lane<6>(h);
}

}  // namespace hgk
