// Row products with a group of lanes per row: the shape shared by the kernels
// that walk a CSR's rows and read whole neuron-major rows per edge.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace ns {

constexpr int kEdgeUnroll = 4;  // edges per lane per round of the backward's edge loops

// The edge kernels of the backward and of the event tick give each row (a source,
// or a destination) a power-of-two group of lanes: LPE lanes per edge, VL
// neighbouring columns each (one 4 * VL byte load of a neuron-major row; VL = 1
// takes any strides), and `edge_lanes` edges at a time, `unroll` rounds of them in
// flight.  The host picks edge_lanes so that a row of average length is about
// one round (edge_lanes_for).  A wavefront per row, every lane walking its edge's columns
// by itself, left two thirds of the lanes idle at 20 edges per row and read
// each gathered row in 4-byte pieces.

template <int VL>
__device__ __forceinline__ void load_row(const float* at, float x[VL]) {
  typedef float vec __attribute__((ext_vector_type(VL == 1 ? 2 : VL)));
  if constexpr (VL == 1) {
    x[0] = *at;
  } else {
    const vec y = *reinterpret_cast<const vec*>(at);
#pragma unroll
    for (int k = 0; k < VL; ++k) x[k] = y[k];
  }
}

// log2 of the edges a row's group takes at a time: the smallest power of two for
// which `unroll` of them cover a row of average length, at most what fits
// one wavefront beside the LPE lanes of an edge.
inline int edge_lanes_for(int64_t edges, int64_t rows, int lpe, int unroll) {
  int lg = 0;
  while ((lpe << lg) < 64 && (int64_t{unroll} << lg) * rows < edges) ++lg;
  return lg;
}

struct EdgeForm {
  int vl, lpe;
};

// The edge kernels' form for a batch: VL = 4 (2 at B = 2) where whole neuron-major
// rows can be loaded, else one column per lane.
inline EdgeForm edge_form(int64_t batch, bool whole_rows) {
  if (whole_rows && batch == 2) return {2, 1};
  if (whole_rows && batch % 4 == 0) return {4, batch == 4 ? 1 : batch == 8 ? 2 : 4};
  return {1, batch <= 1 ? 1 : batch == 2 ? 2 : batch <= 4 ? 4 : batch <= 8 ? 8 : 16};
}

template <typename F>
inline void with_edge_form(EdgeForm form, F&& launch) {
  if (form.vl == 4) {
    if (form.lpe == 1) launch(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
    else if (form.lpe == 2) launch(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
    else launch(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
  } else if (form.vl == 2) {
    launch(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
  } else {
    switch (form.lpe) {
      case 1: launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{}); break;
      case 2: launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{}); break;
      case 4: launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{}); break;
      case 8: launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 8>{}); break;
      default: launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 16>{});
    }
  }
}

}  // namespace ns
