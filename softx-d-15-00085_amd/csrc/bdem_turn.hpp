/*
 * bdem_turn.hpp - the mill's turning lifters, on the device (internal).
 *
 * The reference turns its lifters on the host before every step
 * (Rotate_VolObject_Inc, Input/Processing_Mills.h:7-60, called from
 * UpdateSim, main.cpp:114-121) and re-uploads the whole lifter table to
 * constant memory (Device_Update_DObjectPostions,
 * Device/DeviceInterface.cu:2826-2831).  Here one block turns the lifters
 * inside the parameter block the step kernel reads, on the step's own
 * stream, so a mill run never leaves the device: an extra block of the
 * incremental re-sort, which does not read them, or a launch of its own
 * beside the full sort.  A thread turns one vertex, then one face (a thread
 * per lifter took 6.6 us, and a launch of its own a step).
 *
 * Arithmetic as on the host: the cosine and sine of the double angle
 * (computed once on the host), the two products and their sum in double,
 * rounded once to float; the face centroids, normals and areas re-derived in
 * float in the reference's order.  The build turns off FMA contraction and
 * uses correctly rounded division and square root, so the results are the
 * host's bit for bit.
 */
#pragma once
#include "bdem_kernels.hpp"

namespace bdem {

__device__ __forceinline__ void turn_point(bdem_float3& v, double c, double s, float ax, float ay, float az) {
  const float px = v.x - ax, py = v.y - ay;
  /* vertex.x = cos*point.x + sin*point.y; vertex.y = -sin*point.x + cos*point.y;
   * vertex.z kept; then vertex += about */
  const float x = (float)(c * (double)px + s * (double)py);
  const float y = (float)(-s * (double)px + c * (double)py);
  v.x = x + ax;
  v.y = y + ay;
  v.z = v.z + az;
}

constexpr int TURN_THREADS = 256;
static_assert(TURN_THREADS == 8 * MAX_DOBJ, "a thread per lifter vertex");
/* By the first TURN_THREADS threads of a block, all of whose threads call;
 * tv: 8 x MAX_DOBJ vertices in LDS, as they are after the turn. */
__device__ __forceinline__ void turn_lifters_block(DevParams* __restrict__ P, const TurnArgs& t, bdem_float3* tv) {
  const int k = (int)threadIdx.x >> 3, q = (int)threadIdx.x & 7;
  const bool on = threadIdx.x < TURN_THREADS && k < P->num_dobj && P->dobj[k].is_attached_DWorld;
  if (on) {
    bdem_float3 v = P->dobj[k].vertex[q];
    if (q < P->dobj[k].num_vertex) {
      turn_point(v, t.c, t.s, t.about[0], t.about[1], t.about[2]);
      P->dobj[k].vertex[q] = v;
    }
    tv[threadIdx.x] = v;   /* a face of fewer than four vertices may name any of the eight */
  }
  __syncthreads();
  if (!on) return;
  bdem_DOBJ& d = P->dobj[k];
  if (q < d.num_faces) {
    bdem_Surface& f = d.faces[q];
    auto at = [&](int j) { return cvt(tv[8 * k + f.vertex_Order[j]]); };
    f3 sum = mk3(0.0f, 0.0f, 0.0f);
    for (int j = 0; j < f.num_vertex; ++j) sum = sum + at(j);
    const f3 cen = (1.0f / (float)f.num_vertex) * sum;
    const f3 v0 = at(0), v1 = at(1), v2 = at(2), v3 = at(3);
    const f3 V1 = v1 - v0, V2 = v2 - v1, V3 = v3 - v2, V4 = v0 - v3;
    const f3 n = cross(V2, V1);
    const f3 nn = n / length(n);
    f.centroid = bdem_float3{cen.x, cen.y, cen.z};
    f.normal = bdem_float3{nn.x, nn.y, nn.z};
    f.area = 0.500000f * length(n) + 0.500000f * length(cross(V3, V4));
  } else if (q == 7) {
    turn_point(d.COM, t.c, t.s, t.about[0], t.about[1], t.about[2]);
  }
}

}  // namespace bdem
