/*
 * bdem_state.hip - the state's way in and out: the caller's arrays (float3,
 * quaternion, type and ID per particle) to and from the device's float4
 * streams, converted on the device.
 *
 * The streams were copied whole through pageable vectors (allocated, faulted
 * in and converted particle by particle on each call): 8 of the 10 ms of a
 * 100,003-sphere restart.  Now a kernel packs the state into a buffer of the
 * caller's layout, and the bytes asked for cross through two pinned halves of
 * a small staging buffer, one in flight while the other is copied from or to
 * the caller's memory.
 */
#include "bdem_kernels.hpp"

namespace bdem {

__global__ __launch_bounds__(256) void k_pack_state(int n, const float4* __restrict__ pos,
                                                    const float4* __restrict__ vel, const float4* __restrict__ omg,
                                                    const float4* __restrict__ quat,
                                                    const bdem_poly_shape* __restrict__ shapes, int num_shapes,
                                                    int by_pid, StateArrays out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float4 p = pos[i];
  const float4 v = vel[i], o = omg[i];
  const int packed = __float_as_int(o.w);
  if (shapes) {
    /* Get_SystemState / Get_Particle_PosArray return position - COM for
     * polyhedra (GPU_Memory_Transfer.cuh:461, 504) */
    const int row = by_pid ? max(packed >> 3, 0) : (packed & 7);
    if (row < num_shapes) {
      const bdem_float3 cm = shapes[row].COM;
      p.x -= cm.x; p.y -= cm.y; p.z -= cm.z;
    }
  }
  out.pos[i] = bdem_float3{p.x, p.y, p.z};
  out.vel[i] = bdem_float3{v.x, v.y, v.z};
  out.avel[i] = bdem_float3{o.x, o.y, o.z};
  out.ptype[i] = (unsigned)(packed & 7);
  out.pid[i] = packed >> 3;
  if (quat) {
    const float4 q = quat[i];
    out.quat[i] = bdem_Quaterion{q.x, q.y, q.z, q.w};
  }
}

void launch_pack_state(const StepBuffers& b, const bdem_poly_shape* shapes, int num_shapes, bool by_pid, bool orient,
                       const StateArrays& out, hipStream_t s) {
  if (b.n <= 0) return;
  hipLaunchKernelGGL(k_pack_state, dim3((b.n + 255) / 256), dim3(256), 0, s, b.n, b.pos_cur, b.vel_cur, b.omg_cur,
                     orient ? b.quat_cur : nullptr, shapes, num_shapes, by_pid ? 1 : 0, out);
}

/* Radius and mass come from the type table (the reference's only source),
 * the particle's own shape row, or stay as they are (per-particle values). */
__global__ __launch_bounds__(256) void k_unpack_state(const DevParams* __restrict__ Pp, int n, StateArrays in,
                                                      UnpackMode m, const bdem_poly_shape* __restrict__ shapes,
                                                      float4* __restrict__ pos, float4* __restrict__ vel,
                                                      float4* __restrict__ omg, float4* __restrict__ quat) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const bdem_float3 p = in.pos[i];
  const unsigned t = in.ptype[i];
  const int pid = in.pid[i];
  float r, mass;
  if (m.shape_by_pid) {
    const bdem_poly_shape& sh = shapes[pid > 0 ? pid : 0];
    r = sh.radius;
    mass = sh.mass;
  } else if (m.per_particle) {
    r = pos[i].w;
    mass = vel[i].w;
  } else {
    r = Pp->t_radius[t & 7u];
    mass = Pp->t_mass[t & 7u];
  }
  const bdem_float3 v = m.has_vel ? in.vel[i] : bdem_float3{vel[i].x, vel[i].y, vel[i].z};
  const bdem_float3 w = m.has_avel ? in.avel[i] : bdem_float3{omg[i].x, omg[i].y, omg[i].z};
  pos[i] = make_float4(p.x, p.y, p.z, r);
  vel[i] = make_float4(v.x, v.y, v.z, mass);
  omg[i] = make_float4(w.x, w.y, w.z, __int_as_float(pack_id_type(pid, (int)t)));
  if (quat) {   /* the stream holds (w, x, y, z); Set_Pos: identity where none is given */
    float4 q = make_float4(1.f, 0.f, 0.f, 0.f);
    if (m.has_quat) {
      const bdem_Quaterion g = in.quat[i];
      q = make_float4(g.w, g.x, g.y, g.z);
    }
    quat[i] = q;
  }
}

void launch_unpack_state(const DevParams* dP, const StepBuffers& b, const StateArrays& in, const UnpackMode& m,
                         const bdem_poly_shape* shapes, bool orient, hipStream_t s) {
  if (b.n <= 0) return;
  hipLaunchKernelGGL(k_unpack_state, dim3((b.n + 255) / 256), dim3(256), 0, s, dP, b.n, in, m, shapes, b.pos_cur,
                     b.vel_cur, b.omg_cur, orient ? b.quat_cur : nullptr);
}

__global__ __launch_bounds__(256) void k_set_radii(int n, const float* __restrict__ radius,
                                                   const float* __restrict__ mass, float4* __restrict__ pos,
                                                   float4* __restrict__ vel) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  pos[i].w = radius[i];
  vel[i].w = mass[i];
}

void launch_set_radii(const StepBuffers& b, const float* radius, const float* mass, hipStream_t s) {
  if (b.n <= 0) return;
  hipLaunchKernelGGL(k_set_radii, dim3((b.n + 255) / 256), dim3(256), 0, s, b.n, radius, mass, b.pos_cur, b.vel_cur);
}

}  // namespace bdem
