/*
 * bdem_step.hpp - the pieces of one step that its kernels share: a team's
 * contact search, a contact's force, the contacts past the list, walls and lifters, the
 * integration with the next key, and the changed-list append (internal).
 */
#pragma once
#include "bdem_kernels.hpp"

namespace bdem {

/* ------------------------------------------------------------------------ */
/* Pair forces of one particle (all laws).                                    */
/* ------------------------------------------------------------------------ */
struct PairHistCtx {
  const HistRec* in; int in_cnt; int cursor;
  HistRec* out; int out_cnt;
};

/* Force and torque on particle A from contact partner j (all laws), and the
 * spring record of that contact.  The caller accumulates Fc and Tc. */
template <int LAW>
__device__ __forceinline__ void contact_force(const DevParams& P, int j, const float4* __restrict__ pos_r,
                                              const float4* __restrict__ vel_m,
                                              const float4* __restrict__ omg_t, f3 pa, float ra, f3 va,
                                              float ma, f3 wa, int ta, const HistRec* hin, int hin_cnt,
                                              int cursor, HistRec* hrec, f3& Fc, f3& Tc,
                                              float* tally = nullptr) {
  const float4 pb = pos_r[j];
  const float4 vb = vel_m[j];
  const float4 ob = omg_t[j];
  HistRec first = make_float4(0.f, 0.f, 0.f, 0.f);
  if (LAW != BDEM_LAW_REFERENCE && hin_cnt > 0) first = hin[spring_start(hin_cnt, cursor)];
  if (LAW == BDEM_LAW_REFERENCE) {
    pair_ref(P, pa, ra, va, ma, wa, ta, xyz(pb), pb.w, xyz(vb), vb.w, xyz(ob), packed_type(ob.w), Fc, Tc,
             tally);
  } else {
    const f3 rel = pa - xyz(pb);
    const float d = length(rel);
    const f3 n = rel * (1.0f / d);
    const float delta = (ra + pb.w) - d;
    const f3 la = (-1.0f * n) * ra;
    const f3 lb = n * pb.w;
    const f3 vc = (va + cross(wa, la)) - (xyz(vb) + cross(xyz(ob), lb));
    /* R* and m* from one division */
    const float sr = ra + pb.w, sm = ma + vb.w;
    const float q = 1.0f / (sr * sm);
    const float rstar = ((ra * pb.w) * sm) * q;
    const float mstar = ((ma * vb.w) * sr) * q;
    const int idb = packed_pid(ob.w);
    f3 xi = find_spring_first(hin, hin_cnt, idb, cursor, first);
    /* one type: a wave-uniform address, read by scalar loads that need not
     * wait for the partner's type word */
    float e = 0.0f;
    Fc = history_law(P, n, delta, vc, rstar, mstar, P.one_type ? P.law_pp[0][0] : P.law_pp[ta][packed_type(ob.w)],
                     xi, tally ? &e : nullptr);
    /* half the pair's dissipation from each side (the pair is met from both) */
    if (tally) atomicAdd(tally + TALLY_PP, (0.5f * e) * P.dt);
    Tc = cross(la, Fc);
    if (hrec) *hrec = make_float4(xi.x, xi.y, xi.z, __int_as_float(idb));
  }
}

/* Per-particle (uncompacted) loop over the contacts found by the scan. */
template <int LAW>
__device__ __forceinline__ void particle_contact(const DevParams& P, int j, const float4* __restrict__ pos_r,
                                                 const float4* __restrict__ vel_m,
                                                 const float4* __restrict__ omg_t, f3 pa, float ra, f3 va,
                                                 float ma, f3 wa, int ta, f3& F, f3& T, PairHistCtx* hc,
                                                 float* tally = nullptr) {
  f3 Fc, Tc;
  HistRec* rec = (LAW != BDEM_LAW_REFERENCE && hc->out_cnt < HMAX) ? hc->out + hc->out_cnt : nullptr;
  contact_force<LAW>(P, j, pos_r, vel_m, omg_t, pa, ra, va, ma, wa, ta, hc->in, hc->in_cnt,
                     hc->out_cnt, rec, Fc, Tc, tally);
  if (LAW != BDEM_LAW_REFERENCE && hc->out_cnt < HMAX) ++hc->out_cnt;
  F = F + Fc;
  if (P.rotation) T = T + Tc;
}

constexpr int CLIST = 12;   /* LDS list entries per thread: 12 KiB + wave staging fits 6 blocks per CU */
static_assert(CLIST <= HMAX, "springs of the listed contacts are stored first");
constexpr int STEP_THREADS = 256;

#define BDEM_STEP_PARAMS                                                                            \
  int n, const float4* __restrict__ pos_in, const float4* __restrict__ vel_in,                      \
      const float4* __restrict__ omg_in, const float4* __restrict__ quat_in,                        \
      float4* __restrict__ pos_out, float4* __restrict__ vel_out, float4* __restrict__ omg_out,     \
      float4* __restrict__ quat_out, uint32_t* __restrict__ keys_out,                               \
      const uint32_t* __restrict__ sorted_keys, uint8_t* __restrict__ changed,                      \
      unsigned long long* __restrict__ sbuf, uint32_t* __restrict__ append,                         \
      const uint32_t* __restrict__ hwc_in, uint32_t* __restrict__ hwc_out,                          \
      const HistRec* __restrict__ hr_in, HistRec* __restrict__ hr_out,                              \
      const HistRec* __restrict__ wr_in, HistRec* __restrict__ wr_out, int hist_cap,                \
      float* __restrict__ wall_force, int do_kill, uint32_t *status, int *kill_count
#define BDEM_STEP_ARGS                                                                               \
  n, pos_in, vel_in, omg_in, quat_in, pos_out, vel_out, omg_out, quat_out, keys_out, sorted_keys, changed, \
      sbuf, append, hwc_in, hwc_out, hr_in, hr_out, wr_in, wr_out, hist_cap, wall_force, do_kill, status,  \
      kill_count

/* Contacts beyond the LDS list: rescan, same order (rare).  Springs of
 * contacts CLIST .. HMAX-1 are stored after the list's, as in the
 * restatement.  One live particle per lane; nc its full contact count. */
template <int LAW>
__device__ __forceinline__ void contact_tail(const DevParams& P, const uint2* __restrict__ cells,
                                             const float4* __restrict__ pos_in, const float4* __restrict__ vel_in,
                                             const float4* __restrict__ omg_in, int i, f3 p, float r, f3 v, f3 w,
                                             float m, int ta, int pid, int nc, uint32_t hwc,
                                             const HistRec* __restrict__ hr_in, HistRec* __restrict__ hr_out,
                                             int hist_cap, uint32_t* __restrict__ dbg_list, uint32_t* status, f3& Fpp,
                                             f3& Tpp, float* tally) {
  if (nc > CLIST) {
    PairHistCtx hc{nullptr, 0, 0, nullptr, HMAX};   /* no slot: looked up, not stored */
    if (LAW != BDEM_LAW_REFERENCE && pid < hist_cap) {
      hc.in = hr_in + (size_t)pid * HMAX;
      hc.in_cnt = min((int)(hwc & 0xFFFFu), HMAX);
      hc.out = hr_out + (size_t)pid * HMAX;
      hc.out_cnt = CLIST;
    }
    for_each_contact(P, cells, pos_in, i, p, r, [&](int j, float4, int k) {
      if (k >= CLIST)
        particle_contact<LAW>(P, j, pos_in, vel_in, omg_in, p, r, v, m, w, ta, Fpp, Tpp, &hc, tally);
      if (dbg_list && k >= CLIST && k < LIST_STRIDE) dbg_list[(size_t)i * LIST_STRIDE + k] = (uint32_t)j;
    });
    /* the reference's 32-entry list overflows (Collision_Detection_BroadPhase.cuh:481) */
    if (nc > LIST_STRIDE) atomicOr(status, ST_LIST_OVERFLOW);
  }
  if (LAW != BDEM_LAW_REFERENCE && nc > HMAX) atomicOr(status, ST_HIST_OVERFLOW);
  if (!P.rotation) Tpp = mk3(0.f, 0.f, 0.f);
}

/* Walls (a8) and lifters (a9) of one live particle: they need its own state
 * only.  ltype is the lifter contact type kept for the next step, wcnt the
 * number of wall springs written. */
struct WallOut { f3 Fw, Tw, Fl, Tl; uint32_t ltype; int wcnt; };
template <int LAW>
__device__ __forceinline__ void walls_and_lifters(const DevParams& P, int i, int pid, int ta, f3 p, float r, f3 v,
                                                  f3 w, float m, uint32_t hwc, const HistRec* __restrict__ wr_in,
                                                  HistRec* __restrict__ wr_out, int hist_cap,
                                                  float* __restrict__ wall_force, WallOut& o, float* tally) {
  WallHist wh{nullptr, 0, nullptr, 0};
  if (LAW != BDEM_LAW_REFERENCE) {
    if (pid < hist_cap) {
      wh.in = wr_in + (size_t)pid * WMAX;
      wh.in_cnt = min((int)((hwc >> 16) & 0xFFu), WMAX);
      wh.out = wr_out + (size_t)pid * WMAX;
    } else {
      wh.out = nullptr; wh.out_cnt = WMAX;   /* no slot: springs are not kept (full count: never written) */
    }
  }
  wall_forces(P, ta, p, r, v, w, m, o.Fw, o.Tw, &wh, tally);
  if (wall_force) {
    wall_force[3 * i] = o.Fw.x; wall_force[3 * i + 1] = o.Fw.y; wall_force[3 * i + 2] = o.Fw.z;
  }
  o.wcnt = wh.out_cnt;
  o.Fl = mk3(0.f, 0.f, 0.f);
  o.Tl = o.Fl;
  o.ltype = 0u;
  if (P.num_dobj > 0)
    o.ltype = (uint32_t)lifter_forces(P, ta, p, r, v, w, m, (int)((hwc >> 24) & 3u), o.Fl, o.Tl, tally);
}

/* Integration, discharge, the state's write-back, the next key and changed
 * flag of slot i (< n); returns whether the key changed.  A dead slot is
 * copied through. */
template <int LAW, bool ORIENT, bool SKIN>
__device__ __forceinline__ bool particle_finish(const DevParams& P, uint32_t key_base, int i, bool alive, float4 pr,
                                                float4 vm, float4 ot, uint32_t hwc, int nc, f3 Fpp, f3 Tpp,
                                                const WallOut& wo, uint64_t new_mask, const SkinArgs& sk,
                                                const float4* __restrict__ quat_in, float4* __restrict__ pos_out,
                                                float4* __restrict__ vel_out, float4* __restrict__ omg_out,
                                                float4* __restrict__ quat_out, uint32_t* __restrict__ keys_out,
                                                const uint32_t* __restrict__ sorted_keys,
                                                uint8_t* __restrict__ changed, uint32_t* __restrict__ hwc_out,
                                                int hist_cap, float* __restrict__ wall_force, int do_kill,
                                                uint32_t* status, int* kill_count, uint32_t& new_key, float& dmove) {
  int pid = packed_pid(ot.w);
  const int ta = packed_type(ot.w);
  f3 p = xyz(pr), v = xyz(vm), w = xyz(ot);
  const float r = pr.w, m = vm.w;
  if (alive) {
    /* the contact type of the last lifter check is kept for the next step */
    if (hwc_out) {
      uint32_t h = wo.ltype << 24;
      if (LAW != BDEM_LAW_REFERENCE && pid < hist_cap)
        h |= (uint32_t)(nc < HMAX ? nc : HMAX) | ((uint32_t)wo.wcnt << 16);
      hwc_out[i] = h;
    }

    const float inv_inertia = P.per_particle ? 1.0f / (0.4f * r * r * m) : P.t_inertia[ta];
    QuatF q{1.f, 0.f, 0.f, 0.f};
    if (ORIENT) { const float4 q4 = quat_in[i]; q = QuatF{q4.x, q4.y, q4.z, q4.w}; }
    integrate(P, inv_inertia, m, Fpp, Tpp, wo.Fw, wo.Tw, wo.Fl, wo.Tl, p, v, w, ORIENT ? &q : nullptr);
    if (SKIN) {
      /* |p_new - p_old| <= sum |v dt| (1 + 2^-20) + sum |p| 2^-22 (rounding of p += v dt) */
      dmove = ((fabsf(v.x) + fabsf(v.y) + fabsf(v.z)) * P.dt) * 1.00000095367431640625f +
              (fabsf(p.x) + fabsf(p.y) + fabsf(p.z)) * 2.384185791015625e-07f;
    }

    /* a11: Remove_Silo_Discharged_Particles, GPU_Memory_Transfer.cuh:650-664 */
    if (do_kill && p.y < P.kill_height) {
      p = cvt(P.max_size);
      pid = -1;
      atomicAdd(kill_count, 1);
    }
    pos_out[i] = make_float4(p.x, p.y, p.z, r);
    vel_out[i] = make_float4(v.x, v.y, v.z, m);
    omg_out[i] = make_float4(w.x, w.y, w.z, __int_as_float(pack_id_type(pid, ta)));
    if (ORIENT) quat_out[i] = make_float4(q.w, q.x, q.y, q.z);
    if (SKIN) sk.mask_out[i] = new_mask;
  } else {
    /* dead: inert, copied through */
    pos_out[i] = pr;
    vel_out[i] = vm;
    omg_out[i] = ot;
    if (ORIENT) quat_out[i] = quat_in[i];
    if (SKIN) sk.mask_out[i] = 0ull;
    if (hwc_out) hwc_out[i] = hwc;
    if (wall_force) { wall_force[3 * i] = 0.f; wall_force[3 * i + 1] = 0.f; wall_force[3 * i + 2] = 0.f; }
  }
  new_key = key_base + key_of(P, p, pid, status);
  keys_out[i] = new_key;
  const bool chg = new_key != sorted_keys[i];
  changed[i] = chg ? 1 : 0;
  return chg;
}

/* Append changed slots for the next incremental sort, one atomic per wave;
 * every lane of the wave calls it. */
__device__ __forceinline__ void append_changed(bool chg, uint32_t new_key, int i, int n,
                                               unsigned long long* __restrict__ sbuf, uint32_t* __restrict__ append,
                                               uint32_t* status) {
  const uint64_t mask = __ballot(chg);
  if (mask) {
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((unsigned long long)mask) - 1;
    uint32_t base = 0u;
    if (lane == leader) base = atomicAdd(append, (uint32_t)__popcll(mask));
    base = __shfl(base, leader, 64);
    const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    const uint32_t at = base + (uint32_t)__popcll(mask & lt);
    if (chg) {
      if (at < (uint32_t)n) sbuf[at] = ((unsigned long long)new_key << 32) | (uint32_t)i;
      else atomicOr(status, ST_SORT_ERROR);   /* a counter left uncleared: never write past the list */
    }
  }
}

/* The contacts of one particle by its team (the G consecutive lanes that
 * hold the same arguments): visit(j, k) on the lane that found contact k,
 * k counting in the traversal order of for_each_contact.  Returns the count
 * (team-uniform).  `active` is team-uniform; every lane of the wave calls.
 * cand: the team's LDS list, CAND candidates at a time, numbered over all
 * rows so that short rows share a round of 4 G.  Past 27 G candidates a row
 * fills three quarters of a round on average, and the rows are taken one by
 * one, straight from their run (18 G and 36 G measured the same within 2 %).  The work grows with the candidates whatever their number:
 * a grid's cells are sized for its largest particles, and small ones crowd
 * them (573 spheres a cell: 20,000 of them 293 us a step, 6,441 while every
 * CAND candidates walked all the runs again). */
template <int G, int CAND, class Visit>
__device__ __forceinline__ int team_contacts(const DevParams& P, const uint2* __restrict__ cells,
                                             const float4* __restrict__ pos_r, uint32_t n, int i, f3 pa, float ra,
                                             bool active, uint32_t* cand, Visit&& visit) {
  constexpr int NR = (9 + G - 1) / G;
  const int lane = threadIdx.x & 63, sub = lane & (G - 1), lead = lane & ~(G - 1);
  int g[3];
  grid_pos(P, pa, g);
  const int xs = max(g[0] - 1, 0), xe = min(g[0] + 1, P.nx - 1);
  uint32_t lo[NR], cnt[NR];
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    const int r = sub + G * q;
    const uint32_t y = (uint32_t)g[1] + (uint32_t)(r / 3) - 1u, z = (uint32_t)g[2] + (uint32_t)(r % 3) - 1u;
    lo[q] = 0u;
    cnt[q] = 0u;
    if (active && r < 9 && xs <= xe && y < (uint32_t)P.ny && z < (uint32_t)P.nz) {
      const uint32_t h0 = hash_of(P, xs, (int)y, (int)z), h1 = hash_of(P, xe, (int)y, (int)z);
      if (h1 < P.C) {   /* at most three cells, first and last occupied entry */
        const uint2 none = make_uint2(0xFFFFFFFFu, 0u);
        const uint2 c0 = cells[h0];
        uint2 c1 = none, c2 = none;
        if (h0 + 1u <= h1) c1 = cells[h0 + 1u];
        if (h0 + 2u <= h1) c2 = cells[h0 + 2u];
        const uint32_t a = min(min(c0.x, c1.x), c2.x);
        if (a != 0xFFFFFFFFu) {
          uint32_t b = c2.x != 0xFFFFFFFFu ? c2.y : (c1.x != 0xFFFFFFFFu ? c1.y : c0.y);
          b = min(b, n);   /* table entries never exceed n; kept in range regardless */
          lo[q] = a;
          cnt[q] = b - min(a, b);
        }
      }
    }
  }
  /* offsets of the rows in the numbering of all candidates */
  uint32_t off[NR], total = 0u;
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    uint32_t incl = cnt[q];
#pragma unroll
    for (int o = 1; o < G; o <<= 1) {
      const uint32_t v = (uint32_t)__shfl_up((int)incl, o, G);
      if (sub >= o) incl += v;
    }
    off[q] = total + incl - cnt[q];
    total += (uint32_t)__shfl((int)incl, G - 1, G);
  }
  int count = 0;
  const uint32_t self = i < (int)n ? (uint32_t)i : 0u;
  /* candidates j[u] (self: none), in the order u, then lane */
  auto test = [&](const uint32_t (&j)[4]) {
    float4 pb[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) pb[u] = pos_r[j[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool hit = j[u] != self && overlaps(pa, ra, pb[u]);
      const uint32_t bits = (uint32_t)(__ballot(hit) >> lead) & ((1u << G) - 1u);
      if (hit) visit((int)j[u], count + __popc(bits & ((1u << sub) - 1u)));
      count += __popc(bits);
    }
  };
  constexpr uint32_t ROWS = CAND > 27 * G ? CAND : 27 * G;
  if (__any((int)(total > ROWS))) {   /* row by row, each row by its team */
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      for (int s = 0; s < G && s + G * q < 9; ++s) {
        const uint32_t l = (uint32_t)__shfl((int)lo[q], s, G), m = (uint32_t)__shfl((int)cnt[q], s, G);
        for (uint32_t t0 = 0u; __any((int)(t0 < m)); t0 += 4u * G) {
          uint32_t j[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t t = t0 + (uint32_t)(u * G + sub);
            j[u] = t < m ? l + t : self;
          }
          test(j);
        }
      }
    }
    return count;
  }
  for (uint32_t c0 = 0u; __any((int)(c0 < total)); c0 += (uint32_t)CAND) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      /* the row's part in the window, as signed numbers (a guard on the
       * unsigned difference, c0 + CAND > off ? ... : 0, is dropped by the
       * compiler, which takes the difference as not wrapping) */
      const int at = (int)off[q] - (int)c0, end = min((int)cnt[q], CAND - at);
      for (int k = max(-at, 0); k < end; ++k) cand[at + k] = lo[q] + (uint32_t)k;
    }
    __builtin_amdgcn_wave_barrier();
    const uint32_t m = min(total - min(c0, total), (uint32_t)CAND);
    for (uint32_t t0 = 0u; __any((int)(t0 < m)); t0 += 4u * G) {
      uint32_t j[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t t = t0 + (uint32_t)(u * G + sub);
        j[u] = t < m ? cand[t] : self;
      }
      test(j);
    }
    __builtin_amdgcn_wave_barrier();
  }
  return count;
}

}  // namespace bdem
