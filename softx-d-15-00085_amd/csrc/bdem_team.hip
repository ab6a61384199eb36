/*
 * bdem_team.hip - the fused sphere step with a team of lanes per particle.
 *
 * One lane per particle (k_step) leaves a serial chain in every wave: nine
 * stencil rows one after another, then the force passes, the walls and the
 * integration.  Below a few hundred thousand particles the whole chip holds
 * every wave at once, so a step lasts as long as that chain.  Here a block
 * owns PB consecutive sorted slots; G lanes work on each:
 *
 *   team waves    lane t of a particle's team reads the cells of stencil row
 *                 t, a team prefix over the rows' counts numbers the
 *                 candidates in the reference order, and the lanes then test
 *                 candidates t, t + G, ... with several loads in flight;
 *                 ballots give every contact its place in that order.  Lane
 *                 t computes contact t, and the team adds the results in
 *                 contact order.
 *   one more wave computes the walls and lifters of all PB slots meanwhile,
 *                 then takes the pair sums from LDS, integrates and writes
 *                 back (the same code as k_step).
 *
 * Every float operation and every sum is k_step's, in the same order.
 *
 * What bounds it: memory round trips, about six in a row (state, cells,
 * candidates, partners and springs, the append counter), and past one
 * resident round of waves the address rate of its 16-byte gathers, which
 * k_step avoids by staging whole rows in LDS.  Hence the shapes below: the
 * most lanes per particle whose waves the chip still holds at once.
 * Measured per step with the re-sort and the launch gaps (k_step beside it),
 * random packs of r 0.5 cm at 1.5 to the cm3, about six contacts each: 8,192
 * LSD 29.5 us (62), 20,000 reference law 29.1 (50), 32,000 LSD 37 (64),
 * 60,013 Hertz-Mindlin 51.5 (71), 100,003 reference law 57 (65), 131,000
 * reference law 66.6 (71.4), LSD 77 (87), Hertz-Mindlin 79 (89), 160,000
 * Hertz-Mindlin 85 (92), 262,143 116 (108).  The gathers grow with the
 * candidates: at 3 to the cm3, 12 contacts, 131,000 of the reference law take
 * 153 (132).  TEAM_STEP_MAX lies between the two crossings.
 */
#include "bdem_step.hpp"

namespace bdem {

namespace {

constexpr int TEAM_CAND = 64;   /* candidates listed per particle at a time */

template <int G>
struct TeamScratch {
  static constexpr int NP = 64 / G;   /* particles per wave */
  union {
    uint32_t cand[NP][TEAM_CAND];
    float f[6][64];
  };
  uint32_t clist[NP][CLIST];
};

template <int LAW, bool ORIENT, bool ENERGY, int G, int PB, bool BATCH>
__global__ __launch_bounds__(PB* G + 64) __attribute__((amdgpu_waves_per_eu(6))) void k_step_team(const DevParams* __restrict__ Pp,
                                                          const uint32_t* __restrict__ tile_sim,
                                                          const uint2* __restrict__ cells_all,
                                                          uint32_t* __restrict__ dbg_list,
                                                          uint32_t* __restrict__ dbg_nn, BDEM_STEP_PARAMS) {
  constexpr int NP = 64 / G, TW = PB / NP;   /* particles per team wave, team waves */
  __shared__ TeamScratch<G> scratch[TW];
  __shared__ float sums[6][PB];
  __shared__ int count[PB];
  const int block = xcd_block(blockIdx.x, gridDim.x);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const DevParams& P = BATCH ? Pp[__builtin_amdgcn_readfirstlane(tile_sim[block / (64 / PB)])] : *Pp;
  const uint32_t key_base = BATCH ? P.key_base : 0u;
  const uint2* const cells = cells_all + key_base;
  float* const tally = ENERGY ? P.tally : nullptr;   /* dissipation tallies (EnergyCalc) */
  const bool team = wave < TW;
  const int s = team ? wave * NP + lane / G : (lane < PB ? lane : 0);   /* the lane's particle in the block */
  const int i = block * PB + s;
  const bool in = i < n && (team || lane < PB);
  if (team) {
    TeamScratch<G>& ts = scratch[wave];
    const int sub = lane & (G - 1), lead = lane & ~(G - 1), ps = lane / G;
    /* velocity and spin are read after the scan, beside the partners': held
     * through it they would cost registers (six waves per SIMD: 80) */
    float4 pr = make_float4(0.f, 0.f, 0.f, 0.f);
    int packed = -8;
    uint32_t hwc = 0u;
    if (in) {
      pr = pos_in[i];
      packed = reinterpret_cast<const int*>(omg_in)[4 * (size_t)i + 3];
      if (hwc_in) hwc = hwc_in[i];
    }
    const int pid = packed >> 3;
    const bool alive = in && pid >= 0;
    const f3 p = xyz(pr);
    const float r = pr.w;
    const int nc = team_contacts<G, TEAM_CAND>(P, cells, pos_in, (uint32_t)n, i, p, r, alive, ts.cand[ps], [&](int j, int k) {
      if (k < CLIST) ts.clist[ps][k] = (uint32_t)j;
      if (dbg_list && k < LIST_STRIDE) dbg_list[(size_t)i * LIST_STRIDE + k] = (uint32_t)j;
    });
    float4 vm = make_float4(0.f, 0.f, 0.f, 0.f), ot = vm;
    if (alive) {
      vm = vel_in[i];
      ot = omg_in[i];
    }
    const f3 v = xyz(vm), w = xyz(ot);
    const float m = vm.w;
    const int ta = packed & 7;
    /* gravity first (DEM_Kernels_Compute.cuh:654), then the contacts in order */
    f3 F = alive ? cvt(P.gravity) * m : mk3(0.f, 0.f, 0.f);
    f3 T = mk3(0.f, 0.f, 0.f);
    const int nl = nc < CLIST ? nc : CLIST;
    const HistRec* hin = nullptr;
    int hin_cnt = 0;
    const bool slot = LAW != BDEM_LAW_REFERENCE && pid >= 0 && pid < hist_cap;
    if (slot) {
      hin = hr_in + (size_t)pid * HMAX;
      hin_cnt = min((int)(hwc & 0xFFFFu), HMAX);
    }
    for (int q = 0; __any((int)(q < nl)); q += G) {
      const int k = q + sub;
      f3 Fc = mk3(0.f, 0.f, 0.f), Tc = Fc;
      if (k < nl)
        contact_force<LAW>(P, (int)ts.clist[ps][k], pos_in, vel_in, omg_in, p, r, v, m, w, ta, hin, hin_cnt, k,
                           slot && k < HMAX ? hr_out + (size_t)pid * HMAX + k : nullptr, Fc, Tc, tally);
      ts.f[0][lane] = Fc.x; ts.f[1][lane] = Fc.y; ts.f[2][lane] = Fc.z;
      ts.f[3][lane] = Tc.x; ts.f[4][lane] = Tc.y; ts.f[5][lane] = Tc.z;
      __builtin_amdgcn_wave_barrier();
      const int here = min(nl - q, G);
      for (int c = 0; c < here; ++c) {
        const int l = lead + c;
        F = F + mk3(ts.f[0][l], ts.f[1][l], ts.f[2][l]);
        if (P.rotation) T = T + mk3(ts.f[3][l], ts.f[4][l], ts.f[5][l]);
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (sub == 0) {
      sums[0][s] = F.x; sums[1][s] = F.y; sums[2][s] = F.z;
      sums[3][s] = T.x; sums[4][s] = T.y; sums[5][s] = T.z;
      count[s] = nc;
      if (dbg_nn && in) dbg_nn[i] = (uint32_t)nc;
    }
    __syncthreads();
    return;
  }

  float4 pr = make_float4(0.f, 0.f, 0.f, 0.f), vm = pr, ot = pr;
  uint32_t hwc = 0u;
  if (in) {
    pr = pos_in[i]; vm = vel_in[i]; ot = omg_in[i];
    if (hwc_in) hwc = hwc_in[i];
  }
  const int pid = in ? packed_pid(ot.w) : -1;
  const int ta = packed_type(ot.w);
  const bool alive = in && pid >= 0;
  const f3 p = xyz(pr), v = xyz(vm), w = xyz(ot);
  const float r = pr.w, m = vm.w;
  WallOut wo;
  if (alive)
    walls_and_lifters<LAW>(P, i, pid, ta, p, r, v, w, m, hwc, wr_in, wr_out, hist_cap, wall_force, wo, tally);
  __syncthreads();
  uint32_t new_key = 0u;
  bool chg = false;
  if (in) {
    const int nc = count[s];
    f3 F = mk3(sums[0][s], sums[1][s], sums[2][s]), T = mk3(sums[3][s], sums[4][s], sums[5][s]);
    if (alive)
      contact_tail<LAW>(P, cells, pos_in, vel_in, omg_in, i, p, r, v, w, m, ta, pid, nc, hwc, hr_in, hr_out, hist_cap,
                        dbg_list, status, F, T, tally);
    const SkinArgs none{};
    float dmove = 0.0f;
    chg = particle_finish<LAW, ORIENT, false>(P, key_base, i, alive, pr, vm, ot, hwc, nc, F, T, wo, 0ull, none,
                                              quat_in, pos_out, vel_out, omg_out, quat_out, keys_out, sorted_keys,
                                              changed, hwc_out, hist_cap, wall_force, do_kill, status, kill_count,
                                              new_key, dmove);
  }
  append_changed(chg, new_key, i, n, sbuf, append, status);
}

/* Six waves per SIMD on 1,024 SIMDs hold 6,144 waves at once: five for 16
 * particles at 16 lanes each, five for 32 at 8, three for 32 at 4.  The last
 * shape is kept for two such rounds, up to TEAM_STEP_MAX (the figures above). */
constexpr int TEAM16_MAX = 6144 / 5 * 16, TEAM8_MAX = 6144 / 5 * 32;
static_assert(TEAM_STEP_MAX >= TEAM8_MAX, "team shapes in order");

template <int LAW, bool ORIENT, bool ENERGY, int G, int PB>
void launch_team_g(const DevParams* dP, const StepBuffers& b, const uint32_t* sk, int hp, int ap, bool do_kill,
                   bool want_wf, uint32_t* dl, uint32_t* dn, hipStream_t s) {
  hipLaunchKernelGGL((k_step_team<LAW, ORIENT, ENERGY, G, PB, false>), dim3((b.n + PB - 1) / PB), dim3(PB * G + 64), 0,
                     s, dP, nullptr, b.cells, dl, dn, b.n, b.pos_srt, b.vel_srt, b.omg_srt, b.quat_srt, b.pos_cur,
                     b.vel_cur, b.omg_cur, b.quat_cur, b.keys_new, sk, b.changed, b.sbuf, b.meta + META_APPEND + ap,
                     b.hwc_srt, b.hwc_cur, b.hrec[hp], b.hrec[hp ^ 1], b.wrec[hp], b.wrec[hp ^ 1], b.hist_cap,
                     want_wf ? b.wall_force : nullptr, do_kill ? 1 : 0, b.status, b.kill_count);
}

template <int LAW, bool ORIENT, bool ENERGY>
void launch_team_t(const DevParams* dP, const StepBuffers& b, const uint32_t* sk, int hp, int ap, bool do_kill,
                   bool want_wf, uint32_t* dl, uint32_t* dn, hipStream_t s) {
  if (b.n <= TEAM16_MAX) launch_team_g<LAW, ORIENT, ENERGY, 16, 16>(dP, b, sk, hp, ap, do_kill, want_wf, dl, dn, s);
  else if (b.n <= TEAM8_MAX) launch_team_g<LAW, ORIENT, ENERGY, 8, 32>(dP, b, sk, hp, ap, do_kill, want_wf, dl, dn, s);
  else launch_team_g<LAW, ORIENT, ENERGY, 4, 32>(dP, b, sk, hp, ap, do_kill, want_wf, dl, dn, s);
}

template <int LAW>
void launch_team_l(const DevParams* dP, const StepBuffers& b, const uint32_t* sk, bool orient, int hp, int ap,
                   bool do_kill, bool want_wf, bool energy, uint32_t* dl, uint32_t* dn, hipStream_t s) {
  if (orient) {
    if (energy) launch_team_t<LAW, true, true>(dP, b, sk, hp, ap, do_kill, want_wf, dl, dn, s);
    else launch_team_t<LAW, true, false>(dP, b, sk, hp, ap, do_kill, want_wf, dl, dn, s);
  } else {
    if (energy) launch_team_t<LAW, false, true>(dP, b, sk, hp, ap, do_kill, want_wf, dl, dn, s);
    else launch_team_t<LAW, false, false>(dP, b, sk, hp, ap, do_kill, want_wf, dl, dn, s);
  }
}

template <int LAW, int G, int PB>
void launch_team_batch_g(const BatchLaunch& L, const StepBuffers& b, const uint32_t* sk, int hp, int ap,
                         hipStream_t s) {
  hipLaunchKernelGGL((k_step_team<LAW, false, false, G, PB, true>), dim3(L.ntiles * (64 / PB)), dim3(PB * G + 64), 0, s,
                     L.params, L.tile_sim, L.cells, nullptr, nullptr, b.n, b.pos_srt, b.vel_srt, b.omg_srt, nullptr,
                     b.pos_cur, b.vel_cur, b.omg_cur, nullptr, b.keys_new, sk, b.changed, b.sbuf,
                     b.meta + META_APPEND + ap, b.hwc_srt, b.hwc_cur, b.hrec[hp], b.hrec[hp ^ 1], b.wrec[hp],
                     b.wrec[hp ^ 1], b.hist_cap, nullptr, 0, b.status, b.kill_count);
}

template <int LAW>
void launch_team_batch_l(const BatchLaunch& L, const StepBuffers& b, const uint32_t* sk, int hp, int ap,
                         hipStream_t s) {
  if (b.n <= TEAM16_MAX) launch_team_batch_g<LAW, 16, 16>(L, b, sk, hp, ap, s);
  else if (b.n <= TEAM8_MAX) launch_team_batch_g<LAW, 8, 32>(L, b, sk, hp, ap, s);
  else launch_team_batch_g<LAW, 4, 32>(L, b, sk, hp, ap, s);
}

}  // namespace

void launch_step_team_batch(const BatchLaunch& L, const StepBuffers& b, const uint32_t* sk, int hp, int ap,
                            hipStream_t s) {
  if (L.law == BDEM_LAW_REFERENCE) launch_team_batch_l<BDEM_LAW_REFERENCE>(L, b, sk, hp, ap, s);
  else if (L.law == BDEM_LAW_LSD_COULOMB) launch_team_batch_l<BDEM_LAW_LSD_COULOMB>(L, b, sk, hp, ap, s);
  else launch_team_batch_l<BDEM_LAW_HERTZ_MINDLIN>(L, b, sk, hp, ap, s);
}

void launch_step_team(const DevParams* dP, const StepBuffers& b, const uint32_t* sk, int law, bool orient, int hp,
                      int ap, bool do_kill, bool want_wf, bool energy, uint32_t* dl, uint32_t* dn, hipStream_t s) {
  if (law == BDEM_LAW_REFERENCE)
    launch_team_l<BDEM_LAW_REFERENCE>(dP, b, sk, orient, hp, ap, do_kill, want_wf, energy, dl, dn, s);
  else if (law == BDEM_LAW_LSD_COULOMB)
    launch_team_l<BDEM_LAW_LSD_COULOMB>(dP, b, sk, orient, hp, ap, do_kill, want_wf, energy, dl, dn, s);
  else
    launch_team_l<BDEM_LAW_HERTZ_MINDLIN>(dP, b, sk, orient, hp, ap, do_kill, want_wf, energy, dl, dn, s);
}

}  // namespace bdem
