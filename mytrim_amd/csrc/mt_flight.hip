// One TrimBase::trim() call (trim.C:35-425) on the device, driven by the
// caller's uniform stream in the reference's draw order: r1 at flight start,
// r2 and hh per collision, then the unit-ball rejection loop for the
// azimuth (trim.C:71, 143, 147, 322-333).  Every collision is logged as an
// mt_event so the host can replay the virtual hooks (trim.h:72-84) in order.
// One block runs the flight; this is the compatibility path for callers that
// drive trim() one ion at a time.
#include <hip/hip_runtime.h>

#include "mt_flight.h"
#include "mt_geometry.h"
#include "mt_physics.h"
#include "mt_tables.h"
#include "mytrim_gpu.h"

namespace mt {

enum { kFlightDone = 0, kFlightNeedDraws = 1, kFlightNeedEvents = 2, kFlightRunaway = 3, kFlightNonFinite = 4 };

// What one slot publishes (LDS, two of them in turn)
struct FlightSlot {
  double ls, den, ct, st;    // wave 0: path, energy transfer, deflection,
  double Edisp, Elbind, my;  // and the target element's constants
  double se;                 // wave 1: electronic stopping
  double rd[3], r2, hh;      // wave 2: point in the unit ball, the next collision's draws
  double dir[3], ndir[3];    // wave 3: flight direction, as deflected and normalised
  double rr2, rhh;           // wave 3: the next collision's draws after a redraw
  long long iu, riu;         // draws used by this collision, after a redraw
  int nn, Z, need, redo;     // target element; draws ran out; wave 3 drew again (2: they ran out)
};

// bytes at the start of the tables that are not copied to LDS
constexpr int kFlightSkip = int(sizeof(TableHeader) & ~size_t(15));
static_assert(2 * sizeof(FlightSlot) <= kFlightSkip, "slots within the header's place");

// A collision whose direction and event are still to be worked out
struct FlightPending {
  double E, p1E, den, dee, ls, rE, ct, st, my;
  double at[3], pos[3], rd[3];
  int k, nn, state, fate, vac, mtag;
  int event;  // index of the event, -1: the buffer is full
};

// The flight is one chain of collisions, each some thousand dependent
// instructions on a lane, so it is latency that bounds it.  Four waves of a block
// (one per SIMD) share a collision, with one barrier per collision:
//   wave 0  maximum impact parameter, free path, scattering (the energy chain)
//   wave 1  electronic stopping at the same energy
//   wave 2  the draws: 64 uniforms in one load, the rejection loop of
//           trim.C:322-333 by lane (a triple each), and the next collision's r2, hh
//   wave 3  the previous collision's deflection, new direction, recoil direction
//           and event: an ion moves along the direction it came with
//           (trim.C:313-318), so they are not needed before this one's end
// Every wave then merges the results into its own copy of the ion, so nothing is
// handed back.  A draw parallel to the flight direction (a zero normal) is found
// by wave 3 only; it draws again as the reference does and the slot is repeated
// with the draws that follow.
// A collision took 15 000 cycles on one lane with each uniform loaded where it
// was drawn, and takes 7500 (the call of a 500 keV Cu flight: 3.4 -> 1.8 ms): wave 0's
// 5500, of which the library's power and the divisions are a third, and 1900 of
// merging, mostly LDS latency.  Waves 1, 2 and 3 need 2400, 1500 and 3900.
template <int POT>
__global__ void __launch_bounds__(256) flight_kernel(FlightParams P) {
  // the block copies the ion's tables to LDS; each collision then reads its
  // constants there (about a hundred cycles) instead of from L2.  The header
  // stays behind: the slots take no more than its place, so that the tables
  // alone decide which targets fit the LDS
  extern __shared__ __align__(16) unsigned char lds_tables[];
  __shared__ FlightSlot slots[2];
  const TableHeader* H = (const TableHeader*)P.tables;
  {
    const uint4* src = (const uint4*)(P.tables + kFlightSkip);
    uint4* dst = (uint4*)lds_tables;
    for (int i = threadIdx.x; i < (P.table_bytes - kFlightSkip) / 16; i += blockDim.x) dst[i] = src[i];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  TableView T;
  T.n_species = H->n_species;
  T.n_mat = H->n_mat;
  T.n_el = H->n_el;
  T.potential = H->potential;
  T.mat = (const MatConst*)(lds_tables + (H->off_mat - kFlightSkip));
  T.el = (const ElemConst*)(lds_tables + (H->off_el - kFlightSkip));
  T.stop = (const StopConst*)(lds_tables + (H->off_stop - kFlightSkip));
  const Geometry& G = P.geo;
  // arguments used in every collision, held in vector registers (there are
  // plenty): read from the argument segment one by one they cost a merge some
  // 1500 cycles
  double tau = P.tau, invscale = P.invscale, cw = P.cw, w[3] = {G.w[0], G.w[1], G.w[2]};
  int cut[3] = {G.bc[0] == 2, G.bc[1] == 2, G.bc[2] == 2}, max_ev = P.max_ev;
  asm volatile("" : "+v"(tau), "+v"(invscale), "+v"(cw), "+v"(w[0]), "+v"(w[1]), "+v"(w[2]));
  asm volatile("" : "+v"(cut[0]), "+v"(cut[1]), "+v"(cut[2]), "+v"(max_ev));

  mt_ion ion = *P.ion;
  const int sp = 0;  // the flight's ion is species 0 of its table
  ion.state = 0;
  int status = kFlightDone;
  auto u_at = [&](long long i) { return P.u[i < P.n_u ? i : P.n_u - 1]; };
  const double r1 = u_at(0);
  long long iu = 1;  // draws used
  double r2 = u_at(1), hh0 = u_at(2);
  int nev = 0, ic = 0, mtag = -1;
  auto lookup = [&]() {
    const double pos[3] = {ion.pos[0], ion.pos[1], ion.pos[2]};
    return (G.kind == 0 || G.kind >= 3) ? lookup_material<0>(G, pos, mtag)
           : G.kind == 1 ? lookup_material<1>(G, pos, mtag)
                         : lookup_material<2>(G, pos, mtag);
  };
  auto norm_dir = [](const double d[3], double n[3]) {
    const double inv = 1.0 / sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    for (int i = 0; i < 3; ++i) n[i] = d[i] * inv;
  };
  // wave 3: direction as deflected and as normalised for the next collision
  double dir[3] = {ion.dir[0], ion.dir[1], ion.dir[2]}, ndir[3];
  norm_dir(dir, ndir);
  FlightPending C;
  bool pending = false;
  // wave 3: deflection and event of C (draws used up to iu_c), into slot `s`
  auto deflect = [&](FlightSlot& s, long long iu_c) {
    double perp[3], norm;
    int guard = 0, redo = 0;
    double rd[3] = {C.rd[0], C.rd[1], C.rd[2]};
    while (true) {
      for (int i = 0; i < 3; ++i)
        perp[i] = ndir[(i + 1) % 3] * rd[(i + 2) % 3] - ndir[(i + 2) % 3] * rd[(i + 1) % 3];
      norm = sqrt(perp[0] * perp[0] + perp[1] * perp[1] + perp[2] * perp[2]);
      if (!(norm == 0.0 && ++guard < 1000)) break;
      redo = 1;
      do {
        for (int i = 0; i < 3; ++i) rd[i] = 2.0 * u_at(iu_c + i) - 1.0;
        iu_c += 3;
      } while (rd[0] * rd[0] + rd[1] * rd[1] + rd[2] * rd[2] > 1.0 && iu_c <= P.n_u);
      if (iu_c > P.n_u) {
        redo = 2;
        break;
      }
    }
    if (redo != 2) {
      for (int i = 0; i < 3; ++i) perp[i] /= norm;
      const double p1 = sqrt(2.0 * ion.m * C.p1E);
      const double p2 = sqrt(2.0 * ion.m * C.E);
      double rdir[3];
      const double psi = atan2(C.st, C.ct + C.my);
      const double cpsi = cos(psi), spsi = sin(psi);
      for (int i = 0; i < 3; ++i) {
        dir[i] = fma(perp[i], spsi, ndir[i] * cpsi);
        rdir[i] = fma(ndir[i], p1, -(dir[i] * p2));
      }
      norm_dir(dir, ndir);
      if (lane == 0 && C.event >= 0) {
        mt_event& event = P.ev[C.event];
        event.pka_E = C.E;
        for (int i = 0; i < 3; ++i) {
          event.pka_pos[i] = C.pos[i];
          event.pka_dir[i] = dir[i];
          event.rec_pos[i] = C.at[i];
          event.rec_dir[i] = rdir[i];
        }
        event.ls = C.ls;
        event.dee = C.dee;
        event.den = C.den;
        event.rec_E = C.rE;
        event.material = C.k;
        event.element = C.nn;
        event.pka_state = C.state;
        event.fate = C.fate;
        event.vacancy = C.vac;
        event.mat_tag = C.mtag;
      }
    }
    if (lane == 0) {
      for (int i = 0; i < 3; ++i) {
        s.dir[i] = dir[i];
        s.ndir[i] = ndir[i];
      }
      s.redo = redo;
      s.riu = iu_c;
      s.rr2 = u_at(iu_c);
      s.rhh = u_at(iu_c + 1);
    }
  };

  int k = lookup();
  const bool solid = G.kind == 0;  // one material: no lookup in the loop
  for (int par = 0; k >= 0; par ^= 1) {
    FlightSlot& s = slots[par];
    const MatConst& mc = T.mat[sp * T.n_mat + k];
    const int eb = sp * T.n_el + mc.el_begin;
    if (wave == 0) {
      double eps = ion.E * mc.f;
      const double eeg = sqrt(eps * mc.epsdg);
      const double pmax = mc.a / (eeg + sqrt(eeg) + 0.125 * pow(eeg, 0.1));
      double ls = 1.0 / (M_PI * (pmax * pmax) * mc.arho);
      if (ic == 0) ls = r1 * mn(ls, cw);
      const double p = pmax * sqrt(r2);
      double hh = hh0;
      int nn = 0;
      for (; nn < mc.n_el; ++nn) {
        hh -= T.el[eb + nn].t;
        if (hh <= 0.0) break;
      }
      if (nn >= mc.n_el) nn = mc.n_el - 1;
      const ElemConst& ec = T.el[eb + nn];
      eps = ec.fi * ion.E;
      const double b = p / ec.ai;
      double s2, ct, st;
      int it;
      scatter<double, POT, true>(eps, b, m_log(eps), s2, ct, st, it);
      if (lane == 0) {
        s.ls = ls;
        s.den = ec.ec * s2 * ion.E;
        s.ct = ct;
        s.st = st;
        s.Edisp = ec.Edisp;
        s.Elbind = ec.Elbind;
        s.my = ec.my;
        s.nn = nn;
        s.Z = ec.Z;
      }
    } else if (wave == 1) {
      const double se = getrstop<double>(T, sp, k, ion.E);
      if (lane == 0) s.se = se;
    } else if (wave == 2) {
      // uniforms [at, at + 64): 20 triples, and what follows each; one round
      // accepts a triple but for a 4e-7 chance
      long long at = iu + 2;
      int need = at > P.n_u ? 1 : 0;
      double rd[3], n2 = 0.0, nh = 0.0;
      for (bool found = false; !found;) {
        const double v = u_at(at + lane);
        for (int i = 0; i < 3; ++i) rd[i] = 2.0 * __shfl(v, min(3 * lane + i, 63)) - 1.0;
        const uint64_t ok = __ballot(lane < 20 && !(rd[0] * rd[0] + rd[1] * rd[1] + rd[2] * rd[2] > 1.0));
        found = ok != 0ull;
        const int j = found ? __ffsll((long long)ok) - 1 : 19;
        for (int i = 0; i < 3; ++i) rd[i] = __shfl(rd[i], j);
        n2 = __shfl(v, 3 * j + 3);
        nh = __shfl(v, 3 * j + 4);
        at += 3 * j + 3;
        if (at > P.n_u) need = 1;
        if (need) found = true;
      }
      if (lane == 0) {
        for (int i = 0; i < 3; ++i) s.rd[i] = rd[i];
        s.r2 = n2;
        s.hh = nh;
        s.iu = at;
        s.need = need;
      }
    } else if (pending) {
      deflect(s, iu);
    } else if (lane == 0) {
      for (int i = 0; i < 3; ++i) {
        s.dir[i] = dir[i];
        s.ndir[i] = ndir[i];
      }
      s.redo = 0;
    }
    __syncthreads();
    // merge (trim.C:275-352); one batch of reads, few branches: every wave
    // does this between two collisions
    const FlightSlot r = s;
    pending = false;
    for (int i = 0; i < 3; ++i) ion.dir[i] = r.dir[i];
    if (r.redo | r.need) {
      if (r.redo) {  // the previous collision drew again: this one starts after that
        iu = r.riu;
        r2 = r.rr2;
        hh0 = r.rhh;
        if (r.redo != 2) continue;
        --nev;
      }
      status = kFlightNeedDraws;
      break;
    }
    ++ic;
    double dee = r.ls * r.se;
    double den = r.den;
    if (dee > ion.E) dee = ion.E;
    ion.E -= dee;
    const double p1E = ion.E;
    if (den > ion.E) den = ion.E;
    ion.E -= den;
    const double at[3] = {ion.pos[0], ion.pos[1], ion.pos[2]};
    for (int i = 0; i < 3; ++i) ion.pos[i] += r.ndir[i] * (r.ls - tau) * invscale;
    const double rE = den - r.Elbind;
    int lost = 0;
    for (int i = 0; i < 3; ++i) lost |= cut[i] & ((ion.pos[i] > w[i]) | (ion.pos[i] < 0.0));
    const int above = rE > r.Edisp - r.Elbind, moves = ion.E > r.Edisp;
    const int fate = lost ? 2 : above;
    const int vac = (lost == 0) & above & moves;
    ion.state = lost ? 4 : above ? (moves ? 0 : ion.Z == r.Z ? 1 : 2) : ion.E < ion.Ef ? 3 : 0;
    iu = r.iu;
    r2 = r.r2;
    hh0 = r.hh;
    if (nev >= max_ev) status = kFlightNeedEvents;
    const int at_event = status == kFlightDone ? nev : -1;
    if (at_event >= 0) ++nev;
    if (wave == 3) {
      C.E = ion.E;
      C.p1E = p1E;
      C.den = den;
      C.dee = dee;
      C.ls = r.ls;
      C.rE = rE;
      C.ct = r.ct;
      C.st = r.st;
      C.my = r.my;
      for (int i = 0; i < 3; ++i) {
        C.at[i] = at[i];
        C.pos[i] = ion.pos[i];
        C.rd[i] = r.rd[i];
      }
      C.k = k;
      C.nn = r.nn;
      C.state = ion.state;
      C.fate = fate;
      C.vac = vac;
      C.mtag = mtag;
    }
    C.event = at_event;
    pending = true;
    // a NaN or infinite energy or position would fail every threshold and
    // run to the collision cap (x - x is 0 exactly for finite x)
    const int wild = (!(ion.E - ion.E == 0.0)) | (!(ion.pos[0] - ion.pos[0] == 0.0));
    if (status == kFlightDone) status = ic >= 100000000 ? kFlightRunaway : wild ? kFlightNonFinite : kFlightDone;
    if ((status != kFlightDone) | (ion.state != 0)) break;
    if (!solid) k = lookup();  // vacuum: state stays MOVING (trim.C:80-82)
  }
  if (pending) {  // the last collision's direction and event
    FlightSlot& s = slots[0];
    __syncthreads();
    if (wave == 3) deflect(s, iu);
    __syncthreads();
    for (int i = 0; i < 3; ++i) ion.dir[i] = s.dir[i];
    if (s.redo) iu = s.riu;
    if (s.redo == 2) {
      if (C.event >= 0) --nev;
      status = kFlightNeedDraws;
    }
  }
  if (threadIdx.x != 0) return;
  if (status == kFlightNeedDraws) iu = P.n_u;
  if (status == kFlightDone) *P.ion_out = ion;
  P.n_used[0] = iu;
  P.n_used[1] = nev;
  P.n_used[2] = status;
}

hipError_t flight_launch(const FlightParams& P, int potential, hipStream_t stream) {
  const unsigned lds = unsigned(P.table_bytes - kFlightSkip);
  if (potential == 1)
    hipLaunchKernelGGL(flight_kernel<1>, dim3(1), dim3(256), lds, stream, P);
  else if (potential == 2)
    hipLaunchKernelGGL(flight_kernel<2>, dim3(1), dim3(256), lds, stream, P);
  else
    hipLaunchKernelGGL(flight_kernel<0>, dim3(1), dim3(256), lds, stream, P);
  return hipGetLastError();
}

}  // namespace mt
