// Generic path: the project's own model.cuh, compiled into the library as in
// the reference (src/Makefile:44-45 builds gpu_mcmc.cu with -I$(MODELDIR)).
//
// model() keeps the reference contract (ccalcmodel.h): per datum, per pass,
// results in mc->datm[imd], return 0/1/2/-1.  The kernels here fuse what the
// reference splits into calc_chi2_terms (src/gpu_mcmc.cu:273-325),
// calc_chi2 (:331-350), gen_proposal (:361-411), spmp_mcmc (:426-474) and
// adjust_steps (:480-526).  As in the reference, where the data of one pass
// are threads of one launch (:754), the data of a pass run side by side: a
// chain has 1 to 256 lanes, datum id on lane id % lanes, and between two
// passes its lanes wait for each other, so pass p+1 may read what pass p
// stored in datm.
//
//   k_iter_user  fits with few data: a sequence's whole ladder in one wave,
//                many iterations with their replica exchange in one launch,
//                the random numbers from a second wave
//   k_step_user  the others: one iteration a launch, up to 4 waves a chain
//                (the exchange has a launch of its own, k_exchange)
#include <hip/hip_runtime.h>
#include "mhre_device.h"
#include "fitdesc.h"
#include "engine.h"
#include "ccalcmodel.h"
#include "model.cuh"

#ifndef MHRE_MODEL_NAME
#define MHRE_MODEL_NAME "model.cuh"
#endif

namespace mhre {

// Orders the global and LDS accesses of a chain's lanes: what one stored
// before is read by the others afterwards.  Waves = 1: the lanes share a wave
// (its memory operations keep their order); else they are a work-group.
template <int Waves>
__device__ inline void chain_fence() {
  if (Waves == 1) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  } else {
    __syncthreads();
  }
}

// The lanes of one chain.
template <int Waves>
struct ChainLanes {
  int n;          // lanes of the chain (a power of two; 64 Waves for Waves > 1)
  int j;          // this lane's place among them
  double* xs;     // Waves > 1: work-group LDS, 2 Waves doubles
  int flip;

  // Sum over the chain's lanes, the same on each of them.  Waves > 1: the waves'
  // sums meet in xs, whose two halves take turns, so that one barrier does.
  __device__ double sum(double v) {
    if (Waves == 1) {
      if (n == 64) return wave_sum(v);
      for (int m = n >> 1; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
      return v;
    }
    v = wave_sum(v);
    double* x = xs + flip * Waves;
    flip ^= 1;
    if (lane_id() == 0) x[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = x[0];
#pragma unroll
    for (int w = 1; w < Waves; ++w) s += x[w];
    return s;
  }
};

// The fit's CCalcModel as a local object.  Its fields come from scalar loads
// and its pointers are known to be global, so once model() is inlined no
// field is read again per datum and its arrays take global instead of flat
// accesses.
__device__ inline CCalcModel user_model_args(const FitDesc& f) {
  const CONSTANT CCalcModel* c = wave_const(f.mc);
  CCalcModel m;
  m.imodel = c->imodel; m.ncoor = c->ncoor; m.ndat = c->ndat; m.nicoor = c->nicoor; m.nidat = c->nidat;
  m.ndatm = c->ndatm; m.nptot = c->nptot; m.nbeta = c->nbeta; m.nseq = c->nseq; m.nchi2m = c->nchi2m;
  m.coor = (float*)gptr(c->coor); m.dat = (float*)gptr(c->dat); m.std2r = (float*)gptr(c->std2r);
  m.icoor = (int*)gptr(c->icoor); m.idat = (int*)gptr(c->idat);
  m.datm = (float*)gptr(c->datm); m.chi2m = (float*)gptr(c->chi2m);
  m.pcur = (float*)gptr(c->pcur); m.flag = (int*)gptr(c->flag); m.chi2c = (float*)gptr(c->chi2c);
  return m;
}

// One pass of datum id of chain ch: true and the new chi^2 term, or false if
// the pass gives this datum no result.
__device__ inline bool user_term(const FitDesc& f, CCalcModel* mc, int ch, int id, int ipass, float* term, int* err) {
  const int imd = ch * f.ndat + id;
  const int iret = model(mc, id, ch * f.nptot, imd, ipass);
  if (iret == 0) return false;
  if (iret < 0) { *err = iret; return false; }
  // through mc's pointers, as model() stored it: no load has to wait for the store
  float dif = mc->dat[id] - mc->datm[imd];
  if (iret == 2) dif = atan2f(sinf(dif), cosf(dif));
  *term = (dif * dif) * mc->std2r[id];
  mc->chi2m[imd] = *term;
  return true;
}

// chi^2 of chain ch from the user's model (all passes), its terms in chi2m:
// the sum over all ndat terms (the reference sums every chi2m entry of the
// chain, including entries no pass rewrote), in float64.  OneDatum: the chain has
// at most one datum a lane, whose chi2m entry the lane keeps in term, so that
// the sum needs no load behind the store.
template <int Waves, bool OneDatum>
__device__ inline double user_chi2(const FitDesc& f, CCalcModel* mc, ChainLanes<Waves>& cl, int ch, float* term,
                                   int* err) {
  const int ndat = f.ndat;
  for (int ipass = 0; ipass < f.npass; ++ipass) {
    if (ipass) chain_fence<Waves>();
    if (OneDatum) {
      if (cl.j < ndat) user_term(f, mc, ch, cl.j, ipass, term, err);
    } else {
      float t;
      for (int id = cl.j; id < ndat; id += cl.n) user_term(f, mc, ch, id, ipass, &t, err);
    }
  }
  double s = 0.0;
  if (OneDatum) {
    if (cl.j < ndat) s = (double)*term;
  } else {
    const GLOBAL float* c = gptr(f.chi2m) + (size_t)ch * ndat;
    for (int id = cl.j; id < ndat; id += cl.n) s += (double)c[id];
  }
  return cl.sum(s);
}

// Model data and chi^2 of every chain of the list, one wave per chain.
__global__ void __launch_bounds__(64) k_eval_user(const FitDesc* fits, const WorkItem* work, int nwork,
                                                  int model_only, int respect_flag) {
  const WorkItem w = work[blockIdx.x];
  const FitDesc& f = wave_fit(fits, w.fit);
  const int ch = __builtin_amdgcn_readfirstlane(w.idx);
  CCalcModel mc = user_model_args(f);
  ChainLanes<1> cl{64, lane_id(), nullptr, 0};
  int err = 0;
  if (model_only) {
    // calc_model (src/gpu_mcmc.cu:633-658): pass 0 only, no chi^2
    for (int id = cl.j; id < f.ndat; id += 64) {
      const int iret = model(&mc, id, ch * f.nptot, ch * f.ndat + id, 0);
      if (iret < 0) err = iret;
    }
  } else {
    double s;
    if (respect_flag && f.flag[ch] == 0) {
      s = 0.0;
      for (int id = cl.j; id < f.ndat; id += 64) s += (double)f.chi2m[(size_t)ch * f.ndat + id];
      s = cl.sum(s);
    } else {
      float t;
      s = user_chi2<1, false>(f, &mc, cl, ch, &t, &err);
    }
    if (cl.j == 0) f.chi2c[ch] = (float)s;
  }
  if (err && f.errflag) atomicExch(f.errflag, err);
}

// The random numbers of one iteration of a chain, P entries each.
struct UserDraws {
  double *z, *lu;        // Gaussian steps, log u
  int* k;                // coordinate picks
};
// A chain's state in LDS for the launch, one copy per wave (the waves of a
// chain compute the same, so no wave waits for another's bookkeeping): P
// entries of each array, the draws of two iterations, then two rows of N
// parameters (k_iter_user's exchange writes the one that the iteration did not
// use).
struct UserSlot {
  UserDraws d[2];
  float* stp;
  int *cnt, *nac, *sh;
  uint32_t* hw;          // the history word holding entry cnt % nadj ...
  int* hwi;              // ... and its index
  float* row;
};
__device__ inline UserSlot user_slot(char* lds, int P) {
  UserSlot u;
  double* z = reinterpret_cast<double*>(lds);
  int* k = reinterpret_cast<int*>(z + 4 * P);
  u.d[0] = UserDraws{z, z + P, k};
  u.d[1] = UserDraws{z + 2 * P, z + 3 * P, k + P};
  u.stp = reinterpret_cast<float*>(k + 2 * P);
  u.cnt = reinterpret_cast<int*>(u.stp + P);
  u.nac = u.cnt + P;
  u.sh = u.nac + P;
  u.hw = reinterpret_cast<uint32_t*>(u.sh + P);
  u.hwi = reinterpret_cast<int*>(u.hw + P);
  u.row = reinterpret_cast<float*>(u.hwi + P);
  return u;
}

// Per varied parameter k: ivar[k], its pdescr (as bits), pmint and pmaxt, in the
// wave's LDS: a chain's lanes read them one after the other, each proposal anew.
__device__ inline void user_params(const FitDesc& f, float4* par) {
  const int k = lane_id();
  if (k < f.nprm) {
    const int t = gptr(f.ivar)[k];
    par[k] = make_float4(__int_as_float(t), __int_as_float(gptr(f.pdescr)[t]), gptr(f.pmint)[t], gptr(f.pmaxt)[t]);
  }
}

// Place and number of a wave's lanes of a chain, for work that every wave of
// the chain does by itself.
template <int Waves>
__device__ inline int own_j(const ChainLanes<Waves>& cl) { return Waves == 1 ? cl.j : lane_id(); }
template <int Waves>
__device__ inline int own_n(const ChainLanes<Waves>& cl) { return Waves == 1 ? cl.n : 64; }

// The wave's LDS copy of the chain's state; hist: the launch has burn-in
// iterations.
template <int Waves>
__device__ inline void user_load(const FitDesc& f, const ChainLanes<Waves>& cl, int ch, const UserSlot& u, bool hist) {
  const int C = f.nchain, P = f.nprm, N = f.nptot;
  for (int k = own_j(cl); k < P; k += own_n(cl)) {
    const size_t pk = (size_t)k * C + ch;
    u.stp[k] = gptr(f.pstp)[pk];
    u.nac[k] = gptr(f.n_acpt)[pk];
    const int cnt = gptr(f.n_cnt)[pk];
    u.cnt[k] = cnt;
    if (hist) {
      const int wi = (cnt % f.nadj) >> 5;
      u.sh[k] = gptr(f.sumh)[pk];
      u.hwi[k] = wi;
      u.hw[k] = gptr(f.hbits)[((size_t)ch * f.hwords + wi) * P + k];
    }
  }
  for (int i = own_j(cl); i < N; i += own_n(cl)) u.row[i] = gptr(f.pcur)[(size_t)ch * N + i];
}

template <int Waves>
__device__ inline void user_store(const FitDesc& f, const ChainLanes<Waves>& cl, int ch, const UserSlot& u, bool hist) {
  const int C = f.nchain, P = f.nprm;
  for (int k = cl.j; k < P; k += cl.n) {
    const size_t pk = (size_t)k * C + ch;
    gptr(f.n_acpt)[pk] = u.nac[k];
    if (hist) {
      gptr(f.pstp)[pk] = u.stp[k];
      gptr(f.n_cnt)[pk] = u.cnt[k];
      gptr(f.sumh)[pk] = u.sh[k];
      gptr(f.hbits)[((size_t)ch * f.hwords + u.hwi[k]) * P + k] = u.hw[k];
    }
  }
}

// What the chain's last proposal leaves in flag, ptent and ptentn.
struct LastProposal {
  int flag, t;
  float told;
};

// The draws of iteration it, substep s on the chain's lane s (modulo its lanes).
template <int Waves>
__device__ inline void user_draw(const FitDesc& f, const ChainLanes<Waves>& cl, int ch, int it, const UserDraws& d) {
  const int P = f.nprm;
  for (int s = own_j(cl); s < P; s += own_n(cl)) {
    const U4 r = philox4x32_10((uint32_t)ch, (uint32_t)it, (uint32_t)s, 0u, f.key0, f.key1);
    d.k[s] = pick_with_retry(r.x, P, (uint32_t)ch, (uint32_t)it, (uint32_t)s, 0u, f.key0, f.key1);
    d.z[s] = normal64(r.y, r.z);
    d.lu[s] = log((double)u01(r.w));
  }
}

// The chain's nprm proposals of iteration it on the state in u and chi2c, with its draws d;
// returns the chi^2 evaluations performed.  Every lane of the chain follows
// the same decisions; the data of a chi^2 are split among them.  row: the
// current half of u.row.
template <int Waves, bool OneDatum>
__device__ unsigned user_substeps(const FitDesc& f, CCalcModel* mc, ChainLanes<Waves>& cl, int ch, int it,
                                  const TraceBuf& tr, const UserSlot& u, const UserDraws& d, const float4* par,
                                  double beta, float* row, float& chi2c, float* term, LastProposal& last, int* err) {
  const int C = f.nchain, P = f.nprm, N = f.nptot;
  const bool burn = it < f.nburn;
  const int nadj = f.nadj;
  const float rnadj = 1.0f / (float)nadj;
  GLOBAL float* prow = gptr(f.pcur) + (size_t)ch * N;
  unsigned nev = 0;
  for (int s = 0; s < P; ++s) {
    const int k = d.k[s];
    const float4 pk = par[k];
    const int t = __float_as_int(pk.x);
    const float old = row[t], sd = u.stp[k];
    double pd = (double)old + (double)sd * d.z[s];
    if (__float_as_int(pk.y) == 2) pd = pd - 6.283185307179586 * rint(pd / 6.283185307179586);
    const float pn = (float)pd;
    const bool inprior = !(pn < pk.z || pn > pk.w);
    wave_sync_lds();   // every lane has read its row and step size
    int acc = 0;
    double c2 = 0.0;
    if (inprior) {
      if (cl.j == 0) prow[t] = pn;
      chain_fence<Waves>();   // the chain's lanes read the proposal through mc->pcur
      c2 = user_chi2<Waves, OneDatum>(f, mc, cl, ch, term, err);
      ++nev;
      const double x = -0.5 * beta * (c2 - (double)chi2c);
      if (d.lu[s] <= x) {
        acc = 1;
        chi2c = (float)c2;
        if (own_j(cl) == 0) {
          u.nac[k] += 1;
          row[t] = pn;
        }
      } else if (cl.j == 0) {
        prow[t] = old;   // every lane has used the rejected value: the sum took its term
      }
    }
    last = LastProposal{acc, t, old};
    if (tr.dec && it >= tr.it0 && it < tr.it0 + tr.nit && cl.j == 0) {
      const size_t ti = (size_t)f.tr_dec + ((size_t)(it - tr.it0) * P + s) * C + ch;
      tr.dec[ti] = k | ((inprior ? 1 : 0) << 8) | (acc << 9);
      tr.chi2[ti] = inprior ? (float)c2 : 0.0f;
    }
    if (burn) {
      // history entry cnt % nadj: the oldest one, replaced by this outcome
      // (the division-free forms of mhre_device.h give the reference's bits)
      const int cnt = u.cnt[k], wi = u.hwi[k];
      const int w2 = mod_small(cnt + 1, nadj, rnadj) >> 5;
      if (own_j(cl) == 0) {
        const uint32_t bit = 1u << (mod_small(cnt, nadj, rnadj) & 31);
        const uint32_t word = u.hw[k];
        const int sh = u.sh[k] + acc - ((word & bit) ? 1 : 0);
        u.hw[k] = acc ? (word | bit) : (word & ~bit);
        u.sh[k] = sh;
        const int den = cnt < nadj ? cnt : nadj;
        u.stp[k] = rate_below(sh, den, f.adapt_mid, f.adapt_tie) ? step_shrink(sd) : step_grow(sd);
        u.cnt[k] = cnt + 1;
      }
      if (w2 != wi) {
        // the word is full: on to the next one, which an earlier proposal of
        // this launch may have written (short rings), hence the fences
        GLOBAL uint32_t* h = gptr(f.hbits) + (size_t)ch * f.hwords * P + k;
        chain_fence<Waves>();
        if (cl.j == 0) h[(size_t)wi * P] = u.hw[k];
        chain_fence<Waves>();
        if (own_j(cl) == 0) {
          u.hw[k] = h[(size_t)w2 * P];
          u.hwi[k] = w2;
        }
      }
    }
    wave_sync_lds();
  }
  return nev;
}

// One iteration of every chain of the list.  Waves = 1: lanes lanes a chain, so
// 64 / lanes chains a wave (the list is padded to whole waves); Waves > 1: one
// chain a work-group of Waves waves.  slot_bytes: LDS of one chain's state
// (user_slot at maxp parameters).
template <int Waves>
__global__ void __launch_bounds__(64 * Waves) k_step_user(const FitDesc* fits, const WorkItem* work, int nwork,
                                                       RunClock* clk, TraceBuf tr, int it_off, int lanes,
                                                       int slot_bytes) {
  extern __shared__ __align__(16) char lds[];
  __shared__ double xs[2 * Waves];
  __shared__ float4 par[Waves][MAXP];
  const int lane = lane_id();
  const int per = Waves == 1 ? 64 / lanes : 1;
  const int c = Waves == 1 ? lane / lanes : 0;
  const WorkItem w = work[blockIdx.x * per + c];
  const FitDesc& f = wave_fit(fits, w.fit);
  pass_clock(clk);
  const int it = __builtin_amdgcn_readfirstlane(load_clock(clk, it_off));
  if (it >= f.nburn + f.niter) return;
  const int ch = w.idx;
  const bool live = ch >= 0;   // padding lanes only take part in the counting
  ChainLanes<Waves> cl{Waves == 1 ? lanes : 64 * Waves, Waves == 1 ? lane & (lanes - 1) : (int)threadIdx.x, xs, 0};
  unsigned nev = 0;
  const int wid = Waves == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  user_params(f, par[wid]);
  if (live) {
    const UserSlot u = user_slot(lds + (size_t)(wid * per + c) * slot_bytes, f.nprm);
    const bool hist = it < f.nburn;
    CCalcModel mc = user_model_args(f);
    float chi2c = gptr(f.chi2c)[ch], term;
    LastProposal last{0, 0, 0.0f};
    int err = 0;
    const double beta = (double)gptr(f.beta)[ch / f.nseq];
    user_load(f, cl, ch, u, hist);
    user_draw(f, cl, ch, it, u.d[0]);
    wave_sync_lds();
    nev = user_substeps<Waves, false>(f, &mc, cl, ch, it, tr, u, u.d[0], par[wid], beta, u.row, chi2c, &term, last,
                                      &err);
    chain_fence<Waves>();   // every wave's state is final and no wave reads the arrays any more
    user_store(f, cl, ch, u, hist);
    if (cl.j == 0) {
      gptr(f.chi2c)[ch] = chi2c;
      gptr(f.flag)[ch] = last.flag;
      gptr(f.ptent)[ch] = last.told;
      gptr(f.ptentn)[ch] = last.t;
    }
    if (err && f.errflag) atomicExch(f.errflag, err);
  }
  const bool count = live && cl.j == 0;
  if (Waves == 1 || threadIdx.x < 64) wave_count(f, count ? nev : 0u, count ? (unsigned)f.nprm : 0u);
}

// Iterations it_off .. it_off + iters - 1 of the segment for whole sequences,
// replica exchange included: a wave holds the temperature ladders (at most 64
// rungs) of its sequences, f.ulanes lanes a chain, and nothing couples one
// sequence to another, so no launch has to end between two iterations.  For
// problems of few data such a launch is all latency, and so was the exchange
// launch between two of them.  What is left is the latency of one iteration's
// chain of steps, so a second wave, with the same lanes, draws the random
// numbers of the next iteration meanwhile: none of them depends on the chains.
// Items are (fit, first sequence of the work-group).
template <bool OneDatum>
__global__ void __launch_bounds__(128) k_iter_user(const FitDesc* fits, const WorkItem* work, int nwork, RunClock* clk,
                                                  TraceBuf tr, int it_off, int iters, int slot_bytes) {
  extern __shared__ __align__(16) char lds[];
  __shared__ LadderLds ladder;
  __shared__ SwapDraw swap[2][64];
  __shared__ float4 par[MAXP];
  const WorkItem w = work[blockIdx.x];
  const FitDesc& f = wave_fit(fits, w.fit);
  pass_clock(clk);
  const int it0 = __builtin_amdgcn_readfirstlane(load_clock(clk, it_off));
  const int nit = f.nburn + f.niter;
  if (it0 >= nit) return;
  const int lane = lane_id();
  const int nb = f.nbeta, ns = f.nseq, P = f.nprm, N = f.nptot, n = f.ulanes;
  const int nwseq = 64 / (f.xlanes * n);
  const int c = lane / n, sl = c / nwseq, g = c % nwseq;
  const int iseq = __builtin_amdgcn_readfirstlane(w.idx) + g;
  const bool live = iseq < ns && sl < nb;
  const int ch = live ? sl * ns + iseq : 0;
  ChainLanes<1> cl{n, lane & (n - 1), nullptr, 0};
  const UserSlot u = user_slot(lds + (size_t)c * slot_bytes, P);
  const bool hist = it0 < f.nburn;
  const int end = nit - it0 < iters ? nit - it0 : iters;
  if (__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) != 0) {
    // the second wave: the draws of iteration i, one iteration ahead
    for (int i = 0; i < end; ++i) {
      if (live) {
        user_draw(f, cl, ch, it0 + i, u.d[i & 1]);
        if (cl.j == 0 && nb > 1) swap[i & 1][c] = swap_draw(f, iseq, it0 + i, sl);
      }
      __syncthreads();
    }
    return;
  }
  CCalcModel mc = user_model_args(f);
  float chi2c = 0.0f, term = 0.0f;
  int tc = 0, err = 0, nex = 0;
  unsigned nev = 0, nprop = 0;
  LastProposal last{0, 0, 0.0f};
  if (live) {
    chi2c = gptr(f.chi2c)[ch];
    tc = gptr(f.tcur)[ch];
    if (OneDatum && cl.j < f.ndat) term = gptr(f.chi2m)[(size_t)ch * f.ndat + cl.j];
    user_load(f, cl, ch, u, hist);
  }
  const double hb = swap_factor(f, sl);
  const double beta = live ? (double)gptr(f.beta)[sl] : 0.0;
  user_params(f, par);
  wave_sync_lds();
  float* row = u.row;
  float* other = u.row + N;
  for (int i = 0; i < end; ++i) {
    const int it = it0 + i;
    __syncthreads();   // this iteration's draws are there, the one before's are free
    const bool burn = it < f.nburn;
    if (live) nev += user_substeps<1, OneDatum>(f, &mc, cl, ch, it, tr, u, u.d[i & 1], par, beta, row,
                                                chi2c, &term, last, &err);
    nprop += P;
    int perm = sl;
    if (nb > 1) {
      // the exchange (reference: gpu_mcmc.cu:548-591): slot sl of sequence g is
      // entry c of the ladder LDS, and its first lane has attempt sl
      const SwapDraw d = live ? swap[i & 1][c] : SwapDraw{0, 0.0};
      const double hk = __shfl(hb, (d.k * nwseq + g) * n);
      if (cl.j == 0) {
        ladder.slot[c] = LadderSlot{chi2c, sl};
        ladder.pair[c] = 0;
      }
      const bool attempt = live && cl.j == 0;
      const unsigned long long swapped = ladder_swaps(ladder, attempt, d.k * nwseq + g, nwseq, d.k == 0, d.lu, hk);
      chi2c = ladder.slot[c].c2;
      perm = ladder.slot[c].src;
      tc = __shfl(tc, (perm * nwseq + g) * n);
      if (!burn) nex += __popcll(ladder.pair[c] & swapped);
      if (tr.ex && attempt && it >= tr.it0 && it < tr.it0 + tr.nit)
        tr.ex[(size_t)f.tr_ex + ((size_t)(it - tr.it0) * nb + sl) * ns + iseq] =
            d.k | ((int)((swapped >> lane) & 1ull) << 16);
    }
    if (live) {
      // the row that ends up in this slot, from the LDS of the slot it started in
      const float* src = reinterpret_cast<const float*>(
          reinterpret_cast<const char*>(row) + (ptrdiff_t)((perm * nwseq + g) - c) * slot_bytes);
      const bool moved = perm != sl;
      const bool rec = !burn && f.record;
      const int itr = it - f.nburn;
      for (int q = cl.j; q < N; q += n) {
        const float v = src[q];
        other[q] = v;
        if (moved) gptr(f.pcur)[(size_t)ch * N + q] = v;
        if (rec) {
          const int ip = gptr(f.invar)[q];
          if (ip >= 0) gptr(f.pout)[(((size_t)nb * ip + sl) * ns + iseq) * f.niter + itr] = v;
        }
      }
      if (cl.j == 0) {   // model() may read these
        gptr(f.chi2c)[ch] = chi2c;
        gptr(f.flag)[ch] = last.flag;
      }
      if (rec && cl.j == 0) {
        gptr(f.tout)[(size_t)ch * f.niter + itr] = tc;
        if (sl == 0) gptr(f.chi2)[(size_t)iseq * f.niter + itr] = chi2c;
      }
    }
    wave_sync_lds();
    float* sw = row;
    row = other;
    other = sw;
  }
  if (live) {
    user_store(f, cl, ch, u, hist);
    if (cl.j == 0) {
      gptr(f.tcur)[ch] = tc;
      if (nex) gptr(f.n_exch)[ch] += nex;
      gptr(f.ptent)[ch] = last.told;
      gptr(f.ptentn)[ch] = last.t;
    }
    if (err && f.errflag) atomicExch(f.errflag, err);
  }
  const bool count = live && cl.j == 0;
  wave_count(f, count ? nev : 0u, count ? nprop : 0u);
}

hipError_t launch_eval_user(const FitDesc* fits, const WorkItem* work, int nwork, int model_only,
                            int respect_flag, hipStream_t s) {
  if (nwork <= 0) return hipSuccess;
  k_eval_user<<<nwork, 64, 0, s>>>(fits, work, nwork, model_only, respect_flag);
  return hipGetLastError();
}

hipError_t launch_step_user(const StepLaunch& L, hipStream_t s) {
  if (L.nwork <= 0) return hipSuccess;
  const TraceBuf tr{L.tr_dec, L.tr_chi2, L.tr_ex, L.tr_it0, L.tr_nit};
  const int sb = user_slot_bytes(L.max_prm, L.max_tot), n = L.ulanes;
  switch (n) {
    case 256:
      k_step_user<4><<<L.nwork, 256, 4 * sb, s>>>(L.fits, L.work, L.nwork, L.clk, tr, L.it_off, n, sb);
      break;
    case 128:
      k_step_user<2><<<L.nwork, 128, 2 * sb, s>>>(L.fits, L.work, L.nwork, L.clk, tr, L.it_off, n, sb);
      break;
    default:
      k_step_user<1><<<L.nwork / (64 / n), 64, (64 / n) * sb, s>>>(L.fits, L.work, L.nwork, L.clk, tr, L.it_off, n, sb);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_iter_user(bool one, const StepLaunch& L, hipStream_t s) {
  if (L.nwork <= 0) return hipSuccess;
  const TraceBuf tr{L.tr_dec, L.tr_chi2, L.tr_ex, L.tr_it0, L.tr_nit};
  const int sb = user_slot_bytes(L.max_prm, L.max_tot);
  const int dyn = 64 / L.ulanes * sb;
  if (one) k_iter_user<true><<<L.nwork, 128, dyn, s>>>(L.fits, L.work, L.nwork, L.clk, tr, L.it_off, L.iters, sb);
  else k_iter_user<false><<<L.nwork, 128, dyn, s>>>(L.fits, L.work, L.nwork, L.clk, tr, L.it_off, L.iters, sb);
  return hipGetLastError();
}

const char* user_model_name() { return MHRE_MODEL_NAME; }

}  // namespace mhre
