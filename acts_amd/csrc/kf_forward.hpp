// kf_forward.hpp -- the persistent forward kernel (forward filter, and with
// Rev the reverse filter).
//
// Its instantiations are compiled apart (kf_forward.hip, one object per
// precision, stepper, navigator and field), so that they build in parallel; the
// host code reaches them through forwardVariant.
#pragma once

#include "kf_reverse.hpp"

namespace kf {

constexpr int kBlock = 64;
// geometry kept in LDS by the forward kernel (224 B per surface)
constexpr int kLdsSurfaces = 96;
constexpr int kLdsSlabs = 32;

// The workgroup's field-map cells in LDS, one column per lane: the first
// lookup of an RK step is nearly always in the cell of the previous step's
// last one.
template <bool Mixed>
struct CellStore {
  double v[Mixed ? 1 : kCellValues * kCellCacheStride];
  float vf[Mixed ? kCellValues * kCellCacheStride : 1];
  int32_t idx[kCellCacheStride];
};

// The lane's column of it, empty (no column without a cell-major map).
template <bool Mixed>
__device__ inline CellCache cellCache(CellStore<Mixed>& s, const DevField& F) {
  static_assert(kBlock == kCellCacheStride, "one column per lane of the workgroup");
  CellCache c{nullptr, nullptr, nullptr};
  if (Mixed ? F.cellsF != nullptr : F.cells != nullptr) {
    const int lane = static_cast<int>(threadIdx.x);
    s.idx[lane] = -1;
    c.v = Mixed ? nullptr : s.v + lane;
    c.vf = Mixed ? s.vf + lane : nullptr;
    c.idx = s.idx + lane;
  }
  return c;
}

using ForwardFn = void (*)(FwdArgs, int32_t*, int32_t, int32_t, int32_t, const int32_t*);

// The kernel of a precision, stepper, navigator and kind of field: geometry
// in LDS or in global memory, forward or reverse filter.
template <bool Mixed, bool Sympy, bool Layers, bool Map>
ForwardFn forwardVariant(bool geoInLds, bool rev);

// Forward filter, persistent: each wavefront keeps its 64 lanes busy with
// tracks taken from a global queue (`next`), in the order `order` when given
// (longest surface sequence first, so that long tracks do not start last).
// Per outer iteration: idle lanes
// take new tracks; stepping lanes step until no lane steps towards a surface
// any more, or at least `waitFrac`/64 of the busy lanes wait at one, or
// `maxInner` steps have been taken; then the waiting lanes run the surface
// update together, and finished lanes write their summary and go idle.
// Tracks past their last surface step on beside the others: waiting for
// them, and stepping them with the transport, took 200 000 tracks with holes
// and rejected outliers 7.4 instead of 3.4 ms here.  With Rev
// the kernel runs the reverse filter of the tracks that take one.  The
// navigator is a template parameter (Layers: the layer navigator): its
// option becomes a constant, so the direct navigator's instantiations carry
// none of the layer navigator's code (a run-time choice cost the direct
// fit's forward kernel 4 %).  So is the kind of field (Map): with a step per
// kind in one kernel, ~100 of the ~1 100 vector instructions of a step in a
// uniform field were moves that brought the kinds' results together.
template <bool Mixed, bool GeoInLds, bool Sympy, bool Rev, bool Layers, bool Map>
__global__ __launch_bounds__(kBlock, 1) void fitForwardKernel(
    FwdArgs args, int32_t* __restrict__ next, int32_t maxInner, int32_t waitFrac,
    int32_t quarantine, const int32_t* __restrict__ order) {
  (void)args;  // read through freshArgs
  const FwdArgs& a = freshArgs();
  const int lane = static_cast<int>(threadIdx.x) & 63;
  __shared__ CellStore<Mixed> cells;
  const CellCache cache = cellCache(cells, a.F);
  const uint64_t lanesBelow = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int64_t n = a.in.n;
  // Surfaces and material slabs are read at every step: with GeoInLds (the
  // geometry fits, as it does for the benchmark detectors) the workgroup
  // keeps a copy in LDS.  The choice is a template parameter so that every
  // geometry access compiles to an LDS read: a pointer that may point to
  // either memory needs flat loads, which wait for all outstanding global
  // loads and stores of the wavefront before their data can be used.
  __shared__ DevSurface sGeo[GeoInLds ? kLdsSurfaces : 1];
  __shared__ DevSlab sSlabs[GeoInLds ? kLdsSlabs : 1];
  if constexpr (GeoInLds) {
    const double* src = reinterpret_cast<const double*>(a.geo);
    double* dst = reinterpret_cast<double*>(sGeo);
    const int nd = a.nSurfaces * static_cast<int>(sizeof(DevSurface) / sizeof(double));
    for (int i = static_cast<int>(threadIdx.x); i < nd; i += blockDim.x) dst[i] = src[i];
    const int32_t* ss = reinterpret_cast<const int32_t*>(a.slabs);
    int32_t* sd_ = reinterpret_cast<int32_t*>(sSlabs);
    const int ns = a.nSlabs * static_cast<int>(sizeof(DevSlab) / sizeof(int32_t));
    for (int i = static_cast<int>(threadIdx.x); i < ns; i += blockDim.x) sd_[i] = ss[i];
    __syncthreads();
  }
  const DevSurface* geo = GeoInLds ? sGeo : a.geo;
  const DevSlab* slabs = GeoInLds ? sSlabs : a.slabs;
  Lane L;
  int phase = kPhaseIdle;
  while (true) {
    // a wavefront holding a track that has run longer than `quarantine`
    // steps takes no new tracks until it ends, so that neither slows the
    // other down: the long track waits for the surface updates of fresh ones,
    // and they wait up to `maxInner` of its steps at every surface
    const bool hold =
        quarantine > 0 &&
        __ballot(phase == kPhaseStepping && L.iter > static_cast<uint32_t>(quarantine)) != 0;
    const uint64_t idle = hold ? 0ull : __ballot(phase == kPhaseIdle);
    if (idle) {
      const int cnt = __popcll(idle);
      const int leader = __ffsll(static_cast<long long>(idle)) - 1;
      int base = 0;
      if (lane == leader) base = atomicAdd(next, cnt);
      base = __shfl(base, leader);
      if (phase == kPhaseIdle) {
        const int64_t q = static_cast<int64_t>(base) + __popcll(idle & lanesBelow);
        if (q >= n)
          phase = kPhaseRetired;
        else if constexpr (Rev)
          phase = laneInitReverse<Mixed, Sympy, Layers>(L, q, order ? order[q] : q,
                                                        freshArgs(), geo);
        else
          phase = laneInit<Mixed, Sympy, Layers>(L, q, order ? order[q] : q, freshArgs(), geo);
      }
    }
    if (phase == kPhaseFinished) {
      laneFinish<Rev>(L, freshArgs());
      phase = kPhaseIdle;
    }
    const uint64_t busy = __ballot(phase != kPhaseRetired);
    if (!busy) break;
    const FwdArgs& as = freshArgs();
    const StepArgs sa = stepArgs<Mixed, Map>(as);
    for (int it = 0; it < maxInner; ++it) {
      if (phase == kPhaseStepping)
        phase = laneStep<Mixed, Sympy, Rev, Layers, Map>(L, as, sa, geo, cache);
      const bool stepping = phase == kPhaseStepping;
      const int nStep = __popcll(__ballot(stepping && !pastLastSurface<Rev>(L)));
      const int nWait = __popcll(__ballot(phase == kPhaseSurface || phase == kPhaseFinished));
      if (!__ballot(stepping) ||
          (nWait > 0 && 64 * nWait >= waitFrac * (nStep + nWait)))
        break;
    }
    // a lane that reached a surface while stepping without the transport
    // goes back to its checkpoint and repeats the steps with it; a track
    // that did so once (e.g. a looper that crosses a surface every turn)
    // keeps the transport from then on
    if (phase == kPhaseSurface && L.noTransport) {
      L = freshArgs().ckpt[static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x];
      L.replaying = true;
      L.noSkip = true;
      phase = kPhaseStepping;
    }
    if (phase == kPhaseSurface) phase = laneFilter<Mixed, Sympy, Rev, Layers>(L, freshArgs(), geo, slabs);
    if (phase == kPhaseFinished) {
      laneFinish<Rev>(L, freshArgs());
      phase = kPhaseIdle;
    }
  }
}

}  // namespace kf
