// The tape: what the adjoint needs of every photon's path, written by the forward walk, so the backward reads it
// instead of walking each photon again.
//
// The adjoint's terms (adjoint.h) need of a vertex its lengths, its deposit before the cotangent and the drawn outcome:
// 16 bytes.  The replay walks a photon twice to have them, each walk as long as the forward's: once to total its
// cotangent-weighted deposits, once to add the terms.  Reading 1 to 3 records of a tank photon is a fraction of a walk.
//
// Layout, in 16-byte cells: [control][N first chunks of 4 cells][the pool of longer paths, chunks of 16 cells][the
// replay's list].  The control cell's first word counts the pool chunks handed out.
//   a first chunk, at 4 x the photon's launch index: a head (wavelength at emission, event, records, link) and 3 records
//   a pool chunk: a head (0, 0, 0, link) and 15 records; a link is the next chunk's index in the pool
// A photon's head counts the records up to its last deposit: the ones after it have no deposit ahead, so no term.  Most
// tank photons (1 to 3 vertices) fit their first chunk, one 64-byte line found by the launch index with no allocation;
// 15 records a pool chunk keep the links of the argon box's paths (hundreds to thousands of vertices) at 6 %.
// Pool chunks are handed out to a wavefront 64 at a time (an atomic on one address takes about 12 ns).
//
// Who writes it: the forward, where no surface row can draw a facet path.  Where one can, a walk of the adjoint's own
// writes it, without tallies: the adjoint needs the derivative of the facets' density, and code that computes it rounds
// the path itself another way than the forward's; 1 photon in 10^5 then goes elsewhere, and a gradient of few photons
// moves by 1e-4.  A photon whose path the pool has no chunk for is left to the replay: its head says so, the reader
// lists it.
#pragma once
#include <hip/hip_runtime.h>

#include "adjoint.h"

namespace lh {

constexpr int TAPE_FIRST = 3, TAPE_MORE = 15;        // records of a first chunk, of a pool chunk
constexpr int TAPE_GRAB = 64;                        // pool chunks a wavefront takes at once
constexpr unsigned TAPE_CONTROL = 4;                 // cells before the first chunks
constexpr int TAPE_MAX_CLASSES = 64, TAPE_MAX_SENSORS = 1 << 14;  // what a record's code word holds
constexpr unsigned TAPE_REPLAY = 0xFFFFFFFFu;        // a head's records: the photon is left to the replay
enum { TAPE_SCATTER = 0, TAPE_SURFACE = 1, TAPE_DEPOSIT = 2, TAPE_WAVELENGTH = 3 };

struct Tape {
  uint4 *__restrict__ cells;  // null: none
  unsigned *replay;           // the photons left to the replay: their number, then their launch indices
  unsigned photons;           // N
  unsigned pool;              // pool chunks
};

// a record: the event's length (the free path of a scattering, else the crossing's distance; a new wavelength's nm),
// the deposit q w0 at the crossing (0 none; a step that scatters short of one has a record of its own for it), a
// scattering's channel rate or the facet path's derivative of its log density, and a code: type (2 bits), outcome or
// channel (3), straight pass without a surface (1), class pair (12), sensor (14)
__device__ __forceinline__ unsigned tape_code(int type, int o, bool cont, int pair, int sensor) {
  return (unsigned)type | (unsigned)o << 2 | (unsigned)cont << 5 | (unsigned)pair << 6 | (unsigned)sensor << 18;
}

__device__ __forceinline__ unsigned tape_event(unsigned code, int type, int o) {
  return (code & ~31u) | (unsigned)type | (unsigned)o << 2;
}

struct TapeRec {  // a step's: the crossing's distance, the free path of a scattering, ...
  float len, free, dep, aux;
  unsigned code;
};

// a lane's place on the tape
struct TapePos {
  int n;         // records written; -1: left to the replay
  int last;      // ... up to the last deposit
  unsigned cur;  // the cell of the chunk in use's head
  float lam0;    // the wavelength at emission
};

// per wavefront of the block, its pool chunks in hand: [next, end)
__shared__ unsigned s_pool[16][2];

// append a record (each lane its own; lanes of a wavefront whose chunk is full take their next ones together)
__device__ inline void tape_put(const Tape &T, TapePos &t, uint4 r) {
  if (t.n < 0) return;
  const int more = t.n - TAPE_FIRST;
  const int at = more < 0 ? t.n : more % TAPE_MORE;
  if (more >= 0 && at == 0) {
    const unsigned long long mask = __ballot(1);
    const unsigned cnt = (unsigned)__popcll(mask);
    const unsigned rank =
        __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
    volatile unsigned *hand = s_pool[threadIdx.x >> 6];  // one cell for these lanes: the branches on it are uniform
    unsigned base = hand[0];
    if (base + cnt > hand[1]) {
      // a wavefront whose hand begins in the pool's last chunks would get a later one: it asks no more, so the pool's
      // counter ends at most one grab a wavefront past the pool
      bool out = base + TAPE_GRAB > T.pool;
      if (!out) {
        unsigned got = 0;
        if (rank == 0) got = atomicAdd(&T.cells[0].x, (unsigned)TAPE_GRAB);
        base = (unsigned)__builtin_amdgcn_readfirstlane((int)got);
        out = base + TAPE_GRAB > T.pool;
        if (rank == 0) {
          hand[0] = base;
          hand[1] = out ? base : base + TAPE_GRAB;
        }
      }
      if (out) {
        t.n = -1;
        return;
      }
    }
    if (rank == 0) hand[0] = base + cnt;
    const unsigned chunk = base + rank;
    T.cells[t.cur].w = chunk;
    t.cur = TAPE_CONTROL + 4u * T.photons + 16u * chunk;
  }
  T.cells[t.cur + 1 + at] = r;
  t.n += 1;
}

// after a step: the record of its event or deposit, and of the wavelength a shifter left.  Its values pass a barrier to
// the optimiser: the step before must not be split by what is asked of them here, or it rounds differently
template <bool CHAN, bool PATH>
__device__ __forceinline__ void tape_step(const Tape &T, TapePos &t, TapeRec r, float lam) {
  asm("" : "+v"(r.len), "+v"(r.free), "+v"(r.dep), "+v"(r.aux), "+v"(r.code));
  if (!PATH && (r.code & 31u) == (TAPE_SURFACE | GLOSSY << 2)) t.n = -1;  // no derivative of the facets
  const unsigned type = r.code & 3u;
  if (r.dep != 0.0f || type == TAPE_SURFACE) {
    tape_put(T, t, make_uint4(__float_as_uint(r.len), __float_as_uint(r.dep), __float_as_uint(r.aux),
                              type == TAPE_SCATTER ? tape_event(r.code, TAPE_DEPOSIT, 0) : r.code));
    if (r.dep != 0.0f) t.last = t.n;
  }
  if (type == TAPE_SCATTER) {
    tape_put(T, t, make_uint4(__float_as_uint(r.free), 0u, __float_as_uint(r.aux), r.code));
    if (CHAN && (r.code & 31u) == (TAPE_SCATTER | 2u << 2))
      tape_put(T, t, make_uint4(__float_as_uint(lam), 0u, 0u, TAPE_WAVELENGTH));
  }
}

// a photon begins at launch index gi / ends
__device__ __forceinline__ void tape_begin(TapePos &t, unsigned gi, float lam) {
  t.n = t.last = 0;
  t.cur = TAPE_CONTROL + 4u * gi;
  t.lam0 = lam;
}

__device__ __forceinline__ void tape_end(const Tape &T, const TapePos &t, unsigned gi, int event) {
  unsigned *h = reinterpret_cast<unsigned *>(T.cells + TAPE_CONTROL + 4u * gi);
  if (t.n >= 0 && t.last > 0) {
    h[0] = __float_as_uint(t.lam0);
    h[1] = (unsigned)event;
  }
  h[2] = t.n < 0 ? TAPE_REPLAY : (unsigned)t.last;
}

}  // namespace lh
