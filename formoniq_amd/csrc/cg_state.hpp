// The scalars of a device-resident Jacobi CG run and what its launches read and
// write of them, on the device and on the host.
#pragma once

#include <hip/hip_runtime.h>

namespace feec {

// An iteration's first launch (the direction, or the product that forms it)
// reads the slots of its parity and its lead thread writes the other ones; the
// iteration's later launches read those. So no launch reads a word that it also
// writes, and every wavefront of a launch decides alike, whenever it starts.
struct CgS {
  double rz[2];
  long long iters[2];  // completed when the iteration of this parity starts
  int stop[2];         // the run is over
  double bnorm2, rtol2, res2;
  long long iter, max_iters;
};

__host__ __device__ inline CgS cg_first(double bnorm2, double rtol, long long max_iters) {
  CgS s{};
  s.bnorm2 = bnorm2;
  s.rtol2 = rtol * rtol;
  s.res2 = bnorm2;
  s.max_iters = max_iters;
  s.stop[0] = s.stop[1] = bnorm2 == 0.0 || max_iters <= 0 ? 1 : 0;
  return s;
}

// What an iteration's first launch reads of the state.
struct CgRead {
  double rz, limit;
  long long iters, most;
};
__host__ __device__ inline bool cg_stopped(const CgS& s, int par) { return s.stop[par] != 0; }
__host__ __device__ inline CgRead cg_read(const CgS& s, int par) {
  return {s.rz[par], s.rtol2 * s.bnorm2, s.iters[par], s.max_iters};
}
// Whether an iteration that starts with residual |r|^2 = rr is one too many (the
// first always runs).
__host__ __device__ inline bool cg_stops(const CgRead& q, double rr) {
  return q.iters > 0 && (rr <= q.limit || q.iters >= q.most);
}
// beta of the iteration, rz = r.z at its start
__host__ __device__ inline double cg_beta(const CgRead& q, double rz) { return q.iters > 0 ? rz / q.rz : 0.0; }

// The lead thread's part of the first launch: the run was over before, ends
// here, or goes on.
__host__ __device__ inline void cg_put_stopped(CgS& s, int par) { s.stop[par ^ 1] = 1; }
__host__ __device__ inline void cg_put_stop(CgS& s, int par, const CgRead& q, double rr) {
  s.res2 = rr;
  s.iter = q.iters;
  s.stop[par ^ 1] = 1;
}
__host__ __device__ inline void cg_put_next(CgS& s, int par, const CgRead& q, double rz) {
  s.rz[par ^ 1] = rz;
  s.iters[par ^ 1] = q.iters + 1;
}

// For the iteration's later launches, and for the host after any whole
// iteration: whether the run is over.
__host__ __device__ inline bool cg_over(const CgS& s, int par) { return s.stop[par ^ 1] != 0; }

// Iterations of the host's segment `seg` (even: it starts at parity 0). The next
// one is queued before a segment's state is read, so a run of one iteration (the
// mass of the top grade is diagonal) waits for all launches of the first two. In
// the form of three launches an iteration these are few: 384 k rows 513 us a
// solve with eight and eight iterations in them, 448 with two and six. In the
// form of two, sixteen iterations cost a short run less than the further read
// costs the others (31 k rows, 29 iterations: 460 us and 472).
constexpr int cg_segment(int seg, bool three) { return !three || seg > 1 ? 8 : seg == 0 ? 2 : 6; }

}  // namespace feec
