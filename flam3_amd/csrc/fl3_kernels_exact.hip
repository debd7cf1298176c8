// fl3_kernels_exact.hip - FP64 kernels that must follow the reference's
// arithmetic operation by operation: replay walkers, batched iterate, xform
// preview, point deposit, density estimation, log scaling and the tone map.
// Compiled with FP contraction off (the reference's x86-64 build has no FMA).
#include <type_traits>
#include "fl3_core.h"
#include "fl3_tonemath.h"
#include "fl3_launch.h"

// Replay walkers: walker w is reference iteration thread w (rect.c:253-527)
// with its ISAAC state seeded on the host as rect.c:858-865 does, running
// the same sub-batch loop in FP64 (exact-mode deposits).
template <int BITS>
__global__ __launch_bounds__(64) void k_iter_replay(IterArgs a) {
   unsigned char *lds = fl3_lds;
   GenL<double> G;
   load_genome<double>(a.job, lds, G);
   __syncthreads();
   const int wid = blockIdx.x * blockDim.x + threadIdx.x;
   if (wid >= a.nwalkers) return;
   IsaacRng rng;
   rng.load(a.isaac + 36 * wid);
   uint32_t bad = 0;
   const double bs = a.batch_size;
   const bool use_final = G.final_index >= 0;
   for (double sub = 0; sub < bs; sub += a.sbs) {
      int sbs = (sub + a.sbs > bs) ? (int)(bs - sub) : a.sbs;
      double p[4], q[4];
      p[0] = u11<double>(rng);
      p[1] = u11<double>(rng);
      p[2] = u01<double>(rng);
      p[3] = u01<double>(rng);
      int lastxf = 0, consec = 0;
      for (int i = -a.fuse; i < sbs;) {
         const uint32_t r = rng.next();
         const int fn = select_xform(G, G.chaos_enable ? lastxf : 0, r & 16383u);
         if (apply_xform<double>(G, fn, p, q, rng)) {
            consec++;
            bad++;
            if (consec < 5) {
               p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
               continue;
            }
            consec = 0;
         } else
            consec = 0;
         lastxf = fn + 1;
         p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
         if (use_final) {
            if (G.final_opacity == 1.0 || u01<double>(rng) < G.final_opacity) {
               apply_xform<double>(G, G.final_index, p, q, rng);
               q[3] = p[3];
            }
         }
         if (i >= 0) deposit<double, BITS, true>(G, q, a.buckets, a.sat);
         i++;
      }
   }
   rng.store(a.isaac + 36 * wid);
   if (bad) atomicAdd(a.badvals, (unsigned long long)bad);
}

// Batched flam3_iterate (flam3.c:232-299) in FP64: walker w starts from
// start[4w..4w+3] with ISAAC state w and writes n samples.

__global__ __launch_bounds__(64) void k_iterate_points(PointsArgs a) {
   unsigned char *lds = fl3_lds;
   GenL<double> G;
   load_genome<double>(a.job, lds, G);
   __syncthreads();
   const int wid = blockIdx.x * blockDim.x + threadIdx.x;
   if (wid >= a.nwalkers) return;
   IsaacRng rng;
   rng.load(a.isaac + 36 * wid);
   double p[4], q[4];
   for (int k = 0; k < 4; k++) p[k] = a.start[4 * wid + k];
   int lastxf = 0, consec = 0, bad = 0;
   const bool use_final = G.final_index >= 0;
   double *out = a.out + (size_t)wid * a.n * 4;
   for (int i = -a.fuse; i < a.n;) {
      const uint32_t r = rng.next();
      const int fn = select_xform(G, G.chaos_enable ? lastxf : 0, r & 16383u);
      if (apply_xform<double>(G, fn, p, q, rng)) {
         consec++;
         bad++;
         if (consec < 5) {
            p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
            continue;
         }
         consec = 0;
      } else
         consec = 0;
      lastxf = fn + 1;
      p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
      if (use_final) {
         if (G.final_opacity == 1.0 || u01<double>(rng) < G.final_opacity) {
            apply_xform<double>(G, G.final_index, p, q, rng);
            q[3] = p[3];
         }
      }
      if (i >= 0) {
         out[4 * i + 0] = q[0]; out[4 * i + 1] = q[1];
         out[4 * i + 2] = q[2]; out[4 * i + 3] = q[3];
      }
      i++;
   }
   rng.store(a.isaac + 36 * wid);
   a.badvals[wid] = bad;
}

// ---- one walker per wavefront
//
// A few walkers (the bounding box of a genome is one) are a serial chain of
// FP64 steps, bound by a step's latency.  k_iterate_points takes 33 us a step
// for such a walker: ISAAC's arrays are indexed by their contents, so they
// live in scratch memory, and the 196 KB of apply_xform with every variation
// do not stay in the instruction cache beside it.  Here every lane of a
// wavefront holds the same walker: the xform, the branches and ISAAC run in
// scalar registers (its two arrays across the lanes of a register each), the
// variations are the wavefront's own xform's only, and a genome of classic
// variations runs code that holds no others; the sines and cosines of an
// xform's classic variations are one evaluation (lone_classic).  The arithmetic is apply_xform's,
// operation by operation.  20000 points of a genome of six xforms and a final
// one: 690 -> 62 ms.

// IsaacRng in a wavefront: word k of an array in lane k.
struct WaveIsaac {
   uint32_t rsl, mem, a, b, c, cnt;

   __device__ static uint32_t word(uint32_t v, uint32_t k) {
      return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)k);
   }
   // x into lane k of v
   __device__ __forceinline__ static void put(uint32_t &v, uint32_t x, uint32_t k) {
      v = threadIdx.x == k ? x : v;
   }
   __device__ void load(const uint32_t *s, unsigned lane) {
      rsl = s[1 + (lane & 15u)];
      mem = s[17 + (lane & 15u)];
      cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)s[0]);
      a = (uint32_t)__builtin_amdgcn_readfirstlane((int)s[33]);
      b = (uint32_t)__builtin_amdgcn_readfirstlane((int)s[34]);
      c = (uint32_t)__builtin_amdgcn_readfirstlane((int)s[35]);
   }
   __device__ void store(uint32_t *s, unsigned lane) const {
      if (lane < 16) {
         s[1 + lane] = rsl;
         s[17 + lane] = mem;
      }
      if (lane == 0) {
         s[0] = cnt;
         s[33] = a;
         s[34] = b;
         s[35] = c;
      }
   }
   __device__ __forceinline__ void refill() {
      uint32_t aa = a, bb = b + (++c);
#pragma unroll
      for (uint32_t i = 0; i < 16; i++) {
         const uint32_t x = word(mem, i);
         const uint32_t mixv = (i & 3) == 0 ? aa << 13 : (i & 3) == 1 ? aa >> 6 : (i & 3) == 2 ? aa << 2 : aa >> 16;
         aa = (aa ^ mixv) + word(mem, (i + 8) & 15);
         const uint32_t y = word(mem, (x >> 2) & 15) + aa + bb;
         put(mem, y, i);
         bb = word(mem, (y >> 6) & 15) + x;
         put(rsl, bb, i);
      }
      a = aa;
      b = bb;
   }
   __device__ __forceinline__ uint32_t next() {
      if (cnt-- == 0) {
         refill();
         cnt = 15;
      }
      return word(rsl, cnt);
   }
};

__device__ __forceinline__ double uniform_f64(double v) {
   return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                           __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

__device__ __forceinline__ double lane_f64(double v, int lane) {
   return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                           __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// The classic variations of an xform (weight of variation v: w[v]).  A double
// sine and cosine take some 200 instructions and most variations ask for
// them, each for arguments of its own: lane v takes variation v's (lane 16 + v
// its second), so that all of them cost one evaluation.  Returns how many
// there are.
__device__ __forceinline__ int lone_classic(const double *w, Pre<double> &f, WaveIsaac &rng) {
   const unsigned lane = threadIdx.x, id = lane & 15u;
   const bool second = lane & 16u;
   const double wl = w[id];
   const uint32_t mask = (uint32_t)__builtin_amdgcn_ballot_w64(wl != 0.0) & 0x3fffu;
   const double EPS = 1e-10, PI = M_PI, a = f.atan, r = f.sq;
   uint32_t word = 0;
   if (mask & (1u << 13)) word = rng.next();   // julia's random bit, the classic variations' only draw
   double s = 0.0, c = 0.0;
   if (mask & 0x3bcau) {   // sinusoidal, swirl, handkerchief .. spiral, diamond .. julia
      const double sum = a + r, dif = a - r;
      double ja = 0.5 * a;
      if (word & 1u) ja += PI;
      double x = second ? f.ty : f.tx;                 // 1: sinusoidal
      x = id == 3 ? f.sumsq : x;                       // swirl
      x = id == 6 || id == 12 ? (second ? dif : sum) : x;   // handkerchief, ex
      x = id == 7 ? r * a : x;                         // heart
      x = id == 8 ? PI * r : x;                        // disc
      x = id == 9 ? r + EPS : x;                       // spiral
      x = id == 11 ? r : x;                            // diamond
      x = id == 13 ? ja : x;                           // julia
      m_sincos(x, &s, &c);
   }
#define LONE_VAR(v) if (mask & (1u << (v)))
#define LONE_W(v) const double w = lane_f64(wl, v)
   LONE_VAR(0) {  // linear :142
      LONE_W(0);
      f.p0 += w * f.tx;
      f.p1 += w * f.ty;
   }
   LONE_VAR(1) {  // sinusoidal :153
      LONE_W(1);
      f.p0 += w * lane_f64(s, 1);
      f.p1 += w * lane_f64(s, 17);
   }
   LONE_VAR(2) {  // spherical :164
      LONE_W(2);
      const double r2 = w / (f.sumsq + EPS);
      f.p0 += r2 * f.tx;
      f.p1 += r2 * f.ty;
   }
   LONE_VAR(3) {  // swirl :178
      LONE_W(3);
      const double c1 = lane_f64(s, 3), c2 = lane_f64(c, 3);
      f.p0 += w * (c1 * f.tx - c2 * f.ty);
      f.p1 += w * (c2 * f.tx + c1 * f.ty);
   }
   LONE_VAR(4) {  // horseshoe :202
      LONE_W(4);
      const double h = w / (r + EPS);
      f.p0 += (f.tx - f.ty) * (f.tx + f.ty) * h;
      f.p1 += 2.0 * f.tx * f.ty * h;
   }
   LONE_VAR(5) {  // polar :218
      LONE_W(5);
      f.p0 += w * (a * M_1_PI);
      f.p1 += w * (r - 1.0);
   }
   LONE_VAR(6) {  // handkerchief :232
      LONE_W(6);
      f.p0 += w * r * lane_f64(s, 6);
      f.p1 += w * r * lane_f64(c, 22);
   }
   LONE_VAR(7) {  // heart :246
      LONE_W(7);
      const double h = w * r;
      f.p0 += h * lane_f64(s, 7);
      f.p1 += (-h) * lane_f64(c, 7);
   }
   LONE_VAR(8) {  // disc :264
      LONE_W(8);
      const double h = a * M_1_PI;
      f.p0 += w * lane_f64(s, 8) * h;
      f.p1 += w * lane_f64(c, 8) * h;
   }
   LONE_VAR(9) {  // spiral :282
      LONE_W(9);
      const double r1 = w / (r + EPS);
      f.p0 += r1 * (f.cosa + lane_f64(s, 9));
      f.p1 += r1 * (f.sina - lane_f64(c, 9));
   }
   LONE_VAR(10) {  // hyperbolic :298
      LONE_W(10);
      const double h = r + EPS;
      f.p0 += w * f.sina / h;
      f.p1 += w * f.cosa * h;
   }
   LONE_VAR(11) {  // diamond :311
      LONE_W(11);
      f.p0 += w * f.sina * lane_f64(c, 11);
      f.p1 += w * f.cosa * lane_f64(s, 11);
   }
   LONE_VAR(12) {  // ex :326
      LONE_W(12);
      const double n0 = lane_f64(s, 12), n1 = lane_f64(c, 28);
      const double m0 = n0 * n0 * n0 * r, m1 = n1 * n1 * n1 * r;
      f.p0 += w * (m0 + m1);
      f.p1 += w * (m0 - m1);
   }
   LONE_VAR(13) {  // julia :350
      LONE_W(13);
      const double h = w * m_sqrt(r);
      f.p0 += h * lane_f64(c, 13);
      f.p1 += h * lane_f64(s, 13);
   }
#undef LONE_VAR
#undef LONE_W
   return __popc(mask);
}

// apply_xform<double> for a wavefront whose lanes all hold the same walker
// (wd: the classic weights by xform and variation, 16 each).
template <int TIER>
__device__ __forceinline__ bool lone_apply(const GenL<double> &G, const double *wd, int fn, const double *p, double *q,
                                           WaveIsaac &rng) {
   const XfL<double> &X = G.xf[fn];
   Pre<double> f;
   const double s1 = X.cspeed;
   q[2] = s1 * X.color + (1.0 - s1) * p[2];
   q[3] = X.vis;
   f.tx = X.c[0] * p[0] + X.c[2] * p[1] + X.c[4];
   f.ty = X.c[1] * p[0] + X.c[3] * p[1] + X.c[5];
   const double preblur = uniform_f64(X.preblur);
   if (preblur != 0.0) {
      const double g0 = u01<double>(rng), g1 = u01<double>(rng), g2 = u01<double>(rng), g3 = u01<double>(rng);
      const double rndG = preblur * (g0 + g1 + g2 + g3 - 2.0);
      const double rndA = u01<double>(rng) * 2.0 * M_PI;
      double sA, cA;
      m_sincos(rndA, &sA, &cA);
      f.tx += rndG * cA;
      f.ty += rndG * sA;
   }
   f.sumsq = f.tx * f.tx + f.ty * f.ty;
   f.sq = m_sqrt(f.sumsq);
   f.atan = f.sina = f.cosa = f.atanyx = 0.0;
   const int flags = __builtin_amdgcn_readfirstlane(X.flags);
   if (flags & FL3_PRE_ATAN_XY) f.atan = m_atan2(f.tx, f.ty);
   if (flags & FL3_PRE_ANGLES) {
      f.sina = m_div(f.tx, f.sq);
      f.cosa = m_div(f.ty, f.sq);
   }
   if (flags & FL3_PRE_ATAN_YX) f.atanyx = m_atan2(f.ty, f.tx);
   f.p0 = 0.0;
   f.p1 = 0.0;
   const int classic = lone_classic(wd + fn * 16, f, rng);
   if constexpr (TIER != 0) {
      // (ascending ids: the classic ones come first in the list too)
      const int nv = __builtin_amdgcn_readfirstlane(G.vcount[fn]);
      for (int k = classic; k < nv; k++) {
         const int u = __builtin_amdgcn_readfirstlane((int)G.vlist[fn * G.nunion + k]);
         const int v = __builtin_amdgcn_readfirstlane(G.uid[u]);
         const double w = uniform_f64(G.w[fn * G.nunion + u]);
         fl3_var<double, WaveIsaac, FL3_CLASSIC, FL3_NVAR>(v, w, X, f, rng);
      }
   }
   if (flags & FL3_HAS_POST) {
      q[0] = X.post[0] * f.p0 + X.post[2] * f.p1 + X.post[4];
      q[1] = X.post[1] * f.p0 + X.post[3] * f.p1 + X.post[5];
   } else {
      q[0] = f.p0;
      q[1] = f.p1;
   }
   if (__builtin_amdgcn_ballot_w64(fl3_bad(q[0]) || fl3_bad(q[1]))) {
      q[0] = u11<double>(rng);
      q[1] = u11<double>(rng);
      return true;
   }
   return false;
}

// k_iterate_points, walker w in wavefront w.
template <int TIER>
__global__ __launch_bounds__(64) void k_iterate_lone(PointsArgs a) {
   GenL<double> G;
   load_genome<double>(a.job, fl3_lds, G, false);
   __shared__ double wd[16 * FL3_MAX_XFORMS];
   for (int e = threadIdx.x; e < 16 * G.nxf; e += 64) wd[e] = 0.0;
   __syncthreads();
   for (int e = threadIdx.x; e < G.nxf * G.nunion; e += 64) {
      const int id = G.uid[e % G.nunion];
      if (id < FL3_CLASSIC) wd[e / G.nunion * 16 + id] = G.w[e];
   }
   __syncthreads();
   const int wid = blockIdx.x;
   const unsigned lane = threadIdx.x;
   WaveIsaac rng;
   rng.load(a.isaac + 36 * wid, lane);
   double p[4], q[4];
   for (int k = 0; k < 4; k++) p[k] = a.start[4 * wid + k];
   int lastxf = 0, consec = 0, bad = 0;
   const int final_index = __builtin_amdgcn_readfirstlane(G.final_index);
   double *out = a.out + (size_t)wid * a.n * 4;
   int i = -a.fuse, fn = 0;
   bool fin = false;   // the xform to apply next is the final one, to p's point
   while (i < a.n) {
      if (!fin) {
         // (select_xform, a breakpoint per lane: at most 63 after the first)
         const uint32_t slot = rng.next() & 16383u;
         const int *st = G.starts + (G.chaos_enable ? lastxf : 0) * G.nstd;
         fn = __popcll(__builtin_amdgcn_ballot_w64(lane >= 1 && (int)lane < G.nstd &&
                                                   slot >= (uint32_t)st[min((int)lane, G.nstd - 1)]));
      }
      const bool isbad = lone_apply<TIER>(G, wd, fin ? final_index : fn, p, q, rng);
      if (!fin) {
         if (isbad) {
            consec++;
            bad++;
            if (consec < 5) {
               for (int k = 0; k < 4; k++) p[k] = q[k];
               continue;
            }
         }
         consec = 0;
         lastxf = fn + 1;
         for (int k = 0; k < 4; k++) p[k] = q[k];
         if (final_index >= 0) {
            fin = true;
            if (uniform_f64(G.final_opacity) == 1.0) continue;
            if (u01<double>(rng) < uniform_f64(G.final_opacity)) continue;
         }
      } else
         q[3] = p[3];
      fin = false;
      if (i >= 0 && lane == 0)
         for (int k = 0; k < 4; k++) out[4 * (size_t)i + k] = q[k];
      i++;
   }
   rng.store(a.isaac + 36 * wid, lane);
   if (lane == 0) a.badvals[wid] = bad;
}

// Apply xform xi `depth` times to each point of a grid (flam3.c:301-349).
__global__ __launch_bounds__(64) void k_xform_preview(const unsigned char *job, int xi, double range,
                                                      int numvals, int depth, double *result,
                                                      uint32_t *isaac) {
   unsigned char *lds = fl3_lds;
   GenL<double> G;
   load_genome<double>(job, lds, G);
   __syncthreads();
   if (blockIdx.x != 0 || threadIdx.x != 0) return;
   IsaacRng rng;
   rng.load(isaac);
   const double incr = range / (double)numvals;
   int outi = 0;
   for (int xx = -numvals; xx <= numvals; xx++)
      for (int yy = -numvals; yy <= numvals; yy++) {
         double p[4] = {(double)xx * incr, (double)yy * incr, 0.0, 0.0}, q[4];
         for (int d = 0; d < depth; d++) {
            apply_xform<double>(G, xi, p, q, rng);
            p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
         }
         result[outi] = p[0];
         result[outi + 1] = p[1];
         outi += 2;
      }
   rng.store(isaac);
}

// Deposit a given point stream (stage test of rect.c:411-516).
template <int BITS>
__global__ __launch_bounds__(256) void k_deposit_points(const unsigned char *job, const double *pts, long long n,
                                                        void *buckets, uint32_t *sat) {
   unsigned char *lds = fl3_lds;
   GenL<double> G;
   load_genome<double>(job, lds, G);
   __syncthreads();
   for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
        i += (long long)gridDim.x * blockDim.x) {
      double q[4] = {pts[4 * i], pts[4 * i + 1], pts[4 * i + 2], pts[4 * i + 3]};
      deposit<double, BITS, true>(G, q, buckets, sat);
   }
}

// ------------------------------------------------------------------ density estimation


// ---- density estimation ---------------------------------------------------
//
// The reference scatters each source cell's kernel into the accumulator
// (rect.c:126-173).  Here pass 1 (k_de_prep) picks every source's kernel (the
// hit-count neighbourhood sum and index selection of rect.c:92-117) and pass
// 2 (k_de_gather) gathers, for each output cell, the contributions of the
// sources that reach it.
#define DE_SKIP 0xffffu

// Channel i of the histogram as a double: uint32 cells with a float
// accumulator (bits 33), double cells with a double one (bits 64).
__device__ __forceinline__ double bucket_value(const void *b, long i, float) { return (double)((const uint32_t *)b)[i]; }
__device__ __forceinline__ double bucket_value(const void *b, long i, double) { return ((const double *)b)[i]; }

// Per 16x16 block of cells (one DE workgroup region): 1 + the largest
// kernel radius of its sources (0: no source), so that each gather
// workgroup scans only the halo its neighbourhood's sources can reach from.
// Lanes 16k..16k+15 of a wavefront hold cells of one block (rows of 256
// cells, blocks 16 wide).
__device__ __forceinline__ void de_mark_block(const DEArgs &a, int i, int j, int r1) {
   int m = r1;
   for (int o = 1; o < 16; o <<= 1) m = max(m, __shfl_xor(m, o));
   if ((threadIdx.x & 15) == 0 && m > 0) atomicMax(&a.blkmax[(j >> 4) * a.nbx + (i >> 4)], m);
}

// floor(pow(x, c)) for x > 0 as the double function gives it.  In floats the
// power of up to 2^10, c up to 4, is off by less than 3e-6 of itself (the logarithm times
// c, up to 10, by 2e-6); only where that leaves the integer open, or the power
// is larger (no kernel index is), is the double one formed: 163 -> 142 us for
// the preparation at 1920x1080 with supersample 2 and quality 500.
__device__ __forceinline__ int de_pow_floor(double x, double c) {
   const float p = exp2f((float)c * log2f((float)x)), f = floorf(p), m = p * 1e-5f;
   if (fabs(c) <= 4.0 && p >= 1e-3f && p <= 1024.0f && p - f > m && f + 1.0f - p > m) return (int)f;
   return (int)floor(pow(x, c));
}

// One cell of the DE preparation: its kernel index (DE_SKIP if it is no
// source), per-source values and log term; returns the index.
template <typename BT, typename AT>
__device__ __forceinline__ unsigned de_prep_cell(const DEArgs &a, int i, int j, int os, int ss, bool scf,
                                                 double scfact) {
   const int W = a.width, H = a.height;
   const long cell = i + (long)j * W;
   uint16_t out = DE_SKIP;
   const BT *b = (const BT *)a.buckets;
   // rows (os - 1) .. H - os + 1 (rect.c:979-1000 spans H - 2 (os - 1) + 1
   // rows from os - 1); for os 1 that includes row H, past the histogram,
   // which counts as empty here
   if (i >= os - 1 && i < W - (os - 1) && j >= os - 1 && j <= H - os + 1) {
      const double c4 = (double)b[cell * 5 + 4], c3 = (double)b[cell * 5 + 3];
      if (c4 != 0 && c3 != 0) {
         double fsel = 0.0;
         for (int ii = -ss; ii <= ss; ii++)
            for (int jj = -ss; jj <= ss; jj++) {
               const int y = j + jj;
               if (y < H) fsel += fl3_div255((double)b[((i + ii) + (long)y * W) * 5 + 4]);
            }
         if (scf) fsel *= scfact;
         int fi;
         if (fsel > a.max_filtered_counts)
            fi = a.max_filter_index;
         else if (fsel <= 100)
            fi = (int)ceil(fsel) - 1;
         else
            fi = 100 + de_pow_floor(fsel - 100, a.curve);
         if (fi > a.max_filter_index) fi = a.max_filter_index;
         out = (uint16_t)fi;
         // the per-source factor of rect.c:137, k1 log(1 + c3 k2) / c3,
         // applied to the colour once; the kernel coefficient multiplies
         // it per tap
         const double lnum = a.k1 * log(1.0 + c3 * a.k2);
         if (a.exact) a.srcl[cell] = lnum;
         const double sc = lnum / c3;
         AT *v = (AT *)a.srcv + cell * 4;
         v[0] = (AT)((double)b[cell * 5 + 0] * sc);
         v[1] = (AT)((double)b[cell * 5 + 1] * sc);
         v[2] = (AT)((double)b[cell * 5 + 2] * sc);
         v[3] = (AT)(c3 * sc);
         if constexpr (sizeof(AT) == 8) {
            // (a NaN or an infinity in any of them leaves no zero)
            if (a.nonfinite && v[0] * 0.0 + v[1] * 0.0 + v[2] * 0.0 + v[3] * 0.0 != 0.0) *a.nonfinite = 1;
         }
      }
   }
   a.findex[cell] = out;
   return out;
}

template <typename BT, typename AT>
__device__ __forceinline__ void de_prep_body(const DEArgs &a, int bx, int by) {
   const int os = a.oversample;
   const int ss = os / 2;
   const bool scf = !(os & 1);
   const double scfact = pow(os / (os + 1.0), 2.0);
   const int W = a.width;
   const int i = bx * blockDim.x + threadIdx.x;
   const int j = by;
   if (!a.blkmax && !a.taps) {
      if (i < W) de_prep_cell<BT, AT>(a, i, j, os, ss, scf, scfact);
      return;
   }
   // (every lane takes part in the block and wavefront reductions)
   int r1 = 0;
   if (i < W) {
      const unsigned f = de_prep_cell<BT, AT>(a, i, j, os, ss, scf, scfact);
      if (f != DE_SKIP) r1 = (int)ceil(a.widths[f]);
   }
   if (a.blkmax) de_mark_block(a, i < W ? i : W - 1, j, r1);
   if (a.taps) {
      unsigned long long t = r1 > 0 ? (unsigned long long)(2 * r1 - 1) * (unsigned long long)(2 * r1 - 1) : 0ull;
      for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
      // (64 counters, so that the wavefronts' atomics do not all meet at one address)
      if ((threadIdx.x & 63) == 0 && t) atomicAdd(a.taps + ((blockIdx.x * 4u + (threadIdx.x >> 6)) & 63u), t);
   }
}

#define DG_REGION 16
#define DG_CHUNK 256

// The halo a workgroup's 16x16 region needs: the largest radius among the 16x16 blocks whose widest source can reach it (-1:
// none can), from the preparation pass's per-block maxima; without them the
// widest kernel's.  A smaller halo holds the same reaching sources in the same
// row-major order.  Ends with a barrier.
__device__ __forceinline__ int de_halo(const DEArgs &a, int bx, int by, int rx0, int rx1, int ry0, int ry1) {
   __shared__ int s_ext;
   const int R = a.half;
   if (a.blkmax) {
      if (threadIdx.x == 0) s_ext = -1;
      __syncthreads();
      const int nbx = a.nbx, nby = (a.height + DG_REGION - 1) / DG_REGION;
      const int span = (R + DG_REGION - 1) / DG_REGION, side = 2 * span + 1;
      for (int k = threadIdx.x; k < side * side; k += DG_CHUNK) {
         const int qx = bx + k % side - span, qy = by + k / side - span;
         if (qx < 0 || qy < 0 || qx >= nbx || qy >= nby) continue;
         const int bm = a.blkmax[qy * nbx + qx] - 1;
         const int qx0 = qx * DG_REGION, qy0 = qy * DG_REGION;
         const int gx = max(max(rx0 - (qx0 + DG_REGION - 1), qx0 - rx1), 0);
         const int gy = max(max(ry0 - (qy0 + DG_REGION - 1), qy0 - ry1), 0);
         if (bm >= 0 && gx <= bm && gy <= bm) atomicMax(&s_ext, min(bm, R));
      }
   }
   __syncthreads();
   return a.blkmax ? s_ext : R;
}

// Gather form: each thread owns one output cell and adds, in registers,
// the contribution of every source whose kernel reaches it, sources taken
// in row-major order -- the order in which the reference's single DE thread
// reaches a cell (rect.c:80-173) -- so the sum is deterministic and, in the
// exact mode, formed operation by operation as the reference forms it:
// ls = coef * k1 log(1 + c3 k2) / c3, c *= ls, accumulator += c (float
// accumulator: rounded once per contribution).  A workgroup covers 16x16
// cells (four 8x8 blocks, one per wavefront); it walks its halo in chunks of
// 256 cells, compacts the sources that reach it into LDS in order, and lists
// for each wavefront, in the same order, those that reach its block, so a
// wavefront loops over its own sources only.  No atomics.
// This is the exact form (verification, replay, and sources whose values are
// not finite); production renders take de_taps_body.
template <typename AT>
__device__ __forceinline__ void de_gather_body(const DEArgs &a, int bx, int by) {
   // per source: position, first coefficient of its kernel and radius; its
   // channels and log term
   __shared__ int radius[1024];
   __shared__ int4 s_src[DG_CHUNK];
   __shared__ double s_val[DG_CHUNK][5];
   __shared__ unsigned wave_cnt[DG_CHUNK / 64];
   __shared__ unsigned short s_list[4][DG_CHUNK];   // per 8x8 block: indices into the chunk's sources
   __shared__ unsigned list_cnt[4][DG_CHUNK / 64];  // [block][wavefront that listed them]
   const int W = a.width, H = a.height;
   const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
   const int rx0 = bx * DG_REGION, ry0 = by * DG_REGION;
   const int rx1 = min(rx0 + DG_REGION, W) - 1, ry1 = min(ry0 + DG_REGION, H) - 1;
   const int mx0 = rx0 + 8 * (wave & 1), my0 = ry0 + 8 * (wave >> 1);
   const int x = mx0 + (lane & 7), y = my0 + (lane >> 3);
   const bool live = x < W && y < H;
   AT *accp = (AT *)a.accum + (live ? (x + (long)y * W) * 4 : 0);
   AT acc[4] = {(AT)0, (AT)0, (AT)0, (AT)0};
   if (live)
      for (int c = 0; c < 4; c++) acc[c] = accp[c];
   for (int e = tid; e <= a.max_filter_index && e < 1024; e += DG_CHUNK) radius[e] = (int)ceil(a.widths[e]) - 1;
   const int E = de_halo(a, bx, by, rx0, rx1, ry0, ry1);
   const int hx0 = max(0, rx0 - E), hx1 = min(W, rx1 + 1 + E);
   const int hy0 = max(0, ry0 - E), hy1 = min(H, ry1 + 1 + E);
   const int hw = hx1 - hx0, nh = E < 0 ? 0 : hw * (hy1 - hy0);
   for (int base = 0; base < nh; base += DG_CHUNK) {
      const int s = base + tid;
      int flag = 0, sx = 0, sy = 0, fi = 0;
      if (s < nh) {
         sx = hx0 + s % hw;
         sy = hy0 + s / hw;
         const unsigned f = a.findex[sx + (long)sy * W];
         if (f != DE_SKIP) {
            fi = (int)f;
            const int r = radius[fi];
            const int gx = max(max(rx0 - sx, sx - rx1), 0), gy = max(max(ry0 - sy, sy - ry1), 0);
            flag = gx <= r && gy <= r;
         }
      }
      const unsigned long long m = __ballot(flag);
      const unsigned rank = __popcll(m & ((1ull << lane) - 1ull));
      if (lane == 0) wave_cnt[wave] = (unsigned)__popcll(m);
      __syncthreads();
      unsigned off = 0;
      for (int w = 0; w < wave; w++) off += wave_cnt[w];
      // the blocks (of the four 8x8 ones) this source reaches
      unsigned reach = 0;
      if (flag) {
         const int r = radius[fi];
         for (int b = 0; b < 4; b++) {
            const int bx0 = rx0 + 8 * (b & 1), by0 = ry0 + 8 * (b >> 1);
            reach |= (unsigned)(sx + r >= bx0 && sx - r <= bx0 + 7 && sy + r >= by0 && sy - r <= by0 + 7) << b;
         }
      }
      unsigned brank[4];
      for (int b = 0; b < 4; b++) {
         const unsigned long long mb = __ballot((reach >> b) & 1u);
         brank[b] = (unsigned)__popcll(mb & ((1ull << lane) - 1ull));
         if (lane == 0) list_cnt[b][wave] = (unsigned)__popcll(mb);
      }
      if (flag) {
         const unsigned idx = off + rank;
         const long cell = sx + (long)sy * W;
         s_src[idx] = make_int4(sx, sy, fi * a.kernel_size, radius[fi]);
         for (int c = 0; c < 4; c++) s_val[idx][c] = bucket_value(a.buckets, cell * 5 + c, (AT)0);
         s_val[idx][4] = a.srcl[cell];
      }
      __syncthreads();
      unsigned nb = 0;
      for (int b = 0; b < 4; b++) {
         unsigned boff = 0;
         for (int w = 0; w < DG_CHUNK / 64; w++)
            if (w < wave) boff += list_cnt[b][w];
         if ((reach >> b) & 1u) s_list[b][boff + brank[b]] = (unsigned short)(off + rank);
      }
      for (int w = 0; w < DG_CHUNK / 64; w++) nb += list_cnt[wave][w];
      __syncthreads();
      // (the coefficient is loaded for every listed source, from index 0
      // when the tap misses this cell, so that the loads of consecutive
      // sources overlap; a missed tap adds nothing)
#pragma unroll 4
      for (unsigned i = 0; i < nb; i++) {
         const unsigned k = s_list[wave][i];
         const int4 src = s_src[k];
         const int dx = abs(x - src.x), dy = abs(y - src.y);
         const int hi = max(dx, dy), lo = min(dx, dy);
         const bool tap = live && hi <= src.w;
         const long ci = tap ? (long)src.z + hi * (hi + 1) / 2 + lo : 0;
         const double coef = a.coefs[ci];
         if (tap && coef != 0.0) {
            const double c3 = s_val[k][3];
            const double ls = coef * s_val[k][4] / c3;
            for (int c = 0; c < 4; c++) acc[c] = (AT)((double)acc[c] + s_val[k][c] * ls);
         }
      }
      __syncthreads();
   }
   if (live)
      for (int c = 0; c < 4; c++) accp[c] = acc[c];
}

// The production gather: the sums of de_gather_body in the same row-major
// order, each contribution one fused multiply-add of the kernel's coefficient
// and the source's pre-scaled channels.  Bound by vector instructions, those
// of the taps and those that scan the halo for sources that reach.  A kernel's
// coefficients lie in a square table with a zero row and column at its edge,
// and the distances are clamped to that edge, so a tap costs three
// instructions for its address, without tests (a missed tap adds zero); the tables are in LDS where they fit (a wavefront
// reads 64 scattered coefficients per source).  A lane holds CELLS cells, some
// rows apart, which share the source's read and the x distance (FP64: side by
// side).  In FP32 the
// four channels are one matrix instruction, an outer product of four cells'
// coefficients and four channels whose every sum is one fused multiply-add
// with the bits of fmaf.  Each
// wavefront scans its own block's halo and lists its sources in LDS of its
// own: no barriers, and a tighter halo than a workgroup's.
// At 1920x1080 with 2x2 supersampling (8.4M cells, radius 9): 876 us with a
// workgroup's shared lists and tests per tap, 635 us so (2.75e8 vector
// instructions instead of 5.7e8; LDS is active for 60% of the time); 3840x2160
// with 3x3 in FP64 44.0 ms (each term formed per tap) against 15.3 ms (vector
// instructions and the vector caches' 64 addresses a load).
// Wavefronts of a workgroup (they share the tables).
constexpr int de_waves(int cells) { return cells == 2 ? 8 : 4; }
template <typename AT, int CELLS>
__device__ __forceinline__ void de_taps_body(const DEArgs &a, int bx, int by) {
   constexpr int SH = sizeof(AT) == 4 ? 2 : 3, NW = de_waves(CELLS), TURN = 32, CAP = TURN + 64;
   // a wavefront's block: BW cells across, CELLS times RW down (FP64 tables are
   // read from the vector caches: 21.4 ms with 8 across, 19.5 with 16, 22.4 with 32
   // in the 3840x2160 case above; FP32 ones from LDS: no difference)
   constexpr int BW = sizeof(AT) == 4 ? 8 : 16, ACROSS = 4 * NW / BW;
   // FP64: two cells side by side, so that one load of 16 bytes has both
   // coefficients (in that case two cells rows apart took 19.6 ms, side by side
   // 17.2, two and two 15.3)
   constexpr bool PAIR = sizeof(AT) == 8 && CELLS >= 2;
   constexpr int LW = PAIR ? BW / 2 : BW, RW = 64 / LW, BH = PAIR ? RW * CELLS / 2 : RW * CELLS;
   typedef typename std::conditional<sizeof(AT) == 4, float4, double4>::type V4;
   __shared__ int4 s_src[NW][CAP];   // per wavefront: x, y, its table's place, radius + 1
   __shared__ unsigned s_stride[NW][CAP];   // bytes of a row of its square
   __shared__ V4 s_val[NW][CAP];
   __shared__ int s_ext[NW];
   // the tables (tab_bytes), then per kernel its table's place (LDS address, or
   // byte offset in tab) and radius, and one that reaches nothing
   int2 *s_info = (int2 *)(fl3_lds + a.tab_bytes);
   typedef double two __attribute__((ext_vector_type(2), aligned(8)));
   typedef typename std::conditional<PAIR, two, AT>::type C;
   typedef const __attribute__((address_space(3))) C lds_at;
   const int nf = a.max_filter_index + 1;
   const int lds0 = a.tab_bytes ? (int)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)fl3_lds : 0;
   const int W = a.width, H = a.height;
   const int tid = threadIdx.x, lane = tid & 63;
   const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // (so that what depends on it is scalar)
   const int mx0 = (bx * ACROSS + wave % ACROSS) * BW, my0 = (by * (NW / ACROSS) + wave / ACROSS) * BH;
   const int mx1 = min(mx0 + BW, W) - 1, my1 = min(my0 + BH, H) - 1;
   const int x = mx0 + lane % LW * (BW / LW), y = my0 + lane / LW;
#pragma unroll 4
   for (int e = tid; e < a.tab_bytes / 16; e += 64 * NW) ((uint4 *)fl3_lds)[e] = ((const uint4 *)a.tab)[e];
   for (int e = tid; e <= nf; e += 64 * NW)
      s_info[e] = e < nf ? make_int2((a.info[2 * e] << SH) + lds0, a.info[2 * e + 1]) : make_int2(lds0, -(1 << 20));
   // acc[j][i]: FP32, channel lane & 3 of cell (px + i, y + RW j) of this lane's
   // four, as the matrix instruction leaves them; FP64, channel i of the lane's j-th
   constexpr bool MAT = sizeof(AT) == 4;
   const int px = MAT ? mx0 + (lane & (BW - 4)) : x;
   // from a lane's first cell to its j-th
   auto dxj = [](int j) { return PAIR ? j & 1 : 0; };
   auto dyj = [](int j) { return PAIR ? RW * (j >> 1) : RW * j; };
   typedef AT AV __attribute__((ext_vector_type(4)));
   AV acc[CELLS];
   auto at_acc = [&](int j, int i) {
      return (AT *)a.accum + ((px + dxj(j) + (MAT ? i : 0)) + (long)(y + dyj(j)) * W) * 4 + (MAT ? lane & 3 : i);
   };
   for (int j = 0; j < CELLS; j++)
      for (int i = 0; i < 4; i++)
         acc[j][i] = px + dxj(j) + (MAT ? i : 0) < W && y + dyj(j) < H ? *at_acc(j, i) : (AT)0;
   // this block's halo, as de_halo finds a region's
   int E = a.half;
   if (a.blkmax) {
      if (lane == 0) s_ext[wave] = -1;
      const int span = (a.half + DG_REGION - 1) / DG_REGION;
      const int bx0 = mx0 / DG_REGION - span, by0 = my0 / DG_REGION - span;
      const int cols = 2 * span + 1, rows = (my0 + BH - 1) / DG_REGION + span - by0 + 1;
      const int nby = (H + DG_REGION - 1) / DG_REGION;
      for (int k = lane; k < cols * rows; k += 64) {
         const int qx = bx0 + k % cols, qy = by0 + k / cols;
         if (qx < 0 || qy < 0 || qx >= a.nbx || qy >= nby) continue;
         const int bm = a.blkmax[qy * a.nbx + qx] - 1;
         const int gx = max(max(mx0 - (qx * DG_REGION + DG_REGION - 1), qx * DG_REGION - mx1), 0);
         const int gy = max(max(my0 - (qy * DG_REGION + DG_REGION - 1), qy * DG_REGION - my1), 0);
         if (bm >= 0 && gx <= bm && gy <= bm) atomicMax(&s_ext[wave], min(bm, a.half));
      }
   }
   __syncthreads();
   if (a.blkmax) E = __builtin_amdgcn_readfirstlane(s_ext[wave]);
   const int hx0 = max(0, mx0 - E), hx1 = min(W, mx1 + 1 + E);
   const int hy0 = max(0, my0 - E), hy1 = min(H, my1 + 1 + E);
   const int hw = hx1 - hx0, nh = E < 0 || mx0 >= W || my0 >= H ? 0 : hw * (hy1 - hy0);
   const V4 *srcv = (const V4 *)a.srcv;
   // U sources from the i-th on: all their reads before the first sum (the matrix
   // instruction keeps the compiler from unrolling a loop of single ones)
   auto taps_of = [&](int i, auto count, auto coef_at) {
      constexpr int U = decltype(count)::value;
      AT coef[U][CELLS];
      V4 val[U];
      float chan[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
         const int4 src = s_src[wave][i + u];
         const unsigned w = (unsigned)src.w;
         // (|x - y| of coordinates below 65536, whose high halves are zero)
         unsigned ax = min(__builtin_amdgcn_sad_u16((unsigned)x, (unsigned)src.x, 0u), w);
         if constexpr (PAIR) ax = min(ax, __builtin_amdgcn_sad_u16((unsigned)x + 1u, (unsigned)src.x, 0u));
         const unsigned row = (ax << SH) + (unsigned)src.z, stride = s_stride[wave][i + u];
         if constexpr (PAIR) {
            // the nearer cell's coefficient and the next one: the right cell is
            // the nearer to a source at its right
            for (int j = 0; j < CELLS; j += 2) {
               const unsigned ay = min(__builtin_amdgcn_sad_u16((unsigned)(y + dyj(j)), (unsigned)src.y, 0u), w);
               const auto c = coef_at(__umul24(ay, stride) + row);
               coef[u][j] = src.x > x ? c.y : c.x;
               coef[u][j + 1] = src.x > x ? c.x : c.y;
            }
         } else
            for (int j = 0; j < CELLS; j++) {
               const unsigned ay = min(__builtin_amdgcn_sad_u16((unsigned)(y + RW * j), (unsigned)src.y, 0u), w);
               coef[u][j] = coef_at(__umul24(ay, stride) + row);
            }
         if constexpr (MAT)
            chan[u] = ((const float *)&s_val[wave][i + u])[lane & 3];
         else
            val[u] = s_val[wave][i + u];
      }
#pragma unroll
      for (int u = 0; u < U; u++)
         for (int j = 0; j < CELLS; j++)
            if constexpr (MAT)
               acc[j] = __builtin_amdgcn_mfma_f32_4x4x1f32(coef[u][j], chan[u], acc[j], 0, 0, 0);
            else {
               acc[j][0] = fma(coef[u][j], val[u].x, acc[j][0]);
               acc[j][1] = fma(coef[u][j], val[u].y, acc[j][1]);
               acc[j][2] = fma(coef[u][j], val[u].z, acc[j][2]);
               acc[j][3] = fma(coef[u][j], val[u].w, acc[j][3]);
            }
   };
   auto taps = [&](int n, auto coef_at) {
      int i = 0;
      for (; i + 4 <= n; i += 4) taps_of(i, std::integral_constant<int, 4>(), coef_at);
      for (; i < n; i++) taps_of(i, std::integral_constant<int, 1>(), coef_at);
   };
   auto scan = [&](auto coef_at) {
      // the lane's cell of the next 64 halo cells (its place, its index), and
      // its kernel; the source it found among the 64 before, whose channels are
      // on their way
      int sx = hx0, sy = hy0, stepx = 0, stepy = 0;
      if (nh > 0) {
         sx += lane % hw;
         sy += lane / hw;
         stepx = 64 % hw;
         stepy = 64 / hw;
      }
      unsigned cell = fl3k_de_cell(sx, sy, W);
      const unsigned step = (unsigned)(stepx + stepy * W), wrap = (unsigned)(W - hw);
      auto kernel_at = [&](int k, unsigned c) {
         return k < nh ? (int)*(const uint16_t *)((const unsigned char *)a.findex + fl3k_de_findex_at(c)) : (int)DE_SKIP;
      };
      int fnext = kernel_at(lane, cell);
      int listed = 0, found = 0, at = -1;   // sources in the list, and with the last 64's
      int4 src = make_int4(0, 0, 0, 0);
      V4 val = {(AT)0, (AT)0, (AT)0, (AT)0};
      // (a block reaches as far as its distances from twice its middle)
      const unsigned mid2x = (unsigned)(2 * mx0 + BW - 1), mid2y = (unsigned)(2 * my0 + BH - 1);
      for (int base = 0; base < nh + 64; base += 64) {   // (one turn more for the last 64's)
         const int f = fnext, cx = sx, cy = sy;
         const unsigned cc = cell;
         sx += stepx;
         sy += stepy;
         cell += step;
         if (sx >= hx1) {
            sx -= hw;
            sy++;
            cell += wrap;
         }
         fnext = kernel_at(base + 64 + lane, cell);
         const int2 in = s_info[min(f, nf)];
         if (at >= 0) {
            s_src[wave][at] = src;
            s_stride[wave][at] = (unsigned)(src.w + fl3k_de_cols(sizeof(AT)) - 1) << SH;
            s_val[wave][at] = val;
         }
         listed = found;
         at = -1;
         const int dx2 = abs(2 * cx - (int)mid2x), dy2 = abs(2 * cy - (int)mid2y);
         const bool reach = dx2 <= 2 * in.y + BW - 1 && dy2 <= 2 * in.y + BH - 1;
         const unsigned long long m = __builtin_amdgcn_ballot_w64(reach);
         if (listed >= TURN) {
            __builtin_amdgcn_wave_barrier();
            const int n = listed & ~(TURN - 1);
            taps(n, coef_at);
            __builtin_amdgcn_wave_barrier();
            listed -= n;
            if (lane < listed) {
               s_src[wave][lane] = s_src[wave][n + lane];
               s_stride[wave][lane] = s_stride[wave][n + lane];
               s_val[wave][lane] = s_val[wave][n + lane];
            }
         }
         if (reach) {
            at = listed + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            src = make_int4(cx, cy, in.x, in.y + 1);
            val = srcv[cc];
         }
         found = listed + __popcll(m);
      }
      __builtin_amdgcn_wave_barrier();
      taps(listed, coef_at);
   };
   if (a.tab_bytes)
      scan([&](unsigned o) { return *(lds_at *)(uintptr_t)o; });
   else
      scan([&](unsigned o) { return *(const C *)((const unsigned char *)a.tab + o); });
   for (int j = 0; j < CELLS; j++)
      for (int i = 0; i < 4; i++)
         if (px + dxj(j) + (MAT ? i : 0) < W && y + dyj(j) < H) *at_acc(j, i) = acc[j][i];
}

__global__ __launch_bounds__(256) void k_fill_i32(int *p, long n, int v) {
   const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n) p[i] = v;
}

template <typename BT, typename AT>
__global__ __launch_bounds__(256) void k_de_prep(DEArgs a) {
   de_prep_body<BT, AT>(a, blockIdx.x, blockIdx.y);
}

template <typename AT>
__global__ __launch_bounds__(DG_CHUNK) void k_de_gather(DEArgs a) {
   if (a.nonfinite && !*a.nonfinite) return;   // (the production gather has run)
   de_gather_body<AT>(a, blockIdx.x, blockIdx.y);
}

template <typename AT, int CELLS>
__global__ __launch_bounds__(64 * de_waves(CELLS)) void k_de_taps(DEArgs a) {
   if (a.nonfinite && *a.nonfinite) return;   // (k_de_gather takes over)
   de_taps_body<AT, CELLS>(a, blockIdx.x, blockIdx.y);
}

// Several renders in one launch: workgroup b belongs to the render j with
// first[j] <= b < first[j + 1] and is that render's workgroup b - first[j]
// of a grid `cols` wide.
__device__ __forceinline__ int de_job(const unsigned *first, int n, unsigned b) {
   int lo = 0, hi = n - 1;
   while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (first[mid] <= b) lo = mid;
      else hi = mid - 1;
   }
   return lo;
}

template <typename BT, typename AT>
__global__ __launch_bounds__(256) void k_de_prep_many(const DEArgs *as, const unsigned *first, int n) {
   const int j = de_job(first, n, blockIdx.x);
   const DEArgs a = as[j];
   const unsigned local = blockIdx.x - first[j], cols = (unsigned)(a.width + 255) / 256;
   de_prep_body<BT, AT>(a, (int)(local % cols), (int)(local / cols));
}

template <int CELLS>
__global__ __launch_bounds__(64 * de_waves(CELLS)) void k_de_taps_many(const DEArgs *as, const unsigned *first, int n) {
   const int j = de_job(first, n, blockIdx.x);
   const DEArgs a = as[j];
   const unsigned local = blockIdx.x - first[j], cols = (unsigned)(a.width + 4 * de_waves(CELLS) - 1) / (4 * de_waves(CELLS));
   de_taps_body<float, CELLS>(a, (int)(local % cols), (int)(local / cols));
}

// Byte offset of the kernel index of cell (x, y), as the gather forms it (for
// tests).
extern "C" unsigned long long fl3k_de_findex_offset(int x, int y, int w) { return fl3k_de_findex_at(fl3k_de_cell(x, y, w)); }

// Cells a lane of the production gather holds, for regions of `blocks` 16x16
// blocks of cells in all: two where that leaves every CU several workgroups,
// one otherwise, where the gather is bound by how long a workgroup takes.
// Kernel time with one and two: 640x480 (1271 blocks) 40 and 59 us, 7.7k blocks
// 263 and 235 us, 32k blocks 838 and 672 us.  In FP64 four on large ones; one,
// two and four: 4.1k blocks 837, 660 and 684 us, 8.1k 1614, 1292 and 1356, 10.8k
// 2134, 1743 and 1729, the 3840x2160 case (147k) 17.2 ms with two, 15.3 with four.
extern "C" int fl3k_de_cells(long long blocks, int bits) { return blocks < 4096 ? 1 : bits != 64 || blocks < 16384 ? 2 : 4; }
// Cells across and down of a workgroup's region.
extern "C" void fl3k_de_region(int cells, int *w, int *h) {
   *w = 4 * de_waves(cells);
   *h = 16 * cells;
}

// Density estimation of n renders: per-render arguments in device memory,
// workgroup prefixes prep_first[n + 1] (rows of 256 cells) and
// gather_first[n + 1] (regions of fl3k_de_region(cells) cells).  bits
// 32/33 with the FP32 accumulator (production arithmetic) only.
// blkmax: a device array of nblk ints the renders' blkmax pointers point
// into (cleared here), or nullptr.
extern "C" int fl3k_launch_de_many(const DEArgs *as, const unsigned *prep_first, unsigned prep_blocks,
                                   const unsigned *gather_first, unsigned gather_blocks, int n, hipStream_t s,
                                   int *blkmax, long nblk, size_t gather_lds, int cells) {
   if (n <= 0) return 0;
   if (blkmax)
      hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((nblk + 255) / 256)), dim3(256), 0, s, blkmax, nblk, 0);
   hipLaunchKernelGGL((k_de_prep_many<uint32_t, float>), dim3(prep_blocks), dim3(256), 0, s, as, prep_first, n);
   if (cells == 2)
      hipLaunchKernelGGL(k_de_taps_many<2>, dim3(gather_blocks), dim3(64 * de_waves(2)), gather_lds, s, as, gather_first, n);
   else
      hipLaunchKernelGGL(k_de_taps_many<1>, dim3(gather_blocks), dim3(64 * de_waves(1)), gather_lds, s, as, gather_first, n);
   return hipGetLastError() != hipSuccess;
}

// Log scaling of every cell without DE (rect.c:947-974).
template <typename BT, typename AT>
__global__ __launch_bounds__(256) void k_logscale(const BT *b, AT *acc, long ncells, double k1, double k2) {
   const long cell = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (cell >= ncells) return;
   const double c3 = (double)b[cell * 5 + 3];
   if (c3 == 0.0) return;
   const double ls = (k1 * log(1.0 + c3 * k2)) / c3;
   for (int k = 0; k < 4; k++) {
      const double c = (double)b[cell * 5 + k] * ls;
      AT &d = acc[cell * 4 + k];
      if constexpr (std::is_same<AT, uint32_t>::value) {
         // 32-bit integer accumulator: saturating (flam3.c:3774-3776)
         d = (0xffffffffu - d > c) ? (uint32_t)((double)d + c) : 0xffffffffu;
      } else {
         d = (AT)((double)d + c);
      }
   }
}

// ------------------------------------------------------------------ tone map


__device__ __forceinline__ void tone_pixel(const double *t, double *out_rgb, double &alpha, const TMArgs &a) {
   double ls, newrgb[3];
   const double tmp = fl3_div255(t[3]);
   if (t[3] <= 0) {
      alpha = 0.0;
      ls = 0.0;
   } else {
      alpha = fl3_calc_alpha(tmp, a.g, a.linrange);
      ls = a.vibrancy * 256.0 * alpha / tmp;
      if (alpha < 0.0) alpha = 0.0;
      if (alpha > 1.0) alpha = 1.0;
   }
   fl3_calc_newrgb(t, ls, a.highpow, newrgb);
   // (of vibrancy 1 the term is zero times a power that is finite)
   const bool whole = a.vibrancy == 1.0 && a.g >= 0.0 && a.g <= 1.0;
   for (int k = 0; k < 3; k++) {
      double v = newrgb[k];
      if (!(whole && t[k] >= 0.0 && t[k] <= 1e300))
         v += (1.0 - a.vibrancy) * 256.0 * pow(fl3_div255(t[k]), a.g);
      if (a.nchan <= 3 || a.transp == 0)
         v += ((1.0 - alpha) * a.bg[k]);
      else
         v = (alpha > 0) ? v / alpha : 0;
      if (v > 255) v = 255;
      if (v < 0) v = 0;
      out_rgb[k] = v;
   }
}

// earlyclip: tone map every accumulator cell in place before filtering
// (rect.c:1086-1135).
template <typename AT>
__global__ __launch_bounds__(256) void k_earlyclip(AT *acc, long ncells, TMArgs a) {
   const long cell = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (cell >= ncells) return;
   AT *ac = acc + cell * 4;
   double t[4] = {(double)ac[0], (double)ac[1], (double)ac[2], (double)ac[3]}, rgb[3], alpha;
   tone_pixel(t, rgb, alpha, a);
   for (int k = 0; k < 3; k++) ac[k] = (AT)rgb[k];
   ac[3] = (AT)alpha;
}

// The filtered sum of a pixel from the cells at acc (rows `stride` cells apart).
template <typename AT>
__device__ __forceinline__ void filter_pixel(const TMArgs &a, const AT *acc, long stride, double *t) {
   for (int k = 0; k < 4; k++) t[k] = 0.0;
   for (int ii = 0; ii < a.fw; ii++)
      for (int jj = 0; jj < a.fw; jj++) {
         const double k = a.filter[ii + jj * a.fw];
         const AT *ac = acc + (ii + jj * stride) * 4;
         t[0] += k * (double)ac[0];
         t[1] += k * (double)ac[1];
         t[2] += k * (double)ac[2];
         t[3] += k * (double)ac[3];
      }
}

// Tone maps, clips and writes pixel (i, j) with the filtered sum t.
__device__ __forceinline__ void write_pixel(const TMArgs &a, int i, int j, double *t) {
   if (!a.earlyclip) {
      double rgb[3], alpha;
      tone_pixel(t, rgb, alpha, a);
      t[0] = rgb[0]; t[1] = rgb[1]; t[2] = rgb[2];
      t[3] = alpha;
   }
   unsigned char *p = a.out + (size_t)a.nchan * a.bpc * ((size_t)i + (size_t)j * a.iw);
   for (int k = 0; k < 3; k++) {
      double v = t[k];
      if (v > 255) v = 255;
      if (v < 0) v = 0;
      if (a.bpc == 2)
         ((unsigned short *)p)[k] = (unsigned short)(v * 256.0);
      else
         p[k] = (unsigned char)v;
   }
   if (t[3] > 1) t[3] = 1;
   if (t[3] < 0) t[3] = 0;
   if (a.nchan > 3) {
      if (a.transp == 1) {
         if (a.bpc == 2) ((unsigned short *)p)[3] = (unsigned short)(t[3] * 65535);
         else p[3] = (unsigned char)(t[3] * 255);
      } else {
         if (a.bpc == 2) ((unsigned short *)p)[3] = 65535;
         else p[3] = 255;
      }
   }
}

template <typename AT>
__device__ __forceinline__ void tonemap_body(const TMArgs &a, int bx, int by) {
   const int i = bx * blockDim.x + threadIdx.x;
   const int j = by;
   if (i >= a.iw || j >= a.ih) return;
   const int x = a.de_offset + i * a.os, y = a.de_offset + j * a.os;
   double t[4];
   filter_pixel<AT>(a, (const AT *)a.accum + (x + (long)y * a.W) * 4, a.W, t);
   write_pixel(a, i, j, t);
}

// ------------------------------------------------------------------ launchers

extern "C" int fl3k_launch_replay(const IterArgs *a, unsigned grid, size_t lds, hipStream_t s, int bits) {
   if (bits == 64)
      hipLaunchKernelGGL((k_iter_replay<64>), dim3(grid), dim3(64), lds, s, *a);
   else
      hipLaunchKernelGGL((k_iter_replay<33>), dim3(grid), dim3(64), lds, s, *a);
   return hipGetLastError() != hipSuccess;
}

// Up to this many walkers of a genome whose LDS image without the palette is
// lds_lone bytes one per wavefront (k_iterate_lone), more of them one per lane
// (k_iterate_points), whose time does not depend on their number: some rounds of
// what the chip holds at once, a wavefront a SIMD or fewer where the workgroups'
// LDS leaves no room for four a CU; four rounds for the classic variations, two for
// others, whose wavefronts are slower.  120 steps, ms, per wavefront and per lane:
// six xforms and a final one 1024 walkers 0.40 and 3.8, 4096 1.15 and 3.9; 63 xforms
// (one workgroup a CU) 1024 1.1 and 2.8, 3072 3.2 and 2.8; three xforms of the whole
// library 2048 4.3 and 5.6, 3072 6.4 and 5.6; 40 of 12 variations (one a CU) 512 8.0
// and 25.9, 2048 30.8 and 26.6.
extern "C" int fl3k_lone_walkers(size_t lds_lone, size_t lds_max, int ncu, int tier) {
   const size_t lds = lds_lone + sizeof(double) * 16 * FL3_MAX_XFORMS, at_once = lds < lds_max ? lds_max / lds : 1;
   return (tier == 0 ? 4 : 2) * ncu * (int)(at_once < 4 ? at_once : 4);
}

// lds, lds_lone: the genome's LDS image with and without the palette; lds_max: a CU's
extern "C" int fl3k_launch_points(const PointsArgs *a, size_t lds, size_t lds_lone, size_t lds_max, int ncu,
                                  hipStream_t s, int tier) {
   if (a->nwalkers > fl3k_lone_walkers(lds_lone, lds_max, ncu, tier))
      hipLaunchKernelGGL(k_iterate_points, dim3((a->nwalkers + 63) / 64), dim3(64), lds, s, *a);
   else if (tier == 0)
      hipLaunchKernelGGL(k_iterate_lone<0>, dim3(a->nwalkers), dim3(64), lds_lone, s, *a);
   else
      hipLaunchKernelGGL(k_iterate_lone<FL3_TIER_FULL>, dim3(a->nwalkers), dim3(64), lds_lone, s, *a);
   return hipGetLastError() != hipSuccess;
}

extern "C" int fl3k_launch_preview(const unsigned char *job, int xi, double range, int numvals, int depth,
                                   double *result, uint32_t *isaac, size_t lds, hipStream_t s) {
   hipLaunchKernelGGL(k_xform_preview, dim3(1), dim3(64), lds, s, job, xi, range, numvals, depth, result, isaac);
   return hipGetLastError() != hipSuccess;
}

extern "C" int fl3k_launch_deposit(const unsigned char *job, const double *pts, long long n, void *buckets,
                                   uint32_t *sat, unsigned grid, size_t lds, hipStream_t s, int bits) {
   if (bits == 64)
      hipLaunchKernelGGL(k_deposit_points<64>, dim3(grid), dim3(256), lds, s, job, pts, n, buckets, sat);
   else
      hipLaunchKernelGGL(k_deposit_points<33>, dim3(grid), dim3(256), lds, s, job, pts, n, buckets, sat);
   return hipGetLastError() != hipSuccess;
}

// exact: the reference's contributions one by one; else the production
// gather (a->tab ..., and, for the double accumulator, a->nonfinite)
extern "C" int fl3k_launch_de_tiled(const DEArgs *a, hipStream_t s, int bits, int exact) {
   const dim3 g1((a->width + 255) / 256, a->height), b1(256), b3(DG_CHUNK);
   const dim3 g3((a->width + DG_REGION - 1) / DG_REGION, (a->height + DG_REGION - 1) / DG_REGION);
   const int cells = fl3k_de_cells((long long)g3.x * g3.y, bits);
   int tw, th;
   fl3k_de_region(cells, &tw, &th);
   const dim3 gt((a->width + tw - 1) / tw, (a->height + th - 1) / th), bt(64 * de_waves(cells));
   const size_t lds = exact ? 0 : (size_t)a->tab_bytes + 8 * (size_t)(a->max_filter_index + 2);
   // per-block radii, cleared here and marked by the preparation pass, and
   // the flag behind them
   const long nblk = (a->blkmax ? (long)g3.x * g3.y : 0) + (a->nonfinite ? 1 : 0);
   int *clear = a->blkmax ? a->blkmax : a->nonfinite;
   if (nblk) hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((nblk + 255) / 256)), dim3(256), 0, s, clear, nblk, 0);
   if (bits == 64) {
      hipLaunchKernelGGL((k_de_prep<double, double>), g1, b1, 0, s, *a);
      if (!exact && cells == 4)
         hipLaunchKernelGGL((k_de_taps<double, 4>), gt, bt, lds, s, *a);
      else if (!exact && cells == 2)
         hipLaunchKernelGGL((k_de_taps<double, 2>), gt, bt, lds, s, *a);
      else if (!exact)
         hipLaunchKernelGGL((k_de_taps<double, 1>), gt, bt, lds, s, *a);
      hipLaunchKernelGGL(k_de_gather<double>, g3, b3, 0, s, *a);
   } else {
      hipLaunchKernelGGL((k_de_prep<uint32_t, float>), g1, b1, 0, s, *a);
      if (exact)
         hipLaunchKernelGGL(k_de_gather<float>, g3, b3, 0, s, *a);
      else if (cells == 2)
         hipLaunchKernelGGL((k_de_taps<float, 2>), gt, bt, lds, s, *a);
      else
         hipLaunchKernelGGL((k_de_taps<float, 1>), gt, bt, lds, s, *a);
   }
   return hipGetLastError() != hipSuccess;
}

extern "C" int fl3k_launch_logscale(const void *b, void *acc, long n, double k1, double k2, hipStream_t s,
                                    int bits) {
   const dim3 grid((unsigned)((n + 255) / 256)), block(256);
   if (bits == 64)
      hipLaunchKernelGGL((k_logscale<double, double>), grid, block, 0, s, (const double *)b, (double *)acc, n, k1, k2);
   else if (bits == 33)
      hipLaunchKernelGGL((k_logscale<uint32_t, float>), grid, block, 0, s, (const uint32_t *)b, (float *)acc, n, k1,
                         k2);
   else
      hipLaunchKernelGGL((k_logscale<uint32_t, uint32_t>), grid, block, 0, s, (const uint32_t *)b, (uint32_t *)acc,
                         n, k1, k2);
   return hipGetLastError() != hipSuccess;
}

template <typename AT>
__global__ __launch_bounds__(256) void k_tonemap(TMArgs a) {
   tonemap_body<AT>(a, blockIdx.x, blockIdx.y);
}

// The same by tiles of 32 x 4 pixels whose cells are read once, into LDS.  A
// wavefront of 64 pixels of k_tonemap walks fw rows of 64 os cells for each of
// its fw columns, more than a CU's vector cache holds for all of its wavefronts
// when cells are doubles, so every tap goes out to the L2 (3840x2160,
// supersample 3, 5 x 5 taps: 2.75 ms, 0.67 ms from LDS).
#define TM_TX 32
#define TM_TY 4
template <typename AT>
__global__ __launch_bounds__(TM_TX * TM_TY) void k_tonemap_lds(TMArgs a) {
   typedef AT v16 __attribute__((ext_vector_type(16 / sizeof(AT))));
   constexpr int PARTS = 4 * sizeof(AT) / 16;   // 16-byte loads per cell
   v16 *tile = (v16 *)fl3_lds;
   const int i0 = blockIdx.x * TM_TX, j0 = blockIdx.y * TM_TY;
   // the cells of the tile's pixels inside the image
   const int cols = (min(TM_TX, a.iw - i0) - 1) * a.os + a.fw, rows = (min(TM_TY, a.ih - j0) - 1) * a.os + a.fw;
   const v16 *acc = (const v16 *)a.accum + ((a.de_offset + i0 * a.os) + (long)(a.de_offset + j0 * a.os) * a.W) * PARTS;
   const int rowp = cols * PARTS, n = rows * rowp, step = TM_TX * TM_TY, stepr = step / rowp, stepc = step % rowp;
   int r = (int)threadIdx.x / rowp, c = (int)threadIdx.x % rowp;
   for (int e = threadIdx.x; e < n; e += 8 * step) {
      v16 v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
         if (e + u * step < n) v[u] = acc[(long)r * a.W * PARTS + c];
         r += stepr;
         c += stepc;
         if (c >= rowp) {
            c -= rowp;
            r++;
         }
      }
#pragma unroll
      for (int u = 0; u < 8; u++)
         if (e + u * step < n) tile[e + u * step] = v[u];
   }
   __syncthreads();
   const int lx = threadIdx.x % TM_TX, ly = threadIdx.x / TM_TX;
   if (i0 + lx >= a.iw || j0 + ly >= a.ih) return;
   double t[4];
   filter_pixel<AT>(a, (const AT *)fl3_lds + (lx + ly * cols) * a.os * 4, cols, t);
   write_pixel(a, i0 + lx, j0 + ly, t);
}

// Tone maps of several renders in one launch (workgroup prefixes as for
// k_de_taps_many; rows of 256 pixels).
template <typename AT>
__global__ __launch_bounds__(256) void k_tonemap_many(const TMArgs *as, const unsigned *first, int n) {
   const int j = de_job(first, n, blockIdx.x);
   const TMArgs a = as[j];
   const unsigned local = blockIdx.x - first[j], cols = (unsigned)(a.iw + 255) / 256;
   tonemap_body<AT>(a, (int)(local % cols), (int)(local / cols));
}

extern "C" int fl3k_launch_tonemap_many(const TMArgs *as, const unsigned *first, unsigned blocks, int n,
                                        hipStream_t s, int bits) {
   if (n <= 0 || blocks == 0) return 0;
   if (bits == 64)
      hipLaunchKernelGGL((k_tonemap_many<double>), dim3(blocks), dim3(256), 0, s, as, first, n);
   else if (bits == 33)
      hipLaunchKernelGGL((k_tonemap_many<float>), dim3(blocks), dim3(256), 0, s, as, first, n);
   else
      hipLaunchKernelGGL((k_tonemap_many<uint32_t>), dim3(blocks), dim3(256), 0, s, as, first, n);
   return hipGetLastError() != hipSuccess;
}

extern "C" int fl3k_launch_earlyclip(void *acc, long n, const TMArgs *a, hipStream_t s, int bits) {
   const dim3 grid((unsigned)((n + 255) / 256)), block(256);
   if (bits == 64)
      hipLaunchKernelGGL((k_earlyclip<double>), grid, block, 0, s, (double *)acc, n, *a);
   else if (bits == 33)
      hipLaunchKernelGGL((k_earlyclip<float>), grid, block, 0, s, (float *)acc, n, *a);
   else
      hipLaunchKernelGGL((k_earlyclip<uint32_t>), grid, block, 0, s, (uint32_t *)acc, n, *a);
   return hipGetLastError() != hipSuccess;
}

// Tiles of up to this many bytes, so that three workgroups share a CU; 1920x1080,
// direct and from LDS, us: supersample 1 with 3 x 3 taps 43 and 45 (floats), 49
// and 45 (doubles), 2 with 4 x 4 71 and 52, 147 and 81, 3 with 5 x 5 239 and 89,
// 581 and 186, 1 with 20 x 20 565 and 432, 969 and 518.
#define TM_LDS (52 << 10)
extern "C" int fl3k_launch_tonemap(const TMArgs *a, hipStream_t s, int bits) {
   const dim3 grid((a->iw + 255) / 256, a->ih), block(256);
   const long lds = (((long)TM_TX - 1) * a->os + a->fw) * (((long)TM_TY - 1) * a->os + a->fw) * 4 *
                    (bits == 64 ? sizeof(double) : sizeof(float));
   const dim3 gt((a->iw + TM_TX - 1) / TM_TX, (a->ih + TM_TY - 1) / TM_TY), bt(TM_TX * TM_TY);
   if (bits == 64 && lds <= TM_LDS)
      hipLaunchKernelGGL((k_tonemap_lds<double>), gt, bt, (size_t)lds, s, *a);
   else if (bits == 33 && lds <= TM_LDS)
      hipLaunchKernelGGL((k_tonemap_lds<float>), gt, bt, (size_t)lds, s, *a);
   else if (bits == 64)
      hipLaunchKernelGGL((k_tonemap<double>), grid, block, 0, s, *a);
   else if (bits == 33)
      hipLaunchKernelGGL((k_tonemap<float>), grid, block, 0, s, *a);
   else
      hipLaunchKernelGGL((k_tonemap<uint32_t>), grid, block, 0, s, *a);
   return hipGetLastError() != hipSuccess;
}
