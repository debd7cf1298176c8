// fl3_walker.h - the FP32 production walker kernel, instantiated per
// variation tier by fl3_kernels_fast.hip (full set) and fl3_kernels_tier.hip
// (the classic set and the classic set plus one block).
#ifndef FL3_WALKER_H
#define FL3_WALKER_H
#include "fl3_core.h"

// Record formats of the binned deposit (RECORDS template argument).
#define FL3_REC_DIRECT 0   // no records: deposit with atomics
#define FL3_REC_WIDE 1     // 8-byte records (make_record)
#define FL3_REC_NARROW 2   // 4-byte records: cell | palette index << 24
#define FL3_REC_JOB 3      // 8-byte records: cell, palette index, xform, job
                           // (or cell and the palette entry's four bytes)

// Records: row i of walker (workgroup b, thread t) at (b * rows_out + i) *
// 256 + t, so a workgroup's records are one contiguous block.
// Production walkers.  Walker (lane) w plots nsamples/W (+1 for the first
// nsamples%W walkers) points after `fuse` unplotted steps from a random
// start, the per-sub-batch procedure of rect.c:393-400 with one long
// sub-batch per walker; with WAVE (genomes without xaos) the xform is drawn
// per wavefront and the workgroup's points change lanes after every step.  In
// record mode each workgroup also counts its records per tile in LDS.
// Waves per SIMD the walker kernel is compiled for: the classic tier (the
// variations of most genomes) at 8, which holds it to 64 VGPRs (a few
// spills; 7 waves at its natural 67-78 VGPRs ran 11% slower per launch),
// the larger tiers at their natural register counts.
template <int TIER>
constexpr int walker_waves() { return TIER == 0 ? 8 : 1; }

// ---- one xform per wavefront ------------------------------------------
//
// What bounds these walkers: VALU issue on a full chip, and on a launch of a
// few workgroups the latency of one step (a walker's steps are serial).  The
// wavefront's xform is the same in all lanes, so everything about it lives in
// scalar registers: its constants and a bit mask of the classic variations
// present come in two scalar loads issued before the point exchange of the
// step before, the variations' weights in three more when it is applied (all
// of it ahead took more scalar registers than there are).  The variations are
// taken by tests of that mask in ascending order, each an if without else: a
// loop over a list with a switch over ids compiled to a chain of some
// thirteen scalar branches per variation, most of a lone wavefront's step.
// The hashes of 64 steps' draws are computed at once, a step per lane.
// Measured (kernel trace): a 2.59e8-sample launch of the 1080p still 2.23 ->
// 1.47 ms, 249 -> 184 VALU and 203 -> 103 SALU instructions per
// sample; the 228 steps of a 256 x 256 preview of 28160 walkers, 283 -> 171 us.
typedef uint32_t fl3_u32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t fl3_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t fl3_u32x2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(4))) uint32_t fl3_cu32;
typedef const __attribute__((address_space(4))) fl3_u32x8 fl3_cu32x8;
typedef const __attribute__((address_space(4))) fl3_u32x4 fl3_cu32x4;
typedef const __attribute__((address_space(4))) fl3_u32x2 fl3_cu32x2;
struct WaveXf {   // words 0-7 and 8-11 of the walker table's row
   fl3_u32x8 a;
   fl3_u32x4 b;
   __device__ float f(int k) const { return __uint_as_float(a[k]); }
   __device__ uint32_t u(int k) const { return b[k - 8]; }
};
struct WaveW {    // words 16-29: the classic variations' weights
   fl3_u32x8 a;
   fl3_u32x4 b;
   fl3_u32x2 c;
   __device__ float f(int v) const { return __uint_as_float(v < 8 ? a[v & 7] : v < 12 ? b[v & 3] : c[v & 1]); }
};

__device__ __forceinline__ WaveXf wave_xf(fl3_cu32 *wt, int fn) {
   WaveXf x;
   x.a = *(fl3_cu32x8 *)(wt + fn * FL3_WT_WORDS);
   x.b = *(fl3_cu32x4 *)(wt + fn * FL3_WT_WORDS + 8);
   return x;
}

// The classic variations LO.. HI - 1 of the wavefront's xform.  (The empty
// asm keeps a case behind its branch: without it the short ones are computed
// always and selected.)
template <int LO, int HI, class RNG>
__device__ __forceinline__ void wave_classic(uint32_t mask, const WaveW &w, const XfL<float> &X, Pre<float> &f,
                                             RNG &rng) {
   if constexpr (HI - LO == 1) {
      if (mask & (1u << LO)) {
         asm volatile("");
         fl3_var<float, RNG, LO, HI>(LO, w.f(LO), X, f, rng);
      }
   } else {
      wave_classic<LO, LO + 1>(mask, w, X, f, rng);
      wave_classic<LO + 1, HI>(mask, w, X, f, rng);
   }
}

// apply_xform for the wavefront's xform fn (row x of the walker table), the
// same arithmetic term by term; a bad value is left in q.
template <int TIER>
__device__ __forceinline__ bool wave_apply(const GenL<float> &G, int fn, const WaveXf &x, const float *p, float *q,
                                           WalkerRng &rng) {
   const uint32_t flags = x.u(FL3_WT_FLAGS), mask = x.u(FL3_WT_MASK);
   fl3_cu32 *row = G.wt + fn * FL3_WT_WORDS;
   WaveW w;
   w.a = *(fl3_cu32x8 *)(row + FL3_WT_W);
   w.b = *(fl3_cu32x4 *)(row + FL3_WT_W + 8);
   w.c = *(fl3_cu32x2 *)(row + FL3_WT_W + 12);
   Pre<float> f;
   q[2] = fmaf(x.f(FL3_WT_CSPEED), x.f(FL3_WT_COLOR) - p[2], p[2]);
   q[3] = __uint_as_float(x.u(FL3_WT_VIS));
   f.tx = fmaf(x.f(0), p[0], fmaf(x.f(2), p[1], x.f(4)));
   f.ty = fmaf(x.f(1), p[0], fmaf(x.f(3), p[1], x.f(5)));
   if (flags & FL3_HAS_PREBLUR) {  // pre_blur :1480
      const float g0 = u01<float>(rng), g1 = u01<float>(rng), g2 = u01<float>(rng), g3 = u01<float>(rng);
      const float rndG = __uint_as_float(row[FL3_WT_PREBLUR]) * (g0 + g1 + g2 + g3 - 2.0f);
      const float rndA = u01<float>(rng) * 2.0f * (float)M_PI;
      float sA, cA;
      m_sincos(rndA, &sA, &cA);
      f.tx += rndG * cA;
      f.ty += rndG * sA;
   }
   f.sumsq = f.tx * f.tx + f.ty * f.ty;
   f.sq = m_sqrt(f.sumsq);
   f.atan = f.sina = f.cosa = f.atanyx = 0.0f;
   if (flags & FL3_PRE_ATAN_XY) f.atan = m_atan2(f.tx, f.ty);
   if (flags & FL3_PRE_ANGLES) {
      asm volatile("");
      f.sina = m_div(f.tx, f.sq);
      f.cosa = m_div(f.ty, f.sq);
   }
   if (TIER != 0 && (flags & FL3_PRE_ATAN_YX)) f.atanyx = m_atan2(f.ty, f.tx);
   f.p0 = 0.0f;
   f.p1 = 0.0f;
   const XfL<float> &X = G.xf[fn];
   // Of the classic variations only julia draws, one word; in the classic
   // tier it is drawn here, so that the lane's stream does not change among
   // the variations (the other tiers' variations draw in their order).
   struct WordRng {
      uint32_t w;
      __device__ uint32_t next() { return w; }
   } wr;
   if constexpr (TIER == 0) {
      wr.w = 0u;
      if (flags & FL3_DRAWS_JULIA) wr.w = rng.next();
   }
   auto classic = [&](auto &r) {
      if (mask & 0x000fu) wave_classic<0, 4>(mask, w, X, f, r);
      if (mask & 0x00f0u) wave_classic<4, 8>(mask, w, X, f, r);
      if (mask & 0x3f00u) wave_classic<8, 14>(mask, w, X, f, r);
   };
   if constexpr (TIER == 0)
      classic(wr);
   else {
      classic(rng);
      const __attribute__((address_space(4))) int32_t *vl = G.vlc + fn * (2 + 2 * G.nunion);
      const int nv = (int)x.u(FL3_WT_COUNT);
      const uint32_t xoff = (uint32_t)((const unsigned char *)&X - fl3_lds);
      for (int k = __builtin_popcount(mask); k < nv; k++) {
         const int v = vl[2 + 2 * k];
         const float wv = __int_as_float(vl[3 + 2 * k]);
         uint32_t o = xoff;
         asm volatile("" : "+v"(o));
         opaque_pre(f);
         if constexpr (TIER == FL3_TIER_FULL)
            fl3_var<float, WalkerRng, FL3_CLASSIC, FL3_NVAR>(v, wv, *(const XfL<float> *)(fl3_lds + o), f, rng);
         else
            fl3_var<float, WalkerRng, fl3_tier_lo(TIER), fl3_tier_hi(TIER)>(v, wv, *(const XfL<float> *)(fl3_lds + o),
                                                                            f, rng);
      }
   }
   q[0] = f.p0;
   q[1] = f.p1;
   if (flags & FL3_HAS_POST) {
      auto P = [&](int k) { return __uint_as_float(row[FL3_WT_POST + k]); };
      q[0] = fmaf(P(0), f.p0, fmaf(P(2), f.p1, P(4)));
      q[1] = fmaf(P(1), f.p0, fmaf(P(3), f.p1, P(5)));
   }
   return fl3_bad(q[0]) || fl3_bad(q[1]);
}

// A bad value's random replacement (flam3.c:257-270).
__device__ __forceinline__ void random_point(float *q, WalkerRng &rng) {
   q[0] = u11<float>(rng);
   q[1] = u11<float>(rng);
}

// The hardware's conversion (towards zero, saturating, 0 for NaN) of a value
// that may be out of range.
__device__ __forceinline__ int cvt_i32(float x) {
   int r;
   asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x));
   return r;
}

// The integers a record needs, in vector registers: the scalar ones are all
// taken, and what does not fit there is read back lane by lane at each use.
struct RecordV {
   unsigned width, ncells, m1, cell0, shift, hist;
   __device__ void pin() {
      asm volatile("" : "+v"(width), "+v"(ncells), "+v"(m1), "+v"(cell0), "+v"(shift), "+v"(hist));
   }
};

// make_record for a stepped palette and visibility 1, computed in every lane
// without branches: false if the point has no cell, else its cell and palette
// index.  rot: the camera rotates (a scalar).
__device__ __forceinline__ bool stepped_record(const GenL<float> &G, const RecordV &v, int rot, const float *q,
                                               unsigned &cell, unsigned &ci) {
   float x = q[0], y = q[1];
   if (rot) {
      asm volatile("");
      const float x0 = x - G.rc0, y0 = y - G.rc1;
      x = fmaf(x0, G.rot00, y0 * G.rot01) + G.rc0;
      y = fmaf(x0, G.rot10, y0 * G.rot11) + G.rc1;
   }
   const bool in = x >= G.b0 && y >= G.b1 && x <= G.b2 && y <= G.b3;
   const int ix = cvt_i32(fmaf(G.ws0, x, -G.wb0s0)), iy = cvt_i32(fmaf(G.hs1, y, -G.hb1s1));
   cell = (unsigned)ix + __umul24(v.width, (unsigned)iy);
   const int c = cvt_i32(q[2] * (float)G.cmap_size);
   ci = (unsigned)max(min(c, (int)v.m1), 0);
   return in && cell < v.ncells;
}

// The palette index | xform << 8 | fraction << 16 of make_record's 8-byte records,
// without its branches and 64-bit conversions (47M records of 1021x767 at 2x2
// with a linear palette: the walkers' kernel 539 us, 492 us so).
__device__ __forceinline__ unsigned wide_colour(const GenL<float> &G, const RecordV &v, int linear, float colour, int fn) {
   const float di = colour * (float)G.cmap_size;
   const int c = cvt_i32(di), m1 = (int)v.m1;
   if (!linear) return (unsigned)max(min(c, m1), 0) | (unsigned)fn << 8;
   const float f = c < 0 ? 0.0f : c >= m1 ? 1.0f : di - (float)c;
   return (unsigned)max(min(c, m1 - 1), 0) | (unsigned)fn << 8 |
          (unsigned)(fminf(fmaxf(f, 0.0f), 1.0f) * 65535.0f + 0.5f) << 16;
}

template <int BITS, bool EXACT, int RECORDS, int TIER, bool WAVE>
__global__ __launch_bounds__(256, walker_waves<TIER>()) void k_iter_fast(IterArgs a) {
   unsigned char *lds = fl3_lds;
   GenL<float> G;
   // independent renders: direct deposits, or job or 4-byte records in one
   // cell space
   const bool dmode = RECORDS != FL3_REC_WIDE && a.descs;
   const int djob = dmode ? a.blk_job[blockIdx.x] : 0;
   const JobDesc *dsc = dmode ? a.descs + djob : nullptr;
   const int nj = !dsc && a.njobs > 1 ? a.njobs : 1;
   const int jb = nj > 1 ? (int)(blockIdx.x % nj) : 0;
   // record modes leave the colours to the tile accumulation: no palette in LDS
   load_genome<float>(dsc ? a.jobs + dsc->off : (nj > 1 ? a.jobs + a.job_off[jb] : a.job), lds, G,
                      RECORDS == FL3_REC_DIRECT);
   unsigned *bh = (unsigned *)(lds + a.hist_off);
   if (RECORDS)
      for (int b = threadIdx.x; b < a.nbins; b += blockDim.x) bh[b] = 0;
   uint32_t *pal = (uint32_t *)(lds + a.pal_off);
   if (RECORDS == FL3_REC_JOB && a.pal8) {
      const uint32_t *src = a.pal8 + (size_t)(dsc ? djob : jb) * 256;
      for (int e = threadIdx.x; e < 256; e += blockDim.x) pal[e] = src[e];
   }
   __syncthreads();
   // W, wid: the record matrix and walker-state layout over all jobs (with
   // independent renders the launch may cover only the columns from
   // workgroup blk0 on); Wj, wj: this walker's job-local count and index
   const long long W = a.wtot ? a.wtot : (long long)gridDim.x * blockDim.x;
   const long long blk = (long long)a.blk0 + blockIdx.x;
   const long long wid = blk * blockDim.x + threadIdx.x;
   const long long Wj = dsc ? (long long)dsc->nblocks * blockDim.x : (long long)(gridDim.x / nj) * blockDim.x;
   const long long wj = dsc ? (long long)(blockIdx.x - dsc->block0) * blockDim.x + threadIdx.x
                            : (long long)(blockIdx.x / nj) * blockDim.x + threadIdx.x;
   long long nsj = dsc ? dsc->nsamples : a.nsamples;
   if (!dsc && a.job_ns) {   // this chunk's share of the job's own count
      const long long rem = a.job_ns[jb] - a.ns_row0 * Wj;
      nsj = rem < 0 ? 0 : (rem < nsj ? rem : nsj);
   }
   long long n = nsj / Wj + (wj < nsj % Wj ? 1 : 0);
   // independent renders with records run in chunks of rows [row0, row0 + rows_out)
   if (dsc && RECORDS) n = n - a.row0 < 0 ? 0 : (n - a.row0 < a.rows_out ? n - a.row0 : a.rows_out);
   const unsigned long long cell0 = dsc ? (unsigned long long)dsc->cell0 : 0ull;
   // deposit target and counters: the job's render
   void *const buckets = !dsc ? a.buckets
                         : BITS == 64 ? (void *)((double *)a.buckets + dsc->cell0 * 5)
                                      : (void *)((uint32_t *)a.buckets + dsc->cell0 * 5);
   unsigned long long *const badp = dsc ? a.badvals + 2 * dsc->render : a.badvals;
   uint32_t *const satp = dsc ? (uint32_t *)(a.badvals + 2 * dsc->render + 1) : a.sat;
   WalkerRng rng;
   float p[4], q[4];
   int lastxf = 0, consec = 0;
   uint32_t *ws = a.wstate;
   if (a.resume) {
      for (int k = 0; k < 4; k++) p[k] = __uint_as_float(ws[k * W + wid]);
      rng.s0 = ws[4 * W + wid];
      rng.s1 = ws[5 * W + wid];
      rng.s2 = ws[6 * W + wid];
      rng.s3 = ws[7 * W + wid];
      lastxf = (int)ws[8 * W + wid];
      consec = (int)ws[9 * W + wid];
   } else {
      if (dsc)
         rng.seed(dsc->key0, dsc->key1, (uint64_t)wj);
      else if (nj > 1)
         rng.seed(a.keys[2 * jb], a.keys[2 * jb + 1], (uint64_t)wj);
      else
         rng.seed(a.key0, a.key1, (uint64_t)wid);
      p[0] = u11<float>(rng);
      p[1] = u11<float>(rng);
      p[2] = u01<float>(rng);
      p[3] = u01<float>(rng);
   }
   uint32_t bad = 0;
   const bool use_final = G.final_index >= 0;
   // the record (or deposit) of plotted point v at row i
   auto plot = [&](long long i, const float *v, int fn) {
      if (RECORDS == FL3_REC_WIDE) {
         const unsigned long long r = make_record<float>(G, v, fn);
         a.rec[(blk * a.rows_out + i) * 256 + threadIdx.x] = r;
         if ((unsigned)r != FL3_REC_NONE) atomicAdd(&bh[(unsigned)r >> a.bin_shift], 1u);
      } else if (RECORDS == FL3_REC_JOB) {
         // independent renders: the render's first cell moves the cell
         // into the launch's cell space, the job is the descriptor's
         // (palettes as bytes: every job's palette is stepped and every
         // visibility 1, the 4-byte records' case)
         const unsigned long long r = a.pal8 ? make_record<float, true>(G, v, fn) : make_record<float>(G, v, fn);
         const unsigned cell = (unsigned)r == FL3_REC_NONE ? FL3_REC_NONE : (unsigned)(r + cell0);
         const unsigned long long hi = a.pal8 ? (unsigned long long)pal[(r >> 32) & 0xff] << 32
                                              : (r & 0xffff00000000ull) | ((unsigned long long)(dsc ? djob : jb) << 48);
         a.rec[(blk * a.rows_out + i) * 256 + threadIdx.x] =
             cell == FL3_REC_NONE ? (unsigned long long)FL3_REC_NONE : (hi | cell);
         if (cell != FL3_REC_NONE) atomicAdd(&bh[cell >> a.bin_shift], 1u);
      } else if (RECORDS == FL3_REC_NARROW) {
         // (independent renders sharing one palette: the render's first
         // cell moves the cell into the launch's cell space)
         const unsigned long long r = make_record<float, true>(G, v, 0);   // (4-byte records: a stepped palette)
         const unsigned cell = (unsigned)r == FL3_REC_NONE ? FL3_REC_NONE : (unsigned)(r + cell0);
         ((unsigned *)a.rec)[(blk * a.rows_out + i) * 256 + threadIdx.x] =
             cell == FL3_REC_NONE ? FL3_REC_NONE : (cell | ((unsigned)(r >> 32) & 0xffu) << 24);
         if (cell != FL3_REC_NONE) atomicAdd(&bh[cell >> a.bin_shift], 1u);
      } else
         deposit<float, BITS, EXACT>(G, v, buckets, satp, a.bytes != 0);
   };
   if constexpr (WAVE) {
      // One xform per wavefront and step (drawn from a hash of the
      // wavefront's seed, the step and the draw within the step, in scalar
      // registers), so a wavefront evaluates that xform's variations only; after
      // every step the workgroup's 256 points move to other lanes through a
      // random permutation (slot = m (t ^ x) + o mod 256, m odd, from a hash
      // of the job's key, the job-local workgroup and the step), so the
      // xforms a point meets are independent draws with the xforms'
      // probabilities, as in the per-lane chaos game.  Lanes keep their own
      // streams and sample counts; a lane past its count keeps moving points
      // without plotting until the workgroup is done.
      float *xb = (float *)(lds + a.shuf_off);
      const uint64_t kk = dsc ? dsc->key0 : (nj > 1 ? a.keys[2 * jb] : a.key0);
      const uint32_t bjob = dsc ? (uint32_t)(blockIdx.x - dsc->block0)
                                : (nj > 1 ? (uint32_t)(blockIdx.x / nj) : (uint32_t)blk);
      const uint32_t hseed = ((uint32_t)kk ^ (uint32_t)(kk >> 32) * 0x85ebca6bu) ^ bjob * 0xc2b2ae35u;
      // the wavefront's xform draws: draw k of step st is
      // fmix32(wseed ^ (st * 0xcc9e2d51 + k * 0x1b873593)), the 32-bit
      // finaliser of MurmurHash3 (Appleby), over a seed mixed from the
      // workgroup's and the wavefront's index (so it depends on the job-local
      // workgroup, like the permutation, and not on the launch)
      auto fmix32 = [](uint32_t h) {
         h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
         return h;
      };
      const uint32_t wseed = fmix32(hseed + 0x632be5abu * ((uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + 1u));
      auto wdraw = [&](uint32_t step, uint32_t k) { return fmix32(wseed ^ (step * 0xcc9e2d51u + k * 0x1b873593u)); };
      // The xform at the first slot of each 128-slot bucket of the 14-bit
      // selection slot, and the first slot of the next xform: a draw starts
      // there and rarely has to step over more breakpoints inside its bucket
      // (select_xform's count, in fewer steps).
      uint32_t *sel = (uint32_t *)(xb + 1536);
      if (threadIdx.x < 128) {
         const uint32_t b0 = threadIdx.x * 128u;
         int f = 0;
         for (int j = 1; j < G.nstd; j++) f += b0 >= (uint32_t)G.starts[j] ? 1 : 0;
         sel[threadIdx.x] = (uint32_t)f << 16 | (f + 1 < G.nstd ? min((uint32_t)G.starts[f + 1], 16384u) : 16384u);
      }
      __syncthreads();
      // (per lane)
      auto pick = [&](uint32_t slot) {
         const uint32_t e = sel[slot >> 7];
         int f = (int)(e >> 16);
         if (slot >= (e & 0xffffu)) {
            f++;
            while (f + 1 < G.nstd && slot >= (uint32_t)G.starts[f + 1]) f++;
         }
         return f;
      };
      // What the wavefront needs of step st's draws: the xform << 24 and the
      // point exchange's m, x and o in a byte each.  Lane l of `draws` holds
      // step (st & ~63) + l: the hashes of 64 steps take as many vector
      // instructions as one step's take scalar ones, and a step reads its
      // lane.
      auto draw_block = [&](uint32_t st) {
         st = (st & ~63u) + (threadIdx.x & 63u);
         uint32_t h = st * 0x9E3779B9u ^ hseed;
         h ^= h >> 16; h *= 0x7feb352du; h ^= h >> 15; h *= 0x846ca68bu; h ^= h >> 16;
         return (uint32_t)pick(wdraw(st, 0u) & 16383u) << 24 | (h & 0xffffffu) | 1u;
      };
      // (the step count and the workgroup's step bound are the same in
      // every lane: read from the first lane, they live in scalar registers)
      uint32_t st = a.resume ? (uint32_t)__builtin_amdgcn_readfirstlane(lastxf) : 0u;
      // every lane takes one step at a time, so i is the same in all lanes
      // and the workgroup runs until its first walker (the one with the
      // most samples) is done; the others have that many samples or one fewer
      long long nwg = nsj / Wj + ((wj - (long long)threadIdx.x) < nsj % Wj ? 1 : 0);
      if (dsc && RECORDS) nwg = nwg - a.row0 < 0 ? 0 : (nwg - a.row0 < a.rows_out ? nwg - a.row0 : a.rows_out);
      nwg = (long long)(((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(nwg >> 32)) << 32) |
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)nwg));
      const bool full = n == nwg;
      // bit 0: the camera rotates, 1: a final xform, 2: at every step; then its index
      const int what = __builtin_amdgcn_readfirstlane((G.rotate ? 1 : 0) | (use_final ? 2 : 0) |
                                                      (G.final_opacity == 1.0f ? 4 : 0) | G.final_index << 3);
      const int linear = __builtin_amdgcn_readfirstlane(G.palette_mode == 1);
      // the step's record row (4- and 8-byte records)
      unsigned char *row = (unsigned char *)a.rec + blk * a.rows_out * (RECORDS == FL3_REC_NARROW ? 1024 : 2048);
      RecordV rv = {(unsigned)G.width, (unsigned)G.width * (unsigned)G.height, (unsigned)(G.cmap_size - 1),
                    (unsigned)cell0, (unsigned)a.bin_shift, a.hist_off};
      rv.pin();
      auto count = [&](unsigned cell) { atomicAdd((unsigned *)(lds + (rv.hist + (cell >> rv.shift) * 4u)), 1u); };
      auto wplot = [&](long long i, const float *v, int fn) {
         if constexpr (RECORDS == FL3_REC_NARROW) {
            unsigned cell, ci;
            const bool in = stepped_record(G, rv, what & 1, v, cell, ci);
            cell += rv.cell0;
            *(unsigned *)(row + threadIdx.x * 4u) = in ? (cell | ci << 24) : FL3_REC_NONE;
            if (in) count(cell);
         } else if constexpr (RECORDS == FL3_REC_JOB) {
            if (a.pal8) {
               unsigned cell, ci;
               const bool in = stepped_record(G, rv, what & 1, v, cell, ci);
               cell += rv.cell0;
               const unsigned long long r = (unsigned long long)pal[ci & 0xffu] << 32 | cell;
               *(unsigned long long *)(row + threadIdx.x * 8u) = in ? r : (unsigned long long)FL3_REC_NONE;
               if (in) count(cell);
            } else
               plot(i, v, fn);
         } else if constexpr (RECORDS == FL3_REC_WIDE) {
            unsigned cell, ci;
            bool in = stepped_record(G, rv, what & 1, v, cell, ci);
            in = in && v[3] != 0.0f;
            const unsigned long long r = (unsigned long long)wide_colour(G, rv, linear, v[2], fn) << 32 | cell;
            *(unsigned long long *)(row + threadIdx.x * 8u) = in ? r : (unsigned long long)FL3_REC_NONE;
            if (in) count(cell);
         } else
            plot(i, v, fn);
      };
      long long i = a.resume ? 0 : -a.fuse;
      if (i >= nwg) i = nwg - 1;   // (a chunk past the workgroup's samples: one step, not plotted)
      // (a step's xform is drawn, and its constants loaded, during the step
      // before)
      uint32_t draws = draw_block(st);
      uint32_t draw = (uint32_t)__builtin_amdgcn_readlane((int)draws, (int)(st & 63u));
      int fs = (int)(draw >> 24);
      WaveXf x = wave_xf(G.wt, fs);
      for (;;) {
         int fn = fs;
         // A bad value (flam3.c:257-270): the point restarts from the
         // random replacement apply_xform left in q and the step is retried
         // with a new xform, up to four times; the fifth bad value in a row
         // is kept.  The retries stay inside the step (the lanes without a
         // bad value wait), each retry's xform the step's next wavefront
         // draw, so every lane still plots exactly one point per step and
         // chunked launches follow the single launch.
         // Bad values are counted on plotted steps only: the reference's
         // count holds its fuse steps too (15 per 10000-sample sub-batch,
         // 0.15% of its steps), but a walker fuses 100 steps, which for
         // small renders would be a large share of the count.
         bool pend = wave_apply<TIER>(G, fs, x, p, q, rng);
         if (__builtin_amdgcn_ballot_w64(pend)) {
            int nbad = 0;
            uint32_t kdraw = 0;
            if (pend) random_point(q, rng);
            do {
               // (the retry's xform is drawn outside the branch, like the
               // step's own draw)
               const int f2 = __builtin_amdgcn_readfirstlane(pick(wdraw(st, ++kdraw) & 16383u));
               const WaveXf x2 = wave_xf(G.wt, f2);
               if (pend) {
                  if (i >= 0 && i < n) bad++;
                  if (++nbad < 5) {
                     p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
                     fn = f2;
                     pend = wave_apply<TIER>(G, f2, x2, p, q, rng);
                     if (pend) random_point(q, rng);
                  } else
                     pend = false;
               }
            } while (__builtin_amdgcn_ballot_w64(pend));
         }
         p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
         if (i >= 0) {
            // the final xform's point is only plotted, never iterated on: the
            // fuse steps skip it (the reference applies it there and drops the
            // result, flam3.c:280-291)
            if (what & 2) {
               // (loaded anew at each step: kept over the loop, the row
               // would take the scalar registers the step's own needs, which
               // then spill to vector lanes)
               int fi = what >> 3;
               asm volatile("" : "+s"(fi));
               const WaveXf xf = wave_xf(G.wt, fi);
               bool go = true;
               if (!(what & 4)) go = u01<float>(rng) < G.final_opacity;
               if (go) {
                  if (wave_apply<TIER>(G, fi, xf, p, q, rng)) random_point(q, rng);
                  q[3] = p[3];
               }
            }
            if ((i + 1 != nwg) | full) wplot(i, q, fn);
            row += RECORDS == FL3_REC_NARROW ? 1024 : 2048;
         }
         i++;
         const uint32_t now = draw;
         st++;
         if ((st & 63u) == 0u) draws = draw_block(st);
         draw = (uint32_t)__builtin_amdgcn_readlane((int)draws, (int)(st & 63u));
         fs = (int)(draw >> 24);
         x = wave_xf(G.wt, fs);
         // The points change lanes (the same step in every lane: st counts
         // the workgroup's steps).  (Only the low 8 bits of the slot count: a
         // 24-bit product.)
         unsigned to;
         asm("v_mul_u32_u24 %0, %1, %2" : "=v"(to) : "s"(now & 255u), "v"(threadIdx.x ^ ((now >> 8) & 255u)));
         to = (to + (now >> 16)) & 255u;
         float *buf = xb + (st & 1u) * 768;
         buf[to] = p[0];
         buf[256 + to] = p[1];
         buf[512 + to] = p[2];
         // (two buffers: a wavefront writes buffer st & 1 only after every
         // wavefront has passed the barrier behind its reads of it)
         __syncthreads();
         p[0] = buf[threadIdx.x];
         p[1] = buf[256 + threadIdx.x];
         p[2] = buf[512 + threadIdx.x];
         if (i == nwg) break;   // (64-bit scalars compare for equality only)
      }
      lastxf = (int)st;   // the step count is what resumes here
   } else {
      for (long long i = a.resume ? 0 : -a.fuse; i < n;) {
         const uint32_t r = rng.next();
         const int fn = select_xform(G, G.chaos_enable ? lastxf : 0, r & 16383u);
         if (apply_xform<float, WalkerRng, TIER>(G, fn, p, q, rng)) {
            consec++;
            if (i >= 0) bad++;
            if (consec < 5) {
               p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
               continue;
            }
            consec = 0;
         } else
            consec = 0;
         lastxf = fn + 1;
         p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
         if (use_final && i >= 0) {   // (not in the fuse steps, as above)
            if (G.final_opacity == 1.0f || u01<float>(rng) < G.final_opacity) {
               apply_xform<float, WalkerRng, TIER, true>(G, G.final_index, p, q, rng);
               q[3] = p[3];
            }
         }
         if (i >= 0) plot(i, q, fn);
         i++;
      }
   }
   if (RECORDS == FL3_REC_WIDE || RECORDS == FL3_REC_JOB)
      for (long long i = n; i < a.rows_out; i++) a.rec[(blk * a.rows_out + i) * 256 + threadIdx.x] = FL3_REC_NONE;
   if (RECORDS == FL3_REC_NARROW)
      for (long long i = n; i < a.rows_out; i++)
         ((unsigned *)a.rec)[(blk * a.rows_out + i) * 256 + threadIdx.x] = FL3_REC_NONE;
   if (RECORDS) {
      // tile counts summed over workgroups
      __syncthreads();
      for (int b = threadIdx.x; b < a.nbins; b += blockDim.x) {
         const unsigned c = bh[b];
         if (c) atomicAdd(&a.bin_total[b], c);
      }
   }
   if (ws) {
      for (int k = 0; k < 4; k++) ws[k * W + wid] = __float_as_uint(p[k]);
      ws[4 * W + wid] = rng.s0;
      ws[5 * W + wid] = rng.s1;
      ws[6 * W + wid] = rng.s2;
      ws[7 * W + wid] = rng.s3;
      ws[8 * W + wid] = (uint32_t)lastxf;
      ws[9 * W + wid] = (uint32_t)consec;
   }
   add_bad(badp, bad);
}

// One FP32 application of xform xi to each of n points (x, y, colour) in the
// walkers' arithmetic: out = (x, y, colour, 1 if the result was a bad value).
// Random variations draw from a walker stream keyed by (key, point index).
template <int TIER>
__global__ __launch_bounds__(256) void k_apply_fp32(const unsigned char *job, int xi, const double *pts,
                                                    long long n, double *out, unsigned long long key) {
   unsigned char *lds = fl3_lds;
   GenL<float> G;
   load_genome<float>(job, lds, G);
   __syncthreads();
   for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
        i += (long long)gridDim.x * blockDim.x) {
      WalkerRng rng;
      rng.seed(key, ~key, (uint64_t)i);
      float p[4] = {(float)pts[4 * i], (float)pts[4 * i + 1], (float)pts[4 * i + 2], (float)pts[4 * i + 3]}, q[4];
      const bool bad = apply_xform<float, WalkerRng, TIER>(G, xi, p, q, rng);
      out[4 * i] = q[0];
      out[4 * i + 1] = q[1];
      out[4 * i + 2] = q[2];
      out[4 * i + 3] = bad ? 1.0 : 0.0;
   }
}

#endif
