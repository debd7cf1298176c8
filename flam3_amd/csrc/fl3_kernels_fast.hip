// fl3_kernels_fast.hip - launches of the FP32 production walkers, and the
// binned deposit's kernels (compiled with FP contraction on).
#include "fl3_walker.h"
#include "fl3_launch.h"


template <bool WAVE>
static void launch_full(const IterArgs *a, unsigned grid, size_t lds, hipStream_t s, int bits, int exact) {
   if (a->rec_mode == FL3_REC_JOB)
      hipLaunchKernelGGL((k_iter_fast<33, true, FL3_REC_JOB, FL3_TIER_FULL, WAVE>), dim3(grid), dim3(256), lds, s, *a);
   else if (a->rec_mode == FL3_REC_NARROW)
      hipLaunchKernelGGL((k_iter_fast<33, true, FL3_REC_NARROW, FL3_TIER_FULL, WAVE>), dim3(grid), dim3(256), lds, s,
                         *a);
   else if (a->rec_mode == FL3_REC_WIDE)
      hipLaunchKernelGGL((k_iter_fast<33, true, FL3_REC_WIDE, FL3_TIER_FULL, WAVE>), dim3(grid), dim3(256), lds, s, *a);
   else if (bits == 64)
      hipLaunchKernelGGL((k_iter_fast<64, true, FL3_REC_DIRECT, FL3_TIER_FULL, WAVE>), dim3(grid), dim3(256), lds, s,
                         *a);
   else if (exact)
      hipLaunchKernelGGL((k_iter_fast<33, true, FL3_REC_DIRECT, FL3_TIER_FULL, WAVE>), dim3(grid), dim3(256), lds, s,
                         *a);
   else
      hipLaunchKernelGGL((k_iter_fast<33, false, FL3_REC_DIRECT, FL3_TIER_FULL, WAVE>), dim3(grid), dim3(256), lds, s,
                         *a);
}

// a->wave_xf selects the one-xform-per-wavefront walkers (genomes without
// xaos, exchange buffers at a->shuf_off).
extern "C" int fl3k_launch_iter_fast(const IterArgs *a, unsigned grid, size_t lds, hipStream_t s, int bits,
                                     int exact, int tier) {
   if (tier >= 0 && tier < FL3_TIER_FULL && (a->rec_mode || bits != 64))
      return fl3k_launch_iter_tier(a, grid, lds, s, tier, exact);
   if (a->wave_xf)
      launch_full<true>(a, grid, lds, s, bits, exact);
   else
      launch_full<false>(a, grid, lds, s, bits, exact);
   return hipGetLastError() != hipSuccess;
}

extern "C" int fl3k_launch_apply_fp32(const unsigned char *job, int xi, const double *pts, long long n, double *out,
                                      unsigned long long key, size_t lds, hipStream_t s, int tier) {
   if (tier >= 0 && tier < FL3_TIER_FULL) return fl3k_launch_apply_fp32_tier(job, xi, pts, n, out, key, lds, s, tier);
   const unsigned grid = (unsigned)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
   hipLaunchKernelGGL(k_apply_fp32<FL3_TIER_FULL>, dim3(grid), dim3(256), lds, s, job, xi, pts, n, out, key);
   return hipGetLastError() != hipSuccess;
}

// ------------------------------------------------------------------ binned deposit
//
// The walker kernel writes one record per plotted sample instead of five
// global atomics, and counts its workgroup's records per tile of 1 << shift
// cells.  The records are then grouped by tile (tile offsets from
// those counts, then one pass over the records), and each tile's
// records are accumulated in LDS and added to the histogram once.  Integer
// sums commute, so the histogram is the one the atomic deposit produces; the
// tile flush applies the reference's saturation exactly.

// Threads per accumulation workgroup, and records each thread of the one into
// double buckets loads before working on them.
#ifndef FL3_ACC_THREADS
#define FL3_ACC_THREADS 1024
#endif
#ifndef FL3_ACC_UNROLL
#define FL3_ACC_UNROLL 16
#endif

// One workgroup: exclusive scans of the tile counts and of the work items
// (ceil(count / chunk) per tile), and the list of the tiles of several items
// with the place of their first in the array of partial sums.  It also leaves
// the tile counts at zero for their next use and resets the accumulation's
// item counter.
__global__ __launch_bounds__(1024) void k_bin_scan(BinArgs a) {
   // records | (items of tiles of several) << 32, items | (such tiles) << 32
   __shared__ unsigned long long part[1024], ipart[1024];
   const int t = threadIdx.x, per = (a.nbins + 1023) / 1024;
   if (t == 0) *a.item_counter = 0u;
   const int b0 = t * per, b1 = min(a.nbins, b0 + per);
   unsigned long long s = 0, si = 0;
   for (int b = b0; b < b1; b++) {
      const unsigned n = a.bin_total[b], ni = (unsigned)(((unsigned long long)n + a.chunk - 1) / a.chunk);
      s += n + ((unsigned long long)(ni > 1 ? ni : 0u) << 32);
      si += ni + ((unsigned long long)(ni > 1) << 32);
   }
   part[t] = s;
   ipart[t] = si;
   __syncthreads();
   for (int off = 1; off < 1024; off <<= 1) {
      unsigned long long v = t >= off ? part[t - off] : 0, vi = t >= off ? ipart[t - off] : 0;
      __syncthreads();
      part[t] += v;
      ipart[t] += vi;
      __syncthreads();
   }
   unsigned long long run = t ? part[t - 1] : 0, irun = t ? ipart[t - 1] : 0;
   for (int b = b0; b < b1; b++) {
      const unsigned n = a.bin_total[b], ni = (unsigned)(((unsigned long long)n + a.chunk - 1) / a.chunk);
      a.bin_start[b] = (unsigned)run;
      a.cursor[b] = (unsigned)run;
      if (a.band_cursor && (b & ((1 << FL3_SUPER_SHIFT) - 1)) == 0) a.band_cursor[b >> FL3_SUPER_SHIFT] = (unsigned)run;
      a.item_start[b] = (unsigned)irun;
      a.tile_part[b] = (unsigned)(run >> 32);
      if (ni > 1) a.multi[1 + (unsigned)(irun >> 32)] = (unsigned)b;
      run += n + ((unsigned long long)(ni > 1 ? ni : 0u) << 32);
      irun += ni + ((unsigned long long)(ni > 1) << 32);
      a.bin_total[b] = 0u;
   }
   if (t == 1023) {
      a.bin_start[a.nbins] = (unsigned)part[1023];
      a.item_start[a.nbins] = (unsigned)ipart[1023];
      a.multi[0] = (unsigned)(ipart[1023] >> 32);
   }
}

template <typename RT>
__device__ __forceinline__ unsigned rec_cell(RT v) {
   return sizeof(RT) == 4 ? (unsigned)v & 0xffffffu : (unsigned)v;
}
template <typename RT>
__device__ __forceinline__ bool rec_none(RT v) {
   return (unsigned)v == FL3_REC_NONE;
}
// the record's cell relative to the band being sorted (records of a band
// pass hold that already)
template <typename RT>
__device__ __forceinline__ unsigned rel_cell(const BinArgs &a, RT v) {
   return a.rec_rel ? rec_cell(v) : rec_cell(v) - a.cell_base;
}
// slot idx of the input blocks: past rec_count (when set) there are no records
template <typename RT>
__device__ __forceinline__ RT rec_at(const BinArgs &a, const RT *rec, long long idx) {
   return a.rec_count == 0 || idx < a.rec_count ? rec[idx] : (RT)FL3_REC_NONE;
}

#define FL3_SCATTER_UNROLL 16
// The record as the sort writes it: unchanged, or (OT 4 bytes from 8-byte
// records, the band pass of a histogram of 2^24-cell bands, visibility 1
// and a stepped palette) its cell within the band of 1 << sh cells | palette
// index << 24.
template <typename RT, typename OT>
__device__ __forceinline__ OT sorted_rec(RT v, int sh) {
   if (sizeof(OT) == sizeof(RT)) return (OT)v;
   const unsigned long long x = (unsigned long long)v;
   return (OT)(((unsigned)x & ((1u << sh) - 1u)) | (((unsigned)(x >> 32) & 0xffu) << 24));
}

// The records grouped by tile of 1 << sh cells, for at most MT tiles: a
// workgroup takes NT x P records in walker order, counts them by tile in LDS,
// reserves each tile's slots in a.sorted with one global atomic (cursor holds
// each tile's next one), orders the records by tile in LDS and writes them from
// there, consecutive lanes to consecutive slots.  The order within a tile is
// arbitrary: the accumulation adds integers.  Bound by memory latency in those
// phases, with one workgroup of 16 wavefronts a CU, and by the atomics (512
// records a tile's reservation at 64 tiles, 16 at 2000); a workgroup takes as
// many records as LDS holds, so that a tile's run is some cache lines long.  Two
// passes (to groups of 32 tiles, then to tiles) moved every record twice:
// 3.6M records to 18 tiles 79 us, 12 so; 15M to 75 tiles 156 and 41 us; 184M to
// 900 tiles 745 and 437 us; 2^28 to 2060 tiles 910 and 520 us; 126M of 8
// bytes to 3600 2.8 and 1.5 ms.  (Persistent workgroups that load the next
// records meanwhile: 439 and 601 us; half the records: 532 and 591 us.)
template <typename RT, typename OT, int NT, int P, int MT, bool FEW>
__global__ __launch_bounds__(NT) void k_bin_sort(BinArgs a, int sh, unsigned *cursor) {
   constexpr int N = NT * P, PER = (MT + NT - 1) / NT;
   RT *stage = (RT *)fl3_lds;                 // [N]
   unsigned *gofs = (unsigned *)(stage + N);    // [MT] counts, then the tile's slots less its first place in stage
   uint16_t *lofs = (uint16_t *)(gofs + MT);   // [MT] that place
   __shared__ unsigned wsum[NT / 64];
   const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
   const long long slots = a.rec_count ? a.rec_count : a.walkers * a.rows, r0 = (long long)blockIdx.x * N;
   const RT *in = (const RT *)a.rec + r0;
   const int n = (int)(slots - r0 < N ? slots - r0 : N);
   RT v[P];
   for (int k = 0; k < P; k++) {
      const int r = k * NT + tid;
      v[k] = r < n ? in[r] : (RT)FL3_REC_NONE;
   }
   for (int t = tid; t < MT; t += NT) gofs[t] = 0;
   __syncthreads();
   unsigned rank[P];
   auto counter = [&](RT x) {
      const unsigned t = rel_cell(a, x) >> sh;
      return FEW ? t * 64u + (unsigned)lane : t;
   };
   for (int k = 0; k < P; k++)
      if (!rec_none(v[k])) rank[k] = atomicAdd(&gofs[counter(v[k])], 1u);
   __syncthreads();
   // (the slots are on their way while the counts are scanned)
   unsigned g[PER], c[PER], sum = 0;
   for (int j = 0; j < PER; j++) {
      const int t = j * NT + tid;
      const unsigned ct = t < MT ? gofs[t] : 0u;
      g[j] = 0;
      if (!FEW && ct) g[j] = atomicAdd(&cursor[t], ct);
   }
   for (int j = 0; j < PER; j++) {
      c[j] = PER * tid + j < MT ? gofs[PER * tid + j] : 0u;
      sum += c[j];
   }
   unsigned x = sum;
   for (int o = 1; o < 64; o <<= 1) {
      const unsigned y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
   }
   if (lane == 63) wsum[wave] = x;
   __syncthreads();
   unsigned pre = x - sum, tot = 0;
   for (int w = 0; w < NT / 64; w++) {
      if (w < wave) pre += wsum[w];
      tot += wsum[w];
   }
   for (int j = 0; j < PER; j++)
      if (PER * tid + j < MT) {
         lofs[PER * tid + j] = (uint16_t)pre;
         pre += c[j];
      }
   __syncthreads();
   if (!FEW) {
      for (int j = 0; j < PER; j++)
         if (j * NT + tid < MT) gofs[j * NT + tid] = g[j] - lofs[j * NT + tid];
   } else if (tid < MT / 64) {
      const unsigned l0 = lofs[tid * 64], ct = (tid < MT / 64 - 1 ? lofs[tid * 64 + 64] : tot) - l0;
      gofs[tid] = (ct ? atomicAdd(&cursor[tid], ct) : 0u) - l0;
   }
   for (int k = 0; k < P; k++)
      if (!rec_none(v[k])) stage[lofs[counter(v[k])] + rank[k]] = v[k];
   __syncthreads();
   OT *out = (OT *)a.sorted;
   for (unsigned j = tid; j < tot; j += NT) {
      const RT w = stage[j];
      out[gofs[rel_cell(a, w) >> sh] + j] = sorted_rec<RT, OT>(w, sh);
   }
}

// Accumulation of the sorted records: persistent workgroups take work items (a
// tile's records, or a.chunk of them), sum them in LDS and fold the sums into
// registers, a thread the CPT cells it owns.  The sums of a tile of one work item
// are then added to the histogram; those of the items of a fuller tile go to an
// array of partial sums, which k_bin_merge adds up (or, where there is no room
// for one, to the histogram with atomics).  (Atomic adds from every
// item's 20 channels a thread ran at 1e11 a second: 0.2 us an item.)
//
// ACC_NARROW (4-byte records) and ACC_COLOUR (job records that carry the
// entry's bytes, palettes of entries below 256) are of visibility 1 with a stepped
// palette: a record adds its palette entry and 255 hits.  The tile's cells are
// packed sums, and a round of at most `round` records keeps every field below its
// width.  The others (linear palettes, visibilities below 1, entries too bright for
// a round) take one round, in two 64-bit pairs (R|G, B|A) and a hit count: an item
// adds at most 2^18 deltas of at most 255 to a cell, so no 32-bit half carries.
//
// Bound by LDS atomics, so a record makes as few as its fields allow.  RGB:
// every palette entry is below 256 and has alpha a.alpha, so alpha is a
// multiple of the count and a cell is R:24 | G:24 | count:16 and B:32 (one
// 64-bit and one 32-bit atomic, after a 4-byte read of the palette entry for
// 4-byte records); otherwise R:24 | G:24 | count:16 and B:32 | A:32 (two 64-bit
// atomics after a 16-byte read).  Per 64 records of a tile, that is 22 against
// 31 clocks of a CU's LDS.  The next records are loaded while the ones before
// them are added, and the work item after the next is drawn and the next one
// looked up meanwhile, so that its first records are under way while this
// one's sums are stored.
// At 1920x1080 with 2x2 supersampling (2^28 records of 4 bytes a launch) 606 us
// with 2^18-record items added by atomics, 470 us so with the merge (LDS active
// half of the time, 4 TB/s); 256x256 (3.6M records) 94 and 17 us, 640x480
// (15M) 105 and 48 us; 48 previews' 8-byte records 398 and 339 us; 47M records of
// a linear palette and visibilities below 1 483 us and 242 us.
enum { ACC_NARROW, ACC_COLOUR, ACC_PLAIN4, ACC_WIDE, ACC_JOB };
#define FL3_ACC_AHEAD 8   // records a thread loads ahead
// 16-byte words of an item's partial sums: per cell R, G, B, count, then the
// alphas if they are not a multiple of the count
__host__ __device__ __forceinline__ size_t part_words(unsigned cells, bool rgb) {
   return rgb ? cells : cells + cells / 4;
}
__device__ __forceinline__ uint32_t add_u32_sat(uint32_t x, uint32_t y) {
   const uint32_t t = x + y;
   return t < x ? 0xffffffffu : t;
}
template <int KIND, bool RGB>
__global__ __launch_bounds__(FL3_ACC_THREADS) void k_bin_accum(BinArgs a) {
   constexpr bool PACKED = KIND == ACC_NARROW || KIND == ACC_COLOUR;
   typedef typename std::conditional<KIND == ACC_NARROW || KIND == ACC_PLAIN4, unsigned, unsigned long long>::type RT;
   typedef typename std::conditional<RGB, unsigned, unsigned long long>::type PT;
   const fl3_job_hdr *h = (const fl3_job_hdr *)a.job;
   constexpr int tile_cells = 1 << FL3_TILE_SHIFT, CPT = tile_cells / FL3_ACC_THREADS, U = FL3_ACC_AHEAD, step = U * FL3_ACC_THREADS;
   unsigned long long *p0 = (unsigned long long *)fl3_lds;   // tile_cells
   PT *p1 = (PT *)(p0 + tile_cells);                           // tile_cells
   ulonglong2 *pal = (ulonglong2 *)(p1 + tile_cells);          // 256 (RGB: bytes R, G, B)
   unsigned *pal8 = (unsigned *)pal;
   // (not packed:)
   uint32_t *hits = (uint32_t *)(p1 + tile_cells);             // tile_cells
   uint32_t *dmapu = hits + tile_cells;                        // 1024
   float *dmapf = (float *)(dmapu + 1024);                     // 1024
   float *vis = dmapf + 1024;                                  // 256
   // work items, alternating: the one drawn after the next, and of the next its
   // tile, first record, records, and place among the partial sums + 1 (0: the
   // tile's only item)
   __shared__ unsigned drawn[2];
   __shared__ uint4 found[2];
   const int tid = threadIdx.x;
   const double *pd = (const double *)(a.job + h->off_dmap);
   if (!PACKED) {
      const fl3_xform_pack *px = (const fl3_xform_pack *)(a.job + h->off_xf);
      for (int e = tid; e < 1024; e += FL3_ACC_THREADS) {
         dmapu[e] = (uint32_t)pd[e];
         dmapf[e] = (float)pd[e];
      }
      for (int e = tid; e < h->nxf && e < 256; e += FL3_ACC_THREADS) vis[e] = (float)px[e].vis;
   }
   const int linear = h->palette_mode == 1;
   if (KIND == ACC_NARROW)
      for (int e = tid; e < 256; e += FL3_ACC_THREADS) {
         const uint32_t r = (uint32_t)pd[4 * e], g = (uint32_t)pd[4 * e + 1], bb = (uint32_t)pd[4 * e + 2], al = (uint32_t)pd[4 * e + 3];
         if (RGB)
            pal8[e] = r | g << 8 | bb << 16;
         else {
            ulonglong2 w;
            w.x = (unsigned long long)r | ((unsigned long long)g << 24) | (1ull << 48);
            w.y = (unsigned long long)bb | ((unsigned long long)al << 32);
            pal[e] = w;
         }
      }
   for (int e = tid; e < tile_cells; e += FL3_ACC_THREADS) {
      p0[e] = 0;
      p1[e] = 0;
      if (!PACKED) hits[e] = 0;
   }
   const unsigned total_items = a.item_start[a.nbins];
   const int round_steps = PACKED ? a.round / step : INT_MAX;
   auto look_up = [&](unsigned item, int slot) {
      for (int b = tid; b < a.nbins; b += FL3_ACC_THREADS) {
         const unsigned i0 = a.item_start[b], i1 = a.item_start[b + 1], r0 = a.bin_start[b], r1 = a.bin_start[b + 1];
         const unsigned p = a.tile_part[b];
         if (i0 <= item && item < i1) {
            const unsigned k = item - i0, first = r0 + k * (unsigned)a.chunk;
            found[slot] = make_uint4((unsigned)b, first, min(r1 - first, (unsigned)a.chunk), i1 - i0 == 1 ? 0u : p + k + 1u);
         }
      }
   };
   // (the first two items of a workgroup are its own, the others drawn)
   unsigned item = blockIdx.x, next = gridDim.x + blockIdx.x;
   if (item >= total_items) return;
   look_up(item, 0);
   __syncthreads();
   auto in_item = [&](int slot, int c) { return __builtin_amdgcn_readfirstlane(((const unsigned *)&found[slot])[c]); };
   unsigned b = in_item(0, 0), first = in_item(0, 1), place = in_item(0, 3);
   int n = (int)in_item(0, 2);
   auto fetch = [&](RT(&v)[U], int at) {
      const RT *in = (const RT *)a.sorted + first;
      for (int u = 0; u < U; u++) v[u] = in[min(at + u * FL3_ACC_THREADS + tid, n - 1)];
   };
   RT v[U], nx[U];
   fetch(nx, 0);
   for (int slot = 1;; slot ^= 1) {
      const unsigned cell0 = a.cell_base + (b << a.shift), place_now = place;
      unsigned draw = 0;
      if (tid == 0) draw = 2u * gridDim.x + atomicAdd(a.item_counter, 1u);
      if (next < total_items) look_up(next, slot);
      uint32_t acc[CPT][RGB ? 4 : 5];
      for (int j = 0; j < CPT; j++)
         for (int c = 0; c < (RGB ? 4 : 5); c++) acc[j][c] = 0;
      auto add = [&](RT v) {
         const unsigned local = (unsigned)v & (unsigned)(tile_cells - 1);   // (a tile starts at a multiple of its cells)
         if constexpr (KIND == ACC_COLOUR || (KIND == ACC_NARROW && RGB)) {
            const unsigned c = KIND == ACC_COLOUR ? (unsigned)((unsigned long long)v >> 32) : pal8[(unsigned)v >> 24];
            atomicAdd(&p0[local], (unsigned long long)((c & 0xffu) | ((c >> 8) & 0xffu) << 24) | 1ull << 48);
            atomicAdd(&p1[local], (PT)((c >> 16) & 0xffu) | (RGB ? 0 : (PT)((unsigned long long)(c >> 24) << 32)));
         } else if constexpr (KIND == ACC_NARROW) {
            const ulonglong2 w = pal[(unsigned)v >> 24];
            atomicAdd(&p0[local], w.x);
            atomicAdd(&p1[local], (PT)w.y);
         } else {
            uint32_t d[5];
            const int ci = (int)(((unsigned long long)v >> (KIND == ACC_PLAIN4 ? 24 : 32)) & 0xff);
            const int fn = KIND == ACC_PLAIN4 ? 0 : (int)(((unsigned long long)v >> 40) & 0xff);
            const int top = KIND == ACC_PLAIN4 ? 0 : (int)((unsigned long long)v >> 48);
            if (KIND == ACC_PLAIN4) {
               for (int c = 0; c < 4; c++) d[c] = dmapu[ci * 4 + c];
               d[4] = 255u;
            } else if (KIND == ACC_JOB) {
               // the record's job selects palette and visibility (stepped palette)
               const float vv = a.vis_all[top * a.vis_stride + fn];
               const uint32_t *du = a.dmapu_all + top * 1024 + ci * 4;
               if (vv == 1.0f) {
                  for (int c = 0; c < 4; c++) d[c] = du[c];
                  d[4] = 255u;
               } else {
                  const float *df = a.dmapf_all + top * 1024 + ci * 4;
                  for (int c = 0; c < 4; c++) d[c] = (uint32_t)(vv * df[c]);
                  d[4] = (uint32_t)(vv * 255.0f);
               }
            } else {
               const float vv = vis[fn];
               if (linear) {
                  const float f = (float)top * (1.0f / 65535.0f);
                  for (int c = 0; c < 4; c++) {
                     const float col = dmapf[ci * 4 + c] * (1.0f - f) + dmapf[ci * 4 + 4 + c] * f;
                     d[c] = (uint32_t)(vv == 1.0f ? col : vv * col);
                  }
               } else if (vv == 1.0f) {
                  for (int c = 0; c < 4; c++) d[c] = dmapu[ci * 4 + c];
               } else {
                  for (int c = 0; c < 4; c++) d[c] = (uint32_t)(vv * dmapf[ci * 4 + c]);
               }
               d[4] = vv == 1.0f ? 255u : (uint32_t)(vv * 255.0f);
            }
            atomicAdd(&p0[local], (unsigned long long)d[0] | ((unsigned long long)d[1] << 32));
            atomicAdd(&p1[local], (PT)((unsigned long long)d[2] | ((unsigned long long)d[3] << 32)));
            atomicAdd(&hits[local], d[4]);
         }
      };
      for (int at = 0, steps = 0; at < n; at += step) {
         for (int u = 0; u < U; u++) v[u] = nx[u];
         if (at + step < n) fetch(nx, at + step);
         if (at + step <= n)
            for (int u = 0; u < U; u++) add(v[u]);
         else
            for (int u = 0; u < U; u++)
               if (at + u * FL3_ACC_THREADS + tid < n) add(v[u]);
         if (++steps < round_steps && at + step < n) continue;
         steps = 0;
         if (tid == 0) drawn[slot] = draw;
         __syncthreads();
         for (int j = 0; j < CPT; j++) {
            const int e = tid + j * FL3_ACC_THREADS;
            const unsigned long long x0 = p0[e];
            const PT x1 = p1[e];
            p0[e] = 0;
            p1[e] = 0;
            acc[j][0] += PACKED ? (uint32_t)(x0 & 0xffffffu) : (uint32_t)x0;
            acc[j][1] += PACKED ? (uint32_t)((x0 >> 24) & 0xffffffu) : (uint32_t)(x0 >> 32);
            acc[j][2] += (uint32_t)x1;
            acc[j][3] += PACKED ? (uint32_t)(x0 >> 48) : hits[e];
            if (!PACKED) hits[e] = 0;
            if (!RGB) acc[j][RGB ? 0 : 4] += (uint32_t)((unsigned long long)x1 >> 32);
         }
         __syncthreads();
      }
      const bool more = next < total_items;
      if (more) {
         b = in_item(slot, 0);
         first = in_item(slot, 1);
         n = (int)in_item(slot, 2);
         place = in_item(slot, 3);
         fetch(nx, 0);
      }
      next = __builtin_amdgcn_readfirstlane(drawn[slot]);
      if (place_now && (PACKED || a.partial)) {
         uint4 *out = (uint4 *)a.partial + (size_t)(place_now - 1) * part_words(tile_cells, RGB);
         for (int j = 0; j < CPT; j++) {
            const int e = tid + j * FL3_ACC_THREADS;
            out[e] = make_uint4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
            if (!RGB) ((unsigned *)(out + tile_cells))[e] = acc[j][RGB ? 0 : 4];
         }
      } else {
         uint32_t *bk = (uint32_t *)a.buckets + (size_t)cell0 * 5;
         const int nvalid = (int)min((long long)tile_cells, (long long)a.width * a.height - (long long)cell0);
         uint32_t sum[CPT][5], old[CPT][5];
         for (int j = 0; j < CPT; j++) {
            for (int c = 0; c < 3; c++) sum[j][c] = acc[j][c];
            sum[j][3] = RGB ? acc[j][3] * (unsigned)a.alpha : acc[j][RGB ? 0 : 4];
            sum[j][4] = acc[j][3] * (PACKED ? 255u : 1u);
         }
         if (!PACKED && place_now) {   // (no room for partial sums: others add to the tile too)
            for (int j = 0; j < CPT; j++)
               for (int c = 0; c < 5; c++) {
                  const int e = tid + j * FL3_ACC_THREADS;
                  if (e < nvalid && sum[j][c]) sat_add(bk + (size_t)e * 5 + c, sum[j][c]);
               }
         } else {
            // every load of the thread's cells is issued before any result is
            // used, so that their latencies overlap (adding zero leaves a cell as
            // it is, and the tile is this workgroup's alone)
            for (int j = 0; j < CPT; j++)
               for (int c = 0; c < 5; c++) {
                  const int e = tid + j * FL3_ACC_THREADS;
                  old[j][c] = e < nvalid ? bk[(size_t)e * 5 + c] : 0u;
               }
            // (the sums first, each in a register of its own, so that no store
            // waits for an earlier one to release its data register)
            for (int j = 0; j < CPT; j++)
               for (int c = 0; c < 5; c++) old[j][c] = add_u32_sat(old[j][c], sum[j][c]);
            for (int j = 0; j < CPT; j++)
               for (int c = 0; c < 5; c++) {
                  const int e = tid + j * FL3_ACC_THREADS;
                  if (e < nvalid) bk[(size_t)e * 5 + c] = old[j][c];
               }
         }
      }
      if (!more) break;
   }
}

// Adds up the partial sums of the tiles of several work items and adds them
// to the histogram: a workgroup takes 256 cells of a tile at a time.
template <bool RGB, unsigned HIT>
__global__ __launch_bounds__(256) void k_bin_merge(BinArgs a) {
   const unsigned cells = 1u << a.shift, parts = cells / 256, units = a.multi[0] * parts;
   const size_t words = part_words(cells, RGB);
   for (unsigned u = blockIdx.x; u < units; u += gridDim.x) {
      const unsigned b = a.multi[1 + u / parts], e = u % parts * 256 + threadIdx.x;
      const unsigned n = a.item_start[b + 1] - a.item_start[b];
      const uint4 *in = (const uint4 *)a.partial + (size_t)a.tile_part[b] * words;
      const size_t cell = (size_t)a.cell_base + ((size_t)b << a.shift) + e;
      unsigned long long sum[5] = {0, 0, 0, 0, 0};
#pragma unroll 4
      for (unsigned i = 0; i < n; i++) {
         const uint4 v = in[i * words + e];
         sum[0] += v.x;
         sum[1] += v.y;
         sum[2] += v.z;
         sum[4] += v.w;
         if (!RGB) sum[3] += ((const unsigned *)(in + i * words + cells))[e];
      }
      if (cell >= (size_t)a.width * a.height) continue;
      if (RGB) sum[3] = sum[4] * (unsigned)a.alpha;
      sum[4] *= HIT;
      uint32_t *bk = (uint32_t *)a.buckets + cell * 5;
      uint32_t old[5];
      for (int c = 0; c < 5; c++) old[c] = bk[c];
      for (int c = 0; c < 5; c++) {
         const unsigned long long t = old[c] + sum[c];
         bk[c] = t > 0xffffffffull ? 0xffffffffu : (uint32_t)t;
      }
   }
}

// Counting pass of a band (the walkers' counting for records sorted by band
// first): workgroup k counts the records of its block of rows x 256 slots
// per tile in LDS and adds the counts to bin_total.
template <typename RT>
__global__ __launch_bounds__(256) void k_bin_count(BinArgs a) {
   unsigned *hist = (unsigned *)fl3_lds;   // [nbins]
   for (int b = threadIdx.x; b < a.nbins; b += blockDim.x) hist[b] = 0;
   __syncthreads();
   const RT *rec = (const RT *)a.rec;
   // (the rows' loads are issued in batches before their counts, so that a
   // thread has many loads in flight)
   long long i = 0;
   for (; i + FL3_SCATTER_UNROLL <= a.rows; i += FL3_SCATTER_UNROLL) {
      RT v[FL3_SCATTER_UNROLL];
      for (int k = 0; k < FL3_SCATTER_UNROLL; k++) v[k] = rec_at(a, rec, (blockIdx.x * a.rows + i + k) * 256 + threadIdx.x);
      for (int k = 0; k < FL3_SCATTER_UNROLL; k++)
         if (!rec_none(v[k])) atomicAdd(&hist[rel_cell(a, v[k]) >> a.shift], 1u);
   }
   for (; i < a.rows; i++) {
      const RT v = rec_at(a, rec, (blockIdx.x * a.rows + i) * 256 + threadIdx.x);
      if (!rec_none(v)) atomicAdd(&hist[rel_cell(a, v) >> a.shift], 1u);
   }
   __syncthreads();
   for (int b = threadIdx.x; b < a.nbins; b += blockDim.x)
      if (hist[b]) atomicAdd(&a.bin_total[b], hist[b]);
}

// Accumulation into bits-64 (double) buckets.  Each record adds what the
// direct deposit adds for its point (rect.c:492-497 in double: the palette
// entry, blended for a linear palette, times the xform's visibility, and
// 255 times it to the count), rounded to a multiple of 2^-32 and summed in
// LDS as signed 64-bit integers (integer atomics outpace double ones; a
// work item of at most 2^31 / (largest |entry| + 1) records keeps a cell's
// sum below 2^63 in size); the item's sums are then added to the double
// buckets.  Against the per-sample double atomics a cell's sum differs by
// at most 2^-33 per record (about 1e-12 relative), besides the order of the
// additions.
// 4-byte records (stepped palette, visibility 1; each adds exactly 255 to
// the count, which is then a 32-bit record count scaled at the flush) or
// 8-byte records (make_record).  Persistent workgroups take work items
// (up to a.chunk records of one tile) from a counter; a tile with one item is
// added without atomics.
#define FL3_F64_FIX 4294967296.0    // 2^32: the fixed-point scale of the LDS sums
template <typename RT>
__global__ __launch_bounds__(FL3_ACC_THREADS) void k_bin_accum_f64(BinArgs a) {
   const fl3_job_hdr *h = (const fl3_job_hdr *)a.job;
   const int tile_cells = 1 << a.shift;
   unsigned long long *acc = (unsigned long long *)fl3_lds;   // [5][tile_cells]
   unsigned long long *dfx = acc + 5 * tile_cells;            // [1024] the palette, fixed point
   double *dm = (double *)(dfx + 1024);                       // [1024]
   double *vis = dm + 1024;                                   // [256]
   __shared__ int item_sh;
   const double *pd = (const double *)(a.job + h->off_dmap);
   const fl3_xform_pack *px = (const fl3_xform_pack *)(a.job + h->off_xf);
   for (int e = threadIdx.x; e < 1024; e += blockDim.x) {
      dm[e] = pd[e];
      dfx[e] = (unsigned long long)__double2ll_rn(pd[e] * FL3_F64_FIX);
   }
   // (the walkers carry a visibility as a float)
   for (int e = threadIdx.x; e < 256; e += blockDim.x) vis[e] = e < h->nxf ? (double)(float)px[e].vis : 1.0;
   const int linear = h->palette_mode == 1;
   const unsigned long long hits = (unsigned long long)__double2ll_rn(255.0 * FL3_F64_FIX);
   const long long total_items = a.item_start[a.nbins];
   const RT *sorted = (const RT *)a.sorted;
   for (;;) {
      __syncthreads();
      if (threadIdx.x == 0) item_sh = (int)atomicAdd(a.item_counter, 1u);
      for (int e = threadIdx.x; e < 5 * tile_cells; e += blockDim.x) acc[e] = 0ull;
      __syncthreads();
      const long long item = item_sh;
      if (item >= total_items) break;
      int lo = 0, hi = a.nbins - 1;
      while (lo < hi) {  // last tile whose first item is <= item
         const int mid = (lo + hi + 1) >> 1;
         if ((long long)a.item_start[mid] <= item) lo = mid;
         else hi = mid - 1;
      }
      const int b = lo;
      const long long k = item - a.item_start[b];
      const long long r0 = (long long)a.bin_start[b] + k * a.chunk;
      const long long r1 = min((long long)a.bin_start[b + 1], r0 + a.chunk);
      const bool single = (a.item_start[b + 1] - a.item_start[b]) == 1;
      const unsigned tb = (unsigned)b << a.shift;   // the tile's first cell in the band
      const unsigned cell0 = a.cell_base + tb;
      for (long long rb = r0; rb < r1; rb += FL3_ACC_UNROLL * blockDim.x) {
         RT v[FL3_ACC_UNROLL];
         for (int u = 0; u < FL3_ACC_UNROLL; u++) {
            const long long r = rb + u * blockDim.x + threadIdx.x;
            v[u] = r < r1 ? sorted[r] : (RT)FL3_REC_NONE;
         }
         for (int u = 0; u < FL3_ACC_UNROLL; u++) {
            if (rec_none(v[u])) continue;
            const unsigned local = rel_cell(a, v[u]) - tb;
            unsigned long long d[5];
            if (sizeof(RT) == 4) {
               // (every 4-byte record adds 255 hits: the count channel is a
               // 32-bit record count, times 255 at the flush)
               const unsigned long long *e = dfx + ((unsigned)v[u] >> 24) * 4;
               for (int ch = 0; ch < 4; ch++) atomicAdd(&acc[ch * tile_cells + local], e[ch]);
               atomicAdd((unsigned *)(acc + 4 * tile_cells) + local, 1u);
               continue;
            } else {
               const unsigned long long x = (unsigned long long)v[u];
               const int ci = (int)((x >> 32) & 0xff), fn = (int)((x >> 40) & 0xff);
               const double w = vis[fn];
               if (!linear && w == 1.0) {
                  for (int ch = 0; ch < 4; ch++) d[ch] = dfx[ci * 4 + ch];
                  d[4] = hits;
               } else {
                  const double *e = dm + ci * 4;
                  double c[4];
                  if (linear) {
                     const double f = (double)((float)(x >> 48) * (1.0f / 65535.0f));
                     for (int ch = 0; ch < 4; ch++) c[ch] = e[ch] * (1.0 - f) + e[4 + ch] * f;
                  } else
                     for (int ch = 0; ch < 4; ch++) c[ch] = e[ch];
                  for (int ch = 0; ch < 4; ch++)
                     d[ch] = (unsigned long long)__double2ll_rn((w == 1.0 ? c[ch] : w * c[ch]) * FL3_F64_FIX);
                  d[4] = w == 1.0 ? hits : (unsigned long long)__double2ll_rn(w * 255.0 * FL3_F64_FIX);
               }
            }
            for (int ch = 0; ch < 5; ch++) atomicAdd(&acc[ch * tile_cells + local], d[ch]);
         }
      }
      __syncthreads();
      double *bk = (double *)a.buckets + (size_t)cell0 * 5;
      const long long ncells = (long long)a.width * a.height;
      const int nvalid = (int)min((long long)tile_cells, ncells - (long long)cell0);
      // a thread's values of the tile (at most 5 x 2048 / FL3_ACC_THREADS),
      // their loads all issued before any is used
      constexpr int K = 5 * 2048 / FL3_ACC_THREADS;
      double val[K];
      for (int k = 0; k < K; k++) {
         const int e = threadIdx.x + k * FL3_ACC_THREADS;
         val[k] = e >= nvalid * 5 ? 0.0
                  : sizeof(RT) == 4 && e % 5 == 4
                      ? (double)((const unsigned *)(acc + 4 * tile_cells))[e / 5] * 255.0
                      : (double)(long long)acc[(e % 5) * tile_cells + e / 5] * (1.0 / FL3_F64_FIX);
      }
      if (single) {
         double old[K];
         for (int k = 0; k < K; k++) old[k] = val[k] != 0.0 ? bk[threadIdx.x + k * FL3_ACC_THREADS] : 0.0;
         for (int k = 0; k < K; k++) old[k] += val[k];
         for (int k = 0; k < K; k++)
            if (val[k] != 0.0) bk[threadIdx.x + k * FL3_ACC_THREADS] = old[k];
      } else
         for (int k = 0; k < K; k++)
            if (val[k] != 0.0) unsafeAtomicAdd(bk + threadIdx.x + k * FL3_ACC_THREADS, val[k]);
   }
}

extern "C" size_t fl3k_bin_f64_lds_bytes(int shift) { return (size_t)40 * ((size_t)1 << shift) + 8 * (1024 + 1024 + 256) + 64; }

extern "C" int fl3k_bin_pass_records(void) { return FL3_ACC_AHEAD * FL3_ACC_THREADS; }
template <int KIND, bool RGB = false>
static void launch_accum(const BinArgs *a, int ncu, hipStream_t s) {
   constexpr bool packed = KIND == ACC_NARROW || KIND == ACC_COLOUR;
   const size_t cells = (size_t)1 << FL3_TILE_SHIFT;
   const size_t lds = RGB ? 12 * cells + 1024 : packed ? 16 * cells + 4096 : 20 * cells + 9 * 1024;
   if (lds > 65536)
      (void)hipFuncSetAttribute((const void *)k_bin_accum<KIND, RGB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
   hipLaunchKernelGGL((k_bin_accum<KIND, RGB>), dim3((packed ? 2u : 1u) * (unsigned)ncu), dim3(FL3_ACC_THREADS), lds, s, *a);
   if (a->partial) hipLaunchKernelGGL((k_bin_merge<RGB, packed ? 255 : 1>), dim3(8u * (unsigned)ncu), dim3(256), 0, s, *a);
}
// Bytes of the accumulation's partial sums for `records` in a chunk (a tile of
// several items has more than an item's records, so at most two items for every
// item's worth of records); rgb: the alphas are multiples of the counts.  Tiles
// are those of the accumulation, also where the walkers count larger ones
// (banded histograms).  0 where they would take more than 256 MiB and the
// records' 8 bytes each: items of so few records are those of palette entries too
// bright for more (171 records at 2.5e7, whose sums would take 250 GB for a
// chunk of 2^28), and their sums go to the histogram with atomics.  Items of
// 2^14 to 2^18 records, as the launch's size sets them, take at most 130 MB, or
// 1.3 bytes a record.
extern "C" size_t fl3k_bin_partial_bytes(int rgb, long long chunk, long long records) {
   const double n = 16.0 * (double)part_words(1u << FL3_TILE_SHIFT, rgb != 0) * (2.0 * (double)records / (double)chunk + 1.0);
   if (n > 268435456.0 + 8.0 * (double)records) return 0;
   return 16 * part_words(1u << FL3_TILE_SHIFT, rgb != 0) * (size_t)(2 * records / chunk + 1);
}

// LDS of the accumulation into 32-bit histograms, at most.
extern "C" size_t fl3k_bin_lds_bytes(void) { return (size_t)20 * ((size_t)1 << FL3_TILE_SHIFT) + 9 * 1024 + 256; }

template <typename RT, typename OT, int NT, int P, int MT, bool FEW = false>
static void launch_sort(const BinArgs *a, int sh, unsigned *cursor, hipStream_t s) {
   const size_t lds = sizeof(RT) * NT * P + 6 * (size_t)MT;
   if (lds > 65536)
      (void)hipFuncSetAttribute((const void *)k_bin_sort<RT, OT, NT, P, MT, FEW>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
   const long long slots = a->rec_count ? a->rec_count : a->walkers * a->rows;
   const unsigned g = (unsigned)((slots + (long long)NT * P - 1) / ((long long)NT * P));
   if (g) hipLaunchKernelGGL((k_bin_sort<RT, OT, NT, P, MT, FEW>), dim3(g), dim3(NT), lds, s, *a, sh, cursor);
}

// Scans of the walkers' counts, and the records grouped by tile into a->sorted:
// with 128 KB of records a workgroup, or half that where two workgroups then
// fit a CU (15M records to 75 tiles: 41 us, 63 us with half as many wavefronts)
// and 96 KB where the tiles' counts need the room.
template <typename RT>
static void sort_records(const BinArgs *a, hipStream_t s) {
   constexpr int P = 128 / sizeof(RT);
   hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(1024), 0, s, *a);
   if (a->nbins <= 256)
      launch_sort<RT, RT, 1024, P / 2, 256>(a, a->shift, a->cursor, s);
   else if (a->nbins <= 1024)
      launch_sort<RT, RT, 1024, P, 1024>(a, a->shift, a->cursor, s);
   else if (a->nbins <= 3072)
      launch_sort<RT, RT, 1024, P, 3072>(a, a->shift, a->cursor, s);
   else if (a->nbins <= 5120)
      launch_sort<RT, RT, 1024, P, 5120>(a, a->shift, a->cursor, s);
   else
      launch_sort<RT, RT, 1024, P * 3 / 4, FL3_MAX_BINS>(a, a->shift, a->cursor, s);
}

extern "C" int fl3k_launch_bin_sort(const BinArgs *a, int format, hipStream_t s) {
   if (format == 1 || format == FL3_BIN_F64_NARROW)
      sort_records<unsigned>(a, s);
   else
      sort_records<unsigned long long>(a, s);
   return hipGetLastError() != hipSuccess;
}

template <typename RT>
static void launch_f64(const BinArgs *a, int ncu, hipStream_t s) {
   const size_t lf = fl3k_bin_f64_lds_bytes(a->shift);
   const unsigned gf = (unsigned)ncu * (lf > 81920 ? 1 : (lf > 54000 ? 2 : 3));
   if (lf > 65536)
      (void)hipFuncSetAttribute((const void *)k_bin_accum_f64<RT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lf);
   hipLaunchKernelGGL(k_bin_accum_f64<RT>, dim3(gf), dim3(FL3_ACC_THREADS), lf, s, *a);
}
// The sorted records added to the histogram.
extern "C" int fl3k_launch_bin_accum(const BinArgs *a, int ncu, int format, hipStream_t s) {
   if (format == FL3_BIN_F64_WIDE)
      launch_f64<unsigned long long>(a, ncu, s);
   else if (format == FL3_BIN_F64_NARROW)
      launch_f64<unsigned>(a, ncu, s);
   else if (format == 1 && a->round > 0)
      a->alpha >= 0 ? launch_accum<ACC_NARROW, true>(a, ncu, s) : launch_accum<ACC_NARROW>(a, ncu, s);
   else if (format == 2 && a->round > 0)
      a->alpha >= 0 ? launch_accum<ACC_COLOUR, true>(a, ncu, s) : launch_accum<ACC_COLOUR>(a, ncu, s);
   else if (format == 1)
      launch_accum<ACC_PLAIN4>(a, ncu, s);
   else if (format == 2)
      launch_accum<ACC_JOB>(a, ncu, s);
   else
      launch_accum<ACC_WIDE>(a, ncu, s);
   return hipGetLastError() != hipSuccess;
}

// Banded histograms, first level: scans of the walkers' counts, and the
// walkers' 8-byte records grouped by band (1 << FL3_SUPER_SHIFT of the tiles
// that they counted) into a->sorted.
extern "C" int fl3k_launch_bin_split(const BinArgs *a, int narrow_out, hipStream_t s) {
   typedef unsigned long long u64;
   const int sh = a->shift + FL3_SUPER_SHIFT;
   hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(1024), 0, s, *a);
   // with a few bands nearly all of a wavefront's records meet at one counter: 64
   // counters a band then, one for each lane (4 bands, 2^28 records: 1.1 ms with
   // one, 0.8 ms so)
   const bool few = a->nbins <= 16 << FL3_SUPER_SHIFT;
   if (narrow_out)
      few ? launch_sort<u64, unsigned, 1024, 16, 1024, true>(a, sh, a->band_cursor, s)
          : launch_sort<u64, unsigned, 1024, 16, 256>(a, sh, a->band_cursor, s);
   else
      few ? launch_sort<u64, u64, 1024, 16, 1024, true>(a, sh, a->band_cursor, s)
          : launch_sort<u64, u64, 1024, 16, 256>(a, sh, a->band_cursor, s);
   return hipGetLastError() != hipSuccess;
}

// Banded histograms, second level: per-tile counts of one band's records (a->rec,
// a->rec_count of them, as a->nblk blocks of a->rows x 256; 4 bytes each if
// narrow), before fl3k_launch_bin_sort and fl3k_launch_bin_accum take them.
extern "C" int fl3k_launch_bin_count(const BinArgs *a, int narrow, hipStream_t s) {
   const size_t l = sizeof(unsigned) * (size_t)a->nbins;   // at most FL3_MAX_BINS: 32 KiB
   if (narrow)
      hipLaunchKernelGGL(k_bin_count<unsigned>, dim3(a->nblk), dim3(256), l, s, *a);
   else
      hipLaunchKernelGGL(k_bin_count<unsigned long long>, dim3(a->nblk), dim3(256), l, s, *a);
   return hipGetLastError() != hipSuccess;
}

// A plain copy of n16 16-byte words, one per thread: the reference kernel of
// known traffic for calibrating hardware byte counters.
__global__ __launch_bounds__(256) void k_copy_probe(const uint4 *src, uint4 *dst, long long n16) {
   const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n16) dst[i] = src[i];
}

extern "C" int fl3k_launch_copy_probe(const void *src, void *dst, long long n16, hipStream_t s) {
   hipLaunchKernelGGL(k_copy_probe, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, s, (const uint4 *)src,
                      (uint4 *)dst, n16);
   return hipGetLastError() != hipSuccess;
}
