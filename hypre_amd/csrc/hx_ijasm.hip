// Assembly of an IJ matrix on the device: SetValues / AddToValues calls in call
// order to CSR rows with the diagonal first.
//
// A chunk is one call's arrays (or many small calls' operations, staged on the
// host), uploaded as they are: segments (row, length) of columns and values.
// The segments are grouped by row, each row's in call order, their operations
// laid out row by row, and one wave a row (a block where the row is long) folds
// repeated columns in call order and finds the diagonal.  Each row's entries,
// their order and the order of the additions are those of the serial assembly
// on the host.  What bounds it is the upload: of 0.95 ms for 1.75M operations
// (110,000 rows), 0.65 are the call that brings their 23 MB, 0.3 the kernels,
// their read-backs and the wait for the last one; the serial assembly took 18.3
// ms, and 147 ms for 10.8M operations (6.0 now for 11.1M).
#include "hx_internal.h"

#include <algorithm>
#include <climits>

namespace hx {

constexpr int BS = 256;
constexpr int WPB = BS / 64;

static int ij_grid(long long n, int per) { return (int) std::max<long long>(1, std::min<long long>((n + per - 1) / per, 8192)); }

// Rows that take a block.  One row of 512 operations beside 40,000 of nine: the
// whole assembly 0.52 ms with the row on a wave (0.90 where each operation is a
// segment of its own), 0.46 with it on a block; 4096 operations 8.2 (26.9)
// against 0.49 (0.65); at 256 there is nothing between the two.
constexpr int IJ_LONG = 256;
__device__ __forceinline__ bool ij_long(int r, const int *seg_ia, const int *op_ia)
{
   return seg_ia[r + 1] - seg_ia[r] > IJ_LONG || op_ia[r + 1] - op_ia[r] > IJ_LONG;
}

// per row: segments and operations (rows outside [lo, lo + nrows) have none)
__global__ __launch_bounds__(BS) void k_ij_count(int nseg, const int *__restrict__ rows,
                                                 const int *__restrict__ ncols, int lo, int nrows,
                                                 int *__restrict__ segs, int *__restrict__ ops)
{
   for (int s = blockIdx.x * BS + threadIdx.x; s < nseg; s += gridDim.x * BS) {
      const int r = rows[s] - lo;
      if (r < 0 || r >= nrows) { continue; }
      atomicAdd(segs + r, 1);
      atomicAdd(ops + r, ncols ? ncols[s] : 1);
   }
}

// global segment numbers into their rows' lists, in any order
__global__ __launch_bounds__(BS) void k_ij_scatter(int nseg, int first, const int *__restrict__ rows,
                                                   int lo, int nrows, int *__restrict__ fill,
                                                   int *__restrict__ list)
{
   for (int s = blockIdx.x * BS + threadIdx.x; s < nseg; s += gridDim.x * BS) {
      const int r = rows[s] - lo;
      if (r < 0 || r >= nrows) { continue; }
      list[atomicAdd(fill + r, 1)] = first + s;
   }
}

// the chunks as the kernels see them; segment numbers run through them
struct IjChunks
{
   int           n;
   int           first[IJ_CHUNKS];    // number of the chunk's first segment
   const int    *start[IJ_CHUNKS];    // segment's first operation (nullptr: one each)
   const int    *cols[IJ_CHUNKS];
   const double *vals[IJ_CHUNKS];
   const char   *ops[IJ_CHUNKS];      // per segment (nullptr: op)
   char          op[IJ_CHUNKS];
};

// One wave a row: its segments by rank into call order, and their operations
// laid out at the row's place.  longs, here and below: there are rows to leave to
// blocks (looking at every row's lengths is a tenth of these kernels' time).
__global__ __launch_bounds__(BS) void k_ij_layout(int nrows, bool longs, const IjChunks *__restrict__ Cp, const int *__restrict__ seg_ia,
                                                  const int *__restrict__ list,
                                                  int *__restrict__ sorted,
                                                  const int *__restrict__ op_ia,
                                                  int *__restrict__ ocol, double *__restrict__ oval,
                                                  char *__restrict__ oop)
{
   const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
   for (int r = blockIdx.x * WPB + wv; r < nrows; r += gridDim.x * WPB) {
      const int b = seg_ia[r], ns = seg_ia[r + 1] - b;
      int o = op_ia[r];
      if (ns == 0 || (longs && ij_long(r, seg_ia, op_ia))) { continue; }
      if (ns > 1) {
         for (int k = lane; k < ns; k += 64) {
            const int me = list[b + k];
            int rank = 0;
            for (int j = 0; j < ns; j++) { rank += list[b + j] < me; }
            sorted[b + rank] = me;
         }
         __threadfence_block();
         __builtin_amdgcn_wave_barrier();
      }
      const int *seq = ns > 1 ? sorted : list;
      for (int k0 = 0; k0 < ns; k0 += 64) {
         // a lane's segment, then all lanes copy one segment after the other
         // (64 short ones at once where all have one operation)
         int ch = 0, s = 0, len = 0, st = 0;
         if (k0 + lane < ns) {
            const int g = seq[b + k0 + lane];
            while (ch + 1 < Cp->n && g >= Cp->first[ch + 1]) { ch++; }
            s = g - Cp->first[ch];
            st = Cp->start[ch] ? Cp->start[ch][s] : s;
            len = Cp->start[ch] ? Cp->start[ch][s + 1] - st : 1;
         }
         const int here = min(64, ns - k0);
         if (!__any(len > 1)) {
            // places by the segments' lengths (0 or 1)
            const unsigned long long m = __ballot(len == 1);
            if (len == 1) {
               const int q = o + __popcll(m & ((1ull << lane) - 1));
               ocol[q] = Cp->cols[ch][st];
               oval[q] = Cp->vals[ch][st];
               oop[q] = Cp->ops[ch] ? Cp->ops[ch][s] : Cp->op[ch];
            }
            o += __popcll(m);
            continue;
         }
         for (int k = 0; k < here; k++) {
            const int kc = __shfl(ch, k, 64), kst = __shfl(st, k, 64), kl = __shfl(len, k, 64);
            const int ks = __shfl(s, k, 64);
            const char op = Cp->ops[kc] ? Cp->ops[kc][ks] : Cp->op[kc];
            for (int t = lane; t < kl; t += 64) {
               ocol[o + t] = Cp->cols[kc][kst + t];
               oval[o + t] = Cp->vals[kc][kst + t];
               oop[o + t] = op;
            }
            o += kl;
         }
      }
   }
}

// One wave a row: its operations, 64 at a time, against the columns it has so
// far and against each other; the row's entries are gathered in place (never
// ahead of the operations they come from).  A column's first operation gives
// its place and value, later ones overwrite (0) or add (1) in order.  *bad: a
// column outside [0, ncols).
__global__ __launch_bounds__(BS) void k_ij_fold(int nrows, bool longs, int ncols, int jlo, int diag_shift,
                                                const int *__restrict__ seg_ia,
                                                const int *__restrict__ op_ia, int *ocol, double *oval,
                                                const char *__restrict__ oop, int *__restrict__ cnt,
                                                int *__restrict__ dpos, int *__restrict__ bad)
{
   const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
   for (int r = blockIdx.x * WPB + wv; r < nrows; r += gridDim.x * WPB) {
      const int b = op_ia[r], m = op_ia[r + 1] - b;
      if (longs && ij_long(r, seg_ia, op_ia)) { continue; }
      int have = 0;
      for (int k0 = 0; k0 < m; k0 += 64) {
         const bool act = k0 + lane < m;
         int c = -1;
         double v = 0.0;
         int op = 0;
         if (act) {
            c = ocol[b + k0 + lane] - jlo;
            v = oval[b + k0 + lane];
            op = oop[b + k0 + lane];
            if (c < 0 || c >= ncols) { *bad = 1; }
         }
         // the place among the columns of earlier operations, then the first
         // lane of this batch with the same column
         int place = -1;
         for (int q = 0; q < have; q++) {
            if (ocol[b + q] == c) { place = q; }
         }
         int same = lane;
         const int here = min(64, m - k0);
         for (int j = here - 1; j >= 0; j--) {
            const int cj = __shfl(c, j, 64);
            if (cj == c && j < lane) { same = j; }
         }
         const bool lead = act && same == lane;           // first of its column here
         const bool fresh = lead && place < 0;
         const unsigned long long fm = __ballot(fresh);
         if (fresh) { place = have + __popcll(fm & ((1ull << lane) - 1)); }
         double acc = v;
         if (lead && !fresh) { acc = op == 0 ? v : oval[b + place] + v; }
         if (__any(act && !lead)) {
            for (int j = 0; j < here; j++) {
               const int sj = __shfl(same, j, 64), oj = __shfl(op, j, 64);
               const double vj = __shfl(v, j, 64);
               if (sj == lane && j != lane) { acc = oj == 0 ? vj : acc + vj; }
            }
         }
         // all operations of the batch are in registers: their room may be used
         __builtin_amdgcn_wave_barrier();
         if (lead) {
            ocol[b + place] = c;
            oval[b + place] = acc;
         }
         have += __popcll(fm);
         __threadfence_block();
         __builtin_amdgcn_wave_barrier();
      }
      int d = -1;
      for (int q0 = 0; q0 < have; q0 += 64) {
         const bool hit = q0 + lane < have && ocol[b + q0 + lane] == r + diag_shift;
         const unsigned long long hm = __ballot(hit);
         if (hm) { d = q0 + __ffsll((long long) hm) - 1; }
      }
      if (lane == 0) {
         cnt[r] = have;
         dpos[r] = d;
      }
   }
}

// entries of a row into CSR by the threads t of nt, the diagonal (place dpos)
// first: the entries before it one on, or, with swap, only the first one to its
// place
__device__ __forceinline__ void ij_write_row(int r, int t, int nt, const int *__restrict__ op_ia,
                                             const int *__restrict__ ocol, const double *__restrict__ oval,
                                             const int *__restrict__ dpos, bool swap,
                                             const int *__restrict__ ia, int *__restrict__ ja,
                                             double *__restrict__ a)
{
   const int b = op_ia[r], o = ia[r], m = ia[r + 1] - o, d = dpos[r];
   for (int q = t; q < m; q += nt) {
      int to = q;
      if (d > 0) {
         if (q == d) { to = 0; }
         else if (swap) { to = q == 0 ? d : q; }
         else if (q < d) { to = q + 1; }
      }
      ja[o + to] = ocol[b + q];
      a[o + to] = oval[b + q];
   }
}

__global__ __launch_bounds__(BS) void k_ij_write(int nrows, bool longs, const int *__restrict__ seg_ia,
                                                 const int *__restrict__ op_ia,
                                                 const int *__restrict__ ocol,
                                                 const double *__restrict__ oval,
                                                 const int *__restrict__ dpos, bool swap,
                                                 const int *__restrict__ ia, int *__restrict__ ja,
                                                 double *__restrict__ a)
{
   const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
   for (int r = blockIdx.x * WPB + wv; r < nrows; r += gridDim.x * WPB) {
      if (longs && ij_long(r, seg_ia, op_ia)) { continue; }
      ij_write_row(r, lane, 64, op_ia, ocol, oval, dpos, swap, ia, ja, a);
   }
}

// ------------------------------------------------------------------ long rows
// Rows of more than IJ_LONG operations or segments (constraints, mean values)
// by a block each: the wave kernels above compare a row's segments, and its
// columns, all with all, 1.1 and 0.46 ns times the square of their number.
// Here the segments are sorted and the columns found in a hash table: a row of
// 100,000 columns takes 0.9 ms, 3.9 from single operations (most of it the
// counters that all of them add to); the serial assembly's whole 1.9M operations
// took 17 to 18.
constexpr int BL = 1024;

__global__ __launch_bounds__(BS) void k_ij_long_list(int nrows, const int *__restrict__ seg_ia,
                                                     const int *__restrict__ op_ia, int *__restrict__ rows,
                                                     int *__restrict__ count)
{
   for (int r = blockIdx.x * BS + threadIdx.x; r < nrows; r += gridDim.x * BS) {
      if (ij_long(r, seg_ia, op_ia)) { rows[atomicAdd(count, 1)] = r; }
   }
}

// exclusive prefix sum over the block (wsum: a word a wave); *total: all of it
__device__ __forceinline__ int block_excl_scan(int v, int *wsum, int *total)
{
   const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
   int incl = v;
   for (int d = 1; d < 64; d <<= 1) {
      const int t = __shfl_up(incl, d, 64);
      if (lane >= d) { incl += t; }
   }
   if (lane == 63) { wsum[wv] = incl; }
   __syncthreads();
   int before = 0, all = 0;
   for (int w = 0; w < BL / 64; w++) {
      if (w < wv) { before += wsum[w]; }
      all += wsum[w];
   }
   __syncthreads();
   *total = all;
   return before + incl - v;
}

// A row's segments in call order and their operations at the row's place.  Up
// to IJ_SORT segment numbers are sorted in LDS.  More are marked as bits, 32
// IJ_SORT numbers at a time, and the bits read off in order: that takes the
// list once for every such window between its least and largest number.
constexpr int IJ_SORT = 8192;

__global__ __launch_bounds__(BL) void k_ij_layout_long(int nlong, const int *__restrict__ rows,
                                                       const IjChunks *__restrict__ Cp,
                                                       const int *__restrict__ seg_ia,
                                                       const int *__restrict__ list, int *sorted,
                                                       const int *__restrict__ op_ia,
                                                       int *__restrict__ ocol, double *__restrict__ oval,
                                                       char *__restrict__ oop)
{
   __shared__ int buf[IJ_SORT];
   __shared__ int off[BL], from[BL], seg[BL], wsum[BL / 64];
   __shared__ char chunk[BL];
   const int t = threadIdx.x;
   for (int w = blockIdx.x; w < nlong; w += gridDim.x) {
      const int r = rows[w], b = seg_ia[r], ns = seg_ia[r + 1] - b;
      if (ns <= IJ_SORT) {
         int n2 = 2;
         while (n2 < ns) { n2 <<= 1; }
         for (int k = t; k < n2; k += BL) { buf[k] = k < ns ? list[b + k] : INT_MAX; }
         __syncthreads();
         for (int size = 2; size <= n2; size <<= 1) {
            for (int d = size >> 1; d > 0; d >>= 1) {
               for (int k = t; k < n2 / 2; k += BL) {
                  const int i = 2 * k - (k & (d - 1)), j = i + d;
                  const int x = buf[i], y = buf[j];
                  if ((x > y) == ((i & size) == 0)) {
                     buf[i] = y;
                     buf[j] = x;
                  }
               }
               __syncthreads();
            }
         }
         for (int k = t; k < ns; k += BL) { sorted[b + k] = buf[k]; }
         __syncthreads();
      } else {
         if (t == 0) {
            off[0] = INT_MAX;
            off[1] = -1;
         }
         __syncthreads();
         int lo = INT_MAX, hi = -1;
         for (int k = t; k < ns; k += BL) {
            lo = min(lo, list[b + k]);
            hi = max(hi, list[b + k]);
         }
         atomicMin(off, lo);
         atomicMax(off + 1, hi);
         __syncthreads();
         lo = off[0];
         hi = off[1];
         int put = b;
         constexpr int PER = IJ_SORT / BL;
         for (long long base = lo; base <= hi; base += 32LL * IJ_SORT) {
            for (int k = t; k < IJ_SORT; k += BL) { buf[k] = 0; }
            __syncthreads();
            for (int k = t; k < ns; k += BL) {
               const long long g = list[b + k] - base;
               if (g >= 0 && g < 32LL * IJ_SORT) { atomicOr(buf + (g >> 5), 1 << (g & 31)); }
            }
            __syncthreads();
            int mine = 0, all;
            for (int k = 0; k < PER; k++) { mine += __popc((unsigned) buf[t * PER + k]); }
            int at = put + block_excl_scan(mine, wsum, &all);
            for (int k = 0; k < PER; k++) {
               for (unsigned bits = (unsigned) buf[t * PER + k]; bits; bits &= bits - 1u) {
                  sorted[at++] = (int) (base + 32 * (t * PER + k) + __ffs((int) bits) - 1);
               }
            }
            put += all;
            __syncthreads();
         }
      }
      int o = op_ia[r];
      for (int k0 = 0; k0 < ns; k0 += BL) {
         int len = 0, st = 0, s = 0, ch = 0, all;
         if (k0 + t < ns) {
            const int g = sorted[b + k0 + t];
            while (ch + 1 < Cp->n && g >= Cp->first[ch + 1]) { ch++; }
            s = g - Cp->first[ch];
            st = Cp->start[ch] ? Cp->start[ch][s] : s;
            len = Cp->start[ch] ? Cp->start[ch][s + 1] - st : 1;
         }
         const int place = block_excl_scan(len, wsum, &all);
         off[t] = place;
         from[t] = st;
         seg[t] = s;
         chunk[t] = (char) ch;
         __syncthreads();
         for (int q = t; q < all; q += BL) {
            int j = 0;      // the last segment that starts at or before q
            for (int d = BL / 2; d > 0; d >>= 1) {
               if (off[j + d] <= q) { j += d; }
            }
            const int c = chunk[j], e = from[j] + q - off[j];
            ocol[o + q] = Cp->cols[c][e];
            oval[o + q] = Cp->vals[c][e];
            oop[o + q] = Cp->ops[c] ? Cp->ops[c][seg[j]] : Cp->op[c];
         }
         o += all;
         __syncthreads();
      }
   }
}

// The table of a row: column and, beside it, first the least operation seen of
// the column, then its place (never more than that operation).
struct IjSlot
{
   int col, at;
};

static __host__ __device__ __forceinline__ unsigned long long ij_slots(int m)
{
   unsigned long long c = 64;
   while (c < 2ull * (unsigned) m) { c <<= 1; }
   return c;
}

// A row's operations, BL at a time: each finds its column in the table; the
// columns' first operations, in order, are the entries' places; then repeated
// columns overwrite or add, one wave after the other.
__global__ __launch_bounds__(BL) void k_ij_fold_long(int nlong, const int *__restrict__ rows, int ncols, int jlo,
                                                     int diag_shift, const int *__restrict__ op_ia, int *ocol,
                                                     double *oval, const char *__restrict__ oop,
                                                     IjSlot *__restrict__ tables, unsigned long long table_slots,
                                                     int *__restrict__ cnt, int *__restrict__ dpos,
                                                     int *__restrict__ bad)
{
   __shared__ int wsum[BL / 64];
   __shared__ int dplace;
   constexpr int SCOPE = __HIP_MEMORY_SCOPE_WORKGROUP;
   const int t = threadIdx.x, wv = t >> 6, lane = t & 63;
   IjSlot *table = tables + blockIdx.x * table_slots;
   for (int w = blockIdx.x; w < nlong; w += gridDim.x) {
      const int r = rows[w], b = op_ia[r], m = op_ia[r + 1] - b;
      const unsigned long long slots = ij_slots(m);
      for (unsigned long long k = t; k < slots; k += BL) {
         __hip_atomic_store(&table[k].col, -1, __ATOMIC_RELAXED, SCOPE);
         __hip_atomic_store(&table[k].at, INT_MAX, __ATOMIC_RELAXED, SCOPE);
      }
      if (t == 0) { dplace = -1; }
      __syncthreads();
      int have = 0;
      for (int k0 = 0; k0 < m; k0 += BL) {
         const int k = k0 + t;
         bool act = k < m;
         int c = 0, op = 0;
         double v = 0.0;
         IjSlot *e = table;
         if (act) {
            c = ocol[b + k] - jlo;
            v = oval[b + k];
            op = oop[b + k];
            if (c < 0 || c >= ncols) {
               *bad = 1;
               act = false;
            }
         }
         if (act) {
            unsigned long long h = ((unsigned long long) (unsigned) c * 0x9e3779b97f4a7c15ull >> 20) & (slots - 1);
            while (true) {      // at most half of the slots are ever taken
               int was = -1;
               if (__hip_atomic_compare_exchange_strong(&table[h].col, &was, c, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                        SCOPE) ||
                   was == c) {
                  break;
               }
               h = (h + 1) & (slots - 1);
            }
            e = table + h;
            __hip_atomic_fetch_min(&e->at, k, __ATOMIC_RELAXED, SCOPE);
         }
         __syncthreads();
         const bool fresh = act && __hip_atomic_load(&e->at, __ATOMIC_RELAXED, SCOPE) == k;
         int all;
         int place = have + block_excl_scan(fresh, wsum, &all);
         // all operations of the batch are in registers: their room may be used
         if (fresh) {
            __hip_atomic_store(&e->at, place, __ATOMIC_RELAXED, SCOPE);
            ocol[b + place] = c;
            oval[b + place] = v;
            if (c == r + diag_shift) { dplace = place; }
         }
         have += all;
         const bool again = act && !fresh;
         if (__syncthreads_or(again)) {
            if (again) { place = __hip_atomic_load(&e->at, __ATOMIC_RELAXED, SCOPE); }
            // the first lane of this wave with the same column
            int same = lane;
            const bool any = __any(again);
            for (int j = 63; any && j >= 0; j--) {
               const int pj = __shfl(again ? place : -1, j, 64);
               if (again && pj == place && j < lane) { same = j; }
            }
            const bool lead = again && same == lane, twice = __any(again && !lead);
            for (int turn = 0; turn < BL / 64; turn++) {
               if (turn == wv && any) {
                  double acc = 0.0;
                  if (lead) { acc = op == 0 ? v : oval[b + place] + v; }
                  for (int j = 0; twice && j < 64; j++) {
                     const int sj = __shfl(again ? same : -1, j, 64), oj = __shfl(op, j, 64);
                     const double vj = __shfl(v, j, 64);
                     if (sj == lane && j != lane) { acc = oj == 0 ? vj : acc + vj; }
                  }
                  if (lead) { oval[b + place] = acc; }
               }
               __syncthreads();
            }
         }
      }
      __syncthreads();
      if (t == 0) {
         cnt[r] = have;
         dpos[r] = dplace;
      }
      __syncthreads();
   }
}

__global__ __launch_bounds__(BL) void k_ij_write_long(int nlong, const int *__restrict__ rows,
                                                      const int *__restrict__ op_ia,
                                                      const int *__restrict__ ocol,
                                                      const double *__restrict__ oval,
                                                      const int *__restrict__ dpos, bool swap,
                                                      const int *__restrict__ ia, int *__restrict__ ja,
                                                      double *__restrict__ a)
{
   for (int w = blockIdx.x; w < nlong; w += gridDim.x) {
      ij_write_row(rows[w], threadIdx.x, BL, op_ia, ocol, oval, dpos, swap, ia, ja, a);
   }
}

void IjChunk::free_all()
{
   dfree(rows); dfree(ncols); dfree(cols); dfree(vals); dfree(ops);
   *this = IjChunk();
}

IjChunk ij_chunk(int nseg, long long nops, const int *rows, const int *ncols, const int *cols,
                 const double *vals, const char *ops, char op)
{
   IjChunk c;
   c.nseg = nseg;
   c.nops = nops;
   c.op = op;
   hipStream_t s = stream();
   // hipMemcpyDefault: the caller's arrays are on the host or on the device
   auto up = [&](auto *&d, const auto *h, size_t n) {
      if (!h) { return; }
      d = dalloc_n<std::remove_reference_t<decltype(*d)>>(std::max<size_t>(n, 1));
      HX_HIP(hipMemcpyAsync(d, h, n * sizeof(*h), hipMemcpyDefault, s));
   };
   try {
      up(c.rows, rows, (size_t) nseg);
      up(c.ncols, ncols, (size_t) nseg);
      up(c.cols, cols, (size_t) nops);
      up(c.vals, vals, (size_t) nops);
      up(c.ops, ops, (size_t) nseg);
      sync();   // the caller may reuse its arrays
   } catch (...) {
      c.free_all();
      throw;
   }
   return c;
}

bool ij_assemble_device(const std::vector<IjChunk> &chunks, int ilower, int nrows, int jlower, int ncols,
                        bool swap_diag, Csr &A)
{
   long long nseg = 0, nops = 0;
   for (const IjChunk &c : chunks) {
      nseg += c.nseg;
      nops += c.nops;
   }
   if (nseg > INT_MAX || nops > INT_MAX || (int) chunks.size() > IJ_CHUNKS) {
      fail(HYPRE_ERROR_MEMORY, "too many operations for one assembly");
   }
   std::vector<void *> held;   // returned to the allocator in any case
   struct Free
   {
      std::vector<void *> &v;
      ~Free() { for (void *p : v) { dfree(p); } }
   } guard_held{held};
   auto ints = [&](size_t n) {
      int *p = dalloc_n<int>(std::max<size_t>(n, 1));
      held.push_back(p);
      return p;
   };
   hipStream_t s = stream();
   int *seg_ia = ints((size_t) nrows + 1), *op_ia = ints((size_t) nrows + 1), *fill = ints((size_t) nrows + 1);
   dzero(seg_ia, sizeof(int) * ((size_t) nrows + 1));
   dzero(op_ia, sizeof(int) * ((size_t) nrows + 1));
   IjChunks C{};
   C.n = (int) chunks.size();
   int first = 0;
   for (int k = 0; k < C.n; k++) {
      const IjChunk &c = chunks[(size_t) k];
      C.first[k] = first;
      C.cols[k] = c.cols;
      C.vals[k] = c.vals;
      C.ops[k] = c.ops;
      C.op[k] = c.op;
      if (c.ncols) {
         int *st = ints((size_t) c.nseg + 1);
         exclusive_scan_nowait(c.ncols, st, c.nseg);
         C.start[k] = st;
      }
      k_ij_count<<<ij_grid(c.nseg, BS), BS, 0, s>>>(c.nseg, c.rows, c.ncols, ilower, nrows, seg_ia, op_ia);
      HX_LAUNCH_CHECK();
      first += c.nseg;
   }
   int most_seg = 0, most_op = 0;
   const int total_seg = (int) exclusive_scan(seg_ia, seg_ia, nrows, &most_seg);
   const int total_op = (int) exclusive_scan(op_ia, op_ia, nrows, &most_op);
   d2d(fill, seg_ia, sizeof(int) * ((size_t) nrows + 1));
   int *list = ints((size_t) total_seg), *sorted = ints((size_t) total_seg);
   for (int k = 0; k < C.n; k++) {
      const IjChunk &c = chunks[(size_t) k];
      k_ij_scatter<<<ij_grid(c.nseg, BS), BS, 0, s>>>(c.nseg, C.first[k], c.rows, ilower, nrows, fill, list);
      HX_LAUNCH_CHECK();
   }
   int *ocol = ints((size_t) total_op), *cnt = ints((size_t) nrows + 1), *dpos = ints((size_t) nrows);
   double *oval = dalloc_n<double>((size_t) std::max(total_op, 1));
   held.push_back(oval);
   char *oop = dalloc_n<char>((size_t) std::max(total_op, 1));
   held.push_back(oop);
   int *bad = device_flags() + 76, *nlong_dev = device_flags() + 77;
   dzero(bad, 2 * sizeof(int));
   const int nb = ij_grid(nrows, WPB);
   IjChunks *dC = dalloc_n<IjChunks>(1);
   held.push_back(dC);
   h2d(dC, &C, sizeof(C));
   const bool some_long = most_seg > IJ_LONG || most_op > IJ_LONG;
   k_ij_layout<<<nb, BS, 0, s>>>(nrows, some_long, dC, seg_ia, list, sorted, op_ia, ocol, oval, oop);
   HX_LAUNCH_CHECK();
   k_ij_fold<<<nb, BS, 0, s>>>(nrows, some_long, ncols, jlower, ilower - jlower, seg_ia, op_ia, ocol, oval, oop,
                               cnt, dpos, bad);
   HX_LAUNCH_CHECK();
   int nlong = 0, *longs = nullptr;
   if (some_long) {
      longs = ints((size_t) nrows);
      k_ij_long_list<<<ij_grid(nrows, BS), BS, 0, s>>>(nrows, seg_ia, op_ia, longs, nlong_dev);
      HX_LAUNCH_CHECK();
      d2h(&nlong, nlong_dev, sizeof(int));
      // a table a block, in all no more than some times the operations' memory
      const unsigned long long slots = ij_slots(most_op);
      const int blocks = (int) std::min<unsigned long long>(
         (unsigned long long) std::min(nlong, 512), std::max<unsigned long long>(4ull * (unsigned) total_op / slots, 1));
      IjSlot *tables = dalloc_n<IjSlot>((size_t) (slots * (unsigned) blocks));
      held.push_back(tables);
      k_ij_layout_long<<<std::min(nlong, 512), BL, 0, s>>>(nlong, longs, dC, seg_ia, list, sorted, op_ia, ocol, oval,
                                                           oop);
      HX_LAUNCH_CHECK();
      k_ij_fold_long<<<blocks, BL, 0, s>>>(nlong, longs, ncols, jlower, ilower - jlower, op_ia, ocol, oval, oop,
                                           tables, slots, cnt, dpos, bad);
      HX_LAUNCH_CHECK();
   }
   Csr out;
   out.nrows = nrows;
   out.ncols = ncols;
   int h = 0;
   try {
      out.ia = dalloc_n<int>((size_t) nrows + 1);
      out.nnz = exclusive_scan(cnt, out.ia, nrows);
      d2h(&h, bad, sizeof(int));
      if (h == 0) {
         out.ja = dalloc_n<int>((size_t) std::max<long long>(out.nnz, 1));
         out.a = dalloc_n<double>((size_t) std::max<long long>(out.nnz, 1));
         k_ij_write<<<nb, BS, 0, s>>>(nrows, some_long, seg_ia, op_ia, ocol, oval, dpos, swap_diag, out.ia, out.ja, out.a);
         HX_LAUNCH_CHECK();
         if (nlong > 0) {
            k_ij_write_long<<<std::min(nlong, 512), BL, 0, s>>>(nlong, longs, op_ia, ocol, oval, dpos, swap_diag,
                                                                out.ia, out.ja, out.a);
            HX_LAUNCH_CHECK();
         }
         // an assembled matrix is complete: its arrays are handed out as they
         // are, and no stream of the caller's is ordered after this one
         sync();
      }
   } catch (...) {
      out.free_all();
      throw;
   }
   if (h) {
      out.free_all();
      return false;
   }
   A = out;
   return true;
}

} // namespace hx
