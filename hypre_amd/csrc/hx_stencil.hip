// Stencil copy of a level operator for the solve phase: rows whose columns
// differ from the row by one of at most 32 offsets that the whole matrix
// shares (grid operators in their natural order), stored diagonal first and
// then by ascending column.
//
// What bounds a product with a sliced-ELL copy is the matrix stream, 9 to 10
// bytes per entry.  Here the columns cost four bytes a row (a mask of the
// offsets the row has; the offsets themselves are kernel arguments) and the
// values as little as the slice of 128 rows allows: nothing where every entry
// of an offset has the same value as the offset's table (constant
// coefficients), one byte an entry where the slice holds at most 256 distinct
// values (coefficients constant by regions: its own dictionary, staged in
// LDS), eight (four in the FP32 cycle) otherwise.  All values are kept
// exactly, and each row adds the products of the entries it has in storage
// order, so the results are those of the CSR and sliced-ELL kernels bit for
// bit.  Measured against the sliced-ELL kernels (product / l1-Jacobi sweep):
// 27-point 200^3 constant 511 / 535 -> 73 / 88 us, jumping coefficients
// 513 / 538 -> 107 / 124 us (FP32 sweep 280 -> 88); 7-point 256^3
// 363 / 421 -> 100 / 132 us (3.4 TB/s of the bytes left).  Where rows have few of
// the offsets the copy may not pay (sten_pays).
#include "hx_internal.h"

#include <algorithm>
#include <climits>
#include <cstring>

namespace hx {

constexpr int BS = 256;
constexpr int WPB = BS / 64;
constexpr int ST_MAX = 32;           // offsets (one mask word a row)
constexpr int ST_ROWS = 128;         // rows of a slice, two a lane
constexpr int ST_DICT = 256;         // distinct values of a dictionary slice
constexpr int ST_CONST = 0, ST_CODES = 1, ST_RAW = 2;

// ---------------------------------------------------------------- probing
// Device words of the probe: [0] not a stencil, [1] offsets found, [2] longest
// row, [4..] a hash set of offsets and, beside it, the least entry index seen
// with each offset; then the table as the host reads it.
constexpr int ST_SLOTS = 128;
constexpr int ST_KEY = 4, ST_REP = ST_KEY + ST_SLOTS, ST_WORDS = ST_REP + ST_SLOTS;
constexpr int ST_EMPTY = INT_MIN;    // no column lies 2^31 before its row

__global__ void k_sten_init(int *__restrict__ st)
{
   for (int i = threadIdx.x; i < ST_WORDS; i += blockDim.x) {
      st[i] = (i < ST_KEY) ? 0 : (i < ST_REP) ? ST_EMPTY : INT_MAX;
   }
}

__device__ __forceinline__ int sten_slot(int d) { return (int) (((unsigned) d * 2654435761u) >> 25); }

// the slot of offset d in a set of ST_SLOTS keys, inserted when new (*fresh);
// -1 when the set is full.  At most ST_SLOTS probes.
__device__ __forceinline__ int sten_insert(volatile int *key, int d, bool *fresh)
{
   int h = sten_slot(d);
   *fresh = false;
   for (int t = 0; t < ST_SLOTS; t++) {
      int cur = key[h];
      if (cur == ST_EMPTY) {
         cur = atomicCAS(const_cast<int *>(key) + h, ST_EMPTY, d);
         if (cur == ST_EMPTY) { *fresh = true; return h; }
      }
      if (cur == d) { return h; }
      h = (h + 1) & (ST_SLOTS - 1);
   }
   return -1;
}

// Eight lanes walk a row: the diagonal first, then columns ascending, and the
// row's offsets into the block's set, merged into the global one at the end.
// A matrix of another kind overfills a block's set within its first rows, and
// every block stops at the next look at the global flag.
__global__ __launch_bounds__(BS) void k_sten_probe(int n, const int *__restrict__ ia,
                                                   const int *__restrict__ ja, int *__restrict__ st)
{
   __shared__ int key[ST_SLOTS], rep[ST_SLOTS];
   __shared__ int count, bad, longest;
   for (int i = threadIdx.x; i < ST_SLOTS; i += BS) {
      key[i] = ST_EMPTY;
      rep[i] = INT_MAX;
   }
   if (threadIdx.x == 0) {
      count = 0;
      bad = 0;
      longest = 0;
   }
   __syncthreads();
   constexpr int G = 8, RPB = BS / G;
   const int per = (int) (((long long) n + gridDim.x - 1) / gridDim.x);
   const long long first = (long long) blockIdx.x * per;
   const int r0 = (int) (first < n ? first : n);
   const int r1 = (int) (first + per < n ? first + per : n);
   const int l = threadIdx.x & (G - 1);
   int len = 0;
   bool fail = false;
   int step = 0;
   for (int r = r0 + threadIdx.x / G; r < r1 && !fail; r += RPB, step++) {
      if ((step & 7) == 0 && (*(volatile int *) st != 0 || *(volatile int *) &bad != 0)) { break; }
      const int s = ia[r], e = ia[r + 1];
      len = max(len, e - s);
      if (e <= s || e - s > ST_MAX) { fail = true; break; }
      for (int q = s + l; q < e; q += G) {
         const int c = ja[q];
         if (q == s ? c != r : (c == r || (q > s + 1 && c <= ja[q - 1]))) { fail = true; break; }
         bool fresh;
         const int h = sten_insert(key, c - r, &fresh);
         if (h < 0) { fail = true; break; }
         // rows ascend: seldom once the block has seen the offset
         if (q < *(volatile int *) (rep + h)) { atomicMin(rep + h, q); }
         if (fresh && atomicAdd(&count, 1) >= ST_MAX) { fail = true; break; }
      }
   }
   if (fail) { bad = 1; }
   if (l == 0) { atomicMax(&longest, len); }
   __syncthreads();
   if (bad) {
      if (threadIdx.x == 0) { st[0] = 1; }
      return;
   }
   if (threadIdx.x == 0) { atomicMax(st + 2, longest); }
   for (int i = threadIdx.x; i < ST_SLOTS; i += BS) {
      if (key[i] == ST_EMPTY) { continue; }
      bool fresh;
      const int h = sten_insert(st + ST_KEY, key[i], &fresh);
      if (h < 0 || (fresh && atomicAdd(st + 1, 1) >= ST_MAX)) {
         st[0] = 1;
         continue;
      }
      atomicMin(st + ST_REP + h, rep[i]);
   }
}

// The table: offset 0 first, then ascending, with the value of one entry of
// each offset.  Any entry serves, but slices need no values where they have the
// table's, so it is taken from inside the grid: from the row of the greatest
// length that is nearest to the middle (among ST_LOOK tiles of rows around it),
// for offsets that this row has not the offset's first entry.
constexpr int ST_TABLE = 1024, ST_LOOK = 256;

__global__ __launch_bounds__(ST_TABLE) void k_sten_table(int n, const int *__restrict__ ia,
                                                         const int *__restrict__ ja,
                                                         const double *__restrict__ a,
                                                         const int *__restrict__ st,
                                                         StenHead *__restrict__ out)
{
   __shared__ int key[ST_SLOTS], rep[ST_SLOTS];
   __shared__ int best;
   const int i = threadIdx.x;
   const bool ok = st[0] == 0 && st[1] >= 1 && st[1] <= ST_MAX;
   if (i < ST_SLOTS) {
      key[i] = st[ST_KEY + i];
      rep[i] = st[ST_REP + i];
   }
   if (i == 0) { best = INT_MAX; }
   __syncthreads();
   if (i < ST_MAX) {
      out->off[i] = 0;
      out->v[i] = 0.0;
   }
   if (i == 0) {
      out->ok = ok ? 1 : 0;
      out->D = ok ? st[1] : 0;
      out->wmax = st[2];
      out->raw = 0;
      out->coded = 0;
      out->hops = 0;
   }
   if (!ok) { return; }
   const int mid = n / 2, longest = st[2];
   for (int t = 0; t < ST_LOOK; t++) {
      const int d = t * (ST_TABLE / 2) + (i >> 1);
      const long long r = (i & 1) ? (long long) mid - 1 - d : (long long) mid + d;
      const bool hit = r >= 0 && r < n && ia[r + 1] - ia[r] == longest;
      if (hit) { atomicMin(&best, 2 * d + (i & 1)); }
      if (__syncthreads_or(hit)) { break; }
   }
   if (best != INT_MAX && i < longest) {
      const int r = (best & 1) ? mid - 1 - (best >> 1) : mid + (best >> 1);
      const int q = ia[r] + i, d = ja[q] - r;
      for (int j = 0; j < ST_SLOTS; j++) {
         if (key[j] == d) { rep[j] = q; }
      }
   }
   __syncthreads();
   if (i >= ST_SLOTS || key[i] == ST_EMPTY) { return; }
   int rank = 0;
   for (int j = 0; j < ST_SLOTS; j++) {
      if (j == i || key[j] == ST_EMPTY) { continue; }
      rank += key[i] != 0 && (key[j] == 0 || key[j] < key[i]);
   }
   if (rank < ST_MAX) {
      out->off[rank] = key[i];
      out->v[rank] = a[rep[i]];
   }
}

// distinct sums of two offsets in ascending order, numbered for every pair, by
// comparing all with all (on the side stream, beside the first setup kernels)
__global__ __launch_bounds__(ST_MAX * ST_MAX) void k_sten_hop(StenHead *__restrict__ T,
                                                             StenHop *__restrict__ out)
{
   __shared__ long long sum[ST_MAX * ST_MAX];
   __shared__ unsigned char first[ST_MAX * ST_MAX];
   __shared__ int count;
   const int i = threadIdx.x, k = i / ST_MAX, l = i % ST_MAX;
   const int D = T->D;
   const bool in = T->ok && k < D && l < D;
   const long long NONE = LLONG_MAX;
   sum[i] = in ? (long long) T->off[k] + T->off[l] : NONE;
   if (i == 0) { count = 0; }
   __syncthreads();
   bool f = in;
   for (int j = 0; j < i; j++) { f = f && sum[j] != sum[i]; }
   first[i] = f;
   if (f) { atomicAdd(&count, 1); }
   __syncthreads();
   if (i == 0) { T->hops = count; }
   if (i < ST_MAX) {
      int m = -1;
      for (int j = 0; j < D; j++) {
         if (i < D && T->off[j] == -T->off[i]) { m = j; }
      }
      out->mirror[i] = m;
   }
   if (!in || count > STEN_HOPS) { return; }
   int rank = 0;
   for (int j = 0; j < ST_MAX * ST_MAX; j++) { rank += first[j] && sum[j] < sum[i]; }
   out->id[i] = (unsigned char) rank;
   if (f) { out->hop[rank] = (int) sum[i]; }
}

// ---------------------------------------------------------------- filling
// One wave per slice, 32 rows at a time (at most 1024 entries, staged through
// LDS with coalesced loads).  First lane = row walks the table's steps and
// takes its next entry when that has the step's offset; a slice whose values
// are all the table's needs no more.  Otherwise lane = entry numbers the values
// in an LDS hash (a lane that finds its value reads the number, one that does
// not claims a slot and the next number), three entries a lane in flight, and
// two lanes a row pack the numbers four to a word.  A slice is read once,
// unless its first rows have the table's values and later ones do not.
// 27-point 320^3 with jumps (all slices coded, beside the level's PMIS, 10.5 GB
// read): 14.6 ms by rows, one entry a lane and every slice read twice; 8.6 now.
constexpr int SF_ROWS = 32, SF_PARTS = ST_ROWS / SF_ROWS, SF_CH = SF_ROWS * ST_MAX, SF_HASH = 512, SF_U = 3;

__device__ __forceinline__ void sten_stage(int s0, int s1, int lane, const int *__restrict__ ja,
                                           const double *__restrict__ a, int *sj, double *sa)
{
   __syncthreads();
   for (int q0 = s0; q0 < s1; q0 += 256) {
      int jv[4];
      double av[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
         const int q = min(q0 + u * 64 + lane, s1 - 1);
         jv[u] = __builtin_nontemporal_load(ja + q);
         av[u] = __builtin_nontemporal_load(a + q);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
         const int q = q0 + u * 64 + lane;
         if (q < s1) {
            sj[q - s0] = jv[u];
            sa[q - s0] = av[u];
         }
      }
   }
   __syncthreads();
}

__global__ __launch_bounds__(64) void k_sten_fill(int n, int ns, StenHead T,
                                                  const int *__restrict__ ia,
                                                  const int *__restrict__ ja,
                                                  const double *__restrict__ a,
                                                  unsigned *__restrict__ mask,
                                                  int *__restrict__ info,
                                                  unsigned *__restrict__ codes,
                                                  double *__restrict__ dict, int *__restrict__ nraw,
                                                  int *__restrict__ ncoded)
{
   __shared__ int sj[SF_CH];
   __shared__ double sa[SF_CH];
   __shared__ unsigned long long key[SF_HASH];
   __shared__ unsigned short num[SF_HASH];
   __shared__ int count;
   constexpr unsigned long long FREE = ~0ull;   // a NaN: slices that hold it are stored in full
   const int lane = threadIdx.x;
   const int D = T.D, CW = (D + 3) / 4;
   const unsigned all = D == 32 ? ~0u : (1u << D) - 1u;
   unsigned char *code = reinterpret_cast<unsigned char *>(sj);   // once a part's columns are done
   for (int sl = blockIdx.x; sl < ns; sl += gridDim.x) {
      bool full = true, coding = false, raw = false;
      for (int h = 0; h < SF_PARTS; h++) {
         const int f = (int) min((long long) n, (long long) sl * ST_ROWS + h * SF_ROWS);
         const int r = f + lane;
         const int s0 = ia[f], s1 = ia[(int) min((long long) n, (long long) f + SF_ROWS)];
         const bool row = lane < SF_ROWS && r < n;
         const int q0 = row ? ia[r] - s0 : 0, e = row ? ia[r + 1] - s0 : 0;
         sten_stage(s0, s1, lane, ja, a, sj, sa);
         unsigned m = 0;
         bool same = true;
         int q = q0;
         for (int k = 0; k < D; k++) {
            if (q < e && sj[q] - r == T.off[k]) {
               m |= 1u << k;
               same = same && __double_as_longlong(sa[q]) == __double_as_longlong(T.v[k]);
               q++;
            }
         }
         if (lane < SF_ROWS) {
            mask[(size_t) sl * ST_ROWS + h * SF_ROWS + lane] = m;
            full = full && m == all;
         }
         if (!coding && !__all(same)) {
            // the slice needs codes: from its first part
            coding = true;
            for (int i = lane; i < SF_HASH; i += 64) { key[i] = FREE; }
            if (lane == 0) { count = 0; }
            if (h > 0) {
               h = -1;
               continue;
            }
         }
         if (!coding || raw) { continue; }
         __syncthreads();
         for (int c0 = 0; c0 < s1 - s0 && !raw; c0 += 64 * SF_U) {
            unsigned long long bits[SF_U];
            int at[SF_U];
            bool look[SF_U];
            bool odd = false;
#pragma unroll
            for (int u = 0; u < SF_U; u++) {
               const int i = c0 + u * 64 + lane;
               const bool in = i < s1 - s0;
               bits[u] = in ? (unsigned long long) __double_as_longlong(sa[i]) : 0ull;
               at[u] = (int) ((bits[u] * 0x9e3779b97f4a7c15ull) >> 55);
               look[u] = in && bits[u] != FREE;
               odd = odd || (in && bits[u] == FREE);
            }
            raw = __any(odd);
            // at most 256 + 192 of the 512 slots are ever taken: a free one ends
            // every search
            for (bool more = !raw; more;) {
               unsigned long long cur[SF_U];
#pragma unroll
               for (int u = 0; u < SF_U; u++) { cur[u] = *(volatile unsigned long long *) (key + at[u]); }
               bool left = false;
#pragma unroll
               for (int u = 0; u < SF_U; u++) {
                  if (look[u]) {
                     if (cur[u] == FREE) {
                        cur[u] = atomicCAS(key + at[u], FREE, bits[u]);
                        if (cur[u] == FREE) {
                           num[at[u]] = (unsigned short) atomicAdd(&count, 1);
                           cur[u] = bits[u];
                        }
                     }
                     if (cur[u] == bits[u]) { look[u] = false; }
                     else { at[u] = (at[u] + 1) & (SF_HASH - 1); }
                  }
                  left = left || look[u];
               }
               more = __any(left);
            }
            __syncthreads();
            raw = raw || count > ST_DICT;
            if (raw) { break; }
#pragma unroll
            for (int u = 0; u < SF_U; u++) {
               const int i = c0 + u * 64 + lane;
               if (i < s1 - s0) { code[i] = (unsigned char) num[at[u]]; }
            }
         }
         __syncthreads();
         if (raw) { continue; }
         const int half = lane >> 5, sub = lane & (SF_ROWS - 1);
         const unsigned mr = __shfl(m, sub);
         const int qr = __shfl(q0, sub);
         for (int w = half; w < CW; w += 2) {
            unsigned word = 0;
#pragma unroll
            for (int u = 0; u < 4; u++) {
               const unsigned bit = 4 * w + u < 32 ? 1u << (4 * w + u) : 0u;
               if (mr & bit) { word |= (unsigned) code[qr + __popc(mr & (bit - 1u))] << (u * 8); }
            }
            codes[((size_t) sl * CW + w) * ST_ROWS + h * SF_ROWS + sub] = word;
         }
      }
      const int fl = __all(full) ? 4 : 0;
      if (!coding) {
         if (lane == 0) { info[sl] = ST_CONST | fl; }
         continue;
      }
      __syncthreads();
      if (raw) {
         if (lane == 0) {
            info[sl] = ST_RAW | fl;
            atomicAdd(nraw, 1);
         }
         continue;
      }
      for (int i = lane; i < SF_HASH; i += 64) {
         if (key[i] != FREE) {
            dict[(size_t) sl * ST_DICT + num[i]] = __longlong_as_double((long long) key[i]);
         }
      }
      if (lane == 0) {
         info[sl] = ST_CODES | fl | count << 8;
         atomicAdd(ncoded, 1);
      }
   }
}

// Full values are kept for the slices that need them alone, numbered in order
// (out of order their products take 3% longer); one block, a stretch of slices a
// thread.
constexpr int ST_NUMBER = 1024;

__global__ __launch_bounds__(ST_NUMBER) void k_sten_number(int ns, int *__restrict__ info)
{
   __shared__ int sum[ST_NUMBER];
   const int t = threadIdx.x, per = (ns + ST_NUMBER - 1) / ST_NUMBER;
   const int s0 = (int) min((long long) ns, (long long) t * per), s1 = min(ns, s0 + per);
   int c = 0;
   for (int s = s0; s < s1; s++) { c += (info[s] & 3) == ST_RAW; }
   sum[t] = c;
   __syncthreads();
   for (int d = 1; d < ST_NUMBER; d <<= 1) {
      const int v = t >= d ? sum[t - d] : 0;
      __syncthreads();
      sum[t] += v;
      __syncthreads();
   }
   int at = sum[t] - c;
   for (int s = s0; s < s1; s++) {
      if ((info[s] & 3) == ST_RAW) { info[s] |= at++ << 8; }
   }
}

// the values of those slices, step by step
__global__ __launch_bounds__(64) void k_sten_raw(int n, int ns, StenHead T,
                                                 const int *__restrict__ ia,
                                                 const int *__restrict__ ja,
                                                 const double *__restrict__ a,
                                                 const int *__restrict__ info,
                                                 double *__restrict__ raw, float *__restrict__ raw32)
{
   __shared__ int sj[SF_CH];
   __shared__ double sa[SF_CH];
   const int lane = threadIdx.x;
   const int D = T.D;
   for (int sl = blockIdx.x; sl < ns; sl += gridDim.x) {
      const int in = info[sl];
      if ((in & 3) != ST_RAW) { continue; }
      const size_t base = (size_t) (in >> 8) * D;
      for (int h = 0; h < SF_PARTS; h++) {
         const int f = (int) min((long long) n, (long long) sl * ST_ROWS + h * SF_ROWS);
         const int r = f + lane;
         const int s0 = ia[f], s1 = ia[(int) min((long long) n, (long long) f + SF_ROWS)];
         const bool row = lane < SF_ROWS && r < n;
         int q = row ? ia[r] - s0 : 0, e = row ? ia[r + 1] - s0 : 0;
         sten_stage(s0, s1, lane, ja, a, sj, sa);
         for (int k = 0; k < D; k++) {
            double v = 0.0;
            if (q < e && sj[q] - r == T.off[k]) { v = sa[q++]; }
            if (lane < SF_ROWS) {
               const size_t at = (base + k) * ST_ROWS + h * SF_ROWS + lane;
               raw[at] = v;
               if (raw32) { raw32[at] = (float) v; }
            }
         }
      }
   }
}

void Sten::free_all()
{
   dfree(st); dfree(head); dfree(hop); dfree(mask); dfree(info); dfree(codes); dfree(dict); dfree(raw);
   dfree(raw32);
   *this = Sten();
}

// host side of the probe's result: pinned, one for the library's one stream of
// setups
static StenHead *sten_pinned()
{
   static StenHead *h = nullptr;
   if (!h) { HX_HIP(hipHostMalloc(reinterpret_cast<void **>(&h), sizeof(StenHead), hipHostMallocDefault)); }
   return h;
}

bool sten_probe(const Csr &A, Sten &S, int min_rows, hipStream_t s)
{
   S.free_all();
   if (A.nrows < std::max(min_rows, 1) || A.ncols != A.nrows ||
       A.nnz > (long long) ST_MAX * A.nrows) {
      return false;
   }
   S.st = dalloc_n<int>(ST_WORDS);
   S.head = dalloc_n<StenHead>(1);
   S.hop = dalloc_n<StenHop>(1);
   sten_pinned()->ok = 0;
   k_sten_init<<<1, BS, 0, s>>>(S.st);
   HX_LAUNCH_CHECK();
   // half of the wave slots: with all of them, the first kernels of the strength
   // pass waited for the probe's blocks to end (1.9 ms of 27-point 320^3: setup and
   // solve 224.1 ms, 222.9 now; 7-point of 1.67 M rows 16.03, 15.94)
   const int nb = (int) std::min<long long>(((long long) A.nrows + 255) / 256, 1024);
   k_sten_probe<<<nb, BS, 0, s>>>(A.nrows, A.ia, A.ja, S.st);
   HX_LAUNCH_CHECK();
   k_sten_table<<<1, ST_TABLE, 0, s>>>(A.nrows, A.ia, A.ja, A.a, S.st, S.head);
   HX_LAUNCH_CHECK();
   k_sten_hop<<<1, ST_MAX * ST_MAX, 0, s>>>(S.head, S.hop);
   HX_LAUNCH_CHECK();
   HX_HIP(hipMemcpyAsync(sten_pinned(), S.head, sizeof(StenHead), hipMemcpyDeviceToHost, s));
   return true;
}

bool sten_take(Sten &S)
{
   S.tab = *sten_pinned();
   if (!S.tab.ok) { S.free_all(); }
   return S.tab.ok != 0;
}

// One-wave blocks, eight a CU (9 fit its LDS): the fill runs beside the fine
// level's PMIS, short kernels and waits, and has to be done when they are.
constexpr int SF_GRID = 2048;

void sten_fill(const Csr &A, Sten &S, hipStream_t s)
{
   const int ns = (int) (((long long) A.nrows + ST_ROWS - 1) / ST_ROWS);
   const size_t cw = (size_t) (S.tab.D + 3) / 4;
   S.mask = dalloc_n<unsigned>((size_t) ns * ST_ROWS);
   S.info = dalloc_n<int>((size_t) ns);
   S.codes = dalloc_n<unsigned>((size_t) ns * ST_ROWS * cw);
   S.dict = dalloc_n<double>((size_t) ns * ST_DICT);
   S.nslices = ns;
   k_sten_fill<<<std::min(ns, SF_GRID), 64, 0, s>>>(A.nrows, ns, S.tab, A.ia, A.ja, A.a, S.mask,
                                                    S.info, S.codes, S.dict, &S.head->raw, &S.head->coded);
   HX_LAUNCH_CHECK();
   HX_HIP(hipMemcpyAsync(&sten_pinned()->raw, &S.head->raw, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
}

void sten_counts(Sten &S)
{
   S.tab.raw = sten_pinned()->raw;
   S.tab.coded = sten_pinned()->coded;
   if (S.tab.coded == 0) {
      // no slice reads them
      dfree(S.codes);
      dfree(S.dict);
      S.codes = nullptr;
      S.dict = nullptr;
   }
}

// A slice takes the same time however many of the offsets its rows have, the
// other kernels a time that grows with the entries.  In entries a row (of which
// the other kernels move some 17 G/ms), an offset costs 0.10 in slices without
// values, 0.13 with codes and 0.52 with full values.  Products of 120^3 rows, the
// copy's / the others' by entries a row, us: 27 offsets in full 78 / 107 (26.8),
// 100 (16.5), 62 (11.3), 45 (7.5); 31 offsets without runs in full 99 / 130
// (30.7), 115 (18.8), 74 (12.9); 7 in full 29 / 40 (7), 33 (4.6), 24 (2.8); 27
// with codes 31 / 107, 100, 62, 45 and 33 (4.1); 31 with codes 34 / 39 (4.6); 27
// without values 21 / 33 (4.1).
bool sten_pays(const Csr &A, const Sten &S)
{
   const double bare = S.nslices - S.tab.coded - S.tab.raw;
   const double cost = S.tab.D * (0.10 * bare + 0.13 * S.tab.coded + 0.52 * S.tab.raw) / S.nslices;
   return cost <= (double) A.nnz / A.nrows;
}

void sten_fill_raw(const Csr &A, Sten &S, bool fp32, hipStream_t s)
{
   const size_t words = (size_t) S.tab.raw * ST_ROWS * S.tab.D;
   S.raw = dalloc_n<double>(words);
   if (fp32) { S.raw32 = dalloc_n<float>(words); }
   k_sten_number<<<1, ST_NUMBER, 0, s>>>(S.nslices, S.info);
   HX_LAUNCH_CHECK();
   k_sten_raw<<<std::min(S.nslices, SF_GRID), 64, 0, s>>>(A.nrows, S.nslices, S.tab, A.ia, A.ja, A.a,
                                                          S.info, S.raw, S.raw32);
   HX_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- products
// The table in device memory.  Read through the constant address space it
// stays in scalar registers, and through a pointer that is new to the compiler
// in every slice (sten_rows) only while the slice needs it: hoisted out of the
// slice loop, 27 offsets and values took 160 vector registers for spilled
// scalars.
typedef const __attribute__((address_space(4))) StenHead *StenTab;

struct StenView
{
   const StenHead *tab;
   const unsigned *mask, *codes;
   const int *info;
   const double *dict;
};

// The runs of the usual grid stencils' offsets in ascending order: three
// consecutive ones or a single one (5 and 9 points in 2D; 7, 19 and 27 in 3D).
// Other tables, K = 32, have no known runs.
template <int K>
struct StenRuns
{
   static constexpr int count = 0, mid = -1;
   static constexpr int len[1] = {0};
};
template <>
struct StenRuns<5>
{
   static constexpr int count = 3, mid = 1;
   static constexpr int len[count] = {1, 3, 1};
};
template <>
struct StenRuns<7>
{
   static constexpr int count = 5, mid = 2;
   static constexpr int len[count] = {1, 1, 3, 1, 1};
};
template <>
struct StenRuns<9>
{
   static constexpr int count = 3, mid = 1;
   static constexpr int len[count] = {3, 3, 3};
};
template <>
struct StenRuns<19>
{
   static constexpr int count = 9, mid = 4;
   static constexpr int len[count] = {1, 3, 1, 3, 3, 3, 1, 3, 1};
};
template <>
struct StenRuns<27>
{
   static constexpr int count = 9, mid = 4;
   static constexpr int len[count] = {3, 3, 3, 3, 3, 3, 3, 3, 3};
};

// whether the table's offsets have these runs around zero
template <int K>
static bool sten_has_runs(const StenHead &T)
{
   if (T.D != K) { return false; }
   int at = 1;   // the next step past the diagonal
   for (int r = 0; r < StenRuns<K>::count; r++) {
      if (r == StenRuns<K>::mid) {
         if (T.off[at] != -1 || T.off[at + 1] != 1) { return false; }
         at += 2;
      } else {
         for (int i = 1; i < StenRuns<K>::len[r]; i++) {
            if (T.off[at + i] != T.off[at] + i) { return false; }
         }
         at += StenRuns<K>::len[r];
      }
   }
   return true;
}

// two neighbouring values, loaded as one word of twice the size at any
// address of a value
template <typename X>
struct Two
{
   X a, b;
};
typedef double st_dbl2 __attribute__((ext_vector_type(2), aligned(8)));
typedef float st_flt2 __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned st_uns2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ Two<double> load_two(const double *p)
{
   const st_dbl2 v = *reinterpret_cast<const st_dbl2 *>(p);
   return {v.x, v.y};
}
__device__ __forceinline__ Two<float> load_two(const float *p)
{
   const st_flt2 v = *reinterpret_cast<const st_flt2 *>(p);
   return {v.x, v.y};
}
__device__ __forceinline__ Two<double> load_two_once(const double *p)
{
   const st_dbl2 v = __builtin_nontemporal_load(reinterpret_cast<const st_dbl2 *>(p));
   return {v.x, v.y};
}
__device__ __forceinline__ Two<float> load_two_once(const float *p)
{
   const st_flt2 v = __builtin_nontemporal_load(reinterpret_cast<const st_flt2 *>(p));
   return {v.x, v.y};
}
__device__ __forceinline__ void store_two(double *p, double a, double b)
{
   *reinterpret_cast<st_dbl2 *>(p) = st_dbl2{a, b};
}
__device__ __forceinline__ void store_two(float *p, float a, float b)
{
   *reinterpret_cast<st_flt2 *>(p) = st_flt2{a, b};
}

// The values of step k of a lane's two rows
template <int MODE, typename V, typename X>
__device__ __forceinline__ Two<X> sten_value(int k, int lane, StenTab T, const st_uns2 *cw, const X *sd,
                                             const V *__restrict__ raw)
{
   if (MODE == ST_CONST) {
      const X v = (X) T->v[k];
      return {v, v};
   }
   if (MODE == ST_CODES) {
      const st_uns2 w = cw[k >> 2] >> ((k & 3) * 8);
      return {sd[w.x & 255u], sd[w.y & 255u]};
   }
   const Two<V> v = load_two_once(raw + k * ST_ROWS + 2 * lane);
   return {(X) v.a, (X) v.b};
}

template <bool MASK, typename X>
__device__ __forceinline__ void sten_add(int k, st_uns2 m, Two<X> v, X x0, X x1, Two<X> &t)
{
   const X p0 = v.a * x0, p1 = v.b * x1;
   const X s0 = t.a + p0, s1 = t.b + p1;
   t.a = !MASK || (m.x >> k & 1u) ? s0 : t.a;
   t.b = !MASK || (m.y >> k & 1u) ? s1 : t.b;
}

// A lane's two sums over a table of any size, four steps at a time; CLAMP: the
// columns are held inside [0, n).  codes: the slice's words.
template <int MODE, bool CLAMP, typename V, typename X>
__device__ __forceinline__ Two<X> sten_sum_any(long long f, int lane, int n, StenTab T, st_uns2 m,
                                               const X *__restrict__ x,
                                               const unsigned *__restrict__ codes, const X *sd,
                                               const V *__restrict__ raw)
{
   Two<X> t = {(X) 0, (X) 0};
   const int D = T->D;
   const long long r = f + 2 * lane;
#pragma unroll 1
   for (int k0 = 0; k0 < D; k0 += 4) {
      Two<X> xx[4], vv[4];
      st_uns2 w = {0u, 0u};
      if (MODE == ST_CODES) {
         w = *reinterpret_cast<const st_uns2 *>(codes + (k0 >> 2) * ST_ROWS + 2 * lane);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
         // steps past the table's end re-read its last one; their mask bits are clear
         const int k = min(k0 + u, D - 1);
         const long long j = r + T->off[k];
         if (CLAMP) {
            xx[u].a = x[j < 0 ? 0 : j >= n ? n - 1 : j];
            xx[u].b = x[j < -1 ? 0 : j >= n - 1 ? n - 1 : j + 1];
         } else {
            xx[u] = load_two(x + j);
         }
         vv[u] = sten_value<MODE, V, X>(MODE == ST_CODES ? u : k, lane, T, &w, sd, raw);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
         sten_add<true, X>(0, st_uns2{m.x >> (k0 + u), m.y >> (k0 + u)}, vv[u], xx[u].a, xx[u].b, t);
      }
   }
   return t;
}

// A lane sums rows f + 2 lane and the next one.  The loads' width is what
// counts here: the L1 takes four lanes' addresses a cycle, so with one row a
// lane and 8-byte loads the 27-point sum spent 541 of 622 cycles a slice of 64
// rows on addresses (128 us at 200^3; 73 us now); a run of three offsets needs
// four neighbouring x values for two rows, two 16-byte loads instead of six of
// 8.
template <int K, int MODE, bool MASK, typename V, typename X>
__device__ __forceinline__ Two<X> sten_sum(long long f, int lane, StenTab T, st_uns2 m,
                                           const X *__restrict__ x, const st_uns2 *cw, const X *sd,
                                           const V *__restrict__ raw)
{
   using R = StenRuns<K>;
   Two<X> t = {(X) 0, (X) 0};
   // Two loads of a run: (first, second) and (third, fourth) of its four x
   // values; a single offset needs the first load only.  The x loads run two
   // batches of B runs ahead of the sums and the values one: z is zero, but the
   // compiler takes it to depend on the sums so far.  Without it all loads of
   // the slice are moved to its front: 255 registers, two waves a SIMD.
   constexpr int B = 2, NB = (R::count + B - 1) / B;
   const Two<X> c0 = load_two(x + f - 1 + 2 * lane), c1 = load_two(x + f + 1 + 2 * lane);
   Two<X> lo[NB][B], hi[NB][B];
   int z = 0, kx = 1, k = 1;
   auto issue = [&](int b) {
#pragma unroll
      for (int g = 0; g < B; g++) {
         const int run = b * B + g;
         if (run >= R::count) { break; }
         if (run == R::mid) {
            lo[b][g] = c0;
            hi[b][g] = c1;
            kx += 2;
            continue;
         }
         const X *p = x + f + T->off[kx] + z;
         lo[b][g] = load_two(p + 2 * lane);
         if (R::len[run] == 3) { hi[b][g] = load_two(p + 2 + 2 * lane); }
         kx += R::len[run];
      }
   };
   issue(0);
   sten_add<MASK, X>(0, m, sten_value<MODE, V, X>(0, lane, T, cw, sd, raw), c0.b, c1.a, t);
#pragma unroll
   for (int b = 0; b < NB; b++) {
      if (b + 1 < NB) { issue(b + 1); }
      const X *sdz = MODE == ST_CODES ? sd + z : sd;
      const V *rz = MODE == ST_RAW ? raw + z : raw;
      Two<X> vv[3 * B];
      int kv = k;
#pragma unroll
      for (int g = 0; g < B; g++) {
         const int run = b * B + g;
         if (run >= R::count) { break; }
#pragma unroll
         for (int i = 0; i < R::len[run]; i++) {
            if (run == R::mid && i == 1) { continue; }
            vv[3 * g + i] = sten_value<MODE, V, X>(kv++, lane, T, cw, sdz, rz);
         }
      }
#pragma unroll
      for (int g = 0; g < B; g++) {
         const int run = b * B + g;
         if (run >= R::count) { break; }
         sten_add<MASK, X>(k++, m, vv[3 * g], lo[b][g].a, lo[b][g].b, t);
         if (R::len[run] == 3) {
            if (run != R::mid) { sten_add<MASK, X>(k++, m, vv[3 * g + 1], lo[b][g].b, hi[b][g].a, t); }
            sten_add<MASK, X>(k++, m, vv[3 * g + 2], hi[b][g].a, hi[b][g].b, t);
         }
      }
      if (b + 1 < NB) { asm volatile("" : "+s"(z) : "v"(t.a), "v"(t.b)); }
   }
   return t;
}

// what a slice's sum needs besides x, loaded while the slice before it is
// summed: the rows' masks and epilogue operands and, for a dictionary slice,
// its code words and the first 64 values
template <int CW, typename Ops>
struct StenAhead
{
   int     info;
   st_uns2 m, cw[CW];
   double  d;
   Ops     ops;
};

// the sums of slice sl; edge: some row + offset lies outside [0, n)
template <int K, typename V, typename X, typename A>
__device__ __forceinline__ Two<X> sten_slice(int sl, int lane, int n, bool edge, const A &h, StenTab T,
                                             const StenView &S, const X *__restrict__ x, X *sd,
                                             const V *__restrict__ raw)
{
   const int mode = h.info & 3;
   const long long f = (long long) sl * ST_ROWS;
   const V *rw = mode == ST_RAW ? raw + (size_t) (h.info >> 8) * ST_ROWS * T->D : nullptr;
   const unsigned *codes = S.codes + (size_t) sl * ((T->D + 3) / 4) * ST_ROWS;
   if (mode == ST_CODES) {
      const int nd = h.info >> 8;
      __builtin_amdgcn_wave_barrier();
      sd[lane] = (X) h.d;
      for (int i = 64 + lane; i < nd; i += 64) { sd[i] = (X) S.dict[(size_t) sl * ST_DICT + i]; }
      __builtin_amdgcn_wave_barrier();
   }
   if (edge) {
      return mode == ST_CONST ? sten_sum_any<ST_CONST, true, V, X>(f, lane, n, T, h.m, x, codes, sd, rw)
             : mode == ST_RAW ? sten_sum_any<ST_RAW, true, V, X>(f, lane, n, T, h.m, x, codes, sd, rw)
                              : sten_sum_any<ST_CODES, true, V, X>(f, lane, n, T, h.m, x, codes, sd, rw);
   }
   if constexpr (K == ST_MAX) {
      return mode == ST_CONST ? sten_sum_any<ST_CONST, false, V, X>(f, lane, n, T, h.m, x, codes, sd, rw)
             : mode == ST_RAW ? sten_sum_any<ST_RAW, false, V, X>(f, lane, n, T, h.m, x, codes, sd, rw)
                              : sten_sum_any<ST_CODES, false, V, X>(f, lane, n, T, h.m, x, codes, sd, rw);
   } else if (h.info & 4) {
      return mode == ST_CONST ? sten_sum<K, ST_CONST, false, V, X>(f, lane, T, h.m, x, h.cw, sd, rw)
             : mode == ST_RAW ? sten_sum<K, ST_RAW, false, V, X>(f, lane, T, h.m, x, h.cw, sd, rw)
                              : sten_sum<K, ST_CODES, false, V, X>(f, lane, T, h.m, x, h.cw, sd, rw);
   } else {
      return mode == ST_CONST ? sten_sum<K, ST_CONST, true, V, X>(f, lane, T, h.m, x, h.cw, sd, rw)
             : mode == ST_RAW ? sten_sum<K, ST_RAW, true, V, X>(f, lane, T, h.m, x, h.cw, sd, rw)
                              : sten_sum<K, ST_CODES, true, V, X>(f, lane, T, h.m, x, h.cw, sd, rw);
   }
}

// Slices of this wave, one after the other: pre(row, both) loads the operands
// of the epilogue of a lane's two rows ahead of the sum, epi(row, both, sums,
// operands) ends them; both: row + 1 is a row too.
template <int K, typename V, typename X, class Pre, class Epi>
__device__ __forceinline__ void sten_rows(int n, int ns, const StenView &S,
                                          const X *__restrict__ x, const V *__restrict__ raw, Pre pre,
                                          Epi epi)
{
   __shared__ X sdict[WPB * ST_DICT];
   // Block b of XCD x (blocks are dealt round-robin to the XCDs) takes every
   // nbx-th group of four slices of the XCD's contiguous share, one slice a
   // wave: with all blocks resident the slices in flight on an XCD are one
   // narrow band, whose x and neighbouring planes stay in its L2.
   const int nx = (gridDim.x & 7) ? 1 : 8, nbx = gridDim.x / nx;
   const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
   const int share = ((ns + nx - 1) / nx + WPB - 1) / WPB * WPB;
   const long long first = (long long) (blockIdx.x % nx) * share;
   const int S1 = (int) (first + share < ns ? first + share : ns);
   const int S0 = (int) (first + (blockIdx.x / nx) * WPB < S1 ? first + (blockIdx.x / nx) * WPB + wv : S1);
   const int stride = nbx * WPB;
   if (S0 >= S1) { return; }
   X *sd = sdict + wv * ST_DICT;
   StenTab T = reinterpret_cast<StenTab>(reinterpret_cast<uintptr_t>(S.tab));
   constexpr int CW = (K + 3) / 4;   // words of a row's codes (K exact)
   // the least and the largest offset are the table's second and last
   const long long lo = T->D > 1 ? (T->off[1] < 0 ? T->off[1] : 0) : 0;
   const long long hi = T->D > 1 ? (T->off[T->D - 1] > 0 ? T->off[T->D - 1] : 0) : 0;
   using Ops = decltype(pre(0, true));
   int infos = 0, at = 0;   // of this wave's next 64 slices, one a lane
   auto ahead = [&](int sl, StenAhead<CW, Ops> &h) {
      if ((at & 63) == 0) { infos = S.info[min((long long) sl + (long long) lane * stride, (long long) ns - 1)]; }
      h.info = __builtin_amdgcn_readlane(infos, at & 63);
      at++;
      h.m = *reinterpret_cast<const st_uns2 *>(S.mask + (size_t) sl * ST_ROWS + 2 * lane);
      const long long r = (long long) sl * ST_ROWS + 2 * lane;
      h.ops = pre((int) min(r, (long long) n - 1), r + 1 < n);
      if ((h.info & 3) == ST_CODES) {
#pragma unroll
         for (int w = 0; w < (K < ST_MAX ? CW : 0); w++) {
            h.cw[w] = __builtin_nontemporal_load(reinterpret_cast<const st_uns2 *>(
               S.codes + ((size_t) sl * CW + w) * ST_ROWS + 2 * lane));
         }
         h.d = S.dict[(size_t) sl * ST_DICT + min(lane, (h.info >> 8) - 1)];
      }
   };
   StenAhead<CW, Ops> cur, nxt;
   ahead(S0, cur);
   for (int sl = S0; sl < S1; sl += stride) {
      asm volatile("" : "+s"(T));
      nxt = cur;
      if (sl + stride < S1) { ahead(sl + stride, nxt); }
      const long long f = (long long) sl * ST_ROWS, r = f + 2 * lane;
      const bool edge = f + lo < 0 || f + ST_ROWS - 1 + hi >= n;
      const Two<X> t = sten_slice<K, V, X>(sl, lane, n, edge, cur, T, S, x, sd, raw);
      if (r < n) { epi((int) r, r + 1 < n, t, cur.ops); }
      cur = nxt;
   }
}

// an operand of a lane's two rows
template <typename X>
__device__ __forceinline__ Two<X> sten_pair(const X *__restrict__ p, int row, bool both)
{
   if (both) { return load_two(p + row); }
   return {p[row], (X) 0};
}

template <typename X>
__device__ __forceinline__ void sten_put(X *p, int row, bool both, X a, X b)
{
   if (both) { store_two(p + row, a, b); }
   else { p[row] = a; }
}

template <typename X>
struct StenOps
{
   Two<X> a, b, c;
};

template <int K, typename V, typename X, bool DOT>
__global__ __launch_bounds__(BS) void k_spmv_sten(int n, int ns, StenView S,
                                                  const V *__restrict__ raw,
                                                  const X *__restrict__ x, X alpha, X beta,
                                                  const X *b, X *y, double *__restrict__ part)
{
   double acc = 0.0;
   sten_rows<K, V, X>(
      n, ns, S, x, raw,
      [&](int row, bool both) {
         StenOps<X> o{};
         if (beta != (X) 0) { o.a = sten_pair(b, row, both); }
         if (DOT) { o.b = sten_pair(x, row, both); }
         return o;
      },
      [&](int row, bool both, Two<X> t, const StenOps<X> &o) {
         const X v0 = (beta == (X) 0) ? alpha * t.a : alpha * t.a + beta * o.a.a;
         const X v1 = (beta == (X) 0) ? alpha * t.b : alpha * t.b + beta * o.a.b;
         sten_put(y, row, both, v0, v1);
         if (DOT) {
            acc += (double) v0 * (double) o.b.a;
            if (both) { acc += (double) v1 * (double) o.b.b; }
         }
      });
   if (DOT) {
      __shared__ double sh[BS];
      sh[threadIdx.x] = acc;
      __syncthreads();
      for (int off = BS / 2; off > 0; off >>= 1) {
         if (threadIdx.x < off) { sh[threadIdx.x] += sh[threadIdx.x + off]; }
         __syncthreads();
      }
      if (threadIdx.x == 0) { part[blockIdx.x] = sh[0]; }
   }
}

template <int K, typename V, typename X>
__global__ __launch_bounds__(BS) void k_relax_l1_sten(int n, int ns, StenView S,
                                                      const V *__restrict__ raw,
                                                      const X *__restrict__ f,
                                                      const X *__restrict__ u,
                                                      const X *__restrict__ l1, X w,
                                                      X *__restrict__ uo)
{
   sten_rows<K, V, X>(
      n, ns, S, u, raw,
      [&](int row, bool both) {
         return StenOps<X>{sten_pair(f, row, both), sten_pair(u, row, both), sten_pair(l1, row, both)};
      },
      [&](int row, bool both, Two<X> t, const StenOps<X> &o) {
         const X v0 = w * o.a.a - w * t.a, v1 = w * o.a.b - w * t.b;
         sten_put(uo, row, both, o.b.a + v0 / o.c.a, o.b.b + v1 / o.c.b);
      });
}

// ---------------------------------------------------------------- step masks of the strength pass
// One wave a slice, two rows a lane; the values come from the copy, the C/F
// flags of the neighbours at scalar bases, so a row costs its copy's bytes and
// 16 written (27-point 200^3: 0.26 ms, where the lists of C neighbours from the
// CSR entries take 1.4 ms).
__global__ __launch_bounds__(BS) void k_sten_masks(int n, int ns, StenView S,
                                                   const double *__restrict__ raw,
                                                   const double *__restrict__ thr,
                                                   const int *__restrict__ flg,
                                                   const int *__restrict__ CF, uint4 *__restrict__ q)
{
   __shared__ double sdict[WPB * ST_DICT];
   const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
   double *sd = sdict + wv * ST_DICT;
   const StenTab T = reinterpret_cast<StenTab>(reinterpret_cast<uintptr_t>(S.tab));
   const int D = T->D, CW = (D + 3) / 4;
   const long long lo = D > 1 ? (T->off[1] < 0 ? T->off[1] : 0) : 0;
   const long long hi = D > 1 ? (T->off[D - 1] > 0 ? T->off[D - 1] : 0) : 0;
   for (int sl = blockIdx.x * WPB + wv; sl < ns; sl += gridDim.x * WPB) {
      const int info = __builtin_amdgcn_readfirstlane(S.info[sl]);
      const int mode = info & 3;
      const long long f = (long long) sl * ST_ROWS, r = f + 2 * lane;
      const bool edge = f + lo < 0 || f + ST_ROWS - 1 + hi >= n;
      const st_uns2 m = *reinterpret_cast<const st_uns2 *>(S.mask + r);
      const int r0 = (int) min(r, (long long) n - 1), r1 = (int) min(r + 1, (long long) n - 1);
      const double t0 = thr[r0], t1 = thr[r1];
      const int f0 = flg[r0], f1 = flg[r1];
      if (mode == ST_CODES) {
         __builtin_amdgcn_wave_barrier();
         for (int i = lane; i < (info >> 8); i += 64) { sd[i] = S.dict[(size_t) sl * ST_DICT + i]; }
         __builtin_amdgcn_wave_barrier();
      }
      const double *rw = mode == ST_RAW ? raw + (size_t) (info >> 8) * ST_ROWS * D : nullptr;
      uint4 a = {0u, 0u, 0u, 0u}, b = {0u, 0u, 0u, 0u};
#pragma unroll 1
      for (int k0 = 0; k0 < D; k0 += 4) {
         st_uns2 w = {0u, 0u};
         if (mode == ST_CODES) {
            w = *reinterpret_cast<const st_uns2 *>(S.codes + ((size_t) sl * CW + (k0 >> 2)) * ST_ROWS + 2 * lane);
         }
#pragma unroll
         for (int u = 0; u < 4; u++) {
            const int k = k0 + u;
            if (k == 0 || k >= D) { continue; }   // uniform
            const Two<double> v =
               mode == ST_CONST ? sten_value<ST_CONST, double, double>(k, lane, T, &w, sd, rw)
               : mode == ST_RAW ? sten_value<ST_RAW, double, double>(k, lane, T, &w, sd, rw)
                                : sten_value<ST_CODES, double, double>(u, lane, T, &w, sd, rw);
            const long long j = r + T->off[k];
            int c0, c1;
            if (edge) {
               c0 = CF[j < 0 ? 0 : j >= n ? n - 1 : j];
               c1 = CF[j < -1 ? 0 : j >= n - 1 ? n - 1 : j + 1];
            } else {
               c0 = CF[j];
               c1 = CF[j + 1];
            }
            const unsigned bit = 1u << k;
            auto put = [&](uint4 &z, unsigned mk, double val, double t, int fl, int c) {
               if (!(mk & bit)) { return; }
               const bool neg = fl & 1;
               if (!(fl & 2) && (neg ? !(val <= t) : !(val >= t))) { z.x |= bit; }
               if (c >= 0) { z.y |= bit; }
               if (c == -3) { z.z |= bit; }
               if (neg ? val > 0 : val < 0) { z.w |= bit; }
            };
            put(a, m.x, v.a, t0, f0, c0);
            put(b, m.y, v.b, t1, f1, c1);
         }
      }
      if (r < n) { q[r] = a; }
      if (r + 1 < n) { q[r + 1] = b; }
   }
}

void sten_masks(const Csr &A, const Sten &S, const double *thr, const int *flg, const int *CF, uint4 *q)
{
   const StenView v{S.head, S.mask, S.codes, S.info, S.dict};
   const int nb = (int) std::min<long long>(((long long) S.nslices + WPB - 1) / WPB, 2048);
   k_sten_masks<<<nb, BS, 0, stream()>>>(A.nrows, S.nslices, v, S.raw, thr, flg, CF, q);
   HX_LAUNCH_CHECK();
}

// tables with the runs of a usual grid stencil are unrolled exactly; others
// run 32 masked steps
template <class F>
static void dispatch_steps(const StenHead &T, F f)
{
   if (sten_has_runs<5>(T)) { f(std::integral_constant<int, 5>{}); }
   else if (sten_has_runs<7>(T)) { f(std::integral_constant<int, 7>{}); }
   else if (sten_has_runs<9>(T)) { f(std::integral_constant<int, 9>{}); }
   else if (sten_has_runs<19>(T)) { f(std::integral_constant<int, 19>{}); }
   else if (sten_has_runs<27>(T)) { f(std::integral_constant<int, 27>{}); }
   else { f(std::integral_constant<int, ST_MAX>{}); }
}

// as many blocks as the device holds at once of this kernel, fewer for small ns
template <auto k>
static int sten_grid(int ns)
{
   static const int resident = [&] {
      int per = 0, dev = 0, cus = 0;
      HX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, BS, 0));
      HX_HIP(hipGetDevice(&dev));
      HX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
      return std::max(8, std::min(per * cus, 8192) / 8 * 8);
   }();
   const int nb = (int) std::min<long long>(((long long) ns + WPB - 1) / WPB, resident);
   return nb >= 64 ? std::min((nb + 7) / 8 * 8, resident) : std::max(nb, 1);
}

template <typename V>
static const V *sten_raw_values(const Sten &S)
{
   if constexpr (sizeof(V) == 8) { return S.raw; } else { return S.raw32; }
}

template <typename V, typename X, bool DOT>
int sten_spmv(const Csr &A, X alpha, const X *x, X beta, const X *b, X *y, double *part)
{
   const Sten &S = *A.sten;
   const StenView v{S.head, S.mask, S.codes, S.info, S.dict};
   int nb = 0;
   dispatch_steps(S.tab, [&](auto k) {
      constexpr auto kernel = &k_spmv_sten<decltype(k)::value, V, X, DOT>;
      nb = sten_grid<kernel>(S.nslices);
      kernel<<<nb, BS, 0, stream()>>>(A.nrows, S.nslices, v, sten_raw_values<V>(S), x, alpha, beta, b,
                                      y, part);
   });
   HX_LAUNCH_CHECK();
   return nb;
}

template <typename V, typename X>
void sten_relax_l1(const Csr &A, const X *f, const X *u, const X *l1, X w, X *uo)
{
   const Sten &S = *A.sten;
   const StenView v{S.head, S.mask, S.codes, S.info, S.dict};
   dispatch_steps(S.tab, [&](auto k) {
      constexpr auto kernel = &k_relax_l1_sten<decltype(k)::value, V, X>;
      const int nb = sten_grid<kernel>(S.nslices);
      kernel<<<nb, BS, 0, stream()>>>(A.nrows, S.nslices, v, sten_raw_values<V>(S), f, u, l1, w, uo);
   });
   HX_LAUNCH_CHECK();
}

template int sten_spmv<double, double, false>(const Csr &, double, const double *, double, const double *,
                                              double *, double *);
template int sten_spmv<double, double, true>(const Csr &, double, const double *, double, const double *,
                                             double *, double *);
template int sten_spmv<float, float, false>(const Csr &, float, const float *, float, const float *, float *,
                                            double *);
template void sten_relax_l1<double, double>(const Csr &, const double *, const double *, const double *,
                                            double, double *);
template void sten_relax_l1<float, float>(const Csr &, const float *, const float *, const float *, float,
                                          float *);

} // namespace hx
