// Assembly of an IJ matrix on the device: SetValues / AddToValues calls in call
// order to CSR rows with the diagonal first.
//
// A chunk is one call's arrays (or many small calls' operations, staged on the
// host), uploaded as they are: segments (row, length) of columns and values.
// The segments are grouped by row, each row's in call order, their operations
// laid out row by row, and one wave a row folds repeated columns in call order
// and finds the diagonal.  Each row's entries, their order and the order of the
// additions are those of the serial assembly on the host.  What bounds it is
// the upload: of 0.91 ms for 1.76M operations (110,000 rows), 0.66 are the call
// that brings their 23 MB, 0.25 the kernels and their read-backs; the serial
// assembly took 18.3 ms, and 147 ms for 10.8M operations (5.3 now).
#include "hx_internal.h"

#include <algorithm>
#include <climits>

namespace hx {

constexpr int BS = 256;
constexpr int WPB = BS / 64;

static int ij_grid(long long n, int per) { return (int) std::max<long long>(1, std::min<long long>((n + per - 1) / per, 8192)); }

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
// laid out at the row's place.
__global__ __launch_bounds__(BS) void k_ij_layout(int nrows, const IjChunks *__restrict__ Cp, const int *__restrict__ seg_ia,
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
      if (ns == 0) { continue; }
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
__global__ __launch_bounds__(BS) void k_ij_fold(int nrows, int ncols, int jlo, int diag_shift,
                                                const int *__restrict__ op_ia, int *ocol, double *oval,
                                                const char *__restrict__ oop, int *__restrict__ cnt,
                                                int *__restrict__ dpos, int *__restrict__ bad)
{
   const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
   for (int r = blockIdx.x * WPB + wv; r < nrows; r += gridDim.x * WPB) {
      const int b = op_ia[r], m = op_ia[r + 1] - b;
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

// the rows into CSR, the diagonal (place dpos) first: the entries before it one
// on, or, with swap, only the first one to its place
__global__ __launch_bounds__(BS) void k_ij_write(int nrows, const int *__restrict__ op_ia,
                                                 const int *__restrict__ ocol,
                                                 const double *__restrict__ oval,
                                                 const int *__restrict__ dpos, bool swap,
                                                 const int *__restrict__ ia, int *__restrict__ ja,
                                                 double *__restrict__ a)
{
   const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
   for (int r = blockIdx.x * WPB + wv; r < nrows; r += gridDim.x * WPB) {
      const int b = op_ia[r], o = ia[r], m = ia[r + 1] - o, d = dpos[r];
      for (int q = lane; q < m; q += 64) {
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
   const int total_seg = (int) exclusive_scan(seg_ia, seg_ia, nrows);
   const int total_op = (int) exclusive_scan(op_ia, op_ia, nrows);
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
   int *bad = device_flags() + 76;
   dzero(bad, sizeof(int));
   const int nb = ij_grid(nrows, WPB);
   IjChunks *dC = dalloc_n<IjChunks>(1);
   held.push_back(dC);
   h2d(dC, &C, sizeof(C));
   k_ij_layout<<<nb, BS, 0, s>>>(nrows, dC, seg_ia, list, sorted, op_ia, ocol, oval, oop);
   HX_LAUNCH_CHECK();
   k_ij_fold<<<nb, BS, 0, s>>>(nrows, ncols, jlower, ilower - jlower, op_ia, ocol, oval, oop, cnt, dpos, bad);
   HX_LAUNCH_CHECK();
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
         k_ij_write<<<nb, BS, 0, s>>>(nrows, op_ia, ocol, oval, dpos, swap_diag, out.ia, out.ja, out.a);
         HX_LAUNCH_CHECK();
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
