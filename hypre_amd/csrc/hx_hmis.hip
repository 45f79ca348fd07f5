// HMIS coarsening (coarsen_type 10): src/parcsr_ls/par_coarsen.c:2842-2906.
//
// The reference runs the Ruge-Stueben first pass (hypre_BoomerAMGCoarsenRuge,
// par_coarsen.c:911, with coarsen_type 10) on the host even in its device
// builds, because the pass is sequential: each new C point is the undecided
// point of largest measure that entered that measure's list first, and every
// choice changes the measures of the points around it.  This file does the
// same: S is copied to the host, the pass runs there, and its split seeds the
// device PMIS rounds with CF_init 1 (the pass's C points are the first
// independent set).
//
// The pass keeps undecided points in FIFO buckets, one per measure value
// (the reference keeps a list of lists in decreasing measure,
// src/utilities/amg_linklist.c: a point joins the tail of its measure's list
// and the next C point is the head of the list of largest measure, which is
// the same order).
#include "hx_internal.h"

#include <sys/mman.h>

#include <algorithm>
#include <cstdlib>
#include <new>
#include <vector>

namespace hx {

namespace {

constexpr int kC = 1, kF = -1, kZ = -2, kSF = -3;

// a point's list links, measure and state in 16 bytes: the pass visits points in
// no order that a cache could follow, and each visit needs all four
struct Point
{
   int next, prev, measure, cf;
};

struct MeasureBuckets
{
   std::vector<int> head, tail;   // per measure value
   Point *pt;
   int top = 0;                   // no bucket above `top` holds a point

   explicit MeasureBuckets(Point *p) : head(64, -1), tail(64, -1), pt(p) {}

   void push(int m, int i)
   {
      if (m >= (int) head.size()) {
         head.resize(2 * m + 1, -1);
         tail.resize(2 * m + 1, -1);
      }
      const int t = tail[m];
      pt[i].next = -1;
      pt[i].prev = t;
      if (t >= 0) { pt[t].next = i; } else { head[m] = i; }
      tail[m] = i;
      top = std::max(top, m);
   }

   void erase(int m, int i)
   {
      const int nx = pt[i].next, pv = pt[i].prev;
      if (pv >= 0) { pt[pv].next = nx; } else { head[m] = nx; }
      if (nx >= 0) { pt[nx].prev = pv; } else { tail[m] = pv; }
   }

   // first point of the largest non-empty measure (-1 when all are empty)
   int front()
   {
      while (top > 0 && head[top] < 0) { top--; }
      return top > 0 ? head[top] : -1;
   }
};

// Memory that is not cleared first; arrays from RAW_HUGE on come in large pages
// where they can.  Clearing a large page takes longer than a small level's whole
// pass: 1000 points 0.43 ms with all arrays in large pages, 0.24 without.
constexpr size_t RAW_HUGE = 4000000;

template <class T>
struct Raw
{
   T *p;
   explicit Raw(size_t n)
   {
      const size_t page = size_t(2) << 20, want = std::max<size_t>(n, 1) * sizeof(T);
      if (want < RAW_HUGE) {
         p = static_cast<T *>(std::malloc(want));
      } else {
         const size_t bytes = (want + page - 1) / page * page;
         p = static_cast<T *>(std::aligned_alloc(page, bytes));
         if (p) { (void) madvise(p, bytes, MADV_HUGEPAGE); }
      }
      if (!p) { throw std::bad_alloc(); }
   }
   ~Raw() { std::free(p); }
   Raw(const Raw &) = delete;
   Raw &operator=(const Raw &) = delete;
   T &operator[](size_t i) { return p[i]; }
};

} // namespace

// par_coarsen.c:1060-1391 for one rank, measure_type 0, cut_factor 0.
// STi, STj: S^T, each row ascending.  The pass follows S and S^T from point to
// point and each step needs the one before, so it stays on one host thread; a
// point is one 16-byte record.  AHEAD: rows that come next are asked for early,
// which gains 2% at 6.6M entries and costs a tenth where the arrays fit the caches.
template <bool AHEAD>
static void rs_first_pass(int n, const int *Si, const int *Sj, const int *STi, const int *STj, int *CF)
{
   Raw<Point> pts((size_t) n);
   Point *pt = pts.p;
   int num_left = 0;
   for (int j = 0; j < n; j++) {
      if (Si[j + 1] == Si[j]) {
         pt[j] = Point{-1, -1, 0, kSF};
      } else {
         pt[j] = Point{-1, -1, STi[j + 1] - STi[j], 0};
         num_left++;
      }
   }
   MeasureBuckets B(pt);
   // points nobody depends on become Z; their neighbours' measures grow
   for (int j = 0; j < n; j++) {
      if (pt[j].cf == kSF) { continue; }
      if (pt[j].measure > 0) {
         B.push(pt[j].measure, j);
         continue;
      }
      pt[j].cf = kZ;
      for (int k = Si[j]; k < Si[j + 1]; k++) {
         const int nb = Sj[k];
         if (pt[nb].cf == kSF) { continue; }
         if (nb < j) {
            if (pt[nb].measure > 0) { B.erase(pt[nb].measure, nb); }
            B.push(++pt[nb].measure, nb);
         } else {
            ++pt[nb].measure;
         }
      }
      --num_left;
   }
   // a point that becomes F raises the measures of its undecided influences
   auto raise_influences = [&](int p) {
      const int e = Si[p + 1];
      for (int k = Si[p]; k < e; k++) {
         const int q = Sj[k];
         if (AHEAD && k + 8 < e) { __builtin_prefetch(pt + Sj[k + 8], 1); }
         if (pt[q].cf != 0) { continue; }
         B.erase(pt[q].measure, q);
         B.push(++pt[q].measure, q);
      }
   };
   while (num_left > 0) {
      const int c = B.front();
      if (c < 0) { fail(HYPRE_ERROR_GENERIC, "HMIS first pass: no undecided point left"); }
      pt[c].cf = kC;
      B.erase(pt[c].measure, c);
      pt[c].measure = 0;
      --num_left;
      const int e = STi[c + 1];
      for (int k = STi[c]; AHEAD && k < e; k++) { __builtin_prefetch(Sj + Si[STj[k]]); }
      for (int k = STi[c]; k < e; k++) {
         const int nb = STj[k];
         if (pt[nb].cf != 0) { continue; }
         pt[nb].cf = kF;
         B.erase(pt[nb].measure, nb);
         --num_left;
         raise_influences(nb);
      }
      for (int k = Si[c]; k < Si[c + 1]; k++) {
         const int nb = Sj[k];
         if (pt[nb].cf != 0) { continue; }
         B.erase(pt[nb].measure, nb);
         if (--pt[nb].measure > 0) {
            B.push(pt[nb].measure, nb);
         } else {
            pt[nb].cf = kF;
            --num_left;
            raise_influences(nb);
         }
      }
   }
   for (int j = 0; j < n; j++) { CF[j] = pt[j].cf; }
}

void rs_first_pass_host(int n, const int *Si, const int *Sj, int *CF)
{
   const int nnz = Si[n];
   // S^T (stable counting sort): the points that depend on each point
   std::vector<int> STi((size_t) n + 1, 0);
   Raw<int> STj((size_t) nnz);
   for (int k = 0; k < nnz; k++) { STi[(size_t) Sj[k] + 1]++; }
   for (int i = 0; i < n; i++) { STi[i + 1] += STi[i]; }
   {
      std::vector<int> pos(STi.begin(), STi.end() - 1);
      for (int i = 0; i < n; i++) {
         for (int k = Si[i]; k < Si[i + 1]; k++) { STj[(size_t) pos[Sj[k]]++] = i; }
      }
   }
   rs_first_pass<false>(n, Si, Sj, STi.data(), STj.p, CF);
}

int hmis(const Csr &S, const double *measure_in_dev, int *CF, double *measure_keep_dev,
         const int *st_count)
{
   const int n = S.nrows;
   if (n == 0) { return 0; }
   TimedLaunch tl("setup_hmis_first_pass", 0.0);
   // S^T of large levels comes from the device, whose launches and copies take
   // some 0.2 ms.  The split of one level, S^T on the host / on the device:
   // 27-point 40^3 (1.6M entries) 4.1 / 4.0 ms, 64^3 (6.6M) 21.6 / 18.9; 7-point
   // 48^3 (110,000 points, 0.65M) 3.0 / 3.7, 64^3 (262,000, 1.5M) 11.7 / 9.4;
   // 100,000 rows at random, 2.3M entries 12.8 / 14.5, 9.4M 47 / 43.
   // Where many rows depend on one point the device would sort that point's row
   // in one lane, which the host's counting sort does not mind.
   Csr ST;
   const bool on_device = (S.nnz >= 2500000 || n >= 200000) && transpose(S, ST, false, TRANSPOSE_SORT);
   Raw<int> ia((size_t) n + 1), ja((size_t) S.nnz), cf((size_t) n);
   try {
      d2h(ia.p, S.ia, sizeof(int) * ((size_t) n + 1));
      d2h(ja.p, S.ja, sizeof(int) * (size_t) S.nnz);
      if (on_device) {
         Raw<int> tia((size_t) n + 1), tja((size_t) S.nnz);
         d2h(tia.p, ST.ia, sizeof(int) * ((size_t) n + 1));
         d2h(tja.p, ST.ja, sizeof(int) * (size_t) S.nnz);
         ST.free_all();
         rs_first_pass<true>(n, ia.p, ja.p, tia.p, tja.p, cf.p);
      } else {
         rs_first_pass_host(n, ia.p, ja.p, cf.p);
      }
   } catch (...) {
      ST.free_all();
      throw;
   }
   h2d(CF, cf.p, sizeof(int) * (size_t) n);
   return pmis(S, measure_in_dev, CF, measure_keep_dev, st_count, 1);
}

} // namespace hx
