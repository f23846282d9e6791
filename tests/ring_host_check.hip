// CPU model of k_remap_lean's target ring for the CPU tests: one row of source blocks (its columns
// grouped into work units as k_columns does), 16 lanes in step, with the reconstructions and the
// deposit of the library's header.  The ring has the kernel's rows and its order of opening,
// depositing and storing blocks; beside it every deposit inside its column's target range is
// stored into a plain array.
#include <limits.h>

#include <algorithm>
#include <vector>

#include "../vlasiator_amd/csrc/vacc_lean.h"

constexpr int LANES = 16, RING = 16, W = 4;

// set_geom and column_extent of the column build (cpu_acc_map.cpp:258-338), in FP32
static void extent(int b0, int b1, int ks, int len, float I, float di, float dj, float dv, float vmin, float dk,
                   int maxlen, int& fk, int& lk) {
   float hi = 0, lo = 0;
   for (int q = 0; q < 4; ++q) {
      const float c = (I + (float)(b0 * W + ((q & 2) ? W - 1 : 0)) * di) + (float)(b1 * W + ((q & 1) ? W - 1 : 0)) * dj;
      hi = (q == 0 || hi < c) ? c : hi;
      lo = (q == 0 || c < lo) ? c : lo;
   }
   fk = (int)(((float)(W * ks) * dv + vmin - hi) / dk) / W;
   lk = (int)(((float)(W * (ks + len)) * dv + vmin - lo) / dk) / W;
   fk = std::min(std::max(fk, 0), maxlen - 1);
   lk = std::min(std::max(lk, 0), maxlen - 1);
}

struct Column {
   int ks, len, fk, lk;
};

// counts[0]: deposits outside their column's range that hit a row of an open block; [1]: blocks
// stored before they were finished because the ring was full; [4]: all stored because it was full; [2]: deposits outside the range; [3]: units of several
// columns; stored / plain: [maxlen * 4][16], blocks stored once each (seen)
template <int M>
static void unit(const Column* col, int ncol, int b0, int b1, double I, double di, double dj, double dk, double dv,
                 double vmin, const float* src, int n, float* stored, float* plain, int* seen, long long* counts) {
   using R = vacc::ReconLean<M>;
   const double rdk = 1.0 / dk;
   const float r = (float)(dk / dv), inv_r = (float)(dv * rdk);
   static thread_local float ring[RING][LANES];
   int carry_open = -1;
   for (int ci = 0; ci < ncol; ++ci) {
      const Column& C = col[ci];
      const int nfk = (ci + 1 < ncol) ? col[ci + 1].fk : INT_MAX;
      const int hi = W * C.lk + W - 1;
      int next_flush = C.fk, next_open = (carry_open >= 0) ? carry_open : C.fk;
      auto flush = [&](int b) {
         ++seen[b];
         for (int e = 0; e < W; ++e)
            for (int l = 0; l < LANES; ++l) stored[(W * b + e) * LANES + l] = ring[(W * b + e) & (RING - 1)][l];
      };
      auto emit = [&](int gt, float m, int l) {
         const int row = std::min(gt, hi + 1) & (RING - 1);
         if (gt >= W * C.fk && gt <= hi) {
            plain[gt * LANES + l] = m;
         } else {
            ++counts[2];
            for (int b = next_flush; b < next_open; ++b)
               if (((W * b) & (RING - 1)) == (row & ~(W - 1))) ++counts[0];
         }
         ring[row][l] = m;
      };
      R rc[LANES];
      vacc::Flux<R::NC> fx[LANES];
      std::vector<std::vector<float>> v(LANES, std::vector<float>(W * C.len + 8, 0.0f));
      for (int l = 0; l < LANES; ++l) {
         for (int k = 0; k < W * C.len; ++k) v[l][4 + k] = src[(size_t)l * n + W * C.ks + k];
         const double imin = I + (double)(b0 * W + (l & 3)) * di + (double)(b1 * W + (l >> 2)) * dj;
         fx[l].begin((vmin + (double)(W * C.ks) * dv - imin) * rdk, r);
         rc[l].start(v[l].data() + 4);
      }
      auto cell = [&](int l, int k) {
         float c[R::NC];
         rc[l].coeffs(v[l].data() + 4 + k, c);
         fx[l].cell(c, v[l][4 + k], [&](int gt, float m) { emit(gt, m, l); });
      };
      for (int b = 0; b < C.len; ++b) {
         int openLim = INT_MIN, flushLim = INT_MAX;
         for (int l = 0; l < LANES; ++l) {
            const int reach = fx[l].o + 1 + ((fx[l].t < 4.0f) ? (int)((4.0f - fx[l].t) * inv_r) + 1 : 0);
            openLim = std::max(openLim, std::min(reach, hi));
            flushLim = std::min(flushLim, fx[l].o);
         }
         while (next_open <= C.lk && W * next_open <= openLim) {
            if (next_open - next_flush >= RING / W) {
               if (W * next_flush + W - 1 >= flushLim) ++counts[1];
               ++counts[4];
               flush(next_flush++);
            }
            for (int e = 0; e < W; ++e)
               for (int l = 0; l < LANES; ++l) ring[(W * next_open + e) & (RING - 1)][l] = 0.0f;
            ++next_open;
         }
         for (int l = 0; l < LANES; ++l) cell(l, W * b);
         while (next_flush < next_open && next_flush < nfk && W * next_flush + W - 1 < flushLim) flush(next_flush++);
         for (int k = 1; k < W; ++k)
            for (int l = 0; l < LANES; ++l) cell(l, W * b + k);
      }
      for (int l = 0; l < LANES; ++l) fx[l].end([&](int gt, float m) { emit(gt, m, l); });
      while (next_flush < next_open && next_flush < nfk) flush(next_flush++);
      for (int tb = next_open; tb <= C.lk && tb < nfk; ++tb) ++seen[tb];   // zero_block
      carry_open = (next_open > nfk) ? next_open : -1;
   }
}

// One row: occ[maxlen] source blocks present, src[16][4 maxlen] values (zero where absent).
extern "C" int ring_row(int method, int maxlen, const unsigned char* occ, const float* src, int b0, int b1, double I,
                        double di, double dj, double dk, double dv, double vmin, float* stored, float* plain, int* seen,
                        long long* counts) {
   std::vector<Column> cols;
   for (int p = 0; p < maxlen;) {
      if (!occ[p]) {
         ++p;
         continue;
      }
      int e = p;
      while (e < maxlen && occ[e]) ++e;
      Column C{p, e - p, 0, 0};
      extent(b0, b1, p, e - p, (float)I, (float)di, (float)dj, (float)dv, (float)vmin, (float)dk, maxlen, C.fk, C.lk);
      cols.push_back(C);
      p = e;
   }
   bool overlap = false;
   for (size_t i = 1; i < cols.size(); ++i) overlap |= cols[i].fk <= cols[i - 1].lk;
   auto run = [&](const Column* c, int n) {
      if (method == VACC_PLM) unit<VACC_PLM>(c, n, b0, b1, I, di, dj, dk, dv, vmin, src, W * maxlen, stored, plain, seen, counts);
      else if (method == VACC_PPM) unit<VACC_PPM>(c, n, b0, b1, I, di, dj, dk, dv, vmin, src, W * maxlen, stored, plain, seen, counts);
      else unit<VACC_PQM>(c, n, b0, b1, I, di, dj, dk, dv, vmin, src, W * maxlen, stored, plain, seen, counts);
   };
   if (overlap) {
      ++counts[3];
      run(cols.data(), (int)cols.size());
   } else {
      for (const Column& c : cols) run(&c, 1);
   }
   return (int)cols.size();
}
