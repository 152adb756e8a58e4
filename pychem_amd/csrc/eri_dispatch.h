// generated by gen_eri.py -- do not edit
#pragma once
#include "jk_common.h"
#define ERI_NCLASS 21
void eri_run_0000_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_0000_d();
void jk_run_0000_d(const JkArgs<double>&, hipStream_t);
void scatter_run_0000_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_0000_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_0000_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_0000_f();
void jk_run_0000_f(const JkArgs<float>&, hipStream_t);
void scatter_run_0000_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_0000_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_0000_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_0000_mix();
void eri_run_0000_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_0000_s();
void eri_run_1000_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1000_d();
void jk_run_1000_d(const JkArgs<double>&, hipStream_t);
void scatter_run_1000_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_1000_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_1000_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1000_f();
void jk_run_1000_f(const JkArgs<float>&, hipStream_t);
void scatter_run_1000_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_1000_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_1000_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1000_mix();
void eri_run_1000_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1000_s();
void eri_run_1010_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1010_d();
void jk_run_1010_d(const JkArgs<double>&, hipStream_t);
void scatter_run_1010_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_1010_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_1010_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1010_f();
void jk_run_1010_f(const JkArgs<float>&, hipStream_t);
void scatter_run_1010_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_1010_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_1010_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1010_mix();
void eri_run_1010_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1010_s();
void eri_run_1100_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1100_d();
void jk_run_1100_d(const JkArgs<double>&, hipStream_t);
void scatter_run_1100_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_1100_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_1100_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1100_f();
void jk_run_1100_f(const JkArgs<float>&, hipStream_t);
void scatter_run_1100_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_1100_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_1100_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1100_mix();
void eri_run_1100_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1100_s();
void eri_run_1110_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1110_d();
void jk_run_1110_d(const JkArgs<double>&, hipStream_t);
void scatter_run_1110_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_1110_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_1110_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1110_f();
void jk_run_1110_f(const JkArgs<float>&, hipStream_t);
void scatter_run_1110_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_1110_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_1110_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1110_mix();
void eri_run_1110_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1110_s();
void eri_run_1111_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1111_d();
void jk_run_1111_d(const JkArgs<double>&, hipStream_t);
void scatter_run_1111_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_1111_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_1111_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1111_f();
void jk_run_1111_f(const JkArgs<float>&, hipStream_t);
void scatter_run_1111_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_1111_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_1111_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_1111_mix();
void eri_run_1111_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_1111_s();
void eri_run_2000_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2000_d();
void jk_run_2000_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2000_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2000_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2000_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2000_f();
void jk_run_2000_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2000_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2000_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2000_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2000_mix();
void eri_run_2000_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2000_s();
void eri_run_2010_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2010_d();
void jk_run_2010_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2010_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2010_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2010_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2010_f();
void jk_run_2010_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2010_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2010_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2010_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2010_mix();
void eri_run_2010_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2010_s();
void eri_run_2011_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2011_d();
void jk_run_2011_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2011_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2011_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2011_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2011_f();
void jk_run_2011_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2011_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2011_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2011_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2011_mix();
void eri_run_2011_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2011_s();
void eri_run_2020_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2020_d();
void jk_run_2020_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2020_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2020_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2020_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2020_f();
void jk_run_2020_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2020_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2020_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2020_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2020_mix();
void eri_run_2020_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2020_s();
void eri_run_2100_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2100_d();
void jk_run_2100_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2100_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2100_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2100_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2100_f();
void jk_run_2100_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2100_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2100_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2100_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2100_mix();
void eri_run_2100_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2100_s();
void eri_run_2110_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2110_d();
void jk_run_2110_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2110_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2110_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2110_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2110_f();
void jk_run_2110_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2110_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2110_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2110_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2110_mix();
void eri_run_2110_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2110_s();
void eri_run_2111_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2111_d();
void jk_run_2111_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2111_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2111_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2111_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2111_f();
void jk_run_2111_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2111_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2111_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2111_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2111_mix();
void eri_run_2111_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2111_s();
void eri_run_2120_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2120_d();
void jk_run_2120_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2120_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2120_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2120_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2120_f();
void jk_run_2120_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2120_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2120_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2120_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2120_mix();
void eri_run_2120_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2120_s();
void eri_run_2121_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2121_d();
void jk_run_2121_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2121_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2121_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2121_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2121_f();
void jk_run_2121_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2121_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2121_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2121_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2121_mix();
void eri_run_2121_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2121_s();
void eri_run_2200_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2200_d();
void jk_run_2200_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2200_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2200_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2200_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2200_f();
void jk_run_2200_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2200_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2200_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2200_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2200_mix();
void eri_run_2200_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2200_s();
void eri_run_2210_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2210_d();
void jk_run_2210_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2210_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2210_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2210_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2210_f();
void jk_run_2210_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2210_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2210_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2210_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2210_mix();
void eri_run_2210_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2210_s();
void eri_run_2211_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2211_d();
void jk_run_2211_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2211_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2211_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2211_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2211_f();
void jk_run_2211_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2211_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2211_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2211_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2211_mix();
void eri_run_2211_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2211_s();
void eri_run_2220_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2220_d();
void jk_run_2220_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2220_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2220_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2220_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2220_f();
void jk_run_2220_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2220_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2220_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2220_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2220_mix();
void eri_run_2220_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2220_s();
void eri_run_2221_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2221_d();
void jk_run_2221_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2221_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2221_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2221_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2221_f();
void jk_run_2221_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2221_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2221_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2221_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2221_mix();
void eri_run_2221_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2221_s();
void eri_run_2222_d(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2222_d();
void jk_run_2222_d(const JkArgs<double>&, hipStream_t);
void scatter_run_2222_d(const ScatterArgs<double>&, hipStream_t);
void pairscatter_run_2222_d(const PairScatterArgs<double>&, hipStream_t);
void eri_run_2222_f(const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2222_f();
void jk_run_2222_f(const JkArgs<float>&, hipStream_t);
void scatter_run_2222_f(const ScatterArgs<float>&, hipStream_t);
void pairscatter_run_2222_f(const PairScatterArgs<float>&, hipStream_t);
void eri_run_2222_mix(const EriArgs<double>&, const EriArgs<float>&, hipStream_t);
size_t eri_scratch_2222_mix();
void eri_run_2222_s(const EriArgs<double>&, hipStream_t);
size_t eri_scratch_2222_s();
void onee_fused_run(const OneeFusedArgs& a, hipStream_t st);
// la, lb, lc, ld, components, bra pair class, ket pair class
static const int eri_class_table[ERI_NCLASS][7] = {
  {0, 0, 0, 0, 1, 0, 0},
  {1, 0, 0, 0, 3, 1, 0},
  {1, 0, 1, 0, 9, 1, 1},
  {1, 1, 0, 0, 9, 2, 0},
  {1, 1, 1, 0, 27, 2, 1},
  {1, 1, 1, 1, 81, 2, 2},
  {2, 0, 0, 0, 6, 3, 0},
  {2, 0, 1, 0, 18, 3, 1},
  {2, 0, 1, 1, 54, 3, 2},
  {2, 0, 2, 0, 36, 3, 3},
  {2, 1, 0, 0, 18, 4, 0},
  {2, 1, 1, 0, 54, 4, 1},
  {2, 1, 1, 1, 162, 4, 2},
  {2, 1, 2, 0, 108, 4, 3},
  {2, 1, 2, 1, 324, 4, 4},
  {2, 2, 0, 0, 36, 5, 0},
  {2, 2, 1, 0, 108, 5, 1},
  {2, 2, 1, 1, 324, 5, 2},
  {2, 2, 2, 0, 216, 5, 3},
  {2, 2, 2, 1, 648, 5, 4},
  {2, 2, 2, 2, 1296, 5, 5},
};
// VRR and contraction lines per primitive quartet (of one output group)
static const int eri_body_lines[ERI_NCLASS] = {
  2, 8, 27, 24, 79, 227, 21, 70, 200, 152, 51, 170, 252, 366, 305, 101, 340, 353, 172, 411, 955
};
// the electron-scattering operator's class kernels (FP64)
static void (*const eri_table_s[ERI_NCLASS])(const EriArgs<double>&, hipStream_t) = {
  eri_run_0000_s, eri_run_1000_s, eri_run_1010_s, eri_run_1100_s, eri_run_1110_s, eri_run_1111_s, eri_run_2000_s, eri_run_2010_s, eri_run_2011_s, eri_run_2020_s, eri_run_2100_s, eri_run_2110_s, eri_run_2111_s, eri_run_2120_s, eri_run_2121_s, eri_run_2200_s, eri_run_2210_s, eri_run_2211_s, eri_run_2220_s, eri_run_2221_s, eri_run_2222_s
};
// per-lane scratch (spill) bytes of each class kernel, FP64, FP32, mixed and scattering forms
static size_t (*const eri_scratch_table_d[ERI_NCLASS])() = {
  eri_scratch_0000_d, eri_scratch_1000_d, eri_scratch_1010_d, eri_scratch_1100_d, eri_scratch_1110_d, eri_scratch_1111_d, eri_scratch_2000_d, eri_scratch_2010_d, eri_scratch_2011_d, eri_scratch_2020_d, eri_scratch_2100_d, eri_scratch_2110_d, eri_scratch_2111_d, eri_scratch_2120_d, eri_scratch_2121_d, eri_scratch_2200_d, eri_scratch_2210_d, eri_scratch_2211_d, eri_scratch_2220_d, eri_scratch_2221_d, eri_scratch_2222_d
};
static size_t (*const eri_scratch_table_f[ERI_NCLASS])() = {
  eri_scratch_0000_f, eri_scratch_1000_f, eri_scratch_1010_f, eri_scratch_1100_f, eri_scratch_1110_f, eri_scratch_1111_f, eri_scratch_2000_f, eri_scratch_2010_f, eri_scratch_2011_f, eri_scratch_2020_f, eri_scratch_2100_f, eri_scratch_2110_f, eri_scratch_2111_f, eri_scratch_2120_f, eri_scratch_2121_f, eri_scratch_2200_f, eri_scratch_2210_f, eri_scratch_2211_f, eri_scratch_2220_f, eri_scratch_2221_f, eri_scratch_2222_f
};
static size_t (*const eri_scratch_table_mix[ERI_NCLASS])() = {
  eri_scratch_0000_mix, eri_scratch_1000_mix, eri_scratch_1010_mix, eri_scratch_1100_mix, eri_scratch_1110_mix, eri_scratch_1111_mix, eri_scratch_2000_mix, eri_scratch_2010_mix, eri_scratch_2011_mix, eri_scratch_2020_mix, eri_scratch_2100_mix, eri_scratch_2110_mix, eri_scratch_2111_mix, eri_scratch_2120_mix, eri_scratch_2121_mix, eri_scratch_2200_mix, eri_scratch_2210_mix, eri_scratch_2211_mix, eri_scratch_2220_mix, eri_scratch_2221_mix, eri_scratch_2222_mix
};
static size_t (*const eri_scratch_table_s[ERI_NCLASS])() = {
  eri_scratch_0000_s, eri_scratch_1000_s, eri_scratch_1010_s, eri_scratch_1100_s, eri_scratch_1110_s, eri_scratch_1111_s, eri_scratch_2000_s, eri_scratch_2010_s, eri_scratch_2011_s, eri_scratch_2020_s, eri_scratch_2100_s, eri_scratch_2110_s, eri_scratch_2111_s, eri_scratch_2120_s, eri_scratch_2121_s, eri_scratch_2200_s, eri_scratch_2210_s, eri_scratch_2211_s, eri_scratch_2220_s, eri_scratch_2221_s, eri_scratch_2222_s
};
// tiled J/K: bra tile TA x TB, tiles per quartet, LDS doubles per basis function
static const int jk_tile_table[ERI_NCLASS][4] = {
  {1, 1, 1, 6},
  {3, 1, 1, 10},
  {3, 1, 1, 10},
  {3, 3, 1, 14},
  {3, 3, 1, 14},
  {3, 3, 1, 14},
  {6, 1, 1, 14},
  {6, 1, 1, 14},
  {6, 1, 1, 14},
  {6, 1, 1, 14},
  {6, 3, 1, 18},
  {6, 3, 1, 18},
  {3, 3, 2, 14},
  {6, 3, 1, 18},
  {3, 3, 2, 14},
  {3, 6, 2, 18},
  {3, 6, 2, 18},
  {3, 3, 4, 14},
  {3, 6, 2, 18},
  {3, 3, 4, 14},
  {2, 2, 9, 10},
};
// J/K launch groups
#define JK_NGROUP 4
static const int jk_group_table[ERI_NCLASS] = {
  0, 0, 0, 2, 2, 2, 1, 1, 2, 1, 3, 3, 2, 3, 2, 3, 3, 2, 3, 2, 2
};
void jk_group_run_0(const JkGroupArgs&, int, int, size_t, hipStream_t);
void jk_group_run_1(const JkGroupArgs&, int, int, size_t, hipStream_t);
void jk_group_run_2(const JkGroupArgs&, int, int, size_t, hipStream_t);
void jk_group_run_3(const JkGroupArgs&, int, int, size_t, hipStream_t);
static void (*const jk_group_run[JK_NGROUP])(const JkGroupArgs&, int, int, size_t, hipStream_t) = {
  jk_group_run_0, jk_group_run_1, jk_group_run_2, jk_group_run_3
};
// both lists of a class in one launch
static void (*const eri_table_mix[ERI_NCLASS])(const EriArgs<double>&, const EriArgs<float>&, hipStream_t) = {
  eri_run_0000_mix, eri_run_1000_mix, eri_run_1010_mix, eri_run_1100_mix, eri_run_1110_mix, eri_run_1111_mix, eri_run_2000_mix, eri_run_2010_mix, eri_run_2011_mix, eri_run_2020_mix, eri_run_2100_mix, eri_run_2110_mix, eri_run_2111_mix, eri_run_2120_mix, eri_run_2121_mix, eri_run_2200_mix, eri_run_2210_mix, eri_run_2211_mix, eri_run_2220_mix, eri_run_2221_mix, eri_run_2222_mix
};
static void (*const eri_table_d[ERI_NCLASS])(const EriArgs<double>&, hipStream_t) = {
  eri_run_0000_d, eri_run_1000_d, eri_run_1010_d, eri_run_1100_d, eri_run_1110_d, eri_run_1111_d, eri_run_2000_d, eri_run_2010_d, eri_run_2011_d, eri_run_2020_d, eri_run_2100_d, eri_run_2110_d, eri_run_2111_d, eri_run_2120_d, eri_run_2121_d, eri_run_2200_d, eri_run_2210_d, eri_run_2211_d, eri_run_2220_d, eri_run_2221_d, eri_run_2222_d
};
static void (*const eri_table_f[ERI_NCLASS])(const EriArgs<float>&, hipStream_t) = {
  eri_run_0000_f, eri_run_1000_f, eri_run_1010_f, eri_run_1100_f, eri_run_1110_f, eri_run_1111_f, eri_run_2000_f, eri_run_2010_f, eri_run_2011_f, eri_run_2020_f, eri_run_2100_f, eri_run_2110_f, eri_run_2111_f, eri_run_2120_f, eri_run_2121_f, eri_run_2200_f, eri_run_2210_f, eri_run_2211_f, eri_run_2220_f, eri_run_2221_f, eri_run_2222_f
};
template <typename real> static inline void eri_launch(int cls, const EriArgs<real>& a, hipStream_t st)
{ if (sizeof(real) == 8) eri_table_d[cls]((const EriArgs<double>&)a, st); else eri_table_f[cls]((const EriArgs<float>&)a, st); }
static void (*const jk_table_d[ERI_NCLASS])(const JkArgs<double>&, hipStream_t) = {
  jk_run_0000_d, jk_run_1000_d, jk_run_1010_d, jk_run_1100_d, jk_run_1110_d, jk_run_1111_d, jk_run_2000_d, jk_run_2010_d, jk_run_2011_d, jk_run_2020_d, jk_run_2100_d, jk_run_2110_d, jk_run_2111_d, jk_run_2120_d, jk_run_2121_d, jk_run_2200_d, jk_run_2210_d, jk_run_2211_d, jk_run_2220_d, jk_run_2221_d, jk_run_2222_d
};
static void (*const jk_table_f[ERI_NCLASS])(const JkArgs<float>&, hipStream_t) = {
  jk_run_0000_f, jk_run_1000_f, jk_run_1010_f, jk_run_1100_f, jk_run_1110_f, jk_run_1111_f, jk_run_2000_f, jk_run_2010_f, jk_run_2011_f, jk_run_2020_f, jk_run_2100_f, jk_run_2110_f, jk_run_2111_f, jk_run_2120_f, jk_run_2121_f, jk_run_2200_f, jk_run_2210_f, jk_run_2211_f, jk_run_2220_f, jk_run_2221_f, jk_run_2222_f
};
template <typename real> static inline void jk_launch(int cls, const JkArgs<real>& a, hipStream_t st)
{ if (sizeof(real) == 8) jk_table_d[cls]((const JkArgs<double>&)a, st); else jk_table_f[cls]((const JkArgs<float>&)a, st); }
static void (*const scatter_table_d[ERI_NCLASS])(const ScatterArgs<double>&, hipStream_t) = {
  scatter_run_0000_d, scatter_run_1000_d, scatter_run_1010_d, scatter_run_1100_d, scatter_run_1110_d, scatter_run_1111_d, scatter_run_2000_d, scatter_run_2010_d, scatter_run_2011_d, scatter_run_2020_d, scatter_run_2100_d, scatter_run_2110_d, scatter_run_2111_d, scatter_run_2120_d, scatter_run_2121_d, scatter_run_2200_d, scatter_run_2210_d, scatter_run_2211_d, scatter_run_2220_d, scatter_run_2221_d, scatter_run_2222_d
};
static void (*const scatter_table_f[ERI_NCLASS])(const ScatterArgs<float>&, hipStream_t) = {
  scatter_run_0000_f, scatter_run_1000_f, scatter_run_1010_f, scatter_run_1100_f, scatter_run_1110_f, scatter_run_1111_f, scatter_run_2000_f, scatter_run_2010_f, scatter_run_2011_f, scatter_run_2020_f, scatter_run_2100_f, scatter_run_2110_f, scatter_run_2111_f, scatter_run_2120_f, scatter_run_2121_f, scatter_run_2200_f, scatter_run_2210_f, scatter_run_2211_f, scatter_run_2220_f, scatter_run_2221_f, scatter_run_2222_f
};
template <typename real> static inline void scatter_launch(int cls, const ScatterArgs<real>& a, hipStream_t st)
{ if (sizeof(real) == 8) scatter_table_d[cls]((const ScatterArgs<double>&)a, st); else scatter_table_f[cls]((const ScatterArgs<float>&)a, st); }
static void (*const pairscatter_table_d[ERI_NCLASS])(const PairScatterArgs<double>&, hipStream_t) = {
  pairscatter_run_0000_d, pairscatter_run_1000_d, pairscatter_run_1010_d, pairscatter_run_1100_d, pairscatter_run_1110_d, pairscatter_run_1111_d, pairscatter_run_2000_d, pairscatter_run_2010_d, pairscatter_run_2011_d, pairscatter_run_2020_d, pairscatter_run_2100_d, pairscatter_run_2110_d, pairscatter_run_2111_d, pairscatter_run_2120_d, pairscatter_run_2121_d, pairscatter_run_2200_d, pairscatter_run_2210_d, pairscatter_run_2211_d, pairscatter_run_2220_d, pairscatter_run_2221_d, pairscatter_run_2222_d
};
static void (*const pairscatter_table_f[ERI_NCLASS])(const PairScatterArgs<float>&, hipStream_t) = {
  pairscatter_run_0000_f, pairscatter_run_1000_f, pairscatter_run_1010_f, pairscatter_run_1100_f, pairscatter_run_1110_f, pairscatter_run_1111_f, pairscatter_run_2000_f, pairscatter_run_2010_f, pairscatter_run_2011_f, pairscatter_run_2020_f, pairscatter_run_2100_f, pairscatter_run_2110_f, pairscatter_run_2111_f, pairscatter_run_2120_f, pairscatter_run_2121_f, pairscatter_run_2200_f, pairscatter_run_2210_f, pairscatter_run_2211_f, pairscatter_run_2220_f, pairscatter_run_2221_f, pairscatter_run_2222_f
};
template <typename real> static inline void pairscatter_launch(int cls, const PairScatterArgs<real>& a, hipStream_t st)
{ if (sizeof(real) == 8) pairscatter_table_d[cls]((const PairScatterArgs<double>&)a, st); else pairscatter_table_f[cls]((const PairScatterArgs<float>&)a, st); }
