// Launches of qmv_batch_kernel (vpq_qmv_batch.h): the split of a launch, the choice of an instantiation, and the
// instantiations for 4-bit group-64 packs.
#include <type_traits>

#include "vpq_qmv_batch.h"

namespace vpq {

namespace {

size_t batch_lds_bytes(const BatchPlan& v, int K, const BatchFormat& f)
{
  // (64 more: the unaligned reads of the last row's scales may run past its block)
  return (size_t)kBatchWaves * batch_ring(v.mr, f.bits, v.depth) * batch_slot_bytes(v.tiles, v.mr, f.bits, v.depth) +
         2 * (size_t)batch_scale_bytes(v.tiles, K, f.group) + 64;
}

bool batch_fits(const BatchPlan& v, int K, const BatchFormat& f) { return batch_lds_bytes(v, K, f) <= (size_t)kLdsOfCu; }

}  // namespace

namespace {

int batch_mr(int rows) { return rows <= 4 ? 1 : rows <= 8 ? 2 : rows <= 16 ? 4 : rows <= 32 ? 8 : rows <= 48 ? 12 : 16; }

long batch_blocks(const QmvGroup& g, int tiles)
{
  long n = 0;
  for (int i = 0; i < g.count; ++i) { n += (g.seg[i].N + 16 * tiles - 1) / (16 * tiles); }
  return n;
}

// What a launch of 9 rows and more takes, in microseconds.  A CU gets n workgroups (not a whole number), c = ceil(n) of them one
// after the other, in pairs where two fit it (an odd one alone):
//   start + (c or c % 2) (one + one_k k) + c / 2 (two + two_k k) + n k (x_k rows + codes_k),
// k = K / 4096, half way between K and the whole chunks of its longest wavefront.  Fitted to every plan's time on 4900 drawn
// shapes (512..36000 x 2048..17408, packs from HBM; 4 bits, 4 bits in groups of 32, 8 bits), first to the times (met to 5..9
// %), then to the time of what is chosen: on average 0.2..0.6 % above the fastest plan's.  Over the rule for few rows at
// 9..16 / 17..32 / 33..48 / 49..64 rows: 4 bits 1.08 / 1.16 / 1.25 / 1.13 times as fast, groups of 32 1.09 / 1.19 / 1.34 /
// 1.17, 8 bits 1.05 / 1.13 / 1.22 / 1.12.  Binary16 and Q4_0 take the figures of 4 bits in groups of 64 and of 32, 8 bits in
// groups of 32 those of 8 bits: on 30 drawn shapes at 9..16 rows 1.12, 1.12 and 1.06 times as fast as the kernel before with the
// rule for few rows, the slowest 1.00, 0.97 and 0.98.
struct BatchCost {
  int tiles, mr, depth;
  bool pairs;
  double start, one, one_k, two, two_k, x_k, codes_k;
};
constexpr BatchCost kBatchCost4[] = {
    {1, 1, 1, true, 2.968, 0.496, 1.468, 1.716, 2.500, 0.000, 0.276},
    {1, 2, 1, true, 2.778, 0.677, 1.937, 2.006, 2.600, 0.035, 0.055},
    {1, 4, 1, true, 3.485, 0.062, 2.521, 0.744, 4.114, 0.026, 0.094},
    {1, 4, 2, false, 1.874, 1.866, 2.261, 0.000, 0.000, 0.022, 0.031},
    {1, 8, 1, true, 4.076, 0.487, 3.547, 1.053, 5.211, 0.033, 0.000},
    {2, 1, 1, false, 2.777, 11.438, 0.000, 0.000, 0.000, 0.000, 0.530},
    {2, 1, 1, true, 4.076, 0.144, 2.789, 0.943, 4.319, 0.000, 0.401},
    {2, 2, 1, false, 1.809, 3.396, 2.427, 0.000, 0.000, 0.011, 0.360},
    {2, 2, 1, true, 2.908, 0.555, 2.898, 1.419, 3.580, 0.051, 0.270},
    {2, 4, 1, false, 3.857, 4.195, 2.786, 0.000, 0.000, 0.012, 0.351},
    {2, 4, 1, true, 3.407, 0.391, 3.515, 1.611, 4.388, 0.025, 0.478},
    {2, 4, 2, false, 1.806, 2.212, 3.279, 0.000, 0.000, 0.031, 0.000},
    {2, 8, 1, false, 3.697, 3.573, 4.255, 0.000, 0.000, 0.024, 0.633},
    {2, 8, 1, true, 3.830, 0.326, 4.980, 1.807, 6.773, 0.038, 0.218},
    {2, 12, 1, false, 1.909, 2.380, 6.522, 0.000, 0.000, 0.007, 1.222},
    {2, 16, 1, false, 1.733, 2.750, 7.936, 0.000, 0.000, 0.010, 0.898},
    {3, 8, 1, false, 1.824, 2.436, 6.723, 0.000, 0.000, 0.026, 0.506},
    {3, 12, 1, false, 2.245, 3.388, 8.365, 0.000, 0.000, 0.000, 1.733},
};
constexpr BatchCost kBatchCost32[] = {     // 4 bits, groups of 32
    {1, 1, 1, true, 2.742, 0.214, 1.334, 0.868, 3.899, 0.059, 0.095},
    {1, 2, 1, false, 2.038, 10.170, 0.000, 0.000, 0.000, 0.006, 0.108},
    {1, 2, 1, true, 2.408, 0.429, 2.243, 1.379, 2.874, 0.027, 0.050},
    {1, 4, 1, false, 3.356, 12.535, 0.000, 0.000, 0.000, 0.014, 0.206},
    {1, 4, 1, true, 3.750, 0.464, 2.910, 1.773, 3.930, 0.022, 0.062},
    {1, 4, 2, false, 1.905, 1.968, 2.551, 0.000, 0.000, 0.024, 0.000},
    {1, 8, 1, false, 4.060, 19.161, 0.000, 0.000, 0.000, 0.015, 0.587},
    {1, 8, 1, true, 3.300, 0.280, 4.572, 0.789, 6.335, 0.027, 0.000},
    {2, 1, 1, false, 3.453, 2.382, 1.796, 0.000, 0.000, 0.328, 0.843},
    {2, 1, 1, true, 3.452, 0.056, 2.179, 1.374, 2.567, 0.079, 1.178},
    {2, 2, 1, false, 1.977, 2.063, 3.397, 0.000, 0.000, 0.032, 0.223},
    {2, 2, 1, true, 2.988, 0.680, 3.425, 1.662, 4.143, 0.025, 0.685},
    {2, 4, 1, false, 2.110, 2.232, 4.268, 0.000, 0.000, 0.020, 0.300},
    {2, 4, 1, true, 3.854, 0.359, 4.549, 1.874, 4.679, 0.010, 0.909},
    {2, 4, 2, false, 1.780, 2.251, 4.159, 0.000, 0.000, 0.036, 0.000},
    {2, 8, 1, false, 1.503, 2.346, 6.123, 0.000, 0.000, 0.016, 0.639},
    {2, 8, 1, true, 2.490, 2.275, 5.912, 5.418, 10.461, 0.025, 0.809},
    {2, 12, 1, false, 1.848, 3.002, 8.177, 0.000, 0.000, 0.000, 1.669},
    {2, 16, 1, false, 1.427, 2.545, 10.160, 0.000, 0.000, 0.000, 1.722},
    {3, 8, 1, false, 2.062, 2.392, 8.932, 0.000, 0.000, 0.044, 0.157},
    {3, 12, 1, false, 1.398, 3.767, 11.363, 0.000, 0.000, 0.014, 1.913},
};
constexpr BatchCost kBatchCost8[] = {
    {1, 1, 1, true, 3.268, 0.000, 1.680, 0.078, 3.799, 0.000, 0.208},
    {1, 1, 3, false, 3.205, 0.000, 2.532, 0.000, 0.000, 0.000, 0.415},
    {1, 2, 1, true, 3.354, 0.053, 2.451, 0.296, 3.926, 0.033, 0.046},
    {1, 2, 2, false, 3.509, 0.252, 2.486, 0.000, 0.000, 0.016, 0.000},
    {1, 4, 1, true, 3.329, 0.000, 2.804, 0.101, 5.022, 0.050, 0.072},
    {1, 4, 2, false, 1.995, 1.752, 3.334, 0.000, 0.000, 0.000, 0.319},
    {1, 8, 1, true, 3.543, 0.000, 4.018, 0.000, 5.961, 0.064, 0.000},
    {1, 8, 2, false, 1.900, 1.662, 4.016, 0.000, 0.000, 0.040, 0.000},
    {2, 1, 1, true, 3.409, 0.000, 3.479, 0.062, 6.385, 0.000, 0.729},
    {2, 2, 1, false, 2.717, 7.165, 1.774, 0.000, 0.000, 0.029, 0.798},
    {2, 2, 1, true, 2.920, 0.136, 3.593, 0.770, 6.569, 0.037, 0.463},
    {2, 4, 1, false, 2.122, 1.969, 3.639, 0.000, 0.000, 0.045, 0.498},
    {2, 4, 1, true, 3.129, 0.547, 3.986, 1.006, 7.051, 0.058, 0.312},
    {2, 8, 1, false, 4.236, 1.856, 5.142, 0.000, 0.000, 0.073, 0.275},
    {2, 8, 1, true, 3.795, 0.109, 5.953, 1.031, 8.400, 0.086, 0.050},
    {2, 8, 2, false, 2.114, 2.076, 5.528, 0.000, 0.000, 0.055, 0.000},
    {2, 12, 1, false, 2.169, 2.001, 7.476, 0.000, 0.000, 0.060, 0.350},
    {2, 16, 1, false, 1.559, 2.497, 8.892, 0.000, 0.000, 0.047, 0.267},
    {3, 8, 1, false, 2.214, 2.323, 7.695, 0.000, 0.000, 0.084, 0.000},
    {3, 12, 1, false, 1.876, 2.661, 9.910, 0.000, 0.000, 0.075, 0.476},
};

double batch_us(const BatchCost& c, const BatchPlan& v, const QmvGroup& g, int K, int M, const BatchFormat& f, int cus)
{
  const int rows = (M + v.m_tiles - 1) / v.m_tiles, chunk = 1024 / f.bits;
  const long blocks = batch_blocks(g, v.tiles), wgs = v.m_tiles > 1 ? (blocks + 7) / 8 * 8 * v.m_tiles : blocks;
  const double n = (double)wgs / cus;
  const long whole = (wgs + cus - 1) / cus;
  const int per_wave = ((K + chunk - 1) / chunk + kBatchWaves - 1) / kBatchWaves;
  const double k = (0.5 * K + 0.5 * per_wave * kBatchWaves * chunk) / 4096.0;
  const long ones = c.pairs ? whole % 2 : whole, twos = c.pairs ? whole / 2 : 0;
  return c.start + ones * (c.one + c.one_k * k) + twos * (c.two + c.two_k * k) + n * k * (c.x_k * rows + c.codes_k);
}

bool batch_pairs(const BatchPlan& v, int K, const BatchFormat& f)
{
  return batch_two_per_cu(v.tiles, v.mr, f.group, v.depth) && batch_lds_bytes(v, K, f) <= (size_t)kLdsOfCu / 2;
}

// Up to 32 rows of x a workgroup and up to 8 rows of x altogether: two tiles of 16 weight rows share the fetch of x and
// sum(x); one where the tiles alone do not fill the CUs (us, one / two: 4096 -> 4096 at 2 rows 5.0 / 5.9; 12288 -> 4096 9.6 /
// 11.7; 5120 -> 17408 19.8 / 17.7; 4096 -> 24576 16.9 / 14.6).  8 bits, one workgroup per CU, a long K: several chunks in
// flight (12288 -> 4096 at 4 / 6 rows 16.4 / 15.8 -> 13.1 / 14.4; 4 rows: 2560 -> 2560 5.1 -> 5.25, 3072 -> 3072 level, 4096 ->
// 1024 / 4096 6.0 / 7.3 -> 5.7 / 6.8, 5120 -> 4096 8.4 -> 7.7; 7 rows: 3072 -> 3072 and 4096 -> 1024 level, 3840 -> 3840 6.7 ->
// 6.6, 4096 -> 4096 7.5 -> 7.3, 5120 -> 1280 7.1 -> 6.9; 12 rows: 4096 -> 4096 8.05 -> 8.5; 4 bits: 11.2 -> 11.8 at 12288, 4 rows).
BatchPlan batch_plan_few(const QmvGroup& g, int K, int M, const BatchFormat& f, int cus)
{
  const int m_tiles = (M + 31) / 32, mr = batch_mr((M + m_tiles - 1) / m_tiles);
  const bool narrow = batch_blocks(g, 1) * m_tiles <= cus;
  const BatchPlan deep{1, mr, m_tiles, mr == 1 ? 3 : 2};
  if (f.bits == 8 && narrow && K >= (mr == 1 ? 3072 : mr == 2 ? 3840 : 7680) && batch_fits(deep, K, f)) { return deep; }
  return BatchPlan{narrow || !batch_fits(BatchPlan{2, mr, m_tiles, 1}, K, f) ? 1 : 2, mr, m_tiles, 1};
}

// From 9 rows on, the plan that takes least by the figures above: what counts is how many workgroups a CU gets, and that x
// comes in once per workgroup (us, by the rule for few rows / now: 4096 -> 1024 at 48 rows, 16 rows a workgroup, 7.8 / 6.0;
// 12288 -> 4096 at 24, 16 rows in pieces twice as long, 18.3 / 15.6; 17408 -> 5120 at 48 rows 51 / 34 with three tiles and
// two workgroups along M; 4096 -> 24576 at 48 rows 37 / 30 with three tiles and all rows; 12288 -> 4096 at 16 rows 13.1 /
// 12.1 with long pieces). Within 2 % the rule for few rows stays.
BatchPlan batch_plan(const QmvGroup& g, int K, int M, const BatchFormat& f, int cus)
{
  const BatchPlan few = batch_plan_few(g, K, M, f, cus);
  if (M <= 8 || M > 64) { return few; }                     // (above 64: packs that no GEMM takes)
  BatchPlan best = few;
  double best_us = 1e30, few_us = 1e30;
  auto consider = [&](const BatchCost& c) {
    for (int m_tiles = 1; m_tiles <= 4; ++m_tiles) {
      const BatchPlan v{c.tiles, c.mr, m_tiles, c.depth};
      const int rows = (M + m_tiles - 1) / m_tiles;
      if (batch_mr(rows) != c.mr || (M + rows - 1) / rows != m_tiles) { continue; }
      if (!batch_fits(v, K, f) || batch_pairs(v, K, f) != c.pairs) { continue; }
      const double us = batch_us(c, v, g, K, M, f, cus);
      if (us < best_us) { best_us = us; best = v; }
      if (v.tiles == few.tiles && v.mr == few.mr && m_tiles == few.m_tiles && v.depth == few.depth) { few_us = us; }
    }
  };
  if (f.bits == 8) {
    for (const BatchCost& c : kBatchCost8) { consider(c); }
  } else if (f.group == 32) {
    for (const BatchCost& c : kBatchCost32) { consider(c); }
  } else {
    for (const BatchCost& c : kBatchCost4) { consider(c); }
  }
  return best_us < 0.98 * few_us ? best : few;
}

}  // namespace

bool qmv_batch_supports(int K, int M, const BatchFormat& f)
{
  return M >= 1 && K >= f.group && K % f.group == 0 && batch_fits(BatchPlan{1, 8, 1, 1}, K, f);
}

hipError_t launch_qmv_batch(hipStream_t st, const QmvArgs& a, const QmvGroup& g, const BatchFormat& f)
{
  BatchParams p{};
  p.w = g.seg[0].w; p.scales = g.seg[0].scales; p.biases = g.seg[0].biases; p.x = a.x; p.y = g.seg[0].y;
  p.K = a.K; p.N = g.seg[0].N; p.M = a.M;
  p.residual = a.residual;
  p.gate_act = a.gate_act;
  p.y_f32 = a.y_f32 ? 1 : 0;
  p.nseg = g.count;
  // (the forms for more rows store elements without a residual)
  if (a.M > 16 && (a.residual != nullptr || a.y_f32)) { return hipErrorInvalidValue; }
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  const BatchPlan plan = batch_plan(g, a.K, a.M, f, cus);
  p.rows = (a.M + plan.m_tiles - 1) / plan.m_tiles;
  p.m_tiles = (a.M + p.rows - 1) / p.rows;
  const int tiles = plan.tiles;
  const size_t lds_bytes = batch_lds_bytes(plan, a.K, f);
  int first = 0;
  for (int i = 0; i < g.count; ++i) {
    if (i > 0) {
      p.seg[i - 1] = g.seg[i];
      p.seg_first[i - 1] = first;
    }
    first += (g.seg[i].N + 16 * tiles - 1) / (16 * tiles);
  }
  p.blocks = first;
  const int grid = p.m_tiles > 1 ? (first + 7) / 8 * 8 * p.m_tiles : first;
  if (f.bits == 4 && f.group == 64 && !f.f16) { return batch_launch<4, 64, false>(st, p, plan, lds_bytes, grid); }
  return launch_qmv_batch_twin(st, p, plan, lds_bytes, grid, f);
}

}  // namespace vpq
