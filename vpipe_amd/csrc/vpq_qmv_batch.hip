// Launches of qmv_batch_kernel (vpq_qmv_batch.h): the split of a launch, the choice of an instantiation, and the
// instantiations for 4-bit group-64 packs.
#include <type_traits>

#include "vpq_qmv_batch.h"

namespace vpq {

namespace {

size_t batch_lds_bytes(int tiles, int mr, int K, const BatchFormat& f, bool deep)
{
  // (64 more: the unaligned reads of the last row's scales may run past its block)
  return (size_t)kBatchWaves * batch_ring(tiles, mr, f.bits, deep) * batch_slot_bytes(tiles, mr, f.bits, deep) +
         2 * (size_t)batch_scale_bytes(tiles, K, f.group) + 64;
}

}  // namespace

bool qmv_batch_supports(int K, int M, const BatchFormat& f)
{
  return M >= 1 && K >= f.group && K % f.group == 0 && batch_lds_bytes(1, 8, K, f, false) <= (size_t)kLdsOfCu;
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
  p.m_tiles = (a.M + 31) / 32;
  p.rows = (a.M + p.m_tiles - 1) / p.m_tiles;
  const int mr = p.rows <= 4 ? 1 : p.rows <= 8 ? 2 : p.rows <= 16 ? 4 : 8;
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  // Tiles of 16 weight rows per workgroup.  Two share the fetch of x and sum(x); one where the tiles
  // alone do not fill the CUs.  Measured (us, one / two): 4096 -> 4096 at 2 and 16 rows 5.0 / 5.9 and 6.0 / 6.8;
  // 12288 -> 4096 10.2 / 11.8 and 13.1 / 15.5; 5120 -> 17408 19.8 / 17.7 and 23.2 / 19.4; 17408 -> 5120 15.6 / 14.3
  // and 27.3 / 20.2; 4096 -> 24576 18.8 / 14.5 and 21.4 / 18.1.  (Four: 17.8 and 22.8 on the last, slower everywhere:
  // one workgroup per CU is left.)
  long tiles1 = 0;
  for (int i = 0; i < g.count; ++i) { tiles1 += (g.seg[i].N + 15) / 16; }
  const int tiles = tiles1 * p.m_tiles <= cus || batch_lds_bytes(2, mr, a.K, f, false) > (size_t)kLdsOfCu ? 1 : 2;
  // 8 bits, one workgroup per CU, a long K: more chunks in flight.  us without -> with, groups of 64: 12288 -> 4096 at
  // 4 / 6 / 16 / 32 rows 16.4 / 15.8 / 17.0 / 23.1 -> 13.1 / 14.4 / 16.9 / 22.0; 6144 -> 4096 at 4 / 32 rows 9.6 / 12.5 ->
  // 8.2 / 12.3, at 12 level (groups of 32: 9.9 -> 10.1; 6144 -> 2048 9.2 -> 9.5), so 9..16 rows from 7680 on, at 12 rows
  // 11.3 -> 10.8.  4096 -> 4096: 4 rows 7.4 -> 6.9, 12 rows 8.05 -> 8.5.  4 bits, six chunks at 12288: 11.2 -> 11.8 at 4 rows.
  const bool deep = f.bits == 8 && a.K >= (mr == 4 ? 7680 : 6144) && tiles == 1 && tiles1 * p.m_tiles <= cus &&
                    batch_lds_bytes(1, mr, a.K, f, true) <= (size_t)kLdsOfCu;
  const size_t lds_bytes = batch_lds_bytes(tiles, mr, a.K, f, deep);
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
  if (f.bits == 4 && f.group == 64 && !f.f16) { return batch_launch<4, 64, false>(st, p, tiles, mr, deep, lds_bytes, grid); }
  return launch_qmv_batch_twin(st, p, tiles, mr, deep, lds_bytes, grid, f);
}

}  // namespace vpq
