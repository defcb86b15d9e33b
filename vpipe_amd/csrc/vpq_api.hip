// The C ABI (include/vpq.h): argument validation, device check and kernel
// selection.  Nothing here allocates device memory or synchronises.
#include "../../include/vpq.h"

#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <mutex>

#include "vpq_internal.h"

namespace vpq {
ProfileState& profile_state()
{
  static ProfileState ps;
  return ps;
}
}  // namespace vpq

namespace {

struct DeviceState {
  std::atomic<int> status{1};  // 1 = not initialised, 0 = ok, <0 = vpq_status
  int cu_count = 0;
};

DeviceState g_dev;
std::mutex g_init_mutex;
thread_local char g_last_error[256] = "";

int device_error(hipError_t e)
{
  const char* s = hipGetErrorString(e);
  strncpy(g_last_error, s ? s : "unknown HIP error", sizeof(g_last_error) - 1);
  g_last_error[sizeof(g_last_error) - 1] = '\0';
  return VPQ_ERR_DEVICE;
}

int ensure_init()
{
  int st = g_dev.status.load(std::memory_order_acquire);
  if (st <= 0) { return st; }
  std::lock_guard<std::mutex> lock(g_init_mutex);
  st = g_dev.status.load(std::memory_order_acquire);
  if (st <= 0) { return st; }
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) { return device_error(e); }
  hipDeviceProp_t prop;
  e = hipGetDeviceProperties(&prop, dev);
  if (e != hipSuccess) { return device_error(e); }
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    strncpy(g_last_error, "device is not gfx950", sizeof(g_last_error) - 1);
    g_dev.status.store(VPQ_ERR_UNSUPPORTED, std::memory_order_release);
    return VPQ_ERR_UNSUPPORTED;
  }
  g_dev.cu_count = prop.multiProcessorCount;
  g_dev.status.store(VPQ_OK, std::memory_order_release);
  return VPQ_OK;
}

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

inline int finish(hipError_t e) { return e == hipSuccess ? VPQ_OK : device_error(e); }

int check_pack(const uint32_t* w, const uint16_t* scales, const uint16_t* biases, int K, int N)
{
  if (w == nullptr || scales == nullptr || biases == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (K <= 0 || N <= 0 || (K % 64) != 0) { return VPQ_ERR_BAD_SHAPE; }
  // Rows of codes are K/2 bytes, a multiple of 32: 16-byte alignment of the base
  // makes every 128-bit load of the kernels aligned.  Scales/biases are read
  // with 2-byte loads by the general kernels; the vector paths need 16.
  if (!aligned(w, 16) || !aligned(scales, 2) || !aligned(biases, 2)) { return VPQ_ERR_MISALIGNED; }
  return VPQ_OK;
}

// Rows from which the size-based entrance takes the dequant-once route when the workspace holds the
// expanded weight: the expansion costs ~20 us per 28 MB pack, the dense GEMM then runs ~1.1x faster than the
// fused kernel where the tiles are many (measured at M = 16320: 1.3 against 1.2 PFLOP/s; at M = 2048 the two
// are even on 4096->12288 and the fused kernel is ahead on the N = 4096 shapes).
constexpr int kDenseRouteMinRows = 8192;

// One row of 8-bit codes: below this K the general kernel, a launch a pack; from it on launch_row8, the same bits.  us: 2048 ->
// 512 3.0 / 3.3, 2560 -> 640 4.2 / 4.2, 2560 -> 2560 5.5 / 4.9, 4096 -> 4096 7.8 / 6.8, 12288 -> 4096 19.8 / 15.1; q|k|v of 4096
// in three launches 18.3, in one 9.1.
constexpr int kRow8MinK = 2560;

// Whether `rows` weight rows of 8-bit codes (of all pairs together) are worth the gathers' kernel.  In its fifth pass over K, from
// 4096 on, it holds x in so many registers that a CU has eight wavefronts, of four rows each; one wavefront per weight row, sixteen
// and more a CU, is ahead up to about twelve sets of four rows a CU (us, that / the gathers' kernel, pairs of K -> N: one of 5120
// -> 5120 8.7 / 9.5, 4 of 4160 -> 1536 8.3 / 9.2, 8 of it, twelve sets a CU, 13.0 / 13.6; 8 of 4608 -> 2048 17.7 / 16.9, 8 of 5120
// -> 3072 26.5 / 24.9, 48 of it 142 / 123).  Gated, where the other kernel reads two rows a wavefront, the gathers' kernel always is
// (one token of 4 experts, 4608 -> 1536: 11.6 / 9.5).
bool gather8_takes(int K, long rows, bool gated)
{
  return vpq::qmv_gather_supports(K, 8) && (K <= 4096 || gated || rows > 4 * 12L * g_dev.cu_count);
}

// One row of x against the 8-bit packs of g, each with the bits that it has as an expert's slab of a gather.  (Several packs: a
// wavefront of one row would pay for the choice among them; q|k|v of 5120 13.1 us, on the gathers' kernel 11.1.)
hipError_t launch_row8(hipStream_t hs, const vpq::QmvArgs& a, const vpq::QmvGroup& g)
{
  return gather8_takes(a.K, g.seg[0].N, g.count > 1) ? vpq::launch_qmv_gather_row8(hs, a, g) : vpq::launch_qmv_row8(hs, a, g);
}

// One row of binary16 whose scales are no whole 16-byte pieces: the one-row kernel from the K on from which its error against
// float64 is no larger than that of one wavefront per weight row, which ran these (fp32 output, 1e-7, K = 2112 / 3840 / 9664:
// 1.36 / 1.34 / 1.32 and 1.20 / 1.51 / 2.27; the batch kernel, which takes what is shorter: 0.83 / 0.91 / 1.07).  us, one
// wavefront per row / batch kernel / now: 3840 -> 3840 5.8 / 5.1 / 3.9, 3840 -> 19328 17.4 / 13.0 / 10.5, 9664 -> 3840 11.3 / 9.4 /
// 7.8.  What is shorter, one wavefront per row / batch kernel: 1280 -> 4096 3.8 / 3.7, 1280 -> 16384 8.6 / 6.2, 2496 -> 4096 5.7 /
// 5.1, 2496 -> 16384 14.4 / 9.3, but 1280 -> 1024 2.9 / 3.4 and 2496 -> 1024 3.5 / 4.2: the line may not depend on N, or a narrow
// k or v would have other bits in a launch with q, and the three together gain (2496 -> 2496 | 640 | 640 12.1 / 5.1).
bool flow_narrow_f16(int K, int N, int M) { return K >= 3072 && (K % 512) != 0 && vpq::qmv_flow_narrow_supports(K, N, M, 64); }

// The batch kernel over one pack.
hipError_t launch_batch(hipStream_t hs, const vpq::QmvArgs& a, const vpq::BatchFormat& f)
{
  vpq::QmvGroup g;
  g.count = 1;
  g.seg[0] = vpq::QmvSeg{a.w, a.scales, a.biases, a.y, a.N};
  return vpq::launch_qmv_batch(hs, a, g, f);
}

int qmv_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
               const uint16_t* biases, const uint16_t* x, void* y, bool y_f32, int K, int N, int M,
               const uint16_t* residual, void* ws, size_t ws_bytes, int variant, int gate_act = 0)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16) { return VPQ_ERR_BAD_SHAPE; }
  const bool gelu_mul = gate_act == vpq::kStoreGeluMul;       // `residual` is the multiplier [N]; bf16 store only
  if (gate_act != 0 && gate_act != VPQ_GATE_SWIGLU && gate_act != VPQ_GATE_GEGLU && !gelu_mul) { return VPQ_ERR_BAD_SHAPE; }
  if (gelu_mul && (residual == nullptr || y_f32 || variant != VPQ_QMV_AUTO)) { return residual == nullptr ? VPQ_ERR_NULL_POINTER : VPQ_ERR_BAD_SHAPE; }
  if (gate_act != 0 && !gelu_mul && ((N & 1) != 0 || residual != nullptr || variant == VPQ_QMV_STREAM)) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, y_f32 ? 4 : 2)) { return VPQ_ERR_MISALIGNED; }
  if (residual != nullptr && !aligned(residual, 2)) { return VPQ_ERR_MISALIGNED; }
  if (variant < VPQ_QMV_AUTO || variant > VPQ_QMV_RING_SPLITK || variant == 3) { return VPQ_ERR_BAD_SHAPE; }   // (3 is unassigned)
  st = ensure_init();
  if (st != VPQ_OK) { return st; }

  vpq::QmvArgs a;
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y; a.residual = residual;
  a.K = K; a.N = N; a.M = M; a.y_f32 = y_f32; a.ws = ws; a.ws_bytes = ws_bytes;
  a.cu_count = g_dev.cu_count;
  a.gate_act = gate_act;
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);

  const bool batch_ok = vpq::qmv_batch_supports(K, M, vpq::BatchFormat{}) && aligned(scales, 16) && aligned(biases, 16);
  // what the forced variants of the MFMA kernels take
  const bool mfma_ok = vpq::qmv_ring_supports(K, N, M) && aligned(scales, 16) && aligned(biases, 16);
  const bool flow_ok = vpq::qmv_flow_supports(K, N, M) && aligned(scales, 16) && aligned(biases, 16);
  if (gelu_mul) {        // the two kernels that have this store: the streaming one and the general one
    return finish(flow_ok ? vpq::launch_qmv_flow(hs, a) : vpq::launch_qmv_simple(hs, a));
  }
  if (variant == VPQ_QMV_SIMPLE) { return finish(vpq::launch_qmv_simple(hs, a)); }
  if (variant == VPQ_QMV_FLOW) {
    if (!flow_ok) { return VPQ_ERR_BAD_SHAPE; }
    return finish(vpq::launch_qmv_flow(hs, a));
  }
  if (variant == VPQ_QMV_ROWS) {
    if (!vpq::qmv_rows_supports(K, N, M) || (gate_act != 0 && (N & 1) != 0)) { return VPQ_ERR_BAD_SHAPE; }
    return finish(vpq::launch_qmv_rows(hs, a, 0));
  }
  if (variant == VPQ_QMV_RING) {
    if (!mfma_ok) { return VPQ_ERR_BAD_SHAPE; }
    return finish(vpq::launch_qmv_ring(hs, a, 1));
  }
  if (variant == VPQ_QMV_RING_SPLITK) {
    if (!mfma_ok || K < 1024) { return VPQ_ERR_BAD_SHAPE; }
    if (ws == nullptr || !aligned(ws, 16)) { return ws == nullptr ? VPQ_ERR_WORKSPACE : VPQ_ERR_MISALIGNED; }
    const int parts = K / 512 < 4 ? K / 512 : 4;
    if (ws_bytes < vpq::qmv_ring_workspace_bytes(K, N, M)) { return VPQ_ERR_WORKSPACE; }
    return finish(vpq::launch_qmv_ring(hs, a, parts));
  }
  if (variant == VPQ_QMV_STREAM) {
    if (!mfma_ok || gate_act != 0 || !vpq::qmv_stream_supports(K, N, M)) { return VPQ_ERR_BAD_SHAPE; }
    return finish(vpq::launch_qmv_stream(hs, a));
  }
  if (variant == VPQ_QMV_MFMA) {
    if (!mfma_ok) { return VPQ_ERR_BAD_SHAPE; }
    return finish(batch_ok ? launch_batch(hs, a, vpq::BatchFormat{}) : vpq::launch_qmv_ring(hs, a, 1));
  }
  // One row of x: the streaming kernel that requests the whole pack up front (measured, this / the batch kernel at one
  // row, us: 4096 -> 4096 3.9 / 5.1, 12288 -> 4096 8.0 / 9.5, 4096 -> 24576 12.5 / 14.3, 5120 -> 151936 75 / 89).
  if (flow_ok) { return finish(vpq::launch_qmv_flow(hs, a)); }
  // One row over another K: its form with narrow scales, and for a short K the row-streaming kernel.
  if ((K % 512) != 0 && vpq::qmv_flow_narrow_supports(K, N, M, 64)) { return finish(vpq::launch_qmv_flow_narrow(hs, a, vpq::BatchFormat{})); }
  if (M == 1 && (K % 512) != 0) { return finish(vpq::launch_qmv_rows(hs, a, 0)); }
  if (batch_ok) { return finish(launch_batch(hs, a, vpq::BatchFormat{})); }
  // A K too deep for the batch kernel's LDS (above 114176), or scales or biases off 16-byte alignment.
  if (mfma_ok) { return finish(vpq::launch_qmv_ring(hs, a, 1)); }
  if (vpq::qmv_rows_supports(K, N, M)) { return finish(vpq::launch_qmv_rows(hs, a, 0)); }
  return finish(vpq::launch_qmv_simple(hs, a));
}

}  // namespace

extern "C" {

int vpq_version(void) { return 100; }

const char* vpq_status_string(int status)
{
  switch (status) {
    case VPQ_OK: return "ok";
    case VPQ_ERR_NULL_POINTER: return "a required buffer is NULL";
    case VPQ_ERR_BAD_SHAPE: return "shape outside the supported domain";
    case VPQ_ERR_MISALIGNED: return "pointer not aligned as required";
    case VPQ_ERR_WORKSPACE: return "workspace missing or too small";
    case VPQ_ERR_DEVICE: return "HIP runtime error";
    case VPQ_ERR_UNSUPPORTED: return "device is not gfx950";
    default: return "unknown status";
  }
}

const char* vpq_last_device_error(void) { return g_last_error; }

int vpq_init(void)
{
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  // Also resolves the static scratch of vpq_argmax_bf16_static for the current device, so that the entry point
  // itself has no first-call work left.  Best effort: a failure here concerns that one entry point only, which
  // tries again on its first call and reports it there.
  float* unused = nullptr;
  (void)vpq::argmax_static_scratch(&unused);
  return VPQ_OK;
}

int vpq_device_cu_count(void) { return g_dev.status.load() == VPQ_OK ? g_dev.cu_count : 0; }

int vpq_dequant_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                           const uint16_t* biases, uint16_t* w_deq, int K, int N)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (w_deq == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_dequant(reinterpret_cast<hipStream_t>(stream), w, scales, biases, w_deq, K, N));
}

int vpq_dequant_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                           const uint16_t* biases, uint16_t* w_deq, int K, int N)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (w_deq == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_dequant8(reinterpret_cast<hipStream_t>(stream), w, scales, biases, w_deq, K, N));
}

static int qmv8_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                       const uint16_t* x, void* y, bool y_f32, int K, int N, int M, const uint16_t* residual,
                       int store = 0)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr || (store == vpq::kStoreGeluMul && residual == nullptr)) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, y_f32 ? 4 : 2) || (residual != nullptr && !aligned(residual, 2))) {
    return VPQ_ERR_MISALIGNED;
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y; a.residual = residual;
  a.K = K; a.N = N; a.M = M; a.y_f32 = y_f32; a.cu_count = g_dev.cu_count;
  a.gate_act = store;
  const vpq::BatchFormat f{8, 64, false, false};
  if (M >= 2 && store == 0 && vpq::qmv_batch_supports(K, M, f) && aligned(scales, 16) && aligned(biases, 16)) {
    return finish(launch_batch(reinterpret_cast<hipStream_t>(stream), a, f));
  }
  if (M == 1 && store == 0 && K >= kRow8MinK) {
    return finish(launch_row8(reinterpret_cast<hipStream_t>(stream), a, vpq::QmvGroup{1, {{w, scales, biases, y, N}}}));
  }
  return finish(vpq::launch_qmv_simple8(reinterpret_cast<hipStream_t>(stream), a));
}

int vpq_qmv_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                       const uint16_t* x, uint16_t* y, int K, int N, int M, const uint16_t* residual)
{
  return qmv8_common(stream, w, scales, biases, x, y, false, K, N, M, residual);
}

int vpq_qmv_w8g64_f32out(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                         const uint16_t* x, float* y, int K, int N, int M)
{
  return qmv8_common(stream, w, scales, biases, x, y, true, K, N, M, nullptr);
}

int vpq_qmv_gelu_mul_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                                const uint16_t* x, uint16_t* y, int K, int N, const uint16_t* mul)
{
  return qmv8_common(stream, w, scales, biases, x, y, false, K, N, 1, mul, vpq::kStoreGeluMul);
}

int vpq_moe_gate_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                            const uint16_t* x, uint16_t* gate, int K, int M)
{
  int st = check_pack(w, scales, biases, K, 1);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || gate == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 65535) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(gate, 2)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = gate;
  a.K = K; a.N = 1; a.M = 1; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  a.gate_act = vpq::kStoreSigmoid;
  return finish(vpq::launch_qmv_rows8(reinterpret_cast<hipStream_t>(stream), a, M, nullptr, 1, 1));
}

static int rows8_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                        const uint16_t* x, uint16_t* y, int K, int N, int rows, int gate_act, const int32_t* pair_eid,
                        bool gathered, int x_div, int n_experts)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr || (gathered && pair_eid == nullptr)) { return VPQ_ERR_NULL_POINTER; }
  if (gate_act != 0 && gate_act != VPQ_GATE_SWIGLU && gate_act != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (rows < 1 || rows > 65535 || (gate_act != 0 && (N & 1) != 0)) { return VPQ_ERR_BAD_SHAPE; }
  if (gathered ? (x_div < 1 || n_experts < 1) : rows > 16) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 2) || (gathered && !aligned(pair_eid, 4))) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y;
  a.K = K; a.N = N; a.M = 1; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  a.gate_act = gate_act;
  const vpq::BatchFormat f{8, 64, false, false};
  if (!gathered && rows >= 2 && vpq::qmv_batch_supports(K, rows, f) && aligned(scales, 16) && aligned(biases, 16)) {
    a.M = rows;
    return finish(launch_batch(reinterpret_cast<hipStream_t>(stream), a, f));
  }
  if (gather8_takes(K, (long)N * rows, gate_act != 0)) {
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    if (gathered) { return finish(vpq::launch_qmv_gather(hs, a, 8, pair_eid, rows, x_div, n_experts)); }
    if (rows == 1) { return finish(vpq::launch_qmv_gather_row8(hs, a, vpq::QmvGroup{1, {{w, scales, biases, y, N}}})); }
  }
  return finish(vpq::launch_qmv_rows8(reinterpret_cast<hipStream_t>(stream), a, rows, gathered ? pair_eid : nullptr, x_div,
                                      n_experts));
}

int vpq_gather_qmv_gated_split_bf16(vpq_stream_t stream, const uint32_t* wg, const uint16_t* sg, const uint16_t* bg,
                                    int gate_bits, const uint32_t* wu, const uint16_t* su, const uint16_t* bu, int up_bits,
                                    const uint16_t* x, uint16_t* y, int K, int ffn, const int32_t* pair_eid, int npair,
                                    int top_k, int n_experts, int activation)
{
  if (wg == nullptr || sg == nullptr || bg == nullptr || wu == nullptr || su == nullptr || bu == nullptr || x == nullptr ||
      y == nullptr) {
    return VPQ_ERR_NULL_POINTER;
  }
  if ((gate_bits != 4 && gate_bits != 8) || (up_bits != 4 && up_bits != 8)) { return VPQ_ERR_BAD_SHAPE; }
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (K <= 0 || (K % 64) != 0 || ffn < 1 || npair < 1 || npair > 65535) { return VPQ_ERR_BAD_SHAPE; }
  if (pair_eid != nullptr ? (top_k < 1 || n_experts < 1) : npair > 16) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(wg, 16) || !aligned(wu, 16) || !aligned(x, 16) || !aligned(sg, 2) || !aligned(bg, 2) || !aligned(su, 2) ||
      !aligned(bu, 2) || !aligned(y, 2) || (pair_eid != nullptr && !aligned(pair_eid, 4))) {
    return VPQ_ERR_MISALIGNED;
  }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::SplitGateUp a{};
  a.wg = wg; a.sg = sg; a.bg = bg; a.gate_bits = gate_bits;
  a.wu = wu; a.su = su; a.bu = bu; a.up_bits = up_bits;
  a.x = x; a.y = y; a.K = K; a.F = ffn; a.rows = npair; a.gate_act = activation;
  a.pair_eid = pair_eid; a.x_div = pair_eid != nullptr ? top_k : 1; a.n_experts = n_experts;
  return finish(vpq::launch_qmv_split_gate_up(reinterpret_cast<hipStream_t>(stream), a));
}

int vpq_qmv_gated_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                             const uint16_t* x, uint16_t* y, int K, int N, int M, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return rows8_common(stream, w, scales, biases, x, y, K, N, M, activation, nullptr, false, 1, 1);
}

int vpq_gather_qmv_gated_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                    const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                    const int32_t* pair_eid, int npair, int top_k, int n_experts, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return rows8_common(stream, w, scales, biases, x, y, K, N, npair, activation, pair_eid, true, top_k, n_experts);
}

int vpq_gather_down_qmv_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                   const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                   const int32_t* pair_eid, int npair, int n_experts)
{
  return rows8_common(stream, w, scales, biases, x, y, K, N, npair, 0, pair_eid, true, 1, n_experts);
}

int vpq_qmm_dense_route_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                   const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                   uint16_t* w_deq, int expand)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (w_deq == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || !aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (expand != 0) {
    st = finish(vpq::launch_dequant8(hs, w, scales, biases, w_deq, K, N));
    if (st != VPQ_OK) { return st; }
  }
  std::string why;
  const int rc = vpq::dense_gemm_bf16(hs, x, w_deq, y, M, N, K, g_dev.cu_count, &why);
  if (rc != 0) {
    strncpy(g_last_error, why.c_str(), sizeof(g_last_error) - 1);
    g_last_error[sizeof(g_last_error) - 1] = '\0';
    return VPQ_ERR_DEVICE;
  }
  return VPQ_OK;
}

// ---- 8-bit codes in groups of 32 (GGUF q8 repacked; the codec's int8 path): `affine_dequant_w8g32`
// (affine_dequant.metal:99-131), `affine_qmv_w8g32` (affine_qmv.metal:3053-3069), `affine_qmm_steel_w8g32`
// (affine_qmm_steel.metal:1674-1698) by the dequant-once route, which is how the reference's codec runs it.
namespace {

int check_pack_w8g32(const uint32_t* w, const uint16_t* scales, const uint16_t* biases, int K, int N)
{
  if (w == nullptr || scales == nullptr || biases == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (K <= 0 || N <= 0 || (K % 32) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(w, 16) || !aligned(scales, 2) || !aligned(biases, 2)) { return VPQ_ERR_MISALIGNED; }
  return VPQ_OK;
}

}  // namespace

int vpq_dequant_w8g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                           uint16_t* w_deq, int K, int N)
{
  int st = check_pack_w8g32(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (w_deq == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_dequant8(reinterpret_cast<hipStream_t>(stream), w, scales, biases, w_deq, K, N, 32));
}

int vpq_requant_w8_to_w4_g64_bf16(vpq_stream_t stream, const uint32_t* w8, const uint16_t* s8, const uint16_t* b8,
                                  uint32_t* w4, uint16_t* s4, uint16_t* b4, int K, int N)
{
  int st = check_pack(w8, s8, b8, K, N);
  if (st != VPQ_OK) { return st; }
  if (w4 == nullptr || s4 == nullptr || b4 == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(w4, 16) || !aligned(s4, 2) || !aligned(b4, 2)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_requant_w8_to_w4(reinterpret_cast<hipStream_t>(stream), w8, s8, b8, w4, s4, b4, K, N));
}

int vpq_qmv_w8g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                       const uint16_t* x, uint16_t* y, int K, int N, int M, const uint16_t* residual)
{
  int st = check_pack_w8g32(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16 || (K % 16) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 2) || (residual != nullptr && !aligned(residual, 2))) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y; a.residual = residual;
  a.K = K; a.N = N; a.M = M; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  const vpq::BatchFormat f{8, 32, false, false};
  if (M >= 2 && vpq::qmv_batch_supports(K, M, f) && aligned(scales, 16) && aligned(biases, 16)) {
    return finish(launch_batch(reinterpret_cast<hipStream_t>(stream), a, f));
  }
  return finish(vpq::launch_qmv_simple8(reinterpret_cast<hipStream_t>(stream), a, 32));
}

int vpq_qmm_dense_route_w8g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                   const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                   uint16_t* w_deq, int expand)
{
  int st = check_pack_w8g32(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (w_deq == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || !aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (expand != 0) {
    st = finish(vpq::launch_dequant8(hs, w, scales, biases, w_deq, K, N, 32));
    if (st != VPQ_OK) { return st; }
  }
  std::string why;
  const int rc = vpq::dense_gemm_bf16(hs, x, w_deq, y, M, N, K, g_dev.cu_count, &why);
  if (rc != 0) {
    strncpy(g_last_error, why.c_str(), sizeof(g_last_error) - 1);
    g_last_error[sizeof(g_last_error) - 1] = '\0';
    return VPQ_ERR_DEVICE;
  }
  return VPQ_OK;
}

int vpq_embed_gather_w4g64_bf16(vpq_stream_t stream, const int32_t* ids, const uint32_t* w, const uint16_t* scales,
                                const uint16_t* biases, uint16_t* out, int H, int T, int vocab)
{
  int st = check_pack(w, scales, biases, H, vocab);
  if (st != VPQ_OK) { return st; }
  if (ids == nullptr || out == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (T <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(ids, 4) || !aligned(out, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_embed_gather(reinterpret_cast<hipStream_t>(stream), ids, w, scales, biases, out, H, T, vocab));
}

int vpq_qmv_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                       const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                       const uint16_t* residual, void* ws, size_t ws_bytes, int variant)
{
  return qmv_common(stream, w, scales, biases, x, y, false, K, N, M, residual, ws, ws_bytes, variant);
}

int vpq_qmv_w4g64_f32out(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                         const uint16_t* biases, const uint16_t* x, float* y, int K, int N, int M,
                         void* ws, size_t ws_bytes, int variant)
{
  return qmv_common(stream, w, scales, biases, x, y, true, K, N, M, nullptr, ws, ws_bytes, variant);
}

size_t vpq_qmv_workspace_bytes(int K, int N, int M)
{
  if (K <= 0 || N <= 0 || M < 1 || M > 16) { return 0; }
  return (vpq::qmv_ring_workspace_bytes(K, N, M) + 255) / 256 * 256;
}

int vpq_lora_a_bf16(vpq_stream_t stream, const uint16_t* x, const uint16_t* lora_a, uint16_t* t,
                    int M, int K, int r, float alpha)
{
  if (x == nullptr || lora_a == nullptr || t == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M <= 0 || K <= 0 || (K % 64) != 0 || r < 8 || r > vpq::kLoraMaxRank || (r % 8) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(lora_a, 16) || !aligned(t, 16)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_lora_a(reinterpret_cast<hipStream_t>(stream), x, lora_a, t, M, K, r, alpha));
}

namespace {

// The fused GEMM by size, for every format: the three kernels give the same bits, so it is the one that a model of
// their measured times says is fastest (vpq_qmm_mid.hip).
int gemm_by_size(hipStream_t hs, const vpq::GemmArgs& g)
{
  const vpq::GemmChoice c = vpq::qmm_choose(g);
  if (c.kernel == vpq::GemmKernel::kBig) { return finish(vpq::launch_qmm_big(hs, g, c.width)); }
  return finish(c.kernel == vpq::GemmKernel::kMid ? vpq::launch_qmm_mid(hs, g) : vpq::launch_qmm_tile(hs, g));
}

// tile: 0 = by size, 128 = the 256 x 128 tile kernel, 192 / 256 = the large-tile kernel at that width,
// -128 = the large-tile kernel at width 128
int qmm_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
               const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
               const uint16_t* lora_a, const uint16_t* lora_b, int r, float alpha,
               uint16_t* lora_t_ws, int tile)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16)) { return VPQ_ERR_MISALIGNED; }
  const bool lora = lora_a != nullptr && alpha != 0.0f;
  if (lora) {
    if (lora_b == nullptr) { return VPQ_ERR_NULL_POINTER; }
    if (lora_t_ws == nullptr) { return VPQ_ERR_WORKSPACE; }
    if (r < 8 || r > vpq::kLoraMaxRank || (r % 8) != 0) { return VPQ_ERR_BAD_SHAPE; }
    if (!aligned(lora_a, 16) || !aligned(lora_b, 16) || !aligned(lora_t_ws, 16)) { return VPQ_ERR_MISALIGNED; }
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (lora) {
    st = vpq_lora_a_bf16(stream, x, lora_a, lora_t_ws, M, K, r, alpha);
    if (st != VPQ_OK) { return st; }
  }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = M;
  g.lora_t = lora ? lora_t_ws : nullptr;
  g.lora_b = lora ? lora_b : nullptr;
  g.r = lora ? r : 0;
  g.cu_count = g_dev.cu_count;
  if (tile == 192 || tile == 256 || tile == -128) {
    if (!vpq::qmm_big_supports(g)) { return VPQ_ERR_BAD_SHAPE; }
    return finish(vpq::launch_qmm_big(hs, g, tile < 0 ? -tile : tile));
  }
  if (tile == 0) { return gemm_by_size(hs, g); }
  return finish(vpq::launch_qmm_tile(hs, g));
}

}  // namespace

int vpq_qmm_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                       const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                       const uint16_t* lora_a, const uint16_t* lora_b, int r, float alpha,
                       uint16_t* lora_t_ws)
{
  return qmm_common(stream, w, scales, biases, x, y, K, N, M, lora_a, lora_b, r, alpha, lora_t_ws, 0);
}

int vpq_qmm_tiled_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                             const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                             const uint16_t* lora_a, const uint16_t* lora_b, int r, float alpha,
                             uint16_t* lora_t_ws, int tile_n)
{
  if (tile_n != 128 && tile_n != -128 && tile_n != 192 && tile_n != 256) { return VPQ_ERR_BAD_SHAPE; }
  return qmm_common(stream, w, scales, biases, x, y, K, N, M, lora_a, lora_b, r, alpha, lora_t_ws, tile_n);
}

size_t vpq_linear_workspace_bytes(int K, int N, int M)
{
  if (K <= 0 || N <= 0 || M <= 0 || (K % 64) != 0) { return 0; }
  if (M >= kDenseRouteMinRows) { return ((size_t)N * (size_t)K * 2 + 255) / 256 * 256; }
  return vpq_qmm_workspace_bytes(K, N, M);
}

size_t vpq_qmm_workspace_bytes(int K, int N, int M)
{
  if (K <= 0 || N <= 0 || M <= 0 || (K % 64) != 0) { return 0; }
  if (ensure_init() != VPQ_OK) { return 0; }
  return (vpq::qmm_splitk_workspace_bytes(K, N, M, g_dev.cu_count) + 255) / 256 * 256;
}

int vpq_qmm_plan(int K, int N, int M, int bits, int group, int f16, int gated, int splits)
{
  if (K <= 0 || N <= 0 || M <= 0 || (K % 64) != 0 || splits < 0 || splits > 16 || (gated != 0 && (splits > 1 || (N & 1) != 0)) ||
      !((bits == 4 && (group == 64 || (group == 32 && f16 == 0))) || (bits == 8 && group == 64 && f16 == 0)) ||
      (splits > 1 && (bits != 4 || group != 64 || f16 != 0))) {
    return VPQ_ERR_BAD_SHAPE;
  }
  (void)ensure_init();                     // (without a device: the plan for 256 CUs)
  vpq::GemmArgs g{};
  g.K = K; g.N = N; g.M = M;
  g.bits = bits; g.group = group; g.f16 = f16 != 0;
  g.gate_act = gated != 0 ? VPQ_GATE_SWIGLU : 0;
  g.cu_count = g_dev.cu_count;
  return vpq::qmm_plan(g, splits);
}

int vpq_qmm_splitk_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                              const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                              int splits, void* ws, size_t ws_bytes)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M <= 0 || splits < 0 || splits > 16) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || (ws != nullptr && !aligned(ws, 256))) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  const auto room = [&](int n) { return ws != nullptr && ws_bytes >= (size_t)n * (size_t)M * (size_t)N * sizeof(float); };
  if (splits == 0) {
    splits = vpq::qmm_choose_splits(K, N, M, g_dev.cu_count);
    if (splits > 1 && !room(splits)) { splits = vpq::qmm_required_splits(K, N, M, g_dev.cu_count); }
  }
  if (splits > K / 64) { splits = K / 64; }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = M;
  g.cu_count = g_dev.cu_count;
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (splits <= 1) { return gemm_by_size(hs, g); }
  if (!room(splits)) { return VPQ_ERR_WORKSPACE; }
  return finish(vpq::launch_qmm_splitk(hs, g, splits, static_cast<float*>(ws)));
}

int vpq_qmm_dense_route_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                   const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                   uint16_t* w_deq, int expand)
{
  return vpq_qmm_dense_route_lora_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, w_deq, expand, nullptr, nullptr, 0,
                                             0.0f, nullptr);
}

// The dequant-once route with the runtime adapter: the pre-pass t = bf16(alpha * bf16(x . A^T)), the expansion (or the
// kept one), then the dense GEMM with t . B^T in the same accumulators -- the bits of vpq_qmm_w4g64_bf16 with the
// same adapter.
int vpq_qmm_dense_route_lora_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                        const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                        uint16_t* w_deq, int expand, const uint16_t* lora_a, const uint16_t* lora_b,
                                        int r, float alpha, uint16_t* lora_t_ws)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (w_deq == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || !aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  const bool lora = lora_a != nullptr && alpha != 0.0f;
  if (lora) {
    if (lora_b == nullptr) { return VPQ_ERR_NULL_POINTER; }
    if (lora_t_ws == nullptr) { return VPQ_ERR_WORKSPACE; }
    if (r < 8 || r > vpq::kLoraMaxRank || (r % 8) != 0) { return VPQ_ERR_BAD_SHAPE; }
    if (!aligned(lora_a, 16) || !aligned(lora_b, 16) || !aligned(lora_t_ws, 16)) { return VPQ_ERR_MISALIGNED; }
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (lora) {
    st = finish(vpq::launch_lora_a(hs, x, lora_a, lora_t_ws, M, K, r, alpha));
    if (st != VPQ_OK) { return st; }
  }
  if (expand != 0) {
    st = finish(vpq::launch_dequant(hs, w, scales, biases, w_deq, K, N));
    if (st != VPQ_OK) { return st; }
  }
  std::string why;
  const int rc = vpq::dense_gemm_elt(hs, x, w_deq, y, M, N, K, false, g_dev.cu_count, &why, lora ? lora_t_ws : nullptr,
                                     lora ? lora_b : nullptr, lora ? r : 0);
  if (rc != 0) {
    strncpy(g_last_error, why.c_str(), sizeof(g_last_error) - 1);
    g_last_error[sizeof(g_last_error) - 1] = '\0';
    return VPQ_ERR_DEVICE;
  }
  return VPQ_OK;
}

// ---- IEEE binary16 element type (VPIPE_ELT = half) ----

int vpq_dequant_w4g64_f16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                          uint16_t* w_deq, int K, int N)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (w_deq == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_dequant_f16(reinterpret_cast<hipStream_t>(stream), w, scales, biases, w_deq, K, N));
}

static int qmv_f16_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                          const uint16_t* x, void* y, bool y_f32, int K, int N, int M, const uint16_t* residual,
                          int gate_act)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16) { return VPQ_ERR_BAD_SHAPE; }
  if (gate_act != 0 && ((N & 1) != 0 || residual != nullptr)) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, y_f32 ? 4 : 2) || (residual != nullptr && !aligned(residual, 2))) {
    return VPQ_ERR_MISALIGNED;
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y; a.residual = residual;
  a.K = K; a.N = N; a.M = M; a.y_f32 = y_f32; a.cu_count = g_dev.cu_count;
  a.gate_act = gate_act;
  // one row of x on a K the streaming kernel takes: the same kernel as for bf16, on binary16 arithmetic
  if (vpq::qmv_flow_supports(K, N, M) && aligned(scales, 16) && aligned(biases, 16)) {
    return finish(vpq::launch_qmv_flow_f16(reinterpret_cast<hipStream_t>(stream), a));
  }
  const vpq::BatchFormat f{4, 64, true, false};
  if (flow_narrow_f16(K, N, M)) { return finish(vpq::launch_qmv_flow_narrow(reinterpret_cast<hipStream_t>(stream), a, f)); }
  if (vpq::qmv_batch_supports(K, M, f) && aligned(scales, 16) && aligned(biases, 16)) {
    return finish(launch_batch(reinterpret_cast<hipStream_t>(stream), a, f));
  }
  return finish(vpq::launch_qmv_simple_f16(reinterpret_cast<hipStream_t>(stream), a));
}

int vpq_qmv_w4g64_f16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                      const uint16_t* x, uint16_t* y, int K, int N, int M, const uint16_t* residual)
{
  return qmv_f16_common(stream, w, scales, biases, x, y, false, K, N, M, residual, 0);
}

int vpq_qmv_w4g64_f16_f32out(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                             const uint16_t* x, float* y, int K, int N, int M)
{
  return qmv_f16_common(stream, w, scales, biases, x, y, true, K, N, M, nullptr, 0);
}

int vpq_qmv_gated_w4g64_f16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                            const uint16_t* x, uint16_t* y, int K, int N, int M, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return qmv_f16_common(stream, w, scales, biases, x, y, false, K, N, M, nullptr, activation);
}

namespace {

// The fused GEMM on binary16 elements: the large-tile kernel once its tiles fill the CUs (K % 512 == 0, 16-byte
// aligned scales and biases), the 256 x 128 tile kernel otherwise -- same MFMA, same K order, same bits.
// activation 0 = plain y [M,N], else the gated store of an interleaved gate|up pack, y [M,N/2] (no adapter then).
int qmm_f16_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                   const uint16_t* x, uint16_t* y, int K, int N, int M, int activation, const uint16_t* lora_a,
                   const uint16_t* lora_b, int r, float alpha, uint16_t* lora_t_ws)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (activation != 0 && activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (M <= 0 || (activation != 0 && (N & 1) != 0)) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16)) { return VPQ_ERR_MISALIGNED; }
  const bool lora = lora_a != nullptr && alpha != 0.0f;
  if (lora) {
    if (activation != 0) { return VPQ_ERR_BAD_SHAPE; }
    if (lora_b == nullptr) { return VPQ_ERR_NULL_POINTER; }
    if (lora_t_ws == nullptr) { return VPQ_ERR_WORKSPACE; }
    if (r < 8 || r > vpq::kLoraMaxRank || (r % 8) != 0) { return VPQ_ERR_BAD_SHAPE; }
    if (!aligned(lora_a, 16) || !aligned(lora_b, 16) || !aligned(lora_t_ws, 16)) { return VPQ_ERR_MISALIGNED; }
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (lora) {
    st = finish(vpq::launch_lora_a(hs, x, lora_a, lora_t_ws, M, K, r, alpha, true));
    if (st != VPQ_OK) { return st; }
  }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = M;
  g.lora_t = lora ? lora_t_ws : nullptr;
  g.lora_b = lora ? lora_b : nullptr;
  g.r = lora ? r : 0;
  g.cu_count = g_dev.cu_count;
  g.gate_act = activation;
  g.f16 = true;
  return gemm_by_size(hs, g);
}

}  // namespace

int vpq_qmm_w4g64_f16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                      const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M, int activation)
{
  return qmm_f16_common(stream, w, scales, biases, x, y, K, N, M, activation, nullptr, nullptr, 0, 0.0f, nullptr);
}

int vpq_lora_a_f16(vpq_stream_t stream, const uint16_t* x, const uint16_t* lora_a, uint16_t* t, int M, int K, int r,
                   float alpha)
{
  if (x == nullptr || lora_a == nullptr || t == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M <= 0 || K <= 0 || (K % 64) != 0 || r < 8 || r > vpq::kLoraMaxRank || (r % 8) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(lora_a, 16) || !aligned(t, 16)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_lora_a(reinterpret_cast<hipStream_t>(stream), x, lora_a, t, M, K, r, alpha, true));
}

// The same with a runtime adapter: the pre-pass t = f16(alpha * f16(x . A^T)), then r more values of K from t and B
// in the GEMM's accumulators.  alpha == 0 or lora_a == NULL: no adapter.
int vpq_qmm_lora_w4g64_f16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                           const uint16_t* x, uint16_t* y, int K, int N, int M, const uint16_t* lora_a,
                           const uint16_t* lora_b, int r, float alpha, uint16_t* lora_t_ws)
{
  return qmm_f16_common(stream, w, scales, biases, x, y, K, N, M, 0, lora_a, lora_b, r, alpha, lora_t_ws);
}

int vpq_qmm_dense_route_w4g64_f16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                  const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                  uint16_t* w_deq, int expand)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (w_deq == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || !aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (expand != 0) {
    st = finish(vpq::launch_dequant_f16(hs, w, scales, biases, w_deq, K, N));
    if (st != VPQ_OK) { return st; }
  }
  std::string why;
  const int rc = vpq::dense_gemm_elt(hs, x, w_deq, y, M, N, K, true, g_dev.cu_count, &why);
  if (rc != 0) {
    strncpy(g_last_error, why.c_str(), sizeof(g_last_error) - 1);
    g_last_error[sizeof(g_last_error) - 1] = '\0';
    return VPQ_ERR_DEVICE;
  }
  return VPQ_OK;
}

// Rows up to which the size-based entrances run the GEMV arithmetic: one launch of the batch kernel, or slabs of 16
// rows where it does not run.  The 256-row GEMM tile has one row of tiles and N/128 workgroups there, and its time is
// its K loop's latency (57 us at 4096->4096 for any M <= 256 against 9.5 us at 64 rows).
constexpr int kSlabPlanMaxRows = 64;
constexpr int kSlabPlanSplitRows = 32;   // above, over a narrow N: the split-K GEMM, when the workspace has the room

namespace {

// Whether the batch kernel takes a call of more than 16 rows (what it does not, runs as slabs of 16, which report it).
bool batch_takes(const void* w, const void* scales, const void* biases, const void* x, const void* y, int K, int N, int M,
                 const vpq::BatchFormat& f)
{
  return w != nullptr && scales != nullptr && (f.scale_only || biases != nullptr) && N > 0 && K > 0 &&
         vpq::qmv_batch_supports(K, M, f) && aligned(w, 16) && aligned(scales, 16) && aligned(biases, 16) && aligned(x, 16) &&
         aligned(y, 2);
}

int batch_call(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases, const uint16_t* x,
               uint16_t* y, int K, int N, int M, int activation, const vpq::BatchFormat& f)
{
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y;
  a.K = K; a.N = N; a.M = M; a.cu_count = g_dev.cu_count;
  a.gate_act = activation;
  return finish(launch_batch(reinterpret_cast<hipStream_t>(stream), a, f));
}

}  // namespace

int vpq_linear_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                          const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                          void* ws, size_t ws_bytes)
{
  if (M >= 1 && M <= kSlabPlanMaxRows && x != nullptr && y != nullptr && K > 0 && N > 0) {
    // 33..64 rows over a narrow N: where the batch kernel's workgroups would fill less than a quarter of the CUs, the
    // GEMM with K split over the workgroups, if the workspace lets it split (measured at 48 rows, split GEMM / batch
    // kernel: 20 / 9.5 us at 4096 -> 4096 and 39 / 23 us at 4096 -> 12288, so not on wider ones).
    bool split_gemm = false;
    if (M > kSlabPlanSplitRows && ws != nullptr && aligned(ws, 256) && (K % 64) == 0 && ensure_init() == VPQ_OK &&
        (long)((N + 15) / 16) * ((M + 31) / 32) * 4 < (g_dev.cu_count > 0 ? g_dev.cu_count : 256)) {
      const int splits = vpq::qmm_choose_splits(K, N, M, g_dev.cu_count);
      split_gemm = splits > 1 && ws_bytes >= (size_t)splits * (size_t)M * (size_t)N * sizeof(float);
    }
    if (!split_gemm) {
      if (M > 16 && batch_takes(w, scales, biases, x, y, K, N, M, vpq::BatchFormat{})) {
        return batch_call(stream, w, scales, biases, x, y, K, N, M, 0, vpq::BatchFormat{});
      }
      for (int m0 = 0; m0 < M; m0 += 16) {
        const int rows = M - m0 < 16 ? M - m0 : 16;
        const int st = vpq_qmv_w4g64_bf16(stream, w, scales, biases, x + (size_t)m0 * K, y + (size_t)m0 * N, K, N, rows,
                                          nullptr, ws, ws_bytes, VPQ_QMV_AUTO);
        if (st != VPQ_OK) { return st; }
      }
      return VPQ_OK;
    }
  }
  // Very many rows: expanding the pack once into the workspace and running the dense GEMM on it beats the
  // fused kernels, the reference's own route for large M
  // (generative-models/minimax-h3/metal-minimax-h3-transformer.cc:2020-2160).
  if (ws != nullptr && aligned(ws, 256) && M >= kDenseRouteMinRows && K > 0 && N > 0 && (K % 64) == 0 &&
      ws_bytes >= (size_t)N * (size_t)K * 2 && vpq::dense_gemm_supports(M, N, K)) {
    return vpq_qmm_dense_route_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, static_cast<uint16_t*>(ws), 1);
  }
  // Few tiles and a long K: split K over more workgroups when the caller's workspace has the room.
  if (ws != nullptr && aligned(ws, 256) && K > 0 && N > 0 && M > 0 && (K % 64) == 0 && ensure_init() == VPQ_OK) {
    const int splits = vpq::qmm_choose_splits(K, N, M, g_dev.cu_count);
    if (splits > 1 && ws_bytes >= (size_t)splits * (size_t)M * (size_t)N * sizeof(float)) {
      return vpq_qmm_splitk_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, splits, ws, ws_bytes);
    }
  }
  return vpq_qmm_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, nullptr, nullptr, 0, 0.0f, nullptr);
}

int vpq_interleave_rows(vpq_stream_t stream, const void* a, const void* b, void* out, size_t row_bytes, size_t rows)
{
  if (a == nullptr || b == nullptr || out == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (row_bytes == 0 || (row_bytes & 1) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(a, 2) || !aligned(b, 2) || !aligned(out, 2)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_interleave_rows(reinterpret_cast<hipStream_t>(stream), a, b, out, row_bytes, rows));
}

int vpq_qmv_gated_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                             const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                             int variant, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return qmv_common(stream, w, scales, biases, x, y, false, K, N, M, nullptr, nullptr, 0, variant, activation);
}

int vpq_qmv_gelu_mul_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                const uint16_t* mul)
{
  return qmv_common(stream, w, scales, biases, x, y, false, K, N, 1, mul, nullptr, 0, VPQ_QMV_AUTO, vpq::kStoreGeluMul);
}

int vpq_qmv_gated_w4g64_f32out(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                               const uint16_t* biases, const uint16_t* x, float* y, int K, int N, int M,
                               int variant, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return qmv_common(stream, w, scales, biases, x, y, true, K, N, M, nullptr, nullptr, 0, variant, activation);
}

int vpq_qmm_gated_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                             const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                             int out_stride, int out_off, int activation)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (M <= 0 || (N & 1) != 0 || out_off < 0) { return VPQ_ERR_BAD_SHAPE; }
  if (out_stride > 0 && out_off + N / 2 > out_stride) { return VPQ_ERR_BAD_SHAPE; }
  if (out_stride <= 0 && out_off != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = M;
  g.cu_count = g_dev.cu_count;
  g.gate_act = activation;
  g.out_stride = out_stride;
  g.out_off = out_off;
  return gemm_by_size(reinterpret_cast<hipStream_t>(stream), g);
}

int vpq_linear_gated_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                int activation)
{
  if (M >= 1 && M <= kSlabPlanMaxRows && x != nullptr && y != nullptr && K > 0 && N > 0) {
    if (M > 16 && (N & 1) == 0 && (activation == VPQ_GATE_SWIGLU || activation == VPQ_GATE_GEGLU) &&
        batch_takes(w, scales, biases, x, y, K, N, M, vpq::BatchFormat{})) {
      return batch_call(stream, w, scales, biases, x, y, K, N, M, activation, vpq::BatchFormat{});
    }
    for (int m0 = 0; m0 < M; m0 += 16) {
      const int rows = M - m0 < 16 ? M - m0 : 16;
      const int st = vpq_qmv_gated_w4g64_bf16(stream, w, scales, biases, x + (size_t)m0 * K, y + (size_t)m0 * (N / 2), K, N,
                                              rows, VPQ_QMV_AUTO, activation);
      if (st != VPQ_OK) { return st; }
    }
    return VPQ_OK;
  }
  return vpq_qmm_gated_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, 0, 0, activation);
}

int vpq_qmv_swiglu_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                              const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                              int variant)
{
  return vpq_qmv_gated_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, variant, VPQ_GATE_SWIGLU);
}

int vpq_qmv_swiglu_w4g64_f32out(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                const uint16_t* biases, const uint16_t* x, float* y, int K, int N, int M,
                                int variant)
{
  return vpq_qmv_gated_w4g64_f32out(stream, w, scales, biases, x, y, K, N, M, variant, VPQ_GATE_SWIGLU);
}

int vpq_qmm_swiglu_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                              const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                              int out_stride, int out_off)
{
  return vpq_qmm_gated_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, out_stride, out_off, VPQ_GATE_SWIGLU);
}

int vpq_linear_swiglu_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                 const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M)
{
  return vpq_linear_gated_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, VPQ_GATE_SWIGLU);
}

namespace {

int gather_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                  const uint16_t* x, uint16_t* y, int K, int N, const int32_t* pair_eid, int npair, int x_div,
                  int n_experts, int gate_act)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr || pair_eid == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (npair < 1 || npair > 65535 || x_div < 1 || n_experts < 1) { return VPQ_ERR_BAD_SHAPE; }
  if (gate_act != 0 && (N & 1) != 0) { return VPQ_ERR_BAD_SHAPE; }
  // every slab and every row of x must keep the 16-byte alignment of the base
  if (!aligned(x, 16) || !aligned(y, 2) || !aligned(pair_eid, 4)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y;
  a.K = K; a.N = N; a.M = 1; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  a.gate_act = gate_act;
  if (vpq::qmv_gather_supports(K, 4)) {
    return finish(vpq::launch_qmv_gather(reinterpret_cast<hipStream_t>(stream), a, 4, pair_eid, npair, x_div, n_experts));
  }
  return finish(vpq::launch_qmv_rows_gather(reinterpret_cast<hipStream_t>(stream), a, pair_eid, npair, x_div, n_experts));
}

}  // namespace

int vpq_gather_qmv_gated_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                    const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                    const int32_t* pair_eid, int npair, int top_k, int n_experts, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return gather_common(stream, w, scales, biases, x, y, K, N, pair_eid, npair, top_k, n_experts, activation);
}

int vpq_gather_down_qmv_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                   const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                   const int32_t* pair_eid, int npair, int n_experts)
{
  return gather_common(stream, w, scales, biases, x, y, K, N, pair_eid, npair, 1, n_experts, 0);
}

namespace {

int sorted_qmv_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                      const uint16_t* x, uint16_t* y, int K, int N, int npad, const int32_t* tile2e, const int32_t* srow,
                      int n_experts, int gate_act, bool x_from_srow, int bits = 4)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr || tile2e == nullptr || srow == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (npad < VPQ_QMV_GROUPED_SLOTS || (npad % VPQ_QMV_GROUPED_SLOTS) != 0 || npad / VPQ_QMV_GROUPED_SLOTS > 65535 ||
      n_experts < 1) {
    return VPQ_ERR_BAD_SHAPE;
  }
  if (gate_act != 0 && gate_act != VPQ_GATE_SWIGLU && gate_act != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (gate_act != 0 && (N & 1) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 2) || !aligned(tile2e, 4) || !aligned(srow, 4)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y;
  a.K = K; a.N = N; a.M = VPQ_QMV_GROUPED_SLOTS; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  a.gate_act = gate_act;
  if (bits == 8) {
    return finish(vpq::launch_qmv_rows8_sorted(reinterpret_cast<hipStream_t>(stream), a, tile2e, srow,
                                               npad / VPQ_QMV_GROUPED_SLOTS, n_experts));
  }
  return finish(vpq::launch_qmv_rows_sorted(reinterpret_cast<hipStream_t>(stream), a, tile2e, srow,
                                            npad / VPQ_QMV_GROUPED_SLOTS, x_from_srow, n_experts));
}

}  // namespace

int vpq_qmv_grouped_gated_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                     const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int npad,
                                     const int32_t* tile2e, const int32_t* srow, int n_experts, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return sorted_qmv_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, srow, n_experts, activation, true);
}

int vpq_qmv_grouped_down_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                    const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int npad,
                                    const int32_t* tile2e, const int32_t* srow, int n_experts)
{
  return sorted_qmv_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, srow, n_experts, 0, false);
}

int vpq_qmv_grouped_gated_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                     const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int npad,
                                     const int32_t* tile2e, const int32_t* srow, int n_experts, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return sorted_qmv_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, srow, n_experts, activation, true, 8);
}

int vpq_qmv_grouped_down_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                    const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int npad,
                                    const int32_t* tile2e, const int32_t* srow, int n_experts)
{
  return sorted_qmv_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, srow, n_experts, 0, false, 8);
}

int vpq_sample_topp_bf16(vpq_stream_t stream, const uint16_t* logits, int32_t* out_id, int V, float temp,
                         float top_p, uint32_t seed, uint16_t* ws, int n_iter, float rep_penalty,
                         float presence_penalty, int top_k, float min_p, uint8_t* seen)
{
  if (logits == nullptr || out_id == nullptr || ws == nullptr || seen == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (V < 1 || n_iter < 0 || rep_penalty == 0.0f) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(logits, 2) || !aligned(ws, 2) || !aligned(out_id, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_sample_topp(reinterpret_cast<hipStream_t>(stream), logits, out_id, V, temp, top_p, seed, ws,
                                        n_iter, rep_penalty, presence_penalty, top_k, min_p, seen));
}

size_t vpq_sample_hist_workspace_bytes(int n_slabs)
{
  return n_slabs >= 1 && n_slabs <= 1024 ? vpq::sample_hist_work_words(n_slabs) * sizeof(float) : 0;
}

int vpq_sample_hist_bf16(vpq_stream_t stream, const uint16_t* logits, int32_t* out_id, int V, float temp,
                         float top_p, uint32_t seed, uint16_t* ws, float rep_penalty, float presence_penalty,
                         int top_k, float min_p, uint8_t* seen, int n_slabs, void* work, size_t work_bytes)
{
  if (logits == nullptr || out_id == nullptr || ws == nullptr || seen == nullptr) { return VPQ_ERR_NULL_POINTER; }
  // counts travel as fp32: exact up to 2^24 logits
  if (V < 1 || V > (1 << 24) || rep_penalty == 0.0f || n_slabs < 1 || n_slabs > 1024) { return VPQ_ERR_BAD_SHAPE; }
  // a slab's fixed-point mass of one bin stays below 2^32
  if (((long long)V + n_slabs - 1) / n_slabs > 65535) { return VPQ_ERR_BAD_SHAPE; }
  if (work == nullptr || work_bytes < vpq_sample_hist_workspace_bytes(n_slabs)) { return VPQ_ERR_WORKSPACE; }
  if (!aligned(logits, 2) || !aligned(ws, 2) || !aligned(out_id, 4) || !aligned(work, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_sample_hist(reinterpret_cast<hipStream_t>(stream), logits, out_id, V, temp, top_p, seed, ws,
                                        rep_penalty, presence_penalty, top_k, min_p, seen, n_slabs,
                                        static_cast<float*>(work)));
}

int vpq_qmm_grouped_block_rows(void) { return vpq::kGroupedBlockRows; }

int vpq_qmm_grouped_plan(int N, int npad, int n_experts, int rows, int gated)
{
  if (N <= 0 || npad <= 0 || (npad % vpq::kGroupedBlockRows) != 0 || n_experts < 1 || rows < 1 || (gated != 0 && (N & 1) != 0)) {
    return VPQ_ERR_BAD_SHAPE;
  }
  (void)ensure_init();                     // (without a device: the plan for 256 CUs)
  vpq::GemmArgs g{};
  g.N = N; g.M = npad;
  g.gate_act = gated != 0 ? VPQ_GATE_SWIGLU : 0;
  g.cu_count = g_dev.cu_count;
  vpq::GroupedArgs ga{};
  ga.n_experts = n_experts;
  ga.rows_x = gated != 0 ? rows : npad;
  ga.rows_y = gated != 0 ? npad : rows;
  return vpq::qmm_grouped_wide(g, ga) ? 160 : 64;
}

size_t vpq_moe_sort_workspace_bytes(int n_experts)
{
  return n_experts > 0 ? (size_t)3 * (size_t)n_experts * sizeof(int32_t) : 0;
}

int vpq_moe_sort_pairs(vpq_stream_t stream, const int32_t* pair_eid, int npair, int top_k, int n_experts,
                       int block_rows, int max_tiles, int32_t* tile2e, int32_t* srow, int32_t* sdst,
                       int32_t* ntiles, void* ws, size_t ws_bytes)
{
  if (pair_eid == nullptr || tile2e == nullptr || srow == nullptr || sdst == nullptr || ntiles == nullptr ||
      ws == nullptr) {
    return VPQ_ERR_NULL_POINTER;
  }
  if (npair < 1 || top_k < 1 || n_experts < 1 || block_rows < 1 || max_tiles < 1) { return VPQ_ERR_BAD_SHAPE; }
  if (npair > (1 << 24) || n_experts > 65536) { return VPQ_ERR_BAD_SHAPE; }
  // every expert's share rounded up to whole blocks must fit
  const long long need = ((long long)npair + block_rows - 1) / block_rows + (n_experts < npair ? n_experts : npair);
  if ((long long)max_tiles < need || (long long)max_tiles * block_rows > 0x7fffffffLL) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(pair_eid, 4) || !aligned(tile2e, 4) || !aligned(srow, 4) || !aligned(sdst, 4) || !aligned(ntiles, 4) ||
      !aligned(ws, 4)) {
    return VPQ_ERR_MISALIGNED;
  }
  if (ws_bytes < vpq_moe_sort_workspace_bytes(n_experts)) { return VPQ_ERR_WORKSPACE; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_moe_sort(reinterpret_cast<hipStream_t>(stream), pair_eid, npair, top_k, n_experts,
                                     block_rows, max_tiles, tile2e, srow, sdst, ntiles, static_cast<int*>(ws)));
}

int vpq_moe_scatter_back_bf16(vpq_stream_t stream, const uint16_t* dsorted, const int32_t* sdst, uint16_t* partials,
                              int npad, int H, int npair)
{
  if (dsorted == nullptr || sdst == nullptr || partials == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (npad < 1 || H < 1 || npair < 1 || (long long)npad * (long long)H > 0x3fffffffffLL) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(dsorted, 2) || !aligned(partials, 2) || !aligned(sdst, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  const bool wide = (H % 8) == 0 && aligned(dsorted, 16) && aligned(partials, 16);
  return finish(vpq::launch_moe_scatter_back(reinterpret_cast<hipStream_t>(stream), dsorted, sdst, partials, npad, H, npair,
                                             wide));
}

namespace {

int grouped_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                   const uint16_t* x, uint16_t* y, int K, int N, int npad, const int32_t* tile2e,
                   const int32_t* srow, const int32_t* sdst, int n_experts, int rows, int gate_act, int bits = 4)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr || tile2e == nullptr || (srow == nullptr && sdst == nullptr)) {
    return VPQ_ERR_NULL_POINTER;
  }
  if (npad < vpq::kGroupedBlockRows || (npad % vpq::kGroupedBlockRows) != 0 || n_experts < 1 || rows < 1) {
    return VPQ_ERR_BAD_SHAPE;
  }
  if (gate_act != 0 && (N & 1) != 0) { return VPQ_ERR_BAD_SHAPE; }
  // the kernel addresses rows of x by 32-bit byte offsets
  const long long xrows = srow != nullptr ? rows : npad;
  if (xrows * (long long)K * 2 >= 4000000000LL) { return VPQ_ERR_BAD_SHAPE; }
  // (y rows are stored in 16-byte pieces, at any address)
  if (!aligned(x, 16) || !aligned(y, 8) || !aligned(tile2e, 4) || (srow != nullptr && !aligned(srow, 4)) ||
      (sdst != nullptr && !aligned(sdst, 4))) {
    return VPQ_ERR_MISALIGNED;
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = npad; g.lora_t = nullptr; g.lora_b = nullptr; g.r = 0;
  g.cu_count = g_dev.cu_count;
  g.gate_act = gate_act; g.out_stride = N / 2; g.out_off = 0;
  g.bits = bits;
  vpq::GroupedArgs ga{};
  ga.tile2e = tile2e; ga.srow = srow; ga.sdst = sdst;
  ga.n_experts = n_experts;
  ga.rows_x = srow != nullptr ? rows : npad;
  ga.rows_y = sdst != nullptr ? rows : npad;
  return finish(vpq::launch_qmm_grouped(reinterpret_cast<hipStream_t>(stream), g, ga));
}

}  // namespace

int vpq_qmm_grouped_gated_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                     const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                     int npad, const int32_t* tile2e, const int32_t* srow, int n_experts,
                                     int rows_x, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (srow == nullptr) { return VPQ_ERR_NULL_POINTER; }
  return grouped_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, srow, nullptr, n_experts, rows_x,
                        activation);
}

int vpq_qmm_grouped_down_w4g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                    const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                    int npad, const int32_t* tile2e, const int32_t* sdst, int n_experts,
                                    int rows_y)
{
  if (sdst == nullptr) { return VPQ_ERR_NULL_POINTER; }
  return grouped_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, nullptr, sdst, n_experts, rows_y, 0);
}

// ---- 8-bit twins on the fused kernels ----

namespace {

// The fused GEMM of a format twin (byte codes, groups of 32).  tile: 0 = by size, as for the 4-bit group-64 pack
// (the large-tile kernel once its tiles fill the CUs), 128 = the 256 x 128 tile kernel, 192 / 256 = the large-tile
// kernel at that width, -128 = the large-tile kernel at width 128.
int twin_gemm_launch(vpq_stream_t stream, const vpq::GemmArgs& g, int tile)
{
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (tile == 192 || tile == 256 || tile == -128) {
    // byte codes: up to 192 wide; groups of 32: 256 or 128 wide
    if (!vpq::qmm_big_supports(g) || (tile == 256 && g.bits == 8) || (tile == 192 && g.group == 32)) { return VPQ_ERR_BAD_SHAPE; }
    return finish(vpq::launch_qmm_big(hs, g, tile < 0 ? -tile : tile));
  }
  if (tile == 0) { return gemm_by_size(hs, g); }
  return finish(vpq::launch_qmm_tile(hs, g));
}

}  // namespace

int vpq_qmm_gated_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                             const uint16_t* x, uint16_t* y, int K, int N, int M, int out_stride, int out_off, int activation)
{
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (activation != 0 && activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (M <= 0 || out_off < 0 || (activation != 0 && (N & 1) != 0)) { return VPQ_ERR_BAD_SHAPE; }
  if (activation == 0 && (out_stride != 0 || out_off != 0)) { return VPQ_ERR_BAD_SHAPE; }
  if (out_stride > 0 && out_off + N / 2 > out_stride) { return VPQ_ERR_BAD_SHAPE; }
  if (out_stride <= 0 && out_off != 0) { return VPQ_ERR_BAD_SHAPE; }
  if ((long long)M * (long long)K * 2 >= 4000000000LL) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = M; g.lora_t = nullptr; g.lora_b = nullptr; g.r = 0;
  g.cu_count = g_dev.cu_count;
  g.gate_act = activation; g.out_stride = out_stride; g.out_off = out_off;
  g.bits = 8;
  return twin_gemm_launch(stream, g, 0);
}

int vpq_qmm_tiled_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                             const uint16_t* x, uint16_t* y, int K, int N, int M, int activation, int tile_n)
{
  if (tile_n != 128 && tile_n != -128 && tile_n != 192) { return VPQ_ERR_BAD_SHAPE; }
  int st = check_pack(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (activation != 0 && activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (M <= 0 || (activation != 0 && (N & 1) != 0)) { return VPQ_ERR_BAD_SHAPE; }
  if ((long long)M * (long long)K * 2 >= 4000000000LL) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = M;
  g.cu_count = g_dev.cu_count;
  g.gate_act = activation;
  g.bits = 8;
  return twin_gemm_launch(stream, g, tile_n);
}

int vpq_qmm_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                       const uint16_t* x, uint16_t* y, int K, int N, int M)
{
  return vpq_qmm_gated_w8g64_bf16(stream, w, scales, biases, x, y, K, N, M, 0, 0, 0);
}

// Size-based entrances of the format twins (the ladder of vpq_linear_w4g64_bf16 without a workspace: slabs of
// the GEMV arithmetic up to 64 rows, the fused GEMM above).
int vpq_linear_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                          const uint16_t* x, uint16_t* y, int K, int N, int M)
{
  if (M >= 1 && M <= kSlabPlanMaxRows && x != nullptr && y != nullptr && K > 0 && N > 0) {
    const vpq::BatchFormat f{8, 64, false, false};
    if (M > 16 && batch_takes(w, scales, biases, x, y, K, N, M, f)) {
      return batch_call(stream, w, scales, biases, x, y, K, N, M, 0, f);
    }
    for (int m0 = 0; m0 < M; m0 += 16) {
      const int rows = M - m0 < 16 ? M - m0 : 16;
      const int st = vpq_qmv_w8g64_bf16(stream, w, scales, biases, x + (size_t)m0 * K, y + (size_t)m0 * N, K, N, rows,
                                        nullptr);
      if (st != VPQ_OK) { return st; }
    }
    return VPQ_OK;
  }
  return vpq_qmm_w8g64_bf16(stream, w, scales, biases, x, y, K, N, M);
}

int vpq_qmm_grouped_gated_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                     const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                     int npad, const int32_t* tile2e, const int32_t* srow, int n_experts,
                                     int rows_x, int activation)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (srow == nullptr) { return VPQ_ERR_NULL_POINTER; }
  return grouped_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, srow, nullptr, n_experts, rows_x,
                        activation, 8);
}

int vpq_qmm_grouped_down_w8g64_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                    const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N,
                                    int npad, const int32_t* tile2e, const int32_t* sdst, int n_experts,
                                    int rows_y)
{
  if (sdst == nullptr) { return VPQ_ERR_NULL_POINTER; }
  return grouped_common(stream, w, scales, biases, x, y, K, N, npad, tile2e, nullptr, sdst, n_experts, rows_y, 0, 8);
}


namespace {

int check_pack_g32(const uint32_t* w, const uint16_t* scales, const uint16_t* biases, int K, int N, bool scale_only)
{
  if (w == nullptr || scales == nullptr || (!scale_only && biases == nullptr)) { return VPQ_ERR_NULL_POINTER; }
  if (K <= 0 || N <= 0 || (K % 32) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(w, 16) || !aligned(scales, 2) || (!scale_only && !aligned(biases, 2))) { return VPQ_ERR_MISALIGNED; }
  return VPQ_OK;
}

int qmv_g32_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                   const uint16_t* x, void* y, bool y_f32, int K, int N, int M, const uint16_t* residual,
                   int gate_act, bool scale_only)
{
  int st = check_pack_g32(w, scales, biases, K, N, scale_only);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16) { return VPQ_ERR_BAD_SHAPE; }
  const bool gelu_mul = gate_act == vpq::kStoreGeluMul;       // `residual` is the multiplier [N]
  if (gelu_mul && residual == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (gate_act != 0 && !gelu_mul && ((N & 1) != 0 || residual != nullptr)) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, y_f32 ? 4 : 2) || (residual != nullptr && !aligned(residual, 2))) {
    return VPQ_ERR_MISALIGNED;
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.w = w; a.scales = scales; a.biases = biases; a.x = x; a.y = y; a.residual = residual;
  a.K = K; a.N = N; a.M = M; a.y_f32 = y_f32; a.cu_count = g_dev.cu_count;
  a.gate_act = gate_act;
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (gelu_mul) { return finish(vpq::launch_qmv_simple_g32(hs, a, scale_only)); }    // the kernel that has this store
  // one row of x: the one-row kernel, or for a short K the row-streaming one; more: the batch kernel.  Each takes packs with and
  // without biases, and gives both the same bits.  (us, row-streaming / batch / one-row: one row 4096 -> 24576 16.9 / 17.9 / 13.8,
  // 12288 -> 4096 9.7 / 11.7 / 9.1, 4096 -> 4096 5.8 / 6.0 / 4.2; two rows 23.3 / 17.9, 12.6 / 11.7 and 6.9 / 6.0)
  const vpq::BatchFormat f{4, 32, false, scale_only};
  if (M > 1 && vpq::qmv_batch_supports(K, M, f) && aligned(scales, 16) && (scale_only || aligned(biases, 16))) {
    return finish(launch_batch(hs, a, f));
  }
  if (vpq::qmv_flow_narrow_supports(K, N, M, 32)) { return finish(vpq::launch_qmv_flow_narrow(hs, a, f)); }
  if (M <= 2) { return finish(vpq::launch_qmv_rows_g32(hs, a, scale_only)); }
  return finish(vpq::launch_qmv_simple_g32(hs, a, scale_only));
}

}  // namespace

int vpq_dequant_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                           uint16_t* w_deq, int K, int N)
{
  int st = check_pack_g32(w, scales, biases, K, N, false);
  if (st != VPQ_OK) { return st; }
  if (w_deq == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_dequant_g32(reinterpret_cast<hipStream_t>(stream), w, scales, biases, w_deq, K, N));
}

int vpq_qmv_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                       const uint16_t* x, uint16_t* y, int K, int N, int M, const uint16_t* residual, int scale_only)
{
  return qmv_g32_common(stream, w, scales, biases, x, y, false, K, N, M, residual, 0, scale_only != 0);
}

int vpq_qmv_w4g32_f32out(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                         const uint16_t* x, float* y, int K, int N, int M, int scale_only)
{
  return qmv_g32_common(stream, w, scales, biases, x, y, true, K, N, M, nullptr, 0, scale_only != 0);
}

int vpq_qmv_gelu_mul_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                                const uint16_t* x, uint16_t* y, int K, int N, const uint16_t* mul, int scale_only)
{
  return qmv_g32_common(stream, w, scales, biases, x, y, false, K, N, 1, mul, vpq::kStoreGeluMul, scale_only != 0);
}

int vpq_qmv_gated_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                             const uint16_t* x, uint16_t* y, int K, int N, int M, int activation, int scale_only)
{
  if (activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  return qmv_g32_common(stream, w, scales, biases, x, y, false, K, N, M, nullptr, activation, scale_only != 0);
}

namespace {

int qmm_g32_common(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                   const uint16_t* x, uint16_t* y, int K, int N, int M, int activation, int tile_n)
{
  int st = check_pack_g32(w, scales, biases, K, N, false);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (activation != 0 && activation != VPQ_GATE_SWIGLU && activation != VPQ_GATE_GEGLU) { return VPQ_ERR_BAD_SHAPE; }
  if (M <= 0 || (K % 64) != 0 || (activation != 0 && (N & 1) != 0)) { return VPQ_ERR_BAD_SHAPE; }
  if ((long long)M * (long long)K * 2 >= 4000000000LL) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::GemmArgs g{};
  g.w = w; g.scales = scales; g.biases = biases; g.x = x; g.y = y;
  g.K = K; g.N = N; g.M = M; g.lora_t = nullptr; g.lora_b = nullptr; g.r = 0;
  g.cu_count = g_dev.cu_count;
  g.gate_act = activation; g.out_stride = 0; g.out_off = 0;
  g.group = 32;
  return twin_gemm_launch(stream, g, tile_n);
}

}  // namespace

int vpq_qmm_gated_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                             const uint16_t* x, uint16_t* y, int K, int N, int M, int activation)
{
  return qmm_g32_common(stream, w, scales, biases, x, y, K, N, M, activation, 0);
}

int vpq_qmm_tiled_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                             const uint16_t* x, uint16_t* y, int K, int N, int M, int activation, int tile_n)
{
  if (tile_n != 128 && tile_n != -128 && tile_n != 192 && tile_n != 256) { return VPQ_ERR_BAD_SHAPE; }
  return qmm_g32_common(stream, w, scales, biases, x, y, K, N, M, activation, tile_n);
}

int vpq_qmm_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                       const uint16_t* x, uint16_t* y, int K, int N, int M)
{
  return vpq_qmm_gated_w4g32_bf16(stream, w, scales, biases, x, y, K, N, M, 0);
}

int vpq_linear_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                          const uint16_t* x, uint16_t* y, int K, int N, int M)
{
  // K % 64 != 0 (a group-32 pack may have K % 64 == 32) has no fused GEMM: slabs at every M
  if (M >= 1 && (M <= kSlabPlanMaxRows || (K % 64) != 0) && x != nullptr && y != nullptr && K > 0 && N > 0) {
    const vpq::BatchFormat f{4, 32, false, false};
    if (M > 16 && batch_takes(w, scales, biases, x, y, K, N, M, f)) {
      return batch_call(stream, w, scales, biases, x, y, K, N, M, 0, f);
    }
    for (int m0 = 0; m0 < M; m0 += 16) {
      const int rows = M - m0 < 16 ? M - m0 : 16;
      const int st = vpq_qmv_w4g32_bf16(stream, w, scales, biases, x + (size_t)m0 * K, y + (size_t)m0 * N, K, N, rows,
                                        nullptr, 0);
      if (st != VPQ_OK) { return st; }
    }
    return VPQ_OK;
  }
  return vpq_qmm_w4g32_bf16(stream, w, scales, biases, x, y, K, N, M);
}

int vpq_qmm_dense_route_w4g32_bf16(vpq_stream_t stream, const uint32_t* w, const uint16_t* scales,
                                   const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                   uint16_t* w_deq, int expand)
{
  int st = check_pack_g32(w, scales, biases, K, N, false);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (w_deq == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || !aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (expand != 0) {
    st = finish(vpq::launch_dequant_g32(hs, w, scales, biases, w_deq, K, N));
    if (st != VPQ_OK) { return st; }
  }
  std::string why;
  const int rc = vpq::dense_gemm_bf16(hs, x, w_deq, y, M, N, K, g_dev.cu_count, &why);
  if (rc != 0) {
    strncpy(g_last_error, why.c_str(), sizeof(g_last_error) - 1);
    g_last_error[sizeof(g_last_error) - 1] = '\0';
    return VPQ_ERR_DEVICE;
  }
  return VPQ_OK;
}

size_t vpq_argmax_workspace_bytes(int V, int rows)
{
  if (V <= 0 || rows <= 0) { return 0; }
  return (size_t)rows * (size_t)vpq::argmax_parts(V) * 2 * sizeof(float);
}

int vpq_argmax_bf16(vpq_stream_t stream, const uint16_t* logits, int32_t* out_id, int V, int rows, void* ws,
                    size_t ws_bytes)
{
  if (logits == nullptr || out_id == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (V <= 0 || rows <= 0 || rows > 65535) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(logits, 2) || !aligned(out_id, 4) || (ws != nullptr && !aligned(ws, 4))) { return VPQ_ERR_MISALIGNED; }
  if (ws != nullptr && ws_bytes < vpq_argmax_workspace_bytes(V, rows)) { return VPQ_ERR_WORKSPACE; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (ws == nullptr) { return finish(vpq::launch_argmax_row(hs, logits, out_id, V, rows)); }
  const int parts = vpq::argmax_parts(V);
  const int e = finish(vpq::launch_argmax_partial(hs, logits, static_cast<float*>(ws), V, rows, parts));
  if (e != VPQ_OK) { return e; }
  return finish(vpq::launch_argmax_combine(hs, static_cast<const float*>(ws), out_id, rows, parts));
}

int vpq_argmax_bf16_static(vpq_stream_t stream, const uint16_t* logits, int32_t* out_id, int V, int rows)
{
  if (logits == nullptr || out_id == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (V <= 0 || rows <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (rows > vpq::kArgmaxStaticRows) {
    snprintf(g_last_error, sizeof(g_last_error), "vpq_argmax_bf16_static: %d rows, the static scratch holds %d", rows,
             vpq::kArgmaxStaticRows);
    return VPQ_ERR_WORKSPACE;
  }
  if (!aligned(logits, 2) || !aligned(out_id, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  float* partials = nullptr;
  const hipError_t se = vpq::argmax_static_scratch(&partials);
  if (se != hipSuccess) { return device_error(se); }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  // Every pair the combine reads is written by this call's first stage: nothing of an earlier call is read,
  // so nothing has to be cleared.
  const int parts = vpq::argmax_parts(V);
  const int e = finish(vpq::launch_argmax_partial(hs, logits, partials, V, rows, parts));
  if (e != VPQ_OK) { return e; }
  return finish(vpq::launch_argmax_combine(hs, partials, out_id, rows, parts));
}

int vpq_argmax_partial_bf16(vpq_stream_t stream, const uint16_t* logits, float* partials, int V, int parts)
{
  if (logits == nullptr || partials == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (V <= 0 || parts < 1 || parts > 65535) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(logits, 2) || !aligned(partials, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_argmax_partial(reinterpret_cast<hipStream_t>(stream), logits, partials, V, 1, parts));
}

int vpq_argmax_combine(vpq_stream_t stream, const float* partials, int32_t* out_id, int parts)
{
  if (partials == nullptr || out_id == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (parts < 1) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(partials, 4) || !aligned(out_id, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_argmax_combine(reinterpret_cast<hipStream_t>(stream), partials, out_id, 1, parts));
}

int vpq_qmv_group_w4g64_bf16(vpq_stream_t stream, int count, const uint32_t* const* w,
                             const uint16_t* const* scales, const uint16_t* const* biases,
                             const uint16_t* x, uint16_t* const* y, int K, const int* N, int M)
{
  if (w == nullptr || scales == nullptr || biases == nullptr || y == nullptr || N == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (count < 1 || count > 4) { return VPQ_ERR_BAD_SHAPE; }
  int wides = 0;                                        // packs whose scales and biases allow 16-byte loads
  for (int i = 0; i < count; ++i) {
    int st = check_pack(w[i], scales[i], biases[i], K, N[i]);
    if (st != VPQ_OK) { return st; }
    if (y[i] == nullptr) { return VPQ_ERR_NULL_POINTER; }
    if (!aligned(y[i], 2)) { return VPQ_ERR_MISALIGNED; }
    wides += aligned(scales[i], 16) && aligned(biases[i], 16) ? 1 : 0;
  }
  if (x == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16)) { return VPQ_ERR_MISALIGNED; }
  // The kernels of the single call (qmv_common), each in its grouped form.  Packs of both kinds have the same one only at one row
  // of a K that is no multiple of 512.
  const bool wide = wides == count, mixed = wides != 0 && !wide && !(M == 1 && (K % 512) != 0);
  const bool batch = wide && vpq::qmv_batch_supports(K, M, vpq::BatchFormat{});
  const bool flow = batch && vpq::qmv_flow_supports(K, 1, M);
  const bool narrow = (K % 512) != 0 && vpq::qmv_flow_narrow_supports(K, 1, M, 64);
  const bool rows = !narrow && !mixed && vpq::qmv_rows_supports(K, 1, M) && (!wide || (K % 512) != 0) && (!batch || M == 1);
  if (!flow && !narrow && !rows && !batch) {
    for (int i = 0; i < count; ++i) {
      const int st = vpq_qmv_w4g64_bf16(stream, w[i], scales[i], biases[i], x, y[i], K, N[i], M, nullptr, nullptr, 0,
                                        VPQ_QMV_AUTO);
      if (st != VPQ_OK) { return st; }
    }
    return VPQ_OK;
  }
  int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.x = x; a.K = K; a.M = M; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  vpq::QmvGroup g;
  g.count = count;
  for (int i = 0; i < count; ++i) { g.seg[i] = vpq::QmvSeg{w[i], scales[i], biases[i], y[i], N[i]}; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (flow) { return finish(vpq::launch_qmv_flow_group(hs, a, g)); }
  if (narrow) { return finish(vpq::launch_qmv_flow_narrow_group(hs, a, g, vpq::BatchFormat{})); }
  if (rows) { return finish(vpq::launch_qmv_rows_group(hs, a, g)); }
  return finish(vpq::launch_qmv_batch(hs, a, g, vpq::BatchFormat{}));
}

// The fused-QKV GEMV of the format twins (`affine_qmv_qkv_w4g32`, `affine_qmv_qkv_w8g64`,
// gpu-kernels/metal/quant/affine_qmv.metal:518-559): 1..4 packs that share x, one launch where the kernel of the single
// call has a grouped form; otherwise the packs are separate calls, with the same bits.
int vpq_qmv_group_w4g32_bf16(vpq_stream_t stream, int count, const uint32_t* const* w, const uint16_t* const* scales,
                             const uint16_t* const* biases, const uint16_t* x, uint16_t* const* y, int K, const int* N,
                             int M, int scale_only)
{
  if (w == nullptr || scales == nullptr || y == nullptr || N == nullptr || (biases == nullptr && scale_only == 0)) {
    return VPQ_ERR_NULL_POINTER;
  }
  if (count < 1 || count > 4) { return VPQ_ERR_BAD_SHAPE; }
  if (x == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16) { return VPQ_ERR_BAD_SHAPE; }
  for (int i = 0; i < count; ++i) {
    const int st = check_pack_g32(w[i], scales[i], scale_only ? nullptr : biases[i], K, N[i], scale_only != 0);
    if (st != VPQ_OK) { return st; }
    if (y[i] == nullptr) { return VPQ_ERR_NULL_POINTER; }
    if (!aligned(y[i], 2)) { return VPQ_ERR_MISALIGNED; }
  }
  if (!aligned(x, 16)) { return VPQ_ERR_MISALIGNED; }
  const vpq::BatchFormat f{4, 32, false, scale_only != 0};
  bool batch = M > 1 && vpq::qmv_batch_supports(K, M, f);
  for (int i = 0; i < count; ++i) {
    batch = batch && aligned(scales[i], 16) && (scale_only != 0 || aligned(biases[i], 16));
  }
  if (M > 1 && !batch) {                                // (a pack's own alignment chooses its kernel)
    for (int i = 0; i < count; ++i) {
      const int st = vpq_qmv_w4g32_bf16(stream, w[i], scales[i], scale_only ? nullptr : biases[i], x, y[i], K, N[i], M,
                                        nullptr, scale_only);
      if (st != VPQ_OK) { return st; }
    }
    return VPQ_OK;
  }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.x = x; a.K = K; a.M = M; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  vpq::QmvGroup g;
  g.count = count;
  for (int i = 0; i < count; ++i) { g.seg[i] = vpq::QmvSeg{w[i], scales[i], scale_only ? nullptr : biases[i], y[i], N[i]}; }
  if (batch) { return finish(vpq::launch_qmv_batch(reinterpret_cast<hipStream_t>(stream), a, g, f)); }
  if (vpq::qmv_flow_narrow_supports(K, 1, M, 32)) {
    return finish(vpq::launch_qmv_flow_narrow_group(reinterpret_cast<hipStream_t>(stream), a, g, f));
  }
  return finish(vpq::launch_qmv_rows_group(reinterpret_cast<hipStream_t>(stream), a, g, 32, scale_only != 0));
}

int vpq_qmv_group_w8g64_bf16(vpq_stream_t stream, int count, const uint32_t* const* w, const uint16_t* const* scales,
                             const uint16_t* const* biases, const uint16_t* x, uint16_t* const* y, int K, const int* N,
                             int M)
{
  if (w == nullptr || scales == nullptr || biases == nullptr || y == nullptr || N == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (count < 1 || count > 4) { return VPQ_ERR_BAD_SHAPE; }
  const vpq::BatchFormat f{8, 64, false, false};
  const bool row = M == 1 && K >= kRow8MinK;
  bool one_launch = x != nullptr && aligned(x, 16) && (row || (M >= 2 && M <= 16 && vpq::qmv_batch_supports(K, M, f)));
  for (int i = 0; i < count && one_launch; ++i) {
    one_launch = check_pack(w[i], scales[i], biases[i], K, N[i]) == VPQ_OK && y[i] != nullptr && aligned(y[i], 2) &&
                 (row || (aligned(scales[i], 16) && aligned(biases[i], 16)));
  }
  if (one_launch) {
    const int st = ensure_init();
    if (st != VPQ_OK) { return st; }
    vpq::QmvArgs a{};
    a.x = x; a.K = K; a.M = M; a.y_f32 = false; a.cu_count = g_dev.cu_count;
    vpq::QmvGroup g;
    g.count = count;
    for (int i = 0; i < count; ++i) { g.seg[i] = vpq::QmvSeg{w[i], scales[i], biases[i], y[i], N[i]}; }
    hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    return finish(row ? launch_row8(hs, a, g) : vpq::launch_qmv_batch(hs, a, g, f));
  }
  // one row of a short K, packs that the batch kernel does not take, or something to report: the separate calls
  for (int i = 0; i < count; ++i) {
    const int st = vpq_qmv_w8g64_bf16(stream, w[i], scales[i], biases[i], x, y[i], K, N[i], M, nullptr);
    if (st != VPQ_OK) { return st; }
  }
  return VPQ_OK;
}

int vpq_rmsnorm_bf16(vpq_stream_t stream, const uint16_t* x, const uint16_t* norm_w, uint16_t* out, int K, int M, float eps)
{
  if (x == nullptr || norm_w == nullptr || out == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (K < 1 || M < 1 || M > 65535 || !(eps >= 0.0f)) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 2) || !aligned(norm_w, 2) || !aligned(out, 2)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_rmsnorm(reinterpret_cast<hipStream_t>(stream), x, norm_w, out, K, M, eps));
}

// `affine_qmv_qkv_rms_w4g64` / `_w4g32` / `_w8g64` (gpu-kernels/metal/quant/affine_qmv.metal:671-740): RMSNorm of the
// one row of x, then the fused-QKV GEMV over the normalized row.  format: 0 = 4-bit group-64, 1 = 4-bit group-32,
// 2 = 8-bit group-64.  x_norm_ws: K elements of scratch that receive the normalized row.
int vpq_qmv_qkv_rms_bf16(vpq_stream_t stream, int format, int count, const uint32_t* const* w, const uint16_t* const* scales,
                         const uint16_t* const* biases, const uint16_t* x, const uint16_t* norm_w, uint16_t* const* y,
                         int K, const int* N, float eps, uint16_t* x_norm_ws)
{
  if (format < 0 || format > 2) { return VPQ_ERR_BAD_SHAPE; }
  if (x_norm_ws == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (!aligned(x_norm_ws, 16)) { return VPQ_ERR_MISALIGNED; }
  // (the packs themselves are checked by the format's own grouped entry point below: a refusal there has written the
  // scratch and nothing else)
  if (w == nullptr || scales == nullptr || biases == nullptr || y == nullptr || N == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (count < 1 || count > 4) { return VPQ_ERR_BAD_SHAPE; }
  if (K <= 0 || (K % (format == 1 ? 32 : 64)) != 0) { return VPQ_ERR_BAD_SHAPE; }
  int st = vpq_rmsnorm_bf16(stream, x, norm_w, x_norm_ws, K, 1, eps);
  if (st != VPQ_OK) { return st; }
  if (format == 1) { return vpq_qmv_group_w4g32_bf16(stream, count, w, scales, biases, x_norm_ws, y, K, N, 1, 0); }
  if (format == 2) { return vpq_qmv_group_w8g64_bf16(stream, count, w, scales, biases, x_norm_ws, y, K, N, 1); }
  return vpq_qmv_group_w4g64_bf16(stream, count, w, scales, biases, x_norm_ws, y, K, N, 1);
}

int vpq_qmv_group_w4g64_f16(vpq_stream_t stream, int count, const uint32_t* const* w,
                            const uint16_t* const* scales, const uint16_t* const* biases,
                            const uint16_t* x, uint16_t* const* y, int K, const int* N, int M)
{
  if (w == nullptr || scales == nullptr || biases == nullptr || y == nullptr || N == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (count < 1 || count > 4) { return VPQ_ERR_BAD_SHAPE; }
  const vpq::BatchFormat f{4, 64, true, false};
  const bool narrow = flow_narrow_f16(K, 1, M);
  const bool flow = vpq::qmv_flow_supports(K, 1, M);
  bool one_launch = flow || vpq::qmv_batch_supports(K, M, f);
  for (int i = 0; i < count; ++i) {
    int st = check_pack(w[i], scales[i], biases[i], K, N[i]);
    if (st != VPQ_OK) { return st; }
    if (y[i] == nullptr) { return VPQ_ERR_NULL_POINTER; }
    if (!aligned(y[i], 2)) { return VPQ_ERR_MISALIGNED; }
    one_launch = one_launch && aligned(scales[i], 16) && aligned(biases[i], 16);
  }
  if (x == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (M < 1 || M > 16) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16)) { return VPQ_ERR_MISALIGNED; }
  if (!one_launch && !narrow) {
    for (int i = 0; i < count; ++i) {
      const int st = vpq_qmv_w4g64_f16(stream, w[i], scales[i], biases[i], x, y[i], K, N[i], M, nullptr);
      if (st != VPQ_OK) { return st; }
    }
    return VPQ_OK;
  }
  int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  vpq::QmvArgs a{};
  a.x = x; a.K = K; a.M = M; a.y_f32 = false; a.cu_count = g_dev.cu_count;
  vpq::QmvGroup g;
  g.count = count;
  for (int i = 0; i < count; ++i) { g.seg[i] = vpq::QmvSeg{w[i], scales[i], biases[i], y[i], N[i]}; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (narrow) { return finish(vpq::launch_qmv_flow_narrow_group(hs, a, g, f)); }
  return finish(flow ? vpq::launch_qmv_flow_group(hs, a, g, true) : vpq::launch_qmv_batch(hs, a, g, f));
}

int vpq_quantize_w4g64(vpq_stream_t stream, const uint16_t* src, uint32_t* w, uint16_t* scales_f16,
                       uint16_t* biases_f16, int K, int N, float clip)
{
  if (src == nullptr || w == nullptr || scales_f16 == nullptr || biases_f16 == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (K <= 0 || N <= 0 || (K % 64) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(src, 16) || !aligned(w, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_quantize(reinterpret_cast<hipStream_t>(stream), src, w, scales_f16, biases_f16, K, N, clip));
}

int vpq_quantize(vpq_stream_t stream, int bits, int group, int src_f16, const uint16_t* src, uint32_t* w,
                 uint16_t* scales_f16, uint16_t* biases_f16, int K, int N, float clip)
{
  if (src == nullptr || w == nullptr || scales_f16 == nullptr || biases_f16 == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if ((bits != 4 && bits != 8) || (group != 64 && group != 32)) { return VPQ_ERR_BAD_SHAPE; }
  if (K <= 0 || N <= 0 || (K % group) != 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(src, 16) || !aligned(w, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_quantize(reinterpret_cast<hipStream_t>(stream), src, w, scales_f16, biases_f16, K, N, clip, bits,
                                     group, src_f16 != 0));
}

int vpq_f16_to_bf16(vpq_stream_t stream, const uint16_t* in_f16, uint16_t* out_bf16, size_t count)
{
  if (in_f16 == nullptr || out_bf16 == nullptr) { return VPQ_ERR_NULL_POINTER; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_f16_to_bf16(reinterpret_cast<hipStream_t>(stream), in_f16, out_bf16, count));
}

int vpq_profile_empty_kernel(vpq_stream_t stream, void* sink)
{
  if (sink == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(sink, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_profile_empty(reinterpret_cast<hipStream_t>(stream), static_cast<uint32_t*>(sink)));
}

int vpq_profile_read_kernel(vpq_stream_t stream, const void* src, size_t bytes, void* sink)
{
  if (src == nullptr || sink == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (bytes < 16) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(src, 16) || !aligned(sink, 4)) { return VPQ_ERR_MISALIGNED; }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_profile_read(reinterpret_cast<hipStream_t>(stream), src, bytes, static_cast<uint32_t*>(sink)));
}

int vpq_profile_enable(int max_launches)
{
  vpq::ProfileState& ps = vpq::profile_state();
  if (max_launches <= 0) {
    ps.on = false;
    return VPQ_OK;
  }
  const int st = ensure_init();
  if (st != VPQ_OK) { return st; }
  while (ps.events.size() < (size_t)max_launches * 2) {
    hipEvent_t e;
    const hipError_t err = hipEventCreate(&e);
    if (err != hipSuccess) { return device_error(err); }
    ps.events.push_back(e);
  }
  ps.used = 0;
  ps.on = true;
  return VPQ_OK;
}

int vpq_profile_read(float* kernel_ms, int capacity)
{
  vpq::ProfileState& ps = vpq::profile_state();
  const int n = (int)(ps.used / 2);
  for (int i = 0; i < n && i < capacity; ++i) {
    hipError_t err = hipEventSynchronize(ps.events[2 * i + 1]);
    if (err != hipSuccess) { return device_error(err); }
    float ms = 0.0f;
    err = hipEventElapsedTime(&ms, ps.events[2 * i], ps.events[2 * i + 1]);
    if (err != hipSuccess) { return device_error(err); }
    if (kernel_ms != nullptr) { kernel_ms[i] = ms; }
  }
  ps.used = 0;
  return n;
}

// 8-bit codes on IEEE binary16 elements (the half build's affine_dequant_w8g64 / _w8g32 and affine_qmm_steel_w8g64 /
// _w8g32): the expansion, and the GEMM by the dequant-once route on the binary16 dense GEMM.
int vpq_dequant_w8_f16(vpq_stream_t stream, int group, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                       uint16_t* w_deq, int K, int N)
{
  if (group != 64 && group != 32) { return VPQ_ERR_BAD_SHAPE; }
  int st = group == 64 ? check_pack(w, scales, biases, K, N) : check_pack_w8g32(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (w_deq == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (!aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  return finish(vpq::launch_dequant8(reinterpret_cast<hipStream_t>(stream), w, scales, biases, w_deq, K, N, group, true));
}

int vpq_qmm_dense_route_w8_f16(vpq_stream_t stream, int group, const uint32_t* w, const uint16_t* scales,
                               const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                               uint16_t* w_deq, int expand)
{
  if (group != 64 && group != 32) { return VPQ_ERR_BAD_SHAPE; }
  int st = group == 64 ? check_pack(w, scales, biases, K, N) : check_pack_w8g32(w, scales, biases, K, N);
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (w_deq == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || !aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (expand != 0) {
    st = finish(vpq::launch_dequant8(hs, w, scales, biases, w_deq, K, N, group, true));
    if (st != VPQ_OK) { return st; }
  }
  std::string why;
  const int rc = vpq::dense_gemm_elt(hs, x, w_deq, y, M, N, K, true, g_dev.cu_count, &why);
  if (rc != 0) {
    strncpy(g_last_error, why.c_str(), sizeof(g_last_error) - 1);
    g_last_error[sizeof(g_last_error) - 1] = '\0';
    return VPQ_ERR_DEVICE;
  }
  return VPQ_OK;
}

// The dequant-once route with the runtime adapter for any of the pack formats: the adapter's pre-pass, the format's
// expansion (or the kept one), the dense GEMM with t . B^T in the same accumulators.
int vpq_qmm_dense_route_lora_bf16(vpq_stream_t stream, int format, const uint32_t* w, const uint16_t* scales,
                                  const uint16_t* biases, const uint16_t* x, uint16_t* y, int K, int N, int M,
                                  uint16_t* w_deq, int expand, const uint16_t* lora_a, const uint16_t* lora_b, int r,
                                  float alpha, uint16_t* lora_t_ws)
{
  if (format == VPQ_FORMAT_W4G64) {
    return vpq_qmm_dense_route_lora_w4g64_bf16(stream, w, scales, biases, x, y, K, N, M, w_deq, expand, lora_a, lora_b, r,
                                               alpha, lora_t_ws);
  }
  int st = format == VPQ_FORMAT_W4G32   ? check_pack_g32(w, scales, biases, K, N, false)
           : format == VPQ_FORMAT_W8G64 ? check_pack(w, scales, biases, K, N)
           : format == VPQ_FORMAT_W8G32 ? check_pack_w8g32(w, scales, biases, K, N)
                                        : VPQ_ERR_BAD_SHAPE;
  if (st != VPQ_OK) { return st; }
  if (x == nullptr || y == nullptr) { return VPQ_ERR_NULL_POINTER; }
  if (w_deq == nullptr) { return VPQ_ERR_WORKSPACE; }
  if (M <= 0) { return VPQ_ERR_BAD_SHAPE; }
  if (!aligned(x, 16) || !aligned(y, 16) || !aligned(w_deq, 16)) { return VPQ_ERR_MISALIGNED; }
  const bool lora = lora_a != nullptr && alpha != 0.0f;
  if (lora) {
    if (lora_b == nullptr) { return VPQ_ERR_NULL_POINTER; }
    if (lora_t_ws == nullptr) { return VPQ_ERR_WORKSPACE; }
    // the pre-pass walks K in chunks of 64
    if (r < 8 || r > vpq::kLoraMaxRank || (r % 8) != 0 || (K % 64) != 0) { return VPQ_ERR_BAD_SHAPE; }
    if (!aligned(lora_a, 16) || !aligned(lora_b, 16) || !aligned(lora_t_ws, 16)) { return VPQ_ERR_MISALIGNED; }
  }
  st = ensure_init();
  if (st != VPQ_OK) { return st; }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (lora) {
    st = finish(vpq::launch_lora_a(hs, x, lora_a, lora_t_ws, M, K, r, alpha));
    if (st != VPQ_OK) { return st; }
  }
  if (expand != 0) {
    st = finish(format == VPQ_FORMAT_W4G32   ? vpq::launch_dequant_g32(hs, w, scales, biases, w_deq, K, N)
                : format == VPQ_FORMAT_W8G64 ? vpq::launch_dequant8(hs, w, scales, biases, w_deq, K, N)
                                             : vpq::launch_dequant8(hs, w, scales, biases, w_deq, K, N, 32));
    if (st != VPQ_OK) { return st; }
  }
  std::string why;
  const int rc = vpq::dense_gemm_elt(hs, x, w_deq, y, M, N, K, false, g_dev.cu_count, &why, lora ? lora_t_ws : nullptr,
                                     lora ? lora_b : nullptr, lora ? r : 0);
  if (rc != 0) {
    strncpy(g_last_error, why.c_str(), sizeof(g_last_error) - 1);
    g_last_error[sizeof(g_last_error) - 1] = '\0';
    return VPQ_ERR_DEVICE;
  }
  return VPQ_OK;
}

size_t vpq_weight_bytes(int N, int K) { return (size_t)N * (size_t)(K * 4 / 32) * 4; }
size_t vpq_scale_bytes(int N, int K) { return (size_t)N * (size_t)(K / 64) * 2; }

}  // extern "C"
