// Launches of the int4 experts' streaming kernel (a file of its own: the build compiles it beside w4a16_gemm.hip).
#include "w4a16_stream.h"

namespace ksq {
namespace {

template <typename T, bool PAIRED>
int launch(const SplitKParams& p, uint32_t m_blocks, hipStream_t s) {
  // more dynamic LDS than a kernel may use without asking: once per device
  static std::atomic<uint64_t> configured{0};
  auto kernel = &w4a16_stream_tile_kernel<T, PAIRED>;
  if (int rc = allow_dynamic_lds(configured, reinterpret_cast<const void*>(kernel), kW4StreamLds)) return rc;
  // (a pair of a gate and an up column counts once: the same number either way)
  kernel<<<dim3(static_cast<uint32_t>(div_up(p.N, 256)), m_blocks), 512, kW4StreamLds, s>>>(p);
  return KSQ_OK;
}

template <typename T>
int launch_type(const SplitKParams& p, bool paired, uint32_t m_blocks, hipStream_t s) {
  return paired ? launch<T, true>(p, m_blocks, s) : launch<T, false>(p, m_blocks, s);
}

}  // namespace

int launch_w4a16_stream(const SplitKParams& p, bool paired, uint32_t m_blocks, int dtype, hipStream_t s) {
  return dtype == KSQ_F16 ? launch_type<F16>(p, paired, m_blocks, s) : launch_type<BF16>(p, paired, m_blocks, s);
}

}  // namespace ksq
