// nv_linear's 16-bit products of many rows on the tiles of stream_deep.h: a source of its own, for its compile time.
#include "linear_stream.h"
#include "stream_deep.h"

template <typename TO, int EPI, bool FAR_UPS = false>
static hipError_t linear_deep_as(const LinArgs& p, int64_t total_rows, int batch, hipStream_t s) {
  const auto job = linear_job<TO, EPI, FAR_UPS>(p, batch);
  return launch_stream_deep(job, linear_job_tiles(p, job.nt, total_rows, batch), s);
}
template <typename TO>
static hipError_t linear_deep_to(const LinArgs& p, int epi, int64_t total_rows, int batch, hipStream_t s) {
  switch (epi) {
    case EPI_NONE: return linear_deep_as<TO, EPI_NONE>(p, total_rows, batch, s);
    case EPI_GLU:      // far ups cost scalar registers, which GELU's constants need (2048 rows 2048 -> 2 x 8192: 117 us, 120 with them)
      return 2 * (int64_t)p.N * p.w_rs * 2 < ((int64_t)1 << 32) ? linear_deep_as<TO, EPI_GLU>(p, total_rows, batch, s)
                                                                : linear_deep_as<TO, EPI_GLU, true>(p, total_rows, batch, s);
    case EPI_SOFTCAP: return linear_deep_as<TO, EPI_SOFTCAP>(p, total_rows, batch, s);
    case EPI_ACT: return linear_deep_as<TO, EPI_ACT>(p, total_rows, batch, s);
    default: return linear_deep_as<TO, EPI_ROW_GATE>(p, total_rows, batch, s);
  }
}
hipError_t linear_deep_launch(const LinArgs& p, int epi, bool out_16bit, int64_t total_rows, int batch, hipStream_t s) {
  return out_16bit ? linear_deep_to<bf16_t>(p, epi, total_rows, batch, s) : linear_deep_to<float>(p, epi, total_rows, batch, s);
}
