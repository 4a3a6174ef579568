// nv_linear's 16-bit products whose results take long to form, on the tiles of stream_tiles.h (linear_four_wavefronts says which): a source of
// its own, for its compile time.
#include "linear_stream.h"

template <typename TO, int EPI>
static hipError_t linear_eight_as(const LinArgs& p, int64_t total_rows, int batch, hipStream_t s) {
  const auto job = linear_job<TO, EPI>(p, batch);
  return launch_stream_tiles(job, linear_job_tiles(p, job.nt, total_rows, batch), s);
}
template <typename TO>
static hipError_t linear_eight_to(const LinArgs& p, int epi, int64_t total_rows, int batch, hipStream_t s) {
  switch (epi) {
    case EPI_NONE: return linear_eight_as<TO, EPI_NONE>(p, total_rows, batch, s);
    case EPI_GLU: return linear_eight_as<TO, EPI_GLU>(p, total_rows, batch, s);
    case EPI_SOFTCAP: return linear_eight_as<TO, EPI_SOFTCAP>(p, total_rows, batch, s);
    case EPI_ACT: return linear_eight_as<TO, EPI_ACT>(p, total_rows, batch, s);
    default: return linear_eight_as<TO, EPI_ROW_GATE>(p, total_rows, batch, s);
  }
}
hipError_t linear_eight_launch(const LinArgs& p, int epi, bool out_16bit, int64_t total_rows, int batch, hipStream_t s) {
  return out_16bit ? linear_eight_to<bf16_t>(p, epi, total_rows, batch, s) : linear_eight_to<float>(p, epi, total_rows, batch, s);
}
