// Row-segment wavefront forward (1-4 states per channel; 5-16 with a wave per state): instantiations for f16_t inputs.
#include "snd_wave_fwd_kernel.h"
namespace snd {
int launch_wave_fwd_f16(const snd_fwd_params &p, float *group_ws, hipStream_t stream) { return launch_wave_fwd_t<f16_t>(p, group_ws, stream); }
int launch_wave_states_f16(const snd_fwd_params &p, hipStream_t stream) { return launch_wave_states_t<f16_t>(p, stream); }
}  // namespace snd
