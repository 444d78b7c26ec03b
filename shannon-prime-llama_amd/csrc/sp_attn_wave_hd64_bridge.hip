// sp_attn_wave_hd64_bridge.hip -- the matrix-core decode-attention kernel (sp_attn_wave.h) for
// head_dim 64, K 5/4/4 and V 5.
#include "sp_attn_wave.h"

hipError_t sp_wave_hd64_bridge(const SpWaveLaunch &W) { return wave_launch<WaveHd64Bridge>(W); }
