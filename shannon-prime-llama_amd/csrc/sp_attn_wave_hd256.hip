// sp_attn_wave_hd256.hip -- the matrix-core decode-attention kernel (sp_attn_wave.h) for
// head_dim 256, K 5/5/4/3 and V 3.
#include "sp_attn_wave.h"

hipError_t sp_wave_hd256(const SpWaveLaunch &W) { return wave_launch<WaveHd256>(W); }
