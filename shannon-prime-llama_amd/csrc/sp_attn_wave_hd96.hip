// sp_attn_wave_hd96.hip -- the matrix-core decode-attention kernel (sp_attn_wave.h) for
// head_dim 96, K 5/4/4 and V 5.
#include "sp_attn_wave.h"

hipError_t sp_wave_hd96(const SpWaveLaunch &W) { return wave_launch<WaveHd96>(W); }
