// What the two attention translation units share: the kinds of caches and the launch interface of the 16-bit
// matrix-core kernels (pitch_attn_codes.hip).
#pragma once

#include "pitch_device.h"

namespace pitch {

constexpr float kLn2 = 0x1.62e430p-1f;   // ln(2)

// Kinds of caches: key codec (with or without the key-bias term) and value codec.
#define kAttnKindTurbo 0      // TurboQuant keys and values
#define kAttnKindPolar 1      // PolarQuant keys and values
#define kAttnKindTurboBias 2  // the same with the key-bias term
#define kAttnKindPolarBias 3
#define kAttnKindChanTurbo 4  // per-channel keys, TurboQuant values
#define kAttnKindChanPolar 5  // per-channel keys, PolarQuant values
constexpr int kAttnKinds = 6;

#define PITCH_DECLARE_ATTN_CODES(K)                                                          \
  hipError_t launch_attn_codes_d64_k##K(const AttnArgs& a, uint32_t waves, hipStream_t s);   \
  hipError_t launch_attn_codes_d128_k##K(const AttnArgs& a, uint32_t waves, hipStream_t s);
PITCH_DECLARE_ATTN_CODES(0)
PITCH_DECLARE_ATTN_CODES(1)
PITCH_DECLARE_ATTN_CODES(2)
PITCH_DECLARE_ATTN_CODES(3)
PITCH_DECLARE_ATTN_CODES(4)
PITCH_DECLARE_ATTN_CODES(5)
#undef PITCH_DECLARE_ATTN_CODES

}  // namespace pitch
