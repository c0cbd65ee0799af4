// Host-side helpers of the engine that need no device: configuration checks,
// epsilon tables, 2-bit map packing.
#pragma once
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/crl.h"

namespace crl {

// The calling thread's last failure text, behind crl_last_error().
std::string& last_error();
// Notes `why` as the thread's last failure and returns `code`.
int fail_with(int code, const char* why);

// CRL_OK, or a negative status with the reason in `why`
int validate_config(const crl_config* cfg, std::string& why);

// Epsilon per global step (STEP_MULT) or per episode (EPISODE_*): the values a
// Python float would take under `eps *= decay` (src/train.py:140-141), i.e.
// doubles, rounded to fp32 once.
std::vector<float> build_eps_table(const crl_config& cfg);

// 16 cells per word, cell c in bits [2*(c%16), 2*(c%16)+1] of word c/16
void pack_classes(const uint8_t* cls, size_t n_cells, uint32_t* words);

// n transitions as the update kernels read them: key = s * A + a (-1 for an action outside
// [0, A)), s2d = s' with done in the top bit.  -> false if a state lies outside [0, S); what
// was written is then worthless.  A is 4 or 8, S at most 2^24.
bool pack_transitions(int n, int S, int A, const int32_t* s, const int32_t* a, const int32_t* s_next,
                      const uint8_t* done, int32_t* key, uint32_t* s2d);
// The same in one word each: key in bits 0..15 (all ones: an action outside [0, A)), s' in bits
// 16..30, done in bit 31.  S * A is below 65535.
bool pack_transitions_short(int n, int S, int A, const int32_t* s, const int32_t* a, const int32_t* s_next,
                            const uint8_t* done, uint32_t* words);

}  // namespace crl
