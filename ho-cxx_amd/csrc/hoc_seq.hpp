// hoc_seq.hpp - numbers of the Krylov iterations of a handle and the status word that carries one to the
// host.  The numbers run modulo 2^30: never negative (a negative one stands for the device's counter),
// beside two flag bits in 32, and without an end however long a handle lives (32-bit arithmetic without the
// wrap ended after 2^29 iterations, some 6 hours of marching on 32 x 32 elements).
#pragma once

#include <cstdint>

namespace hoc {

constexpr int kSeqMod = 1 << 30;
// The first number of a handle: close to the wrap, so that every run passes it.
constexpr int kSeqStart = kSeqMod - 64;

constexpr int seq_add(int seq, int d) { return (seq + d) & (kSeqMod - 1); }
// Whether seq is target or one of the 2^29 - 1 numbers after it.
constexpr bool seq_reached(int seq, int target) { return ((seq - target) & (kSeqMod - 1)) < kSeqMod / 2; }

constexpr uint32_t status_word(int seq, bool near, bool active) {
  return (uint32_t)seq * 4u + (near ? 2u : 0u) + (active ? 1u : 0u);
}
constexpr int status_seq(uint32_t v) { return (int)(v >> 2); }
constexpr bool status_near(uint32_t v) { return (v & 2u) != 0; }
constexpr bool status_active(uint32_t v) { return (v & 1u) != 0; }

}  // namespace hoc
