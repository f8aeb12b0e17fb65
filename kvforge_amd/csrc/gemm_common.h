// What the bf16 products of gemm_bf16.hip and gemm_tile.hip share.
#pragma once
#include "common.h"

namespace {
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

struct RopeEpi {
  const int* positions;
  const int* seq_of_token;
  const float* cos_t;
  const float* sin_t;
  const int* block_table;
  bf16_t* k_pages;
  bf16_t* v_pages;
  int H, KV, d, rot, table_len, block_size, table_stride, num_blocks, write_kv, n_seqs;
  // EPI 3: how a pair is joined (GateForm's act and limit), what it is multiplied by, and fp32 biases
  // of the gate and up columns (by pair, may be null)
  int act;
  float act_limit, act_scale;
  const float* gate_bias;
  const float* up_bias;
};

// Compute units of the current device, asked once per device.
int compute_units() {
  static int known[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (known[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    known[dev] = n;
  }
  return known[dev];
}
}  // namespace
