// Heads as a fused projection left them, for decode attention to take.
#pragma once
// Rows of q | k | v heads of 128, one of each sequence: bf16 (parts 0, in q), or f32
// sums [parts, seqs, width] of a split GEMM, which are added up.
struct DecodeHeads {
  const float* sums;
  const int* positions;                 // [seqs]
  const int* slots;                     // [seqs], where the new key goes; -1: nowhere
  const float* cos_sin;                 // [positions, 128] = cos | sin
  const void* q_norm;                   // bf16 [128] each, or null
  const void* k_norm;
  float eps;
  int parts;
};
