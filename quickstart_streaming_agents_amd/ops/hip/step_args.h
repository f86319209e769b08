// Arguments of the mixers' step kernels, as the bindings fill them in.
#pragma once

typedef unsigned short bf16_t;

struct ConvStep {
  const int* item;   // portion of a chunk of rows; null: chunk c is row c,
  const int* t0;     //   one token at position start[c] - 1
  const int* off;
  const int* start;
  const int* len;
  const int* slots;
};

// The attention's short convolutions (short_conv.h)
struct ConvQkv {
  const void* x;
  long long xstride;
  const float* w;
  int taps;
  void* tails;
  ConvStep step;
  const float *cos_t, *sin_t;
  int rot, table_len;
  const int* cache_slots;
  void *q, *kc, *vc;
  int H, G, D, E;
};

// One token per row of a state-space layer (ssd.hip)
struct SsdStep {
  const bf16_t* u;                     // [z | x | B | C | dt] of a row
  long long ustride;
  int zoff, xoff, dtoff;
  const float *w, *bias;               // filters [taps, C]
  int taps;
  bf16_t* tails;                       // [slots, taps - 1, C]
  const float *A, *dt_bias, *Dskip, *norm;
  float* state;
  const int *slots, *seq_lens;
  bf16_t* out;
  long long ostride;
  int B, H, N, P, G;
  float eps;
  int conv_blocks;                     // of a row, of the attention
  ConvQkv conv;
};
