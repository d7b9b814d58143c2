// Launches of the warm-start U-Net kernels (unet_kernels.hip) for the host
// orchestration (unet.cpp).  Plain pointers; every function returns 0 or a
// HIP error code.  bfloat16 tensors are uint16 bit patterns, channels-last.
#pragma once

#include <cstdint>

namespace hlbn {

struct ConvGeom {
  int N, D, H, W;
};

// The input of a convolution may come in two parts where conv_takes_parts:
// channels [0, cu) from xu, a tensor of half the resolution read at
// (d/2, h/2, w/2), the others from x (xu null: all ci from x).
bool conv_takes_parts(const ConvGeom& g, int ci);
// y[p][yoff + o] = (relu)(sum_t,c x[p + off_t][c] w[t][o][c] + bias[o]) into
// a binary32 and/or bfloat16 tensor with yc channels.  ci, co multiples of 16.
// ws: conv_fwd_ws(g, ci, co) floats of workspace for the K slices of coarse
// levels (null when that is 0).
int conv_fwd(const ConvGeom& g, const uint16_t* x, const uint16_t* xu, int cu, int ci,
             const uint16_t* w,
             const float* bias, int co, float* y32, uint16_t* y16, int yc, int yoff, int relu,
             float* ws, void* stream);
int64_t conv_fwd_ws(const ConvGeom& g, int ci, int co);
// Position chunk of the backward-weight partial sums.
int64_t wgrad_chunk(const ConvGeom& g);
// dw[t][o][c] = sum_p dy[p][o] x[p + off_t][c]; part holds
// wgrad_parts(g, ci, co) floats (partial sums over runs of positions, added
// in a fixed order).
int conv_wgrad(const ConvGeom& g, const uint16_t* x, const uint16_t* xu, int cu, int ci,
               const uint16_t* dy, int co,
               float* part, float* dw, void* stream);
int64_t wgrad_parts(const ConvGeom& g, int ci, int co);
// out[c] = sum_p a[p][c] (chunked, fixed order); part holds ceil(P/chunk)*C.
int channel_sum(const float* a, int64_t P, int C, float* part, int64_t chunk, float* out,
                void* stream);
// bfloat16 copies of every layer's weights w [27][co][ci] and of their flipped
// transposes wt[26 - t][ci][co] (the weights of the backward-data convolution).
struct WeightLayers {
  static constexpr int kCount = 14;
  struct Layer {
    int64_t woff;   // first weight in the parameter vector
    int co, ci;
    uint16_t *w16, *wt16;
  } layer[kCount];
  uint32_t first_tile[kCount];   // of each layer's 16 x 16 tiles (set by refresh_weights)
};
int refresh_weights(WeightLayers layers, const float* params, void* stream);
// ReLU backward with the bias gradient: dpre16 = bf16 of dpost where post > 0,
// db[c] = sum_p of its binary32 values (part: ceil(P / wgrad_chunk) * C), for
// C dividing 256 (dpre_fused).  dpost by kind:
//   0: a[p][C];  1: sum_o a[p][o] b[o][c], o < n (the head);
//   2: sum of the 8 children of p in channels [0, C) of a, n channels wide, at
//      twice g's resolution;
//   3: a[p][off + c], n channels wide, plus b[parent][c] / 8.
struct DpreSrc {
  const float* a;
  const float* b;
  int n, off;
};
enum { kDprePlain, kDpreHead, kDpreUp, kDpreSkip };
bool dpre_fused(int C);
int dpre(const ConvGeom& g, int C, int kind, const DpreSrc& src, const uint16_t* post,
         uint16_t* dpre16, float* part, float* db, void* stream);
int relu_bwd(const float* dpost, const uint16_t* post, int64_t n, uint16_t* dpre16,
             float* dpre32, void* stream);
int pool(const ConvGeom& fine, int C, const uint16_t* x, uint16_t* y, void* stream);
int pool_bwd_add(const ConvGeom& fine, int C, const float* dy, float* dx, void* stream);
int up(const ConvGeom& coarse, int C, const uint16_t* x, uint16_t* y, int yc, int yoff,
       void* stream);
int up_bwd(const ConvGeom& coarse, int C, const float* dy, int dyc, int dyoff, float* dx,
           void* stream);
int copy_channels(int64_t P, int C, const uint16_t* x, uint16_t* y, int yc, int yoff,
                  void* stream);
int take_channels(int64_t P, int C, const float* dy, int dyc, int dyoff, float* dx, int add,
                  void* stream);
int pack_input(int64_t P, int cin, const float* in, uint16_t* x, void* stream);
int head_fwd(int64_t P, int K, int O, const uint16_t* h, const float* W, const float* b,
             float* out, void* stream);
int head_bwd_data(int64_t P, int K, int O, const float* dout, const float* W, float* dh,
                  void* stream);
int head_wgrad(int64_t P, int K, int O, const float* dout, const uint16_t* h, float* part,
               int64_t chunk, float* dW, float* db, void* stream);
// Loss weights of up to 16 output channels, passed with the launch.
struct ChannelWeights {
  float w[16];
};
int mse(int64_t P, int O, const float* out, const float* target, const uint8_t* mask,
        const ChannelWeights& wc, float inv_count, float* dout, float* lterm, void* stream);
int adam(int64_t n, float* p, const float* g, float* m, float* v, float lr, float b1, float b2,
         float eps, float wd, float c1, float c2, void* stream);

}  // namespace hlbn
